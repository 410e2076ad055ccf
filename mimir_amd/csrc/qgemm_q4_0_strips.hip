// Products of some rows of x, bfloat16 or float32, by Q4_0 weights on the bfloat16 matrix cores of gfx950, with x and W read
// where they lie and no workspace: what mi355x_qgemm_bf16 takes up to some hundreds of rows, and mi355x_qgemv for rows of W
// that the fixed-point forms do not take (an odd number of blocks, or W on two bytes).
//
// A workgroup has 32 rows of x and one or two strips of 32 rows of W; its eight wavefronts take runs of eight blocks of K in
// turn and add their sums up in order. A chain of steps over all of K, in which one workgroup a tile of the result
// takes 0.9 us for every 64 of K however few the rows, is what bounded these shapes before. W passes through a private slab of LDS as in
// qgemv_q8_0_mfma.hip (144 bytes a row, rows end to end); x, of which an MFMA's operand is sixteen consecutive bytes of each
// of 32 rows, comes straight from memory some blocks ahead. Two v_mfma_f32_32x32x16_bf16 make a block: their operands are
// n - 8 of the lower and of the upper nibbles, exact in bfloat16 (as sixteenths, the scale times sixteen), and one FMA a result adds the
// block's sum by its scale. A float32 x is the sum of three bfloat16, exactly, and a block six MFMAs.
//
// What bounds it, by the counters: 75 vector instructions (30 of unpacking, 16 FMAs) and two MFMAs of 32 cycles a block and strip, half and a tenth of the SIMDs' cycles at
// 128 x 14336 x 4096, the rest waits for loads, of which W's come past the L2 once for every 32 rows of x; with float32 310 instructions a block and two strips, some 150 of them
// splitting x (for two strips where they fill the chip), and twelve MFMAs, 61 % and 19 % at 128 x 4096 x 4064. From some 1800 workgroups on the tile
// kernels, which unpack W once for 128 rows, are the faster. Whole calls, us, before and now:
//   bfloat16   16 x 4096 x 4096    61 -> 10      float32   16 x 4096 x 4064      31 -> 20
//             256 x 4096 x 4096    62 -> 38               128 x 4096 x 4064     215 -> 30
//             128 x 4096 x 14336  200 -> 70               512 x 14336 x 4064   3860 -> 370
// Errors against 64 bits, of the result: bfloat16 5.5e-7 -> 6.6e-8 at K = 4096, 1.05e-6 -> 6.5e-8 at 14336;
// float32 1.96e-7 -> 9.1e-8 at K = 4064, 2.0e-7 -> 1.34e-7 at 14368. With the runs' and the wavefronts' sums of bfloat16 in 32 bits it was
// 8.3e-8 at K = 4064, more than the 7.4e-8 of the float32 kernel that such rows took before.
#include <atomic>

#include "device_util.h"
#include "kernels.h"

namespace mimir {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 8;
constexpr int kRunBlocks = 8;
constexpr int kRunBytes = 18 * kRunBlocks;         // 144: nine pieces of sixteen bytes a row
constexpr int kPieces = kRunBytes / 16;
constexpr int kStripBytes = 32 * kRunBytes;        // a strip's run in LDS, rows end to end: their starts fall on sixteen banks
constexpr int kLoads = (32 * kPieces + 63) / 64;   // 5: the last one half full

template <typename X>
constexpr int kParts = sizeof(X) == 4 ? 3 : 1;

__device__ __forceinline__ uint32_t upper_halves(uint32_t odd, uint32_t even) { return __builtin_amdgcn_perm(odd, even, 0x07060302u); }

// Eight x of a row as the MFMA's operands, the least part first. A float32 is three bfloat16 that add up to it: its upper
// sixteen bits (eight of its 24 significant ones), those of what is left, and of what is left then. An infinity's rest is
// nought, a NaN's NaN.
__device__ __forceinline__ void split(const u32x4* v, bf16x8* parts, __bf16) { __builtin_memcpy(parts, v, 16); }
__device__ __forceinline__ void split(const u32x4* v, bf16x8* parts, float) {
    uint32_t p[3][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t b[3][2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t u = v[i >> 1][2 * (i & 1) + j];
            const float x = __uint_as_float(u), upper = __uint_as_float(u & 0xffff0000u);
            const float rest = __builtin_fabsf(x) == __builtin_inff() ? 0.f : x - upper;
            const float low = rest - __uint_as_float(__float_as_uint(rest) & 0xffff0000u);
            b[2][j] = u;
            b[1][j] = __float_as_uint(rest);
            b[0][j] = __float_as_uint(low);
        }
#pragma unroll
        for (int q = 0; q < 3; q++) p[q][i] = upper_halves(b[q][1], b[q][0]);
    }
#pragma unroll
    for (int q = 0; q < 3; q++) __builtin_memcpy(&parts[q], p[q], 16);
}

// What x's parts and a block's sum do not hold. The matrix cores take subnormal operands for nought, which the lesser parts of
// a float32 below 2^-103 are; and 32 numbers above 2^122 may add up to more than a float32 holds, where their product with the
// scale is none. Where a float32 is below 2^-100, or a bfloat16 subnormal (other than nought; the tile kernel takes these for
// nought too, so they are looked for in its stead only where it does not go), or a result no finite number, a workgroup reads such rows
// of x again, and if one has a block whose largest x is below 2^-60 (in the others what is lost is 2^-66 of
// the largest), or a finite x from 2^100 on, it goes over its share again and takes the former times 2^64, the latter times 2^-64. Rows with a
// NaN or an infinity, and products that no float32 holds, are what they are the first time (us without, with a NaN in one row, and when it went over all of it again:
// bfloat16 16 x 4096 x 4096 10.2, 13.5, 28; 128 x 14336 x 4096 63, 68, 149; float32 128 x 4096 x 4064 32, 34, 61).
constexpr uint32_t kTiny = ((127u - 100u) << 24) - 1;
__device__ __forceinline__ void note_least(const u32x4 (*v)[2], uint32_t* least) {
#pragma unroll
    for (int i = 0; i < 16; i++) *least = min(*least, (v[i >> 3][(i >> 2) & 1][i & 3] << 1) - 1);  // nought: the largest number
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void note_least(const u32x4 (*v)[1], uint32_t* least) {  // two halves a word
    u16x2 most, one;
    __builtin_memcpy(&most, least, 4);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t bits = v[i >> 2][0][i & 3] & 0x7fff7fffu;
        __builtin_memcpy(&one, &bits, 4);
        most = __builtin_elementwise_min(most, one - (uint16_t)1);
    }
    __builtin_memcpy(least, &most, 4);
}
__device__ __forceinline__ bool tiny(uint32_t least, float) { return least < kTiny; }
__device__ __forceinline__ bool tiny(uint32_t least, __bf16) { return (least & 0xffffu) < 0x7f || (least >> 16) < 0x7f; }

// Whether any of the rows in `rows` has what is to be gone over again: pieces of sixteen bytes, a thread each, a block's to neighbours.
template <typename X>
__device__ __forceinline__ bool needs_suit(const X* x, int64_t x_row_stride, uint32_t rows, int K, bool small_too, int tid) {
    constexpr int kPer = 16 / sizeof(X), kTogether = 4;
    const int pieces = K / kPer;
    bool need = false;
    for (int p = tid; rows != 0;) {
        u32x4 v[kTogether];
#pragma unroll
        for (int u = 0; u < kTogether; u++) {
            while (p >= pieces && rows != 0) p -= pieces, rows &= rows - 1;
            const int row = rows != 0 ? __builtin_ctz(rows) : -1;
            v[u] = u32x4{0, 0, 0, 0};
            if (row >= 0) v[u] = *(const u32x4*)(x + row * x_row_stride + (int64_t)kPer * p);
            p += 64 * kWaves;
        }
#pragma unroll
        for (int u = 0; u < kTogether; u++) {
            float most = 0.f;
#pragma unroll
            for (int i = 0; i < kPer; i++) {
                const float a = __builtin_fabsf(__uint_as_float(sizeof(X) == 4 ? v[u][i & 3] : i & 1 ? v[u][(i >> 1) & 3] & 0xffff0000u : v[u][(i >> 1) & 3] << 16));
                need |= a >= 0x1p100f && a < __builtin_inff();
                most = a > most || a != a ? a : most;
            }
#pragma unroll
            for (int o = 1; o < 32 / kPer; o <<= 1) {
                const float other = __shfl_xor(most, o);
                most = other > most || other != other ? other : most;
            }
            need |= small_too && most > 0.f && most < 0x1p-60f;
        }
    }
    return need;
}

// Sixteen x of a row, eight of each half of the block, by the power of two that suits it; returns what takes the row's sum back.
__device__ __forceinline__ float factor(float most) {
    const float other = __shfl_xor(most, 32);  // the other lane's half of the row
    const float all = other > most || other != other ? other : most;
    return all < 0x1p-60f ? 0x1p64f : all >= 0x1p100f ? 0x1p-64f : 1.f;
}
__device__ __forceinline__ float suit(u32x4 (*v)[2]) {
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float a = __builtin_fabsf(__uint_as_float(v[i >> 3][(i >> 2) & 1][i & 3]));
        most = a > most || a != a ? a : most;
    }
    const float by = factor(most);
#pragma unroll
    for (int i = 0; i < 16; i++) v[i >> 3][(i >> 2) & 1][i & 3] = __float_as_uint(__uint_as_float(v[i >> 3][(i >> 2) & 1][i & 3]) * by);
    return 1.f / by;
}
__device__ __forceinline__ float suit(u32x4 (*v)[1]) {
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const uint32_t u = v[i >> 3][0][(i >> 1) & 3];
        const float a = __builtin_fabsf(__uint_as_float(i & 1 ? u & 0xffff0000u : u << 16));
        most = a > most || a != a ? a : most;
    }
    const float by = factor(most);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t u = v[i >> 2][0][i & 3];
        v[i >> 2][0][i & 3] = upper_halves(__float_as_uint(__uint_as_float(u & 0xffff0000u) * by), __float_as_uint(__uint_as_float(u << 16) * by));
    }
    return 1.f / by;
}

__device__ double acc_of(__bf16);
__device__ float acc_of(float);

// SW: strips of 32 rows of W a workgroup. RAGGED: the blocks of a row need be no multiple of eight, and subnormal bfloat16 count.
template <typename X, int SW, bool RAGGED, typename Y>
__global__ __launch_bounds__(64 * kWaves, sizeof(X) == 2 && !RAGGED ? 4 : 2) void qgemm_q4_0_strips_kernel(const uint8_t* __restrict__ W, const X* __restrict__ x, Y* __restrict__ y, int M, int N,
                                                                            int nb, int64_t x_row_stride) {
    constexpr int kP = kParts<X>;
    constexpr int kWords = sizeof(X) == 4 ? 2 : 1;  // sixteen-byte loads of eight x
    constexpr int kAhead = SW == 1 ? 4 : 2;  // blocks of x in registers: of bfloat16 with eight, two wavefronts a SIMD instead of four (256 x 4096 x 4096: 55 us, 38)
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ngroups = (M + 31) / 32, group = (int)(blockIdx.x % (unsigned)ngroups);
    const int n0 = (int)(blockIdx.x / (unsigned)ngroups) * 32 * SW;
    const int nruns = (nb + kRunBlocks - 1) / kRunBlocks;
    uint8_t* slab = smem + wave * SW * kStripBytes;  // this wavefront's alone
    x += (int64_t)32 * group * x_row_stride;
    y += (int64_t)32 * group * N;
    M = M - 32 * group < 32 ? M - 32 * group : 32;

    // piece p = 64 i + lane of a strip's run: row p / 9 of the 32, bytes 16 (p % 9).. of its 144
    uint32_t goff[SW][kLoads];
#pragma unroll
    for (int s = 0; s < SW; s++) {
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            int p = 64 * i + lane;
            p = p < 32 * kPieces ? p : 32 * kPieces - 1;  // the last load's upper lanes repeat the last piece
            const int r = p / kPieces, c = p - kPieces * r;
            const int row = n0 + 32 * s + r < N ? n0 + 32 * s + r : N - 1;
            goff[s][i] = (uint32_t)(row - n0) * (uint32_t)(nb * 18) + 16 * c;  // 64 rows of W within 4 GB (checked by the host)
        }
    }
    const uint8_t* wbase = W + (int64_t)n0 * nb * 18;
    const X* xrow = x + (int64_t)(l32 < M ? l32 : M - 1) * x_row_stride + 8 * lh;  // rows past M: the last one again, not stored

    auto start_of = [&](int run) { return kRunBlocks * run < nb - kRunBlocks ? kRunBlocks * run : nb - kRunBlocks; };  // the last run reaches back
    u32x4 w[SW][kLoads];
    u32x4 xs[kAhead][2][kWords];
    auto fetch_w = [&](int at) {
        const uint8_t* p = wbase + (int64_t)at * 18;
#pragma unroll
        for (int s = 0; s < SW; s++) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) w[s][i] = load_u32x4_unaligned(p + goff[s][i]);
        }
    };
    auto fetch_x = [&](int slot, int block) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int i = 0; i < kWords; i++) xs[slot][h][i] = *((const u32x4*)(xrow + 32 * (int64_t)block + 16 * h) + i);
        }
    };

    // A block's product of a strip and sixteen times its scale. A block is a scale and sixteen bytes, of which this lane takes eight: their
    // lower nibbles are weights 8 lh .., the upper ones 16 + 8 lh .. It starts on a dword for even b, two bytes into one for odd b.
    auto product = [&](int s, int b, const bf16x8 (&xp)[2][kP], float* scale) {
        const uint8_t* block = slab + s * kStripBytes + l32 * kRunBytes + 18 * b;
        uint32_t q[2];
        float d;
        if (b & 1) {
            const uint32_t* p = (const uint32_t*)(block + 2 + 8 * lh);
            q[0] = p[0];
            q[1] = p[1];
            d = f16_bits_to_f32((uint16_t)(*(const uint32_t*)(block - 2) >> 16));
        } else {
            const uint32_t* p = (const uint32_t*)(block + 8 * lh);
            const uint32_t r0 = p[0], r1 = p[1], r2 = p[2];
            q[0] = __builtin_amdgcn_alignbit(r1, r0, 16);
            q[1] = __builtin_amdgcn_alignbit(r2, r1, 16);
            d = f16_bits_to_f32((uint16_t)(*(const uint32_t*)block & 0xffffu));
        }
        *scale = d * 16.f;
        f32x16 c;
#pragma unroll
        for (int i = 0; i < 16; i++) c[i] = 0.f;
        bf16x8 wp[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint32_t packed[4];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint32_t t = (h ? q[k] >> 4 : q[k]) ^ 0x08080808u;  // a nibble n as the four-bit integer n - 8, converted as sixteenths
                float f[4];
#pragma unroll
                for (int i = 0; i < 4; i++) f[i] = __builtin_amdgcn_cvt_off_f32_i4((int)((t >> (8 * i)) & 0xffu));
                packed[2 * k] = upper_halves(__float_as_uint(f[1]), __float_as_uint(f[0]));
                packed[2 * k + 1] = upper_halves(__float_as_uint(f[3]), __float_as_uint(f[2]));
            }
            __builtin_memcpy(&wp[h], packed, 16);
        }
#pragma unroll
        for (int p = 0; p < kP; p++) {
#pragma unroll
            for (int h = 0; h < 2; h++) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xp[h][p], wp[h], c, 0, 0, 0);
        }
        return c;  // register 4 g + j: row 8 g + 4 lh + j of x
    };
    // a wavefront's LDS operations complete in order
    auto store_w = [&]() {
#pragma unroll
        for (int s = 0; s < SW; s++) {
#pragma unroll
            for (int i = 0; i < kLoads; i++) {
                if (64 * i + lane < 32 * kPieces) *(u32x4*)(slab + s * kStripBytes + 16 * (64 * i + lane)) = w[s][i];
            }
        }
    };

    // A run's sums by themselves, the runs' in 64 bits (of float32 x, whose blocks' sums err by more, in 32)
    using Acc = decltype(acc_of(X()));
    Acc acc[SW][16];
#pragma unroll
    for (int s = 0; s < SW; s++) {
#pragma unroll
        for (int i = 0; i < 16; i++) acc[s][i] = 0;
    }
    uint32_t least = 0xffffffffu;
    if (wave < nruns) {
        fetch_w(start_of(wave));
#pragma unroll
        for (int b = 0; b < kAhead; b++) fetch_x(b, start_of(wave) + b);
    }
    for (int run = wave; run < nruns; run += kWaves) {
        const int at = start_of(run), next = start_of(run + kWaves < nruns ? run + kWaves : run), done = kRunBlocks * run - at;
        store_w();
        fetch_w(next);
        float part[SW][16];
#pragma unroll
        for (int b = 0; b < kRunBlocks; b++) {
            bf16x8 xp[2][kP];
            u32x4 v[2][kWords];
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int i = 0; i < kWords; i++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) v[h][i][j] = RAGGED && b < done ? 0u : xs[b % kAhead][h][i][j];  // blocks that the run before has taken
                }
                split(v[h], xp[h], X());
            }
            if constexpr (kP == 3 || RAGGED) note_least(v, &least);
            fetch_x(b % kAhead, b + kAhead < kRunBlocks ? at + b + kAhead : next + b + kAhead - kRunBlocks);
#pragma unroll
            for (int s = 0; s < SW; s++) {
                float d;
                const f32x16 c = product(s, b, xp, &d);
                if (RAGGED) d = b < done ? 0.f : d;
#pragma unroll
                for (int i = 0; i < 16; i++) part[s][i] = b == 0 ? d * c[i] : fmaf(d, c[i], part[s][i]);
            }
        }
#pragma unroll
        for (int s = 0; s < SW; s++) {
#pragma unroll
            for (int i = 0; i < 16; i++) acc[s][i] += part[s][i];
        }
    }
    bool beyond = tiny(least, X());
#pragma unroll
    for (int s = 0; s < SW; s++) {
#pragma unroll
        for (int i = 0; i < 16; i++) beyond = beyond || !(__builtin_fabsf((float)acc[s][i]) < __builtin_inff());
    }
    bool again = false;
    if (__syncthreads_or(beyond)) {  // seldom
        uint32_t rows = tiny(least, X()) ? 1u << l32 : 0u;  // of x
#pragma unroll
        for (int s = 0; s < SW; s++) {
#pragma unroll
            for (int i = 0; i < 16; i++) rows |= __builtin_fabsf((float)acc[s][i]) < __builtin_inff() ? 0u : 1u << (8 * (i >> 2) + 4 * lh + (i & 3));
        }
        uint32_t* all = (uint32_t*)smem;  // every wavefront is done with its slab
        if (tid == 0) *all = 0;
        __syncthreads();
        atomicOr(all, rows);
        __syncthreads();
        again = __syncthreads_or(needs_suit(x, x_row_stride, M < 32 ? *all & ((1u << M) - 1) : *all, 32 * nb, kP == 3 || RAGGED, tid));
    }
    if (again) {  // block after block
#pragma unroll
        for (int s = 0; s < SW; s++) {
#pragma unroll
            for (int i = 0; i < 16; i++) acc[s][i] = 0;
        }
#pragma unroll 1
        for (int run = wave; run < nruns; run += kWaves) {
            const int at = start_of(run);
            fetch_w(at);
            store_w();
#pragma unroll 1
            for (int b = kRunBlocks * run - at; b < kRunBlocks; b++) {
                fetch_x(0, at + b);
                const float back = suit(xs[0]);
                bf16x8 xp[2][kP];
#pragma unroll
                for (int h = 0; h < 2; h++) split(xs[0][h], xp[h], X());
#pragma unroll
                for (int s = 0; s < SW; s++) {
                    float d;
                    const f32x16 c = product(s, b, xp, &d);
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[s][i] += (Acc)(d * c[i]) * (Acc)__shfl(back, 8 * (i >> 2) + 4 * lh + (i & 3));
                }
            }
        }
    }

    __syncthreads();  // every wavefront is done with its slab
    float* red = (float*)smem;  // [wave][16][lane], a strip at a time
#pragma unroll
    for (int s = 0; s < SW; s++) {
        if (s > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; i++) red[(wave * 16 + i) * 64 + lane] = (float)acc[s][i];
        __syncthreads();
        for (int i = wave; i < 16; i += kWaves) {
            double sum = red[i * 64 + lane];
#pragma unroll
            for (int o = 1; o < kWaves; o++) sum += red[(o * 16 + i) * 64 + lane];
            const float v = (float)sum;
            const int m = 8 * (i >> 2) + 4 * lh + (i & 3), n = n0 + 32 * s + l32;
            if (n < N && m < M) {
                if constexpr (sizeof(Y) == 4) y[(int64_t)m * N + n] = v;
                else y[(int64_t)m * N + n] = f32_to_bf16_bits(v);
            }
        }
    }
}

std::atomic<int> g_strips{0};  // measurement aid: 1 = wherever the kernel takes the shape, 2 = never

template <typename X, int SW, bool RAGGED, typename Y>
hipError_t launch(const void* W, const void* x, void* y, int64_t M, int64_t N, int64_t K, int64_t x_row_stride, hipStream_t st) {
    const int64_t wgs = ((N + 32 * SW - 1) / (32 * SW)) * ((M + 31) / 32);
    if (wgs > 0x7fffffff) return hipErrorInvalidValue;
    constexpr int kLds = kWaves * SW * kStripBytes;
    static_assert(kLds >= kWaves * 16 * 64 * 4, "the sums take the slabs' place");
    if (kLds > 64 * 1024) {
        static LdsLimit limit;
        if (hipError_t e = limit.raise(kLds, {(const void*)qgemm_q4_0_strips_kernel<X, SW, RAGGED, Y>})) return e;
    }
    hipLaunchKernelGGL((qgemm_q4_0_strips_kernel<X, SW, RAGGED, Y>), dim3((unsigned)wgs), dim3(64 * kWaves), kLds, st, (const uint8_t*)W, (const X*)x, (Y*)y, (int)M,
                       (int)N, (int)(K / 32), x_row_stride);
    return hipGetLastError();
}

template <typename X, int SW, typename Y>
hipError_t dispatch(const void* W, const void* x, void* y, int64_t M, int64_t N, int64_t K, int64_t x_row_stride, hipStream_t st) {
    const bool tiles = K % (32 * kRunBlocks) == 0 && (sizeof(X) == 4 || qgemm_q4_0_ok(W, x, M, N, K, x_row_stride));
    return SW == 2 || !tiles ? launch<X, SW, true, Y>(W, x, y, M, N, K, x_row_stride, st) : launch<X, 1, false, Y>(W, x, y, M, N, K, x_row_stride, st);
}

}  // namespace

void set_q4_0_strips(int v) { g_strips = v; }

bool qgemm_q4_0_strips_ok(const void* W, const void* x, bool bf16, int64_t M, int64_t N, int64_t K, int64_t x_row_stride) {
    return M >= 1 && M <= 65535 && N > 0 && N <= ((int64_t)1 << 30) && K >= 32 * kRunBlocks && K % 32 == 0 && 64 * (K / 32) * 18 < ((int64_t)1 << 32) &&
           ((uintptr_t)W & 1) == 0 && ((uintptr_t)x & 15) == 0 && x_row_stride % (bf16 ? 8 : 4) == 0;
}

// float32, against the float32 kernel for one row after another (us there, here): from sixteen rows, 8192 results (16 x 512 x
// 4064 20, 19; 64 x 128 x 1056 14, 11; 16 x 256 x 1056 8, 10); nine to fifteen, 1000 rows of W (9 x 4096 x 1056 10.2, 10.0; 12 x
// 512 x 4064 16, 19); five to eight, 32 M weights (6 x 4096 x 8224 47, 35; 6 x 4096 x 4064 14, 19; four rows 33, 35). Past K =
// 32768 its sums, which are longer than that kernel's, would be the less exact.
// bfloat16. Rows of W of an odd number of blocks: against that kernel and two conversions, but for a few rows by few long
// ones of W (8 x 1024 x 8224 34, 20; 2 x 4096 x 14368 35, 33; 2 x 1024 x 8224 14, 20). Where there is a tile
// kernel (K a multiple of 256): up to 1792 workgroups here, fewer of shorter rows (there, here: 256 x 4096 x 4096, 1024
// workgroups, 62, 38; 128 x 14336 x 4096, 1792, 64, 62; 96 x 14336 x 1024, 1344, 21, 20; 256 x 4096 x 512 13.4, 12.5; 192 x
// 4096 x 256, 768, 9.0, 9.2). Else, against the fixed-point forms and two conversions: up to 512.
bool qgemm_q4_0_strips_pays(const void* W, const void* x, bool bf16, int64_t M, int64_t N, int64_t K, int64_t x_row_stride) {
    if (g_strips == 2 || !qgemm_q4_0_strips_ok(W, x, bf16, M, N, K, x_row_stride)) return false;
    if (g_strips == 1) return true;
    if (!bf16) {
        if (K > 32768) return false;
        if (M >= 16) return M * N >= 8192;
        return M >= 9 ? N >= 1000 : M >= 5 && N * K >= ((int64_t)32 << 20);
    }
    const int64_t wgs = ((N + 31) / 32) * ((M + 31) / 32);
    if (K % 64 != 0) return M >= 6 || N >= 4096 || K <= 4096;
    if (!qgemm_q4_0_ok(W, x, M, N, K, x_row_stride)) return wgs <= 512;
    return wgs <= (K >= 2048 ? 1792 : K >= 1024 ? 1344 : K >= 512 ? 1024 : 512);
}

hipError_t qgemm_q4_0_strips(const void* W, const void* x, bool bf16, void* y, bool out_bf16, int64_t M, int64_t N, int64_t K, int64_t x_row_stride, hipStream_t st) {
    if (!qgemm_q4_0_strips_ok(W, x, bf16, M, N, K, x_row_stride) || (out_bf16 && !bf16)) return hipErrorInvalidValue;
    if (bf16 && out_bf16) return dispatch<__bf16, 1, uint16_t>(W, x, y, M, N, K, x_row_stride, st);
    if (bf16) return dispatch<__bf16, 1, float>(W, x, y, M, N, K, x_row_stride, st);
    const int64_t pairs = ((N + 63) / 64) * ((M + 31) / 32);
    return pairs >= 256 ? dispatch<float, 2, float>(W, x, y, M, N, K, x_row_stride, st) : dispatch<float, 1, float>(W, x, y, M, N, K, x_row_stride, st);
}

}  // namespace mimir
