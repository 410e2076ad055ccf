// Products of some rows of x (nine to a few hundred) with Q4_K and Q6_K weights
// on the int8 matrix cores of gfx950, between the kernel that takes eight rows a
// pass over W (qgemv_kquant_rows.hip) and the one of tall tiles
// (qgemm_kquant.hip): x already rounded to int8 per super-block of 256, in the
// order of the lanes (kq_act.h), the results the CPU's bit for bit (qdotQ4KGo and
// qdotQ6KGo, backend/cpu/qmatmul.go:148-200): everything inside a super-block is
// integer, and its float32 terms are added in the super-blocks' order.
//
// A workgroup of eight wavefronts owns sixteen rows of W by up to 64 rows of x.
// Sixteen, because 4096 rows of W are then a workgroup for every compute unit;
// tall tiles are 64 workgroups there, each of which splits 64 rows of W a step.
// The wavefronts take the super-blocks round robin: one reads its 16 x 256
// weights once, splits them into two planes of int8 as the tall tiles do (Q4_K by
// the scale, Q6_K by the product's bytes), and multiplies all rows of x by them.
// Rows of W are the first operand of v_mfma_i32_16x16x64_i8, so that a lane ends
// up with four rows of W by one of x: one scale of x a lane, four of W for all
// tiles. Q4_K's mins are a third plane, their products' sum exact as well. The
// terms of a round of eight super-blocks go through LDS, two buffers of them, one
// barrier a round; a wavefront owns one tile's sums (of Q4_K one of the tile's
// two) and adds the round's terms in order.
//
// What bounds it: the cache's front end and the vector instructions, two
// wavefronts a SIMD. x in the order of the lanes is loads of a whole kilobyte;
// from plain rows, 64 bytes of sixteen each, 64 x 4096 x 14336 Q4_K took 43 us,
// not 26.4. Blocks of Q6_K through LDS in aligned pieces: 27.4 us for 33.8 with
// aligned loads straight into the lanes. With the rounding of x, us, here and by
// the kernels that had them, 16 / 32 / 64 / 128 rows: Q4_K 4096 x 4096 7.7 / 8.9 /
// 11.1 / 19.1 for 7.7 / 12.1 / 18.6 / 32.6; 4096 x 14336 13.3 / 19.3 / 26.6 / 49
// for 19.5 / 32.7 / 59.7 / 98; Q6_K 4096 x 14336 17.4 / 20.2 / 27.4 / 49 for 24.4 /
// 45 / 83 / 100, where 48 MB of W take 9.4 us at the rate of a large copy.
#include "device_util.h"
#include "kernels.h"
#include "kq_act.h"

namespace mimir {

#pragma clang fp contract(off)

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;
constexpr int kStrip = 16;  // rows of W a workgroup, rows of x a tile

// Two 16-bit products a lane, their low halves.
__device__ __forceinline__ uint32_t mul_pairs(uint32_t a, uint32_t b) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b)); }

// Four quants in the bytes of q (each below 64) times the int8 scale s, less 32 s each, as the digits of 256 a + b, both int8 (split_q6k of
// qgemm_kquant.hip): q s + (128 - 32 s) in 16 bits has a in its upper byte and b + 128 in its lower. s and bias: the two numbers in both halves.
__device__ __forceinline__ void split_six(uint32_t q, uint32_t s, uint32_t bias, int& a, int& b) {
    const s16x2 sc = __builtin_bit_cast(s16x2, s), c = __builtin_bit_cast(s16x2, bias);
    const uint32_t even = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, q, 0x0c020c00u)) * sc + c);
    const uint32_t odd = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, q, 0x0c030c01u)) * sc + c);
    a = (int)__builtin_amdgcn_perm(odd, even, 0x07030501u);
    b = (int)(__builtin_amdgcn_perm(odd, even, 0x06020400u) ^ 0x80808080u);
}

// Lane 16 kq + n of an operand holds, of step s, elements 64 s + 16 kq .. + 15 of row n's super-block.
template <int DT>
struct Raw;
template <>
struct Raw<kQ4_K> {  // d, dmin and the scales; 16 bytes of nibbles of each half
    u32x4 hdr, q[2];
};
// Sixteen bytes from an even address in LDS, as the aligned dwords that hold them.
struct Even16 {
    uint32_t w[5];
    __device__ __forceinline__ uint32_t at(int i, uint32_t off) const { return __builtin_amdgcn_alignbyte(w[i + 1], w[i], off); }
};
template <>
struct Raw<kQ6_K> {  // per half: 16 bytes of low nibbles, the 16 bytes of high bits that go with them; the scales; d
    Even16 q[2], high[2], scales;
    uint32_t d, off;
};

// Q6_K's blocks of 210 bytes start on even addresses: loads of them straight into the lanes, off 16-byte boundaries, are eleven that take the cache's front end longer each
// than the four of the aligned 16-byte pieces of sixteen rows' blocks, 14 a row (each holds at least a byte of the block, so that it lies in memory that is there). Those pass
// through a slab of LDS of the wavefront's own.
constexpr int kPieces = 14, kSlabRow = 16 * kPieces + 16;
struct Pieces {
    u32x4 p[4];
};

__device__ __forceinline__ void fetch(Raw<kQ4_K>& f, const uint8_t* block, int kq) {
    f.hdr = *(const u32x4*)block;
#pragma unroll
    for (int p = 0; p < 2; p++) f.q[p] = *(const u32x4*)(block + 16 + 64 * p + 16 * kq);
}
struct Planes {
    i32x4 a[4], b[4];
};

// Sub-block 2 s + (kq / 2) is a lane's in step s. A lane's 16 bytes hold low nibbles of one sub-block and high nibbles of the next: the halves of the
// wavefront trade those (v_permlane32_swap), which puts neighbouring sub-blocks into one step.
__device__ __forceinline__ void split(const Raw<kQ4_K>& f, int kq, Planes& p) {
    // the eight scales (scale_min_k4, backend/cpu/quant.go:129-134), four to a dword, as 8 s1 + s0
    const uint32_t lo4 = f.hdr[1] & 0x3f3f3f3fu, hi4 = (f.hdr[3] & 0x0f0f0f0fu) | ((f.hdr[1] >> 2) & 0x30303030u);
    const uint32_t first = 0x0c000c00u + (uint32_t)(kq >> 1) * 0x00010001u;  // byte kq / 2 into both halves; two more for the next step
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const uint32_t four = s < 2 ? lo4 : hi4, sel = first + (s & 1 ? 0x00020002u : 0u);
        const uint32_t s1 = __builtin_amdgcn_perm(0u, (four >> 3) & 0x07070707u, sel), s0 = __builtin_amdgcn_perm(0u, four & 0x07070707u, sel);
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const uint32_t x = f.q[s >> 1][d];
            const auto r = __builtin_amdgcn_permlane32_swap(x & 0x0F0F0F0Fu, (x >> 4) & 0x0F0F0F0Fu, false, false);
            const uint32_t r0 = r[0], r1 = r[1];
            const uint32_t w = s & 1 ? r1 : r0;
            p.a[s][d] = (int)mul_pairs(w, s1);  // at most 15 x 7 a byte
            p.b[s][d] = (int)mul_pairs(w, s0);
        }
    }
}
__device__ __forceinline__ void split(const Raw<kQ6_K>& f, int kq, Planes& p) {
    const uint32_t byte = 0x0c000c00u + (uint32_t)kq * 0x00010001u;
#pragma unroll
    for (int s = 0; s < 4; s++) {  // scale 4 s + kq
        const uint32_t pair = __builtin_amdgcn_perm(0u, f.scales.at(s, f.off), byte);  // the byte in both halves
        const uint32_t sc = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(s16x2, pair) << 8) >> 8);
        const uint32_t bias = __builtin_bit_cast(uint32_t, (s16x2){128, 128} - (__builtin_bit_cast(s16x2, sc) << 5));
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const uint32_t q = f.q[s >> 1].at(d, f.off), h = f.high[s >> 1].at(d, f.off) >> (kq & 2);
            const uint32_t six = s & 1 ? ((q >> 4) & 0x0F0F0F0Fu) | (h & 0x30303030u) : (q & 0x0F0F0F0Fu) | ((h & 0x03030303u) << 4);
            int a, b;
            split_six(six, sc, bias, a, b);
            p.a[s][d] = a;
            p.b[s][d] = b;
        }
    }
}

// Q4_K's mins as a third plane: of step s, that of sub-block 2 s + kq / 2 for each of its elements.
__device__ __forceinline__ void mins(const Raw<kQ4_K>& f, int kq, int m[4]) {
    const uint32_t lo4 = f.hdr[2] & 0x3f3f3f3fu, hi4 = ((f.hdr[3] >> 4) & 0x0f0f0f0fu) | ((f.hdr[2] >> 2) & 0x30303030u);
    const uint32_t first = (uint32_t)(kq >> 1) * 0x01010101u;
#pragma unroll
    for (int s = 0; s < 4; s++) m[s] = (int)__builtin_amdgcn_perm(0u, s < 2 ? lo4 : hi4, first + (s & 1 ? 0x02020202u : 0u));
}

template <int DT, int MT>
constexpr int kBufferBytes = kWaves * (DT == kQ4_K ? 2 : 1) * MT * 1024;
template <int DT, int MT>
constexpr int kLds = 2 * kBufferBytes<DT, MT> + (DT == kQ6_K ? kWaves * kStrip * kSlabRow : 0);

// MT tiles of sixteen rows of x. groups: workgroups a strip of W, each with rows 16 MT apart.
template <int DT, int MT>
__global__ __launch_bounds__(64 * kWaves) void qgemm_kquant_shared_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ act, void* yv,
                                                                         const float* resid, int M, int N, int nsb, int groups, int y_bf16) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int BB = DT == kQ4_K ? 144 : 210, KINDS = DT == kQ4_K ? 2 : 1;
    static_assert(MT * KINDS <= kWaves, "a wavefront owns one tile's sums");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, kq = lane >> 4;
    // A die's workgroups are every eighth: those of one strip of W follow each other there and find it in its L2.
    const int strips = (N + kStrip - 1) / kStrip, on_die = blockIdx.x >> 3;
    const int strip = (on_die / groups) * 8 + (blockIdx.x & 7), m0 = (on_die % groups) * MT * kStrip;
    if (strip >= strips) return;
    const int n0 = strip * kStrip, last_n = N - 1 - n0;
    const uint8_t* w_strip = W + (int64_t)n0 * nsb * BB;
    const uint32_t row_bytes = (uint32_t)(nsb * BB), w_row = (uint32_t)(l16 < last_n ? l16 : last_n) * row_bytes;
    const int last_tile = (M + kStrip - 1) / kStrip - 1;
    const uint8_t* x_tile[MT];  // past the last tile: it again
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int tile = m0 / kStrip + t;
        x_tile[t] = act + (int64_t)(tile < last_tile ? tile : last_tile) * nsb * kLanesBlock;
    }

    struct X {
        i32x4 q[4];
        float d;
    };
    X x[MT];
    Raw<DT> raw;
    // Q6_K: this lane's pieces of a super-block of the strip, relative to the 16-byte boundary before the strip
    Pieces pieces;
    const uint32_t lead = (uint32_t)(uintptr_t)w_strip & 15;
    const uint8_t* boundary = w_strip - lead;
    uint8_t* slab = smem + 2 * kBufferBytes<DT, MT> + wave * kStrip * kSlabRow;
    uint32_t piece_row[4], piece_at[4];
    if constexpr (DT == kQ6_K) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int piece = 64 * i + lane < kStrip * kPieces ? 64 * i + lane : 0, r = piece / kPieces;
            piece_row[i] = lead + (uint32_t)(r < last_n ? r : last_n) * row_bytes;
            piece_at[i] = (uint32_t)r << 16 | (uint32_t)(piece % kPieces);
        }
    }
    auto fetch_w = [&](int sb) {
        if constexpr (DT == kQ4_K) {
            fetch(raw, w_strip + w_row + (uint32_t)(sb * BB), kq);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) pieces.p[i] = *(const u32x4*)(boundary + ((piece_row[i] + (uint32_t)(sb * BB)) & ~15u) + 16 * (piece_at[i] & 0xffff));
        }
    };
    auto unpack_w = [&](int sb) {  // what fetch_w brought, into raw
        if constexpr (DT == kQ6_K) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (i < 3 || lane < kStrip * kPieces - 192) *(u32x4*)(slab + (piece_at[i] >> 16) * kSlabRow + 16 * (piece_at[i] & 0xffff)) = pieces.p[i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const uint32_t start = (lead + w_row + (uint32_t)(sb * BB)) & 15;
            raw.off = start & 2;
            const uint8_t* mine = slab + l16 * kSlabRow + (start & ~3u);
            auto read = [&](Even16& e, int at) {
#pragma unroll
                for (int i = 0; i < 5; i++) e.w[i] = *(const uint32_t*)(mine + at + 4 * i);
            };
#pragma unroll
            for (int h = 0; h < 2; h++) {
                read(raw.q[h], 64 * h + 16 * kq);
                read(raw.high[h], 128 + 32 * h + 16 * (kq & 1));
            }
            read(raw.scales, 192);
            raw.d = __builtin_amdgcn_alignbyte(0u, raw.scales.w[4], raw.off) & 0xffff;
            __builtin_amdgcn_wave_barrier();
        }
    };
    auto fetch_x = [&](int t, int sb) {
        const uint8_t* p = x_tile[t] + (int64_t)sb * kLanesBlock;
#pragma unroll
        for (int s = 0; s < 4; s++) x[t].q[s] = *(const i32x4*)(p + 1024 * s + 16 * lane);
        x[t].d = *(const float*)(p + 4096 + 4 * l16);
    };
    const int rounds = (nsb + kWaves - 1) / kWaves;
    int sb = wave < nsb ? wave : nsb - 1;  // past the last: it again, its terms left out
    fetch_w(sb);
#pragma unroll
    for (int t = 0; t < MT; t++) fetch_x(t, sb);

    f32x4 sum = {0.f, 0.f, 0.f, 0.f};  // of slice `wave`: kind wave / MT of tile wave % MT
    for (int r = 0; r < rounds; r++) {
        uint8_t* buffer = smem + (r & 1) * kBufferBytes<DT, MT>;
        const int next = (r + 1) * kWaves + wave, sbn = next < nsb ? next : nsb - 1;
        Planes w;
        unpack_w(sb);
        split(raw, kq, w);
        int mn[4] = {};
        uint32_t scales;
        if constexpr (DT == kQ4_K) {
            mins(raw, kq, mn);
            scales = raw.hdr[0];
        } else {
            scales = raw.d;
        }
        float dw[4], dmin[4];  // of rows 4 kq + i of the strip
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t s = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (4 * kq + i), (int)scales);
            dw[i] = f16_bits_to_f32((uint16_t)s);
            dmin[i] = DT == kQ4_K ? f16_bits_to_f32((uint16_t)(s >> 16)) : 0.f;
        }
        fetch_w(sbn);
        sb = sbn;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            i32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0}, least = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                a = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.a[s], x[t].q[s], a, 0, 0, 0);
                b = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.b[s], x[t].q[s], b, 0, 0, 0);
                if (DT == kQ4_K) least = __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{mn[s], mn[s], mn[s], mn[s]}, x[t].q[s], least, 0, 0, 0);
            }
            const float dx = x[t].d;
            fetch_x(t, sbn);
            f32x4 term, under;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int sumi = (a[i] << (DT == kQ4_K ? 3 : 8)) + b[i];
                const float dd = dw[i] * dx;
                term[i] = dd * (float)sumi;
                const float dm = dmin[i] * dx;
                under[i] = dm * (float)least[i];  // below 2^24: exact, as the sum of the products of sums is
            }
            uint8_t* to = buffer + ((wave * KINDS * MT + t) * 64 + lane) * 16;
            *(f32x4*)to = term;
            if constexpr (DT == kQ4_K) *(f32x4*)(to + MT * 1024) = under;
        }
        // the terms are there; the other buffer's have been added
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (wave < MT * KINDS) {
            const int live = nsb - r * kWaves;
            f32x4 part[kWaves];
#pragma unroll
            for (int u = 0; u < kWaves; u++) part[u] = *(const f32x4*)(buffer + ((u * KINDS * MT + wave) * 64 + lane) * 16);
#pragma unroll
            for (int u = 0; u < kWaves; u++) {
                if (u >= live) break;
#pragma unroll
                for (int i = 0; i < 4; i++) sum[i] = sum[i] + part[u][i];
            }
        }
    }
    if constexpr (DT == kQ4_K) {  // the mins' sums to the wavefront of the tile
        __syncthreads();
        if (wave >= MT && wave < 2 * MT) *(f32x4*)(smem + ((wave - MT) * 64 + lane) * 16) = sum;
        __syncthreads();
        if (wave < MT) {
            const f32x4 under = *(const f32x4*)(smem + (wave * 64 + lane) * 16);
#pragma unroll
            for (int i = 0; i < 4; i++) sum[i] = sum[i] - under[i];
        }
    }
    const int m = m0 + kStrip * wave + l16, n = n0 + 4 * kq;
    if (wave >= MT || m >= M) return;
    const int64_t at = (int64_t)m * N + n;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (n + i >= N) break;
        float v = sum[i];
        if (!y_bf16 && resid) v = v + resid[at + i];
        if (y_bf16) ((uint16_t*)yv)[at + i] = f32_to_bf16_bits(v);
        else ((float*)yv)[at + i] = v;
    }
}

int tiles_of(int64_t M, int64_t* groups) {
    const int64_t tiles = (M + kStrip - 1) / kStrip;
    *groups = (tiles + 3) / 4;
    return (int)((tiles + *groups - 1) / *groups);
}

template <int DT, int MT>
hipError_t launch(const QGemvArgs& a, int64_t groups, bool y_bf16, hipStream_t st) {
    const auto kernel = qgemm_kquant_shared_kernel<DT, MT>;
    static LdsLimit limit;
    constexpr int bytes = kLds<DT, MT>;
    if (bytes > 48 * 1024)
        if (hipError_t e = limit.raise(bytes, {(const void*)kernel})) return e;
    const int64_t strips = (a.N + kStrip - 1) / kStrip;
    note_kernel("qgemm_kquant_shared_kernel<%d>", MT);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((strips + 7) / 8 * 8 * groups)), dim3(64 * kWaves), bytes, st, (const uint8_t*)a.W, (const uint8_t*)a.act,
                       (void*)a.y, a.resid, (int)a.M, (int)a.N, (int)(a.K / 256), (int)groups, y_bf16 ? 1 : 0);
    return hipGetLastError();
}

template <int DT>
hipError_t launch_tiles(const QGemvArgs& a, bool y_bf16, hipStream_t st) {
    int64_t groups;
    switch (tiles_of(a.M, &groups)) {
    case 1: return launch<DT, 1>(a, groups, y_bf16, st);
    case 2: return launch<DT, 2>(a, groups, y_bf16, st);
    case 3: return launch<DT, 3>(a, groups, y_bf16, st);
    default: return launch<DT, 4>(a, groups, y_bf16, st);
    }
}

}  // namespace

static std::atomic<int> g_kq_shared{0};  // measurement aid: 1 = never, 2 = wherever the kernel takes the product
void set_kquant_shared(int v) { g_kq_shared = v; }

// W as the other kernels on the matrix cores read it.
bool qgemm_kquant_shared_ok(int dt, const void* W, int64_t M, int64_t N, int64_t K) {
    return (dt == kQ4_K || dt == kQ6_K) && K > 0 && K % 256 == 0 && K <= (1 << 20) && M > 0 && M <= 65535 && N > 0 && N <= (1 << 24) &&
           ((N + 127) / 128) * ((M + 15) / 16) < (1 << 24) && ((uintptr_t)W & (dt == kQ4_K ? 15 : 1)) == 0;
}

// Beyond eight rows (which one pass of the rows kernel takes), by what the kernels take, the rounding of x to int8 apart: here, for as many turns as the busiest of 256 compute
// units has workgroups, 0.7 us and per eight super-blocks 0.3 (Q4_K) or 0.6 (Q6_K) and 0.68 for each tile of rows. On 1350 products of 9 to 512 rows, 384 to 24768 x 512 to 14848,
// the choice takes 0.6 % (Q4_K) or 1.6 % (Q6_K) longer than the faster side in the mean. us, here | by the kernel that had them: Q4_K 16 x 4096 x 14336 13.4 | 19.5, 64 x 4096 x 4096 11.2 | 18.6,
// 64 x 4096 x 14336 26.9 | 59.7, 128 x 14336 x 4096 56 | 34, 256 x 4096 x 14336 92 | 100, 512 x 4096 x 4096 65 | 38; Q6_K 16 x 14336 x 4096 17.7 | 22.4, 64 x 4096 x 14336 27.4 | 83, 128 x 14336 x 4096 56 | 36.
// Not where one tile of rows leaves half the compute units idle (16 x 2048 x 14336 Q4_K 13.4 | 11.9, Q6_K 18.2 | 14.8), nor where seven turns and more are one round of super-blocks each, whose
// beginnings take longer than the model's (64 x 28672 x 2048 Q4_K 45.7 | 37.5, 9 rows 21.3 | 18.4; Q6_K 64 45.8 | 41.7, but 48 37 | 40).
bool qgemm_kquant_shared_pays(int dt, const void* W, int64_t M, int64_t N, int64_t K) {
    if (M > kSharedRows || !qgemm_kquant_shared_ok(dt, W, M, N, K) || g_kq_shared == 1 || !kquant_by_rule()) return false;
    if (g_kq_shared == 2) return true;
    if (M <= 8) return false;
    int64_t groups;
    const int tiles = tiles_of(M, &groups);
    const int64_t turns = ((N + 127) / 128 * 8 * groups + 255) / 256, rounds = (K / 256 + kWaves - 1) / kWaves;
    if (M <= kStrip && N <= 2048) return false;
    if (rounds == 1 && turns > 6 && (dt == kQ4_K || tiles == 4)) return false;
    return 2 + (double)turns * (0.7 + (double)rounds * ((dt == kQ4_K ? 0.3 : 0.6) + 0.68 * tiles)) < qgemv_kquant_us(dt, M, N, K);
}

hipError_t qgemm_kquant_shared(int dt, const QGemvArgs& a, hipStream_t st, bool y_bf16) {
    return dt == kQ4_K ? launch_tiles<kQ4_K>(a, y_bf16, st) : launch_tiles<kQ6_K>(a, y_bf16, st);
}

}  // namespace mimir
