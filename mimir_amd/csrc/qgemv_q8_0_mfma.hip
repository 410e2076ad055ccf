// Products of two and more rows of x with Q8_0 weights on the int8 matrix cores of gfx950, W read once for eight rows
// (the output projection of a batch's decoding step) or for 32 (a prompt's rows). What it computes is qdotQ8_0Go's sum
// (backend/cpu/qmatmul.go:125-139, see qgemv_q8_0.hip), in one of two orders:
//   - a block's int32 sum, exact, once times the product of the two scales;
//   - FOUR: the CPU's four sums a block, one for every fourth group of four values, each times the product of the scales (a
//     multiply, then an add) into a float32 sum of its own, added (0 + 2) + (1 + 3) at the end. It serves two to eight rows by the
//     largest matrices, the output projections, whose results stay what they were before there was the other (8 x 32768 x 4096: 36.1 us by the other, 36.7).
//
// One v_mfma_i32_32x32x32_i8 per block: its first operand has 32 rows of x, or eight rows four times (FOUR: each time with everything but the
// values of one of the four sums zeroed, which of the 16 values a lane holds are one dword), its other operand
// 32 rows of W. A lane ends up with its row of W's sums for sixteen rows of x, or for four (and three times again,
// which it leaves, or the four sums of each). A workgroup's wavefronts take runs of eight blocks in turn and add their sums up in order.
//
// W stays in ggml's layout. As in qgemv_q4_0_rows.hip, a wavefront loads a run of its 32 rows as 16-byte pieces in row
// order (272 bytes a row), passes them through a private LDS slab and reads its 16 int8 of each block back as dwords.
// Where K is no multiple of 256 the pieces start on two bytes, which the hardware takes, and the last run reaches back
// over blocks whose scale is then nought. x comes converted by q8_convert_act: of eight rows a lane loads its row's
// sixteen bytes of a block, again for the next run as soon as it has used them; of 32, whose rows would be 64 lines a
// load, x goes through LDS as W does, and a block's MFMA is issued before the sums of the block ahead of it (512 x 4096
// x 14336 without: 236 us, with: 191).
//
// What bounds it. Eight rows: the loads (143 MB of 32768 x 4096: 27 us at the rate of a copy), with four wavefronts
// too few for them where the matrix is small. 32 rows: a conversion, a product and an fma for each sum and block, 192
// cycles beside the MFMA's 32 and some 50 of unpacking (61 vector instructions a block by the counters, 57 % of the SIMDs' cycles at
// 512 x 4096 x 14336, where LDS spends 28 % of them in bank conflicts); 315 TFLOP/s there. Whole calls, us, with W read for eight rows
// by the vector unit (and by four zeroed copies of x on the matrix cores: 2 and 8 x 32768 x 4096) and now:
//   2, 8 x 32768 x 4096    40, 43 -> 35, 37        8 x 4096 x 14336     71 -> 29
//   32 x 32768 x 4096         122 -> 49            64 x 1024 x 4096     34 -> 14
//   512 x 4096 x 14336       3511 -> 191           128 x 4096 x 4096   229 -> 24
// Errors against 64 bits, of the result: K = 256: 7.2e-8 -> 6.0e-8, 4096: 9.1e-8 -> 8.5e-8 (FOUR: 1.25e-7 as ever), 14336: 1.02e-7 -> 9.8e-8, 28672: 1.13e-7 -> 1.03e-7, 57344: 1.3e-7 .. 3.9e-7 -> 1.1e-7.
#include "device_util.h"
#include "kernels.h"

namespace mimir {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int kRunBlocks = 8;
constexpr int kRunBytes = 34 * kRunBlocks;     // 272: seventeen pieces a row
constexpr int kPieces = kRunBytes / 16;
constexpr int kSlabStride = kRunBytes + 32;    // 304 bytes = 76 dwords: rows fall on eight banks, four to each
constexpr int kSlabBytes = 32 * kSlabStride;
constexpr int kLoads = (32 * kPieces + 63) / 64;  // 9: the last one half full
constexpr int kManyRows = 32;
constexpr int kRunsTogether = 8;

// LDS of a wavefront: the slab, the scales of x of a run [block][row] and, of 32 rows, x's pieces [row][half][block],
// the block's place turned by the row so that a block's reads fall on all banks.
template <int XR>
constexpr int kWaveLds = kSlabBytes + kRunBlocks * XR * 4 + (XR == kManyRows ? XR * kRunBlocks * 32 : 0);

// XR: rows of x a workgroup (8 or 32); WAVES: its wavefronts, among which the runs of K go round. AHEAD: a run's loads stay a run ahead, which takes the
// registers of two wavefronts: for so few workgroups that no more are on a compute unit (four sums, us, without and with: 4 x 8192 x 14336 48, 33).
template <int XR, int WAVES, bool FOUR = false, bool AHEAD = false>
__global__ __launch_bounds__(64 * WAVES, XR == kManyRows || AHEAD ? 2 : 4) void qgemv_q8_0_mfma_kernel(const uint8_t* __restrict__ W, const uint8_t* act, void* yv, int M,
                                                                                             int N, int nb, int64_t act_row_bytes, int y_bf16) {
    constexpr bool kMany = XR == kManyRows;
    constexpr int kSums = FOUR ? 16 : XR / 2;  // of a lane
    static_assert(!FOUR || XR == 8, "four sums of each of a lane's four rows");
    extern __shared__ __align__(16) uint8_t smem[];  // per wavefront; later the wavefronts' sums
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The grid runs over the groups of rows of x first: the workgroups that read the same 32 rows of W are handed
    // out together, so the rows come from HBM once and from the memory-side cache for the other groups.
    const int ngroups = (M + XR - 1) / XR, group = (int)(blockIdx.x % (unsigned)ngroups);
    const int n0 = (int)(blockIdx.x / (unsigned)ngroups) * 32, n = n0 + l32;
    const int nruns = (nb + kRunBlocks - 1) / kRunBlocks, nbp = nb | 1;
    uint8_t* slab = smem + wave * kWaveLds<XR>;
    float* dxs = (float*)(slab + kSlabBytes);
    uint8_t* xslab = slab + kSlabBytes + kRunBlocks * XR * 4;
    act += (int64_t)XR * group * act_row_bytes;
    const int64_t y0 = (int64_t)XR * group * N;
    M = M - XR * group < XR ? M - XR * group : XR;

    // piece p = 64 i + lane of a run: row p / 17 of the 32, bytes 16 (p % 17).. of its 272
    uint32_t goff[kLoads], loff[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        int p = 64 * i + lane;
        p = p < 32 * kPieces ? p : 32 * kPieces - 1;  // the last load's upper lanes repeat the last piece
        const int r = p / kPieces, c = p - kPieces * r;
        const int row = n0 + r < N ? n0 + r : N - 1;
        goff[i] = (uint32_t)(row - n0) * (uint32_t)(nb * 34) + 16 * c;  // 32 rows of W within 4 GB (checked by the host)
        loff[i] = r * kSlabStride + 16 * c;
    }
    const uint8_t* wbase = W + (int64_t)n0 * nb * 34;
    // rows past M: the last one again, not stored
    auto row_of = [&](int r) { return act + (int64_t)(r < M ? r : M - 1) * act_row_bytes; };
    const i32x4* xq = (const i32x4*)row_of(l32 & (XR - 1)) + (int64_t)lh * nbp;  // + b: half lh of block b of this lane's operand row
    const int sum = l32 >> 3;                                                    // FOUR: which sum's values it keeps, a dword of a half
    uint32_t xoff[8];  // of 32 rows: this lane's pieces of a run, of row 4 i + lane / 16 half (lane / 8) % 2 of block lane % 8
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (kMany) xoff[i] = (uint32_t)((row_of(4 * i + (lane >> 4)) - act) + (((lane >> 3) & 1) * nbp + (lane & 7)) * 16);
    auto x_piece = [](int row, int half, int block) { return ((2 * row + half) * kRunBlocks + (block ^ (row & 7))) * 16; };
    // The scales of x of a run: of 32 rows a lane brings four blocks' of row l32, of eight one block's of row 4 lh + l32 % 4.
    const float* own_scales = (const float*)(row_of(kMany ? l32 : 4 * lh + (l32 & 3)) + (int64_t)nbp * 32) + (kMany ? 4 * lh : l32 >> 2);

    auto start_of = [&](int run) { return kRunBlocks * run < nb - kRunBlocks ? kRunBlocks * run : nb - kRunBlocks; };  // the last run reaches back
    u32x4 w[kLoads];
    i32x4 x[FOUR ? 1 : 8];  // eight rows: the operands of a run's blocks; 32: this lane's pieces of it
    int kept[FOUR ? 8 : 1];
    auto fetch_x = [&](int b, int block) {  // of eight rows
        if constexpr (FOUR) kept[b] = ((const int*)(xq + block))[sum];
        else x[b] = xq[block];
    };
    float own[kMany ? 4 : 1];
    auto fetch = [&](int at) {
        const uint8_t* p = wbase + (int64_t)at * 34;
#pragma unroll
        for (int i = 0; i < kLoads; i++) w[i] = load_u32x4_unaligned(p + goff[i]);
        if constexpr (kMany) {
#pragma unroll
            for (int i = 0; i < 8; i++) x[i] = *(const i32x4*)(act + xoff[i] + 16 * at);
        }
        __builtin_memcpy(own, own_scales + at, sizeof(own));
    };

    // A run's sums by themselves, those of eight runs, and the eights': short chains, whose errors stay below those of
    // the one-row kernel's 64 lanes with four sums each (one chain for all of a wavefront's blocks: 2.0e-7 at K = 14336).
    float acc[kSums], total[kSums];
#pragma unroll
    for (int i = 0; i < kSums; i++) acc[i] = total[i] = 0.f;
    if (wave < nruns) {
        fetch(start_of(wave));
#pragma unroll
        for (int b = 0; b < kRunBlocks; b++)
            if (!kMany) fetch_x(b, start_of(wave) + b);
    }
    const uint8_t* mine = slab + l32 * kSlabStride + 16 * lh;  // the lane's 16 int8 of block b: bytes 34 b + 2 + 16 lh
    for (int run = wave; run < nruns; run += WAVES) {
        const int nrun = run + WAVES < nruns ? run + WAVES : run, next = start_of(nrun), done = kRunBlocks * run - start_of(run);
        // slabs and scales are this wavefront's alone, and a wavefront's LDS operations complete in order
#pragma unroll
        for (int i = 0; i < kLoads - 1; i++) *(u32x4*)(slab + loff[i]) = w[i];
        if (lane < 32 * kPieces - 64 * (kLoads - 1)) *(u32x4*)(slab + loff[kLoads - 1]) = w[kLoads - 1];
        if constexpr (kMany) {
#pragma unroll
            for (int i = 0; i < 4; i++) dxs[(4 * lh + i) * XR + l32] = own[i % (kMany ? 4 : 1)];
#pragma unroll
            for (int i = 0; i < 8; i++) *(i32x4*)(xslab + x_piece(4 * i + (lane >> 4), (lane >> 3) & 1, lane & 7)) = x[i];
        } else {
            dxs[(l32 >> 2) * XR + 4 * lh + (l32 & 3)] = own[0];
        }
        fetch(next);
        if (AHEAD) __builtin_amdgcn_sched_barrier(0);
        // The block's product of this lane's row of W (scale into dw).
        auto multiply = [&](int b, float* dw) {
            // bytes 34 b + 2 ..: on a dword for odd b, two bytes into one for even b
            i32x4 wop;
            if (b & 1) {
                const uint8_t* p = mine + 34 * b + 2;
#pragma unroll
                for (int i = 0; i < 4; i++) wop[i] = (int)*(const uint32_t*)(p + 4 * i);
                *dw = f16_bits_to_f32((uint16_t)(*(const uint32_t*)(slab + l32 * kSlabStride + 34 * b - 2) >> 16));
            } else {
                const uint8_t* p = mine + 34 * b;
                uint32_t r[5];
#pragma unroll
                for (int i = 0; i < 5; i++) r[i] = *(const uint32_t*)(p + 4 * i);
#pragma unroll
                for (int i = 0; i < 4; i++) wop[i] = (int)__builtin_amdgcn_alignbit(r[i + 1], r[i], 16);
                *dw = f16_bits_to_f32((uint16_t)(*(const uint32_t*)(slab + l32 * kSlabStride + 34 * b) & 0xffffu));
            }
            *dw = b < done ? 0.f : *dw;  // blocks that the run before has taken
            i32x4 xop;
            if constexpr (FOUR) {
#pragma unroll
                for (int i = 0; i < 4; i++) xop[i] = sum == i ? kept[b] : 0;  // operand row 8 l + m: sum l of row m
            } else {
                xop = kMany ? *(const i32x4*)(xslab + x_piece(l32, lh, b)) : x[b];
            }
            i32x16 zero;
#pragma unroll
            for (int i = 0; i < 16; i++) zero[i] = 0;
            return __builtin_amdgcn_mfma_i32_32x32x32_i8(xop, wop, zero, 0, 0, 0);
        };
        float part[kSums];
        float dw;
        i32x16 c = multiply(0, &dw);
#pragma unroll
        for (int b = 0; b < kRunBlocks; b++) {
            float dw_next = 0.f;
            i32x16 c_next = c;
            if (b + 1 < kRunBlocks) c_next = multiply(b + 1, &dw_next);  // under the sums of block b
            if (kMany) __builtin_amdgcn_sched_barrier(0);
            if (!kMany) fetch_x(b, next + b);
            // register 4 g + j: row 8 g + 4 lh + j of x
#pragma unroll
            for (int g = 0; g < kSums / 4; g++) {
                const f32x4 dx = *(const f32x4*)(dxs + b * XR + (FOUR ? 0 : 8 * g) + 4 * lh);
                if (FOUR) {  // register 4 l + j: sum l of row 4 lh + j
#pragma clang fp contract(off)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float dd = dw * dx[j], t = dd * (float)c[4 * g + j];
                        acc[4 * g + j] = acc[4 * g + j] + t;
                    }
                    continue;
                }
#pragma unroll
                for (int j = 0; j < 4; j++) part[4 * g + j] = b == 0 ? dw * dx[j] * (float)c[4 * g + j] : fmaf(dw * dx[j], (float)c[4 * g + j], part[4 * g + j]);
            }
            c = c_next;
            dw = dw_next;
        }
        if constexpr (FOUR && AHEAD) {  // the next run's loads are under way by here: the compiler issues them where they are used otherwise
#pragma unroll
            for (int i = 0; i < kLoads; i++) asm volatile("" : "+v"(w[i]));
#pragma unroll
            for (int b = 0; b < kRunBlocks; b++) asm volatile("" : "+v"(kept[b]));
        }
        if (FOUR) continue;
#pragma unroll
        for (int i = 0; i < kSums; i++) acc[i] += part[i];
        if ((run / WAVES) % kRunsTogether == kRunsTogether - 1) {
#pragma unroll
            for (int i = 0; i < kSums; i++) {
                total[i] += acc[i];
                acc[i] = 0.f;
            }
        }
    }
    if (!FOUR) {
#pragma unroll
        for (int i = 0; i < kSums; i++) acc[i] += total[i];
    }

    __syncthreads();  // every wavefront is done with its slab
    float* red = (float*)smem;  // [wave][sum][lane]
#pragma unroll
    for (int i = 0; i < kSums; i++) red[(wave * kSums + i) * 64 + lane] = acc[i];
    __syncthreads();
    auto sum_of = [&](int s) {
        float v = red[s * 64 + lane];
#pragma unroll
        for (int o = 1; o < WAVES; o++) v = v + red[(o * kSums + s) * 64 + lane];
        return v;
    };
    // the wavefronts share the sums
    for (int s = wave; s < (FOUR ? 4 : kSums); s += WAVES) {
        const float v = FOUR ? (sum_of(s) + sum_of(8 + s)) + (sum_of(4 + s) + sum_of(12 + s)) : sum_of(s);
        const int m = 8 * (s >> 2) + 4 * lh + (s & 3);
        if (n < N && m < M) {
            const int64_t at = y0 + (int64_t)m * N + n;
            if (y_bf16) ((uint16_t*)yv)[at] = f32_to_bf16_bits(v);
            else ((float*)yv)[at] = v;
        }
    }
}

constexpr int kFewRows = 8;

}  // namespace

// Rows of x converted beforehand (q8_convert_act), eight blocks and more a row.
bool qgemv_q8_0_mfma_ok(const QGemvArgs& a) {
    const int64_t nb = a.K / 32;
    return a.M >= 2 && a.M <= 8 * 65535 && a.act && ((uintptr_t)a.act & 15) == 0 && !a.resid && nb >= kRunBlocks && ((uintptr_t)a.W & 1) == 0 &&
           32 * nb * 34 < ((int64_t)1 << 32) && 32 * (int64_t)q8_act_bytes(a.K) < ((int64_t)1 << 31) && a.N > 0 && a.N <= (1ll << 30);
}

static std::atomic<int> g_q8_mfma{0};  // measurement aid: 1 = wherever the kernel takes the shape, 2 = never
void set_q8_mfma(int v) { g_q8_mfma = v; }

// Up to eight rows: matrices of 32 M weights and more that give the chip 128 workgroups, for two and three rows 192 (us by the vector unit, here; 8 rows: 8192 x 4096 34, 13; 4 rows:
// 4096 x 8192 19, 17, 2048 x 16384 18, 28; 2 rows: 6144 x 8192 20, 18, 4096 x 14336 24, 26), and of short rows, of which the vector unit has as much to do whatever their length: eight rows
// 14336 x 1024 29.7, 8.1, 14336 x 2048 49.7, 12.1, 4096 x 1024 10.5, 6.5; four 4096 x 1024 6.4, 6.4, 8192 x 2048 12.6, 8.3; three 8192 x 1024 8.4, 6.7, but 4096 x 2048 6.3, 7.3; two 14336 x
// 1024 9.3, 7.9, but 12288 x 2048 10.9, 11.0, 8192 x 2048 7.8, 8.2. Other few rows keep the bits that a row alone has.
// More rows, of which the vector unit takes eight a pass over W: from 64 rows of W on nearly always; nine rows 512 x 1024 10.6, 7.5, 64 x 2048 10.3, 8.3, 1280 x 4096 15.6, 11.7, 3072 x 14336 46, 30,
// 17 rows 1024 x 4096 17.2, 12.1; of an odd number of blocks, which the vector unit takes a row of x at a time, from 12000 results on (17 rows 874 x 672 8.8, 7.8, 12 rows 1408 x 352 8.4, 7.0, but 26 x 192 x 1696
// 6.3, 9.9, 9 x 1088 x 1184 7.5, 8.7); but sixteen 1024 x 4096 11.3, 12.0, 512 x 8192 10.8, 17.5, twelve 1536 x 8192 16.8, 17.7 (2048 x 8192 19.8, 17.7), nine 2048 x 14336 27.5, 29.4 (twelve 32.7, 29.7).
bool qgemv_q8_0_mfma_pays(const QGemvArgs& a) {
    if (g_q8_mfma == 2 || !qgemv_q8_0_mfma_ok(a)) return false;
    if (g_q8_mfma == 1) return true;
    if (a.M > kFewRows) return a.M * a.N >= 32768 || (a.N >= 64 && (a.K <= 2048 ? qgemv_q8_0_rows_ok(a) || a.M * a.N >= 12000 : (a.K <= 6144 ? a.N >= 1280 || a.M * a.N >= 17000 : a.M * a.N >= 24000)));
    if (a.K <= 2048 && a.N >= (a.M == 2 ? 14336 : a.M == 3 ? 6144 : 4096)) return true;
    return a.N * a.K >= ((int64_t)32 << 20) && a.N >= (a.M >= 4 ? 4096 : 6144);
}

template <int XR, int WAVES, bool FOUR = false, bool AHEAD = false>
static hipError_t launch(const QGemvArgs& a, int64_t wgs, bool bf16, hipStream_t st) {
    constexpr int kLds = WAVES * kWaveLds<XR>;
    if (kLds > 64 * 1024) {
        static LdsLimit limit;
        if (hipError_t e = limit.raise(kLds, {(const void*)qgemv_q8_0_mfma_kernel<XR, WAVES, FOUR, AHEAD>})) return e;
    }
    hipLaunchKernelGGL((qgemv_q8_0_mfma_kernel<XR, WAVES, FOUR, AHEAD>), dim3((unsigned)wgs), dim3(64 * WAVES), kLds, st, (const uint8_t*)a.W, (const uint8_t*)a.act, (void*)a.y,
                       (int)a.M, (int)a.N, (int)(a.K / 32), (int64_t)q8_act_bytes(a.K), bf16 ? 1 : 0);
    return hipGetLastError();
}

// Eight wavefronts a workgroup where all workgroups then are on the chip at once, two a compute unit of eight rows, one of 32
// (us with four, with eight: 2 x 14336 x 4064 21, 20; 32 x 4096 x 14336 65, 45; past it, 64 x 8192 x 4096 26, 30), else four.
hipError_t qgemv_q8_0_mfma(const QGemvArgs& a, hipStream_t st, bool bf16) {
    const int rows = a.M > kFewRows ? kManyRows : 8;
    const int64_t wgs = ((a.N + 31) / 32) * ((a.M + rows - 1) / rows);
    if (wgs > 0x7fffffff) return hipErrorInvalidValue;
    // from 64 M weights on, of whole runs: sums in the order in which they always were
    if (a.M <= kFewRows && a.N * a.K >= ((int64_t)64 << 20) && a.K % 256 == 0 && ((uintptr_t)a.W & 15) == 0)
        return wgs <= 512 ? launch<8, 4, true, true>(a, wgs, bf16, st) : launch<8, 4, true>(a, wgs, bf16, st);
    if (rows == 8) return wgs <= 512 ? launch<8, 8>(a, wgs, bf16, st) : launch<8, 4>(a, wgs, bf16, st);
    return wgs <= 256 ? launch<kManyRows, 8>(a, wgs, bf16, st) : launch<kManyRows, 4>(a, wgs, bf16, st);
}

}  // namespace mimir
