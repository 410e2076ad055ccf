// The exact form of the prompt-sized Q4_0 product with bfloat16 activations (qgemm_q4_0.hip: no operand is rounded,
// float32 sums), for products large enough to pay for a pass over W first, with one MFMA a weight instead of two.
//
// The tile kernel multiplies x by the weights (n - 8) d, which have up to 15 significant bits and so enter the
// bfloat16 matrix cores as two halves. Here the scale stays out of the matrix cores: the weights enter as their
// integers n - 8, exact in bfloat16, so that a block's products x (n - 8) are exact (8 by 4 significant bits) and
// v_mfma_f32_32x32x16_bf16 leaves the block's sum in float32; one FMA per output and block then adds d times that sum
// (d, the block's binary16 scale, is exact in float32, and W's row is a lane's column of the MFMA's result, so the scale
// is one register a lane). Nothing is rounded but float32 sums, as in the tile kernel; which sums are formed differs, so
// the results differ in the last bits like two orders of addition do (the tests' bound is the same for both).
//
// Two launches. blocks_panel_kernel writes W's integers once as bfloat16 and its scales as float32, and X, which the caller
// has row by row, both in the order in which a stage of LDS holds them and an MFMA's lanes read them: granules of 32 rows by one block, 2 KB.
// So every load of qgemm_q4_0_blocks_kernel is a whole KB from contiguous memory straight into LDS (global_load_lds_dwordx4)
// and a fragment read is 1 KB in a row. A workgroup of eight wavefronts owns a tile of Y of 256 x 256 (a wavefront 128 x
// 64), 256 x 192 (64 x 96) or 128 x 256 (64 x 64), cut as tile_plan.h says so that the last round of tiles leaves few
// compute units idle; a stage is one block of 32 of K, four stages are in LDS and three of them on their way while one is multiplied.
// The two MFMAs of a 32 x 32 sub-tile and block are issued with the FMAs of the sub-tile before it.
//
// What bounds it: 64 cycles of MFMA and 64 of FMA per sub-tile and block, which hardly overlap on a SIMD, and the pass over W (28 us at
// 14336 x 4096: 150 MB at the rate of a copy). Stages of a pair of blocks, two of them, with operands in rows and fragments read behind each
// barrier, before; whole calls then and now: 512 x 14336 x 4096 135 -> 124 us, 512 x 28672 x 4096 235 -> 206, 2048 x 4096 x
// 4096 102 -> 94, 2048 x 14336 x 4096 312 -> 297 (810 TFLOP/s), 4096 x 14336 x 4096 607 -> 555. Of the tenth, the stages gave half and
// the fragments read a block ahead the other.
//
// Reference semantics: Tensor.MatMulT for a half-precision x and block-quantized w, tensor/quant.go:45-48.
#include "device_util.h"
#include "kernels.h"
#include "q4_halves.h"
#include "tile_plan.h"

namespace mimir {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kGranule = 1024;  // bfloat16 of 32 rows by a block: two halves of the block, each in the order of an operand's lanes
constexpr int kStages = 4;

// A workgroup's tile of Y: WM x (8 / WM) wavefronts of (32 MT) x (32 NT) each.
template <int WM, int MT_, int NT_>
struct Shape {
    static constexpr int WN = 8 / WM, MT = MT_, NT = NT_;
    static constexpr int BM = WM * 32 * MT, BN = WN * 32 * NT;
    static constexpr int kChunksX = BM / 32 * 2, kChunksP = BN / 32 * 2;             // KB of a stage
    static constexpr int kX = kChunksX / 8, kLoads = kX + (kChunksP + 7) / 8;         // a wavefront issues: kX of X, then P's (the last may do one twice)
    static constexpr int stage = (kChunksX + kChunksP) * 1024;
    static constexpr int kEarly = MT * NT >= 8 ? 1 : MT;  // sub-tiles of X whose fragments two blocks have registers for
    static constexpr int sw = kStages * stage;                                       // float [2 groups][BN / 32][kGroup][32]
    static constexpr int sw_group = BN / 32 * 1024;
    static constexpr int total = sw + 2 * sw_group;
    static_assert(kChunksX % 8 == 0 && BN <= 256 && kLoads <= MT * NT && NT + kEarly <= MT * NT, "a load with a sub-tile, a strip's scales a wavefront");
};
using Wide = Shape<2, 4, 2>;    // 256 x 256
using Narrow = Shape<4, 2, 3>;  // 256 x 192: to fill a last round that wide tiles would leave partly empty
using Low = Shape<2, 2, 2>;     // 128 x 256: for products with too few wide tiles for the device
constexpr size_t kLdsBytes = Wide::total;
static_assert(Narrow::total <= Wide::total && Low::total <= Wide::total, "");

// A wavefront takes a strip's block, lane r + 32 q what row r has of eights q and 2 + q: of W the eight bytes q, whose low nibbles are
// eight q and whose high nibbles 2 + q, as the bfloat16 integers n - 8; of X sixteen bytes each.
__global__ __launch_bounds__(256) void blocks_panel_kernel(const uint8_t* __restrict__ W, const uint16_t* __restrict__ X, int64_t x_row_stride, uint16_t* __restrict__ P,
                                                           uint16_t* __restrict__ XG, float* __restrict__ SW, int M, int N, int nb, int strips) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, q = lane >> 5;
    const int groups = (nb + 31) >> 5, task = (int)blockIdx.x / groups, first = ((int)blockIdx.x - task * groups) * 32 + 8 * wave;  // of blocks
    const bool of_w = task < strips;
    const int strip = of_w ? task : task - strips, at = strip * 32 + r, last = (of_w ? N : M) - 1;
    const int row = at < last ? at : last;  // past the matrix: its last row again
    if (first >= nb) return;
    uint16_t* out = (of_w ? P : XG) + ((int64_t)strip * nb + first) * kGranule + lane * 8;
    if (!of_w) {
        u32x4 v[8][2];
        const uint16_t* from = X + (int64_t)row * x_row_stride + q * 8;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int half = 0; half < 2; half++) v[i][half] = *(const u32x4*)(from + (first + i < nb ? first + i : nb - 1) * 32 + half * 16);
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int half = 0; half < 2; half++)
                if (first + i < nb) *(u32x4*)(out + i * kGranule + 512 * half) = v[i][half];
        return;
    }
    const uint8_t* blocks = W + ((int64_t)row * nb + first) * 18;
    const bool aligned = ((uintptr_t)W & 3) == 0;
    PairBytes pair[4];  // nb is even
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (first + 2 * i < nb) pair[i] = load_pair(blocks + 36 * i, q, aligned);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (first + i >= nb) return;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            u32x4 v;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                // a small integer's float32 has nothing below its upper 16 bits: those are its bfloat16
                const uint32_t two = (k < 2 ? pair[i / 2].lo[i & 1] : pair[i / 2].hi[i & 1]) >> (16 * (k & 1) + 4 * half);
                const float lo = (float)((int)(two & 15) - 8), hi = (float)((int)((two >> 8) & 15) - 8);
                v[k] = (__builtin_bit_cast(uint32_t, lo) >> 16) | (__builtin_bit_cast(uint32_t, hi) & 0xffff0000u);
            }
            *(u32x4*)(out + i * kGranule + 512 * half) = v;
        }
        if (q == 0) SW[((int64_t)strip * scale_blocks(nb) + first + i) * kGranuleS + r] = f16_bits_to_f32((uint16_t)pair[i / 2].scale[i & 1]);
    }
}

// One tile: Y [m0 .. m0 + BM) x [n0 .. n0 + BN).
template <class S, bool OUT_F32>
__device__ __forceinline__ void tile_body(const uint16_t* __restrict__ P, const uint16_t* __restrict__ XG, const float* __restrict__ SW, void* __restrict__ Yv,
                                          int M, int N, int nb, int m0, int n0, char* lds) {
    constexpr int MT = S::MT, NT = S::NT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::WN, wn = wave % S::WN;

    // This wavefront's loads: KB kX wave + j of X's granules, then as many of P's. Strips past the matrix re-read its last
    // strip (their results are not stored).
    const char* from[S::kLoads];
    uint32_t into[S::kLoads];
#pragma unroll
    for (int j = 0; j < S::kLoads; j++) {
        const bool of_x = j < S::kX;
        int c = of_x ? S::kX * wave + j : (S::kLoads - S::kX) * wave + j - S::kX;
        if (!of_x && c >= S::kChunksP) c = S::kChunksP - 1;  // the same KB to the same place twice
        const int strip = (of_x ? m0 : n0) / 32 + c / 2, last = ((of_x ? M : N) - 1) / 32;
        from[j] = (const char*)((of_x ? XG : P) + (int64_t)(strip < last ? strip : last) * nb * kGranule) + (c & 1) * 1024;
        into[j] = (of_x ? c : c + S::kChunksX) * 1024;
    }
    const uint32_t lane16 = lane * 16;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    // W's scales: wavefront w brings strip w of the tile's, a group of blocks at a time
    const bool has_sw = wave < S::BN / 32;
    const char* sw_from;
    {
        const int strip = n0 / 32 + (has_sw ? wave : 0), last = (N - 1) / 32;
        sw_from = (const char*)(SW + (int64_t)(strip < last ? strip : last) * scale_blocks(nb) * kGranuleS);
    }
    const uint32_t sw_into = lds0 + S::sw + wave * 1024;

    const int r32 = lane & 31, hi = lane >> 5;
    const int a_off = wm * MT * 2048 + lane * 16, b_off = S::kChunksX * 1024 + wn * NT * 2048 + lane * 16;

    f32x16 acc[MT][NT], zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = zero;

    auto load = [&](int j, uint32_t slot, int step) {
        load_to_lds(from[j], lane16, lds0 + slot + into[j]);
        from[j] += kGranule * 2 * step;
    };
    if (has_sw) load_to_lds(sw_from, lane16, sw_into);
    // Stages on their way or in use: while a block is multiplied its own stage is refilled, its fragments being in registers, or, where
    // some are read late, the stage of the block before.
    constexpr int kDepth = MT > S::kEarly ? kStages - 1 : kStages;
    uint32_t slot = 0;
    for (int i = 0; i < kDepth; i++) {
#pragma unroll
        for (int j = 0; j < S::kLoads; j++) load(j, slot, i + 1 < nb ? 1 : 0);
        slot += S::stage;
    }
    // Fragments: those of W and of the first kEarly sub-tiles of X are read while the block before is multiplied, so that a block's
    // first products do not wait behind its barrier for every wavefront's reads at once.
    constexpr int kEarly = S::kEarly;
    bf16x8 early[2][kEarly][2], b[2][NT][2], late[MT > kEarly ? MT - kEarly : 1][2];  // [sub-tile][half of the block]
    float dw[2][NT];
    auto read_w = [&](int set, int nt, const char* st, int i) {
#pragma unroll
        for (int h = 0; h < 2; h++) b[set][nt][h] = *(const bf16x8*)(st + b_off + nt * 2048 + h * 1024);
        dw[set][nt] = *(const float*)(lds + S::sw + (i / kGroup & 1) * S::sw_group + (wn * NT + nt) * 1024 + (i & (kGroup - 1)) * 128 + r32 * 4);
    };
    auto read_x = [&](bf16x8 to[2], int mt, const char* st) {
#pragma unroll
        for (int h = 0; h < 2; h++) to[h] = *(const bf16x8*)(st + a_off + mt * 2048 + h * 1024);
    };
    wait_loads<S::kLoads*(kDepth - 1)>();
    lds_barrier();
#pragma unroll
    for (int nt = 0; nt < NT; nt++) read_w(0, nt, lds, 0);
#pragma unroll
    for (int mt = 0; mt < kEarly; mt++) read_x(early[0][mt], mt, lds);
    f32x16 c[2];  // the sums of a sub-tile, finished with the next one's products
    c[1] = zero;
    float dlast = 0.f;
    uint32_t use = 0;  // the stage of block i
    auto block = [&](int i, int set) {
        wait_loads<S::kLoads*(kDepth - 2)>();  // this wavefront's part of block i + 1 has landed, and W's scales
        lds_barrier();                           // everyone's has, and everyone has read the block before for the last time
        const int step = i + kDepth + 1 < nb ? 1 : 0;
        const uint32_t next = use + S::stage == S::sw ? 0 : use + S::stage;
        const uint32_t fill = MT > kEarly ? (use ? use - S::stage : S::sw - S::stage) : use;
        const int ahead = i + 1 < nb ? i + 1 : i;
        if (has_sw && (i & (kGroup - 1)) == 0 && i + kGroup < nb) {  // the next group of W's scales, over the one before this
            sw_from += 1024;
            load_to_lds(sw_from, lane16, sw_into + ((i / kGroup + 1) & 1) * S::sw_group);
        }
#pragma unroll
        for (int mt = kEarly; mt < MT; mt++) read_x(late[mt - kEarly], mt, lds + use);
        // Sub-tile s = NT mt + nt: its two MFMAs are issued with the FMAs of the sub-tile before it, so that the
        // vector unit works while the matrix cores do.
#pragma unroll
        for (int sub = 0; sub < MT * NT; sub++) {
            const int mt = sub / NT, nt = sub % NT, was = (sub + MT * NT - 1) % (MT * NT);
            if (sub < S::kLoads) load(sub, fill, step);
            const bf16x8* a = mt < kEarly ? early[set][mt < kEarly ? mt : 0] : late[mt < kEarly ? 0 : mt - kEarly];
            c[sub & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[set][nt][0], zero, 0, 0, 0);
            c[sub & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[set][nt][1], c[sub & 1], 0, 0, 0);
            if (sub < NT) read_w(set ^ 1, sub, lds + next, ahead);
            else if (sub < NT + kEarly) read_x(early[set ^ 1][sub - NT], sub - NT, lds + next);
            const float d = sub == 0 ? dlast : dw[set][was % NT];
#pragma unroll
            for (int e = 0; e < 16; e++) acc[was / NT][was % NT][e] = fmaf(d, c[(sub + 1) & 1][e], acc[was / NT][was % NT][e]);
            __builtin_amdgcn_sched_barrier(0);
        }
        dlast = dw[set][NT - 1];
        use = next;
    };
    for (int i = 0; i + 1 < nb; i += 2) {  // K is a multiple of 64
        block(i, 0);
        block(i + 1, 1);
    }
#pragma unroll
    for (int e = 0; e < 16; e++) acc[MT - 1][NT - 1][e] = fmaf(dlast, c[1][e], acc[MT - 1][NT - 1][e]);
    wait_loads<0>();  // nothing of this tile's is on its way into LDS any more

    // One rounding to the output's dtype (f32ToBF16, backend/cpu/half.go:42-51). An MFMA leaves a lane one column of Y
    // and four consecutive rows per group of four registers; a 4 x 4 transposition within each quad of lanes turns that
    // into one row and four consecutive columns a lane, stored with one 8-byte (bfloat16) or 16-byte (float32) store.
    const bool wide_ok = (N & 3) == 0 && ((uintptr_t)Yv & 15) == 0;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int m = m0 + wm * 32 * MT + mt * 32 + q * 8 + hi * 4 + (lane & 3);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                float v[4] = {acc[mt][nt][4 * q], acc[mt][nt][4 * q + 1], acc[mt][nt][4 * q + 2], acc[mt][nt][4 * q + 3]};
                quad_transpose(v, lane);
                const int n = n0 + wn * 32 * NT + nt * 32 + (r32 & ~3);
                if (m >= M || n >= N) continue;
                if (wide_ok && n + 3 < N) {
                    if (OUT_F32) {
                        const f32x4 o = {v[0], v[1], v[2], v[3]};
                        *(f32x4*)((float*)Yv + (int64_t)m * N + n) = o;
                    } else {
                        const u32x2 o = {(uint32_t)f32_to_bf16_bits(v[0]) | (uint32_t)f32_to_bf16_bits(v[1]) << 16,
                                         (uint32_t)f32_to_bf16_bits(v[2]) | (uint32_t)f32_to_bf16_bits(v[3]) << 16};
                        *(u32x2*)((uint16_t*)Yv + (int64_t)m * N + n) = o;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if (n + k >= N) continue;
                        if (OUT_F32) ((float*)Yv)[(int64_t)m * N + n + k] = v[k];
                        else ((uint16_t*)Yv)[(int64_t)m * N + n + k] = f32_to_bf16_bits(v[k]);
                    }
                }
            }
        }
}

template <bool OUT_F32>
__global__ __launch_bounds__(512) void qgemm_q4_0_blocks_kernel(const uint16_t* __restrict__ P, const uint16_t* __restrict__ XG, const float* __restrict__ SW,
                                                                void* __restrict__ Yv, int M, int N, int nb, PanelPlan plan) {
    extern __shared__ __align__(1024) char lds[];
    int b = (int)blockIdx.x;
    if (plan.low) {
        const int ntiles = plan.tiles_m * plan.wide_cols;
        const int t = tile_of(b, ntiles);
        if (t >= ntiles) return;  // the whole workgroup
        tile_body<Low, OUT_F32>(P, XG, SW, Yv, M, N, nb, (t % plan.tiles_m) * Low::BM, (t / plan.tiles_m) * Low::BN, lds);
        return;
    }
    const int nwide = plan.tiles_m * plan.wide_cols;
    const int wide_wgs = ((nwide + 7) >> 3) << 3;
    if (b < wide_wgs) {
        const int t = tile_of(b, nwide);
        if (t >= nwide) return;
        tile_body<Wide, OUT_F32>(P, XG, SW, Yv, M, N, nb, (t % plan.tiles_m) * Wide::BM, (t / plan.tiles_m) * Wide::BN, lds);
        return;
    }
    b -= wide_wgs;
    const int nnarrow = plan.tiles_m * plan.narrow_cols;
    const int t = tile_of(b, nnarrow);
    if (t >= nnarrow) return;
    tile_body<Narrow, OUT_F32>(P, XG, SW, Yv, M, N, nb, (t % plan.tiles_m) * Narrow::BM, plan.wide_cols * Wide::BN + (t / plan.tiles_m) * Narrow::BN, lds);
}

// Costs in wide tiles' time, measured: a tile of 256 x 192 has three quarters of the work, one of 128 x 256 half.
constexpr double kNarrowCost = 0.78, kLowCost = 0.56;

std::atomic<int> g_blocks{1};  // measurement aid: 0 keeps every product on the tile kernel, 2 takes this one whatever the shape

}  // namespace

void set_q4_0_blocks(int v) { g_blocks = v; }
bool q4_0_blocks_chosen() { return g_blocks != 1; }

// W's integers and X in granules, W's scales.
static size_t granules_bytes(int64_t rows, int64_t K) { return (size_t)((rows + 31) / 32) * (size_t)(K / 32) * kGranule * 2; }
size_t qgemm_q4_0_blocks_ws_bytes(int64_t M, int64_t N, int64_t K) {
    return granules_bytes(N, K) + granules_bytes(M, K) + (size_t)((N + 31) / 32) * (size_t)scale_blocks((int)(K / 32)) * kGranuleS * 4;
}

// Whether the product is the faster here than in the tile kernel, the pass over W included: from about 200 tiles of
// 128 x 256 on (measured at K = 4096: 512 x 14336 484 against 404 TFLOP/s, 2048 x 4096 569 against 438, 2048 x 14336 757
// against 435; 1024 x 4096, 128 tiles, 327 against 362).
bool qgemm_q4_0_blocks_pays(int64_t M, int64_t N, int64_t K) {
    if (g_blocks == 0 || M <= 0 || N <= 0 || K <= 0 || K % 64 != 0) return false;
    if (g_blocks == 2) return true;
    return M >= 256 && ((M + 127) / 128) * ((N + 255) / 256) >= 192;
}

// X [M, K] bfloat16 (16-byte aligned, rows x_row_stride elements apart, a multiple of 8), W [N, K] Q4_0, Y [M, N] bfloat16
// or float32; ws: qgemm_q4_0_blocks_ws_bytes(M, N, K) bytes, 16-byte aligned.
hipError_t qgemm_q4_0_blocks(const void* W, const void* X, int64_t x_row_stride, void* Y, int64_t M, int64_t N, int64_t K, bool out_f32, void* ws,
                             hipStream_t st) {
    if (!ws || ((uintptr_t)ws & 15) != 0 || ((uintptr_t)X & 15) != 0 || x_row_stride % 8 != 0 || x_row_stride < K || ((uintptr_t)W & 1) != 0 ||
        M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || M >= (1 << 24) || N >= (1 << 24) || K > (1 << 24))
        return hipErrorInvalidValue;
    static LdsLimit limit;
    if (hipError_t e = limit.raise((int)kLdsBytes, {(const void*)qgemm_q4_0_blocks_kernel<true>, (const void*)qgemm_q4_0_blocks_kernel<false>})) return e;
    const int nb = (int)(K / 32), strips = (int)((N + 31) / 32), x_strips = (int)((M + 31) / 32);
    uint16_t* P = (uint16_t*)ws;
    uint16_t* XG = P + granules_bytes(N, K) / 2;
    float* SW = (float*)(XG + granules_bytes(M, K) / 2);
    hipLaunchKernelGGL(blocks_panel_kernel, dim3((unsigned)((nb + 31) / 32 * (strips + x_strips))), dim3(256), 0, st, (const uint8_t*)W, (const uint16_t*)X,
                       x_row_stride, P, XG, SW, (int)M, (int)N, nb, strips);
    PanelPlan plan;
    plan_panel(M, N, kNarrowCost, kLowCost, &plan);
    const int first = plan.tiles_m * plan.wide_cols, then = plan.tiles_m * plan.narrow_cols;
    const dim3 grid((unsigned)(((first + 7) / 8) * 8 + ((then + 7) / 8) * 8));
    if (out_f32)
        hipLaunchKernelGGL(qgemm_q4_0_blocks_kernel<true>, grid, dim3(512), kLdsBytes, st, P, XG, SW, Y, (int)M, (int)N, nb, plan);
    else
        hipLaunchKernelGGL(qgemm_q4_0_blocks_kernel<false>, grid, dim3(512), kLdsBytes, st, P, XG, SW, Y, (int)M, (int)N, nb, plan);
    note_kernel("qgemm_q4_0_blocks_kernel: %d x %d tiles of %s, %d x %d tiles of 256 x 192", plan.tiles_m, plan.wide_cols, plan.low ? "128 x 256" : "256 x 256",
                plan.tiles_m, plan.narrow_cols);
    return hipGetLastError();
}

}  // namespace mimir
