// y = act(x . W^T) for two to eight rows of float32 x and bfloat16 weights, W read once, on the bfloat16 matrix cores: the
// product of a decoding step of several sequences. v_mfma_f32_16x16x32_bf16 multiplies sixteen rows of W by sixteen
// columns; the columns are the rows of x twice, once their bfloat16 value and once what rounding left of them (a float32's
// first sixteen bits of significand), whose results are added at the end: near float32's accuracy for the price of one
// product. The wavefronts of a workgroup (eight, or sixteen for long rows) share its rows of W and cut K into pieces; W goes from memory straight into
// the operand registers (a lane's sixteen bytes of one row), x is converted on the way, through LDS.
#include "device_util.h"
#include "product_store.h"
#include "stack_ops.h"

#include <type_traits>

namespace mimir {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// A step of 64 along K of x for a wavefront: a lane converts PASSES fours of it, neighbouring lanes neighbouring ones, and the operands are read back from
// LDS of the wavefront's own. Converted by the lanes that use them, in registers, an element cost four loads and conversions (every
// column of the operand, twice for up to four rows): 4 x 2048 x 8192 took 16.3 us, now 9.8, 4 x 2048 x 2048 5.9 and 5.0.
template <int PASSES>
struct XStep {
    static constexpr int kRow = 72;  // of bfloat16, eight of them so that sixteen rows' pieces fall on all banks
    f32x4 v[PASSES];

    __device__ __forceinline__ void load(const float* x, int64_t ldx, int M, int k, int lane) {
#pragma unroll
        for (int p = 0; p < PASSES; p++) {
            const int m = 4 * p + (lane >> 4);
            v[p] = *(const f32x4*)(x + (int64_t)(m < M ? m : M - 1) * ldx + k + 4 * (lane & 15));
        }
    }
    // rows 0..7 of `to` are x's bfloat16, 8..15 what these leave; of up to four rows of x the others stay as they are: columns that are not stored
    __device__ __forceinline__ void put(uint16_t* to, int lane) const {
#pragma unroll
        for (int p = 0; p < PASSES; p++) {
            uint16_t* at = to + (4 * p + (lane >> 4)) * kRow + 4 * (lane & 15);
            const uint32_t high[2] = {pack_bf16(v[p][0], v[p][1]), pack_bf16(v[p][2], v[p][3])};
            const uint32_t low[2] = {pack_bf16(low_part(v[p][0]), low_part(v[p][1])), pack_bf16(low_part(v[p][2]), low_part(v[p][3]))};
            __builtin_memcpy(__builtin_assume_aligned(at, 8), high, 8);
            __builtin_memcpy(__builtin_assume_aligned(at + 8 * kRow, 8), low, 8);
        }
    }
    static __device__ __forceinline__ bf16x8 operand(const uint16_t* from, int s, int lane) {  // of half s of the step
        return __builtin_bit_cast(bf16x8, *(const u32x4*)(from + (lane & 15) * kRow + 32 * s + 8 * (lane >> 4)));
    }
};

// T: groups of sixteen rows of W a workgroup; PASSES: fours of rows of x.
template <int T, int kWaves, int PASSES, Out KIND>
__global__ __launch_bounds__(64 * kWaves, 4) void gemv_bf16_rows_kernel(const uint16_t* __restrict__ W, int64_t ldw, const float* __restrict__ x, int64_t ldx,
                                                                     int M, int N, int K, ProductOut out) {
    __shared__ float red[kWaves][T * 16][17];
    __shared__ __align__(16) uint16_t operands[kWaves][16 * XStep<PASSES>::kRow];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16 * T;
    uint16_t* stage = operands[wave];
    // steps of 32 along K, in pieces of whole pairs (64) a wavefront
    const int pairs = K / 64, per = (pairs + kWaves - 1) / kWaves;
    const int k0 = wave * per * 64, k1 = k0 + per * 64 < K ? k0 + per * 64 : K;
    const uint16_t* wp[T];
#pragma unroll
    for (int t = 0; t < T; t++) wp[t] = W + (int64_t)(n0 + t * 16 + r16 < N ? n0 + t * 16 + r16 : N - 1) * ldw + g * 8;
    f32x4 acc[T];
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // under way: with three or four, fewer wavefronts fit a SIMD (4 x 8192 x 2048 10.3 us, 11.2 with four). An odd last step by itself: in a whole pair the
    // one before it was fetched again, a third more of W where a wavefront has three (2 x 8192 x 1536 8.2 us, so 7.2; of five, 2 x 8192 x 2560 12.0 and 11.2).
    constexpr int kSteps = 2;
    auto sum_of = [&](int from, int to) {
        const int n = (to - from) / 64;
        if (n <= 0) return;
        u32x4 w[kSteps][2][T];
        XStep<PASSES> xs[kSteps];
        auto load = [&](int i, int slot) {
            const int k = from + 64 * i;
            xs[slot].load(x, ldx, M, k, lane);
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int s = 0; s < 2; s++) w[slot][s][t] = *(const u32x4*)(wp[t] + k + 32 * s);
        };
        auto multiply = [&](int slot) {
            xs[slot].put(stage, lane);
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const bf16x8 q = XStep<PASSES>::operand(stage, s, lane);
#pragma unroll
                for (int t = 0; t < T; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[slot][s][t]), q, acc[t], 0, 0, 0);
            }
        };
#pragma unroll
        for (int u = 0; u < kSteps; u++)
            if (u < n) load(u, u);
        int base = 0;
        for (; base + kSteps < n - 1; base += kSteps)  // whole pairs of steps: no step of W is asked for twice
#pragma unroll
            for (int u = 0; u < kSteps; u++) {
                multiply(u);
                load(base + kSteps + u, u);
            }
        multiply(0);
        if (base + 2 < n) load(base + 2, 0);
        if (base + 1 < n) multiply(1);
        if (base + 2 < n) multiply(0);
    };
    int from = k0;
    if (KIND == Out::Scaled && out.mid) {  // what of this wavefront's piece lies below split has a factor of its own
        const int to = out.split < k1 ? (int)out.split : k1;
        sum_of(k0, to);
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int n = n0 + t * 16 + 4 * g + i;
                acc[t][i] *= out.mid[n < N ? n : N - 1];
            }
        if (to > from) from = to;
    }
    sum_of(from, k1);
    // a lane holds column r16 of rows 4 g .. 4 g + 3
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[wave][t * 16 + 4 * g + i][r16] = acc[t][i];
    __syncthreads();
    for (int o = tid; o < T * 128; o += 64 * kWaves) {
        const int row = o >> 3, col = o & 7, n = n0 + row;
        if (col >= M || n >= N) continue;
        auto sum = [&](int r) {
            float v = 0.f;
#pragma unroll
            for (int i = 0; i < kWaves; i++) v += red[i][r][col] + red[i][r][col + 8];
            return v;
        };
        if (KIND != Out::Pairs || n < out.pair_from) store_column<KIND>(out, col, n, sum(row));
        else if ((row & 1) == 0) store_pair(out, col, n, sum(row), sum(row + 1));
    }
}

// Eight rows of W a workgroup, for matrices whose sixteens are fewer than the compute units: what a unit draws from memory is
// bounded (13 to 16 GB/s measured in the kernels that read weights once, whatever is under way), so every one of them has to.
// The operand's other eight rows are the same rows of W 32 of K further on: a lane's sixteen bytes of eight rows are whole lines of 128.
// They are multiplied by x of either step, and of each product the half is kept whose step it is; the matrix cores have the time.
// 4 x 2048 x 8192: 19.3 us in sixteens on 128 units, 15.5 in eights (9.8 since x is converted once a wavefront, XStep; 33.5 MB, 3.4 TB/s).
template <int kWaves, int PASSES, Out KIND>
__global__ __launch_bounds__(64 * kWaves) void gemv_bf16_rows_eight_kernel(const uint16_t* __restrict__ W, int64_t ldw, const float* __restrict__ x, int64_t ldx,
                                                                           int M, int N, int K, ProductOut out) {
    __shared__ float red[kWaves][16][17];
    __shared__ __align__(16) uint16_t operands[kWaves][16 * XStep<PASSES>::kRow];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 8, row8 = r16 & 7, step = r16 >> 3;
    uint16_t* stage = operands[wave];
    const int pairs = K / 64, per = (pairs + kWaves - 1) / kWaves;
    const int k0 = wave * per * 64, k1 = k0 + per * 64 < K ? k0 + per * 64 : K;
    const uint16_t* wp = W + (int64_t)(n0 + row8 < N ? n0 + row8 : N - 1) * ldw + step * 32 + g * 8;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    // kSteps steps of 64 are under way, W and x; each one's registers are refilled as it is multiplied
    constexpr int kSteps = PASSES == 1 ? 8 : 5;
    auto sum_of = [&](int from, int to) {
        const int n = (to - from) / 64;
        if (n <= 0) return;
        u32x4 w[kSteps];
        XStep<PASSES> xs[kSteps];
        auto load = [&](int i, int slot) {
            const int k = from + 64 * (i < n ? i : n - 1);
            w[slot] = *(const u32x4*)(wp + k);
            xs[slot].load(x, ldx, M, k, lane);
        };
        auto multiply = [&](int slot) {
            xs[slot].put(stage, lane);
#pragma unroll
            for (int s = 0; s < 2; s++)
                acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[slot]), XStep<PASSES>::operand(stage, s, lane), acc[s], 0, 0, 0);
        };
#pragma unroll
        for (int u = 0; u < kSteps; u++) load(u, u);
        int base = 0;
        for (; base + kSteps < n; base += kSteps)
#pragma unroll
            for (int u = 0; u < kSteps; u++) {
                multiply(u);
                load(base + kSteps + u, u);
            }
#pragma unroll
        for (int u = 0; u < kSteps; u++)
            if (base + u < n) multiply(u);
    };
    int from = k0;
    if (KIND == Out::Scaled && out.mid) {  // what of this wavefront's piece lies below split has a factor of its own
        const int to = out.split < k1 ? (int)out.split : k1;
        sum_of(k0, to);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = n0 + ((4 * g + i) & 7);
            const float f = out.mid[n < N ? n : N - 1];
            acc[0][i] *= f;
            acc[1][i] *= f;
        }
        if (to > from) from = to;
    }
    sum_of(from, k1);
    // a lane holds column r16 of rows 4 g .. 4 g + 3; rows 8 and up are the second step's
#pragma unroll
    for (int i = 0; i < 4; i++) red[wave][4 * g + i][r16] = g < 2 ? acc[0][i] : acc[1][i];
    __syncthreads();
    if (tid < 64) {
        const int row = tid >> 3, col = tid & 7, n = n0 + row;
        if (col >= M || n >= N) return;
        auto sum = [&](int r) {
            float v = 0.f;
#pragma unroll
            for (int i = 0; i < kWaves; i++) v += (red[i][r][col] + red[i][r][col + 8]) + (red[i][r + 8][col] + red[i][r + 8][col + 8]);
            return v;
        };
        if (KIND != Out::Pairs || n < out.pair_from) store_column<KIND>(out, col, n, sum(row));
        else if ((row & 1) == 0) store_pair(out, col, n, sum(row), sum(row + 1));
    }
}

}  // namespace

hipError_t gemv_bf16_rows(const uint16_t* W, int64_t ldw, const float* x, int64_t ldx, int64_t M, int64_t N, int64_t K, const ProductOut& out, hipStream_t st) {
    if (M == 0 || N == 0) return hipSuccess;
    if (M > kGemvRows || ldw % 8 || ldx % 4) return hipErrorInvalidValue;
    const int k = (int)((K + 63) / 64 * 64);
    auto launch = [&](auto kernel, int rows, int waves) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((N + rows - 1) / rows)), dim3(64 * waves), 0, st, W, ldw, x, ldx, (int)M, (int)N, k, out);
    };
    auto by_kind = [&](auto t, auto waves, auto passes) {
        constexpr int T = decltype(t)::value, kWaves = decltype(waves)::value, P = decltype(passes)::value;
        const Out kind = out_kind(out, N);
        if (kind == Out::Plain) launch(gemv_bf16_rows_kernel<T, kWaves, P, Out::Plain>, 16 * T, kWaves);
        else if (kind == Out::Pairs) launch(gemv_bf16_rows_kernel<T, kWaves, P, Out::Pairs>, 16 * T, kWaves);
        else launch(gemv_bf16_rows_kernel<T, kWaves, P, Out::Scaled>, 16 * T, kWaves);
    };
    auto eight_by_kind = [&](auto waves, auto passes) {
        constexpr int kWaves = decltype(waves)::value, P = decltype(passes)::value;
        const Out kind = out_kind(out, N);
        if (kind == Out::Plain) launch(gemv_bf16_rows_eight_kernel<kWaves, P, Out::Plain>, 8, kWaves);
        else if (kind == Out::Pairs) launch(gemv_bf16_rows_eight_kernel<kWaves, P, Out::Pairs>, 8, kWaves);
        else launch(gemv_bf16_rows_eight_kernel<kWaves, P, Out::Scaled>, 8, kWaves);
    };
    using std::integral_constant;
    // sixteens of up to 2048 rows are at most 128 workgroups (4 x 2048 x 2048: 6.9 us in sixteens, 6.0 in eights, 5.0 now)
    // thirty-twos of which a few are left for a last round of the compute units (4 x 8224 x 2048: 257; 13.2 us, in sixteens 11.5)
    const int64_t thirties = (N + 31) / 32, over = thirties % 256;
    const bool tail = over > 0 && over <= 64 && thirties > 256;
    auto by_size = [&](auto passes) {
        if (N <= 2048 && k >= 8192) eight_by_kind(integral_constant<int, 16>{}, passes);
        else if (N <= 2048) eight_by_kind(integral_constant<int, 8>{}, passes);
        else if (N >= 8192 && !tail) by_kind(integral_constant<int, 2>{}, integral_constant<int, 8>{}, passes);
        else if (k >= 8192) by_kind(integral_constant<int, 1>{}, integral_constant<int, 16>{}, passes);
        else by_kind(integral_constant<int, 1>{}, integral_constant<int, 8>{}, passes);
    };
    if (M <= 4) by_size(integral_constant<int, 1>{});
    else by_size(integral_constant<int, 2>{});
    return hipGetLastError();
}

}  // namespace mimir
