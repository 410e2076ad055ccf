// The Q4_0 product of many rows of float32 x, from some tens of rows on, on the binary16 matrix cores. x enters as a pair of
// binary16 numbers an element, x 2^-e = h0 + h1 (to 2^-23 of the element; e the row's exponent), W as the integers n - 8, whose scales stay
// out of the matrix cores: v_mfma_f32_32x32x16_f16 sums a block's products of h1 and of h0 (exact, added in float32) into
// one c, and acc = fma(d, c, acc) is left to the vector unit, one instruction per output and block; 2^e follows at the end.
//
// What bounds it: four MFMAs of 32 cycles and sixteen FMAs of 4 per 32 x 32 outputs and block of 32, which hardly overlap
// on a SIMD (128 + 64 cycles; one wide tile alone takes 1.3 us a block, those cycles at the full clock; with every unit at work
// the clock falls and it was 1.75 us. Counters, with the barrier between blocks: 3097 cycles a block, 2048 of MFMA and 1426 of all vector instructions, 1024 of them FMAs). The form with the int8 form's bits (x as two 12-bit integer
// digits with a float32 scale a block: two sums, an MFMA for dw dx and two FMAs an output: 128 + 32 + 128 cycles) is taken where mi355x_qgemv_noalloc
// multiplies in that form. Whole calls, conversion and the pass over W included, fifty of a shape back to back (among other shapes, as bench.py has them, a
// tenth more: 498 us for the first), digits and halves:
//   2048 x 14336 x 4096   647 -> 461 us (521 TFLOP/s)      4096 x 28672 x 4096   2430 -> 1667 us (577 TFLOP/s)
//   4096 x 4096 x 14336  1286 -> 910 us                    512 x 4096 x 14336    506 (int8 268) -> 155 us
//   2048 x 4096 x 4096    184 -> 149 us                    512 x 14336 x 4096    183 -> 149 us
// The error against 64 bits is no larger: 2.11e-7 of the result at K = 4096 (digits 2.31e-7), 3.84e-7 at 14336 (3.95e-7).
//
// Two launches, three where K is cut into shares. fx16_panel_kernel writes W's integers as binary16 and its scales as float32,
// in the order in which a stage of LDS holds them; the conversion of x (fx16_halves_kernel, with a norm before it
// where the decoder has one) does the same for x. So every load of the product is a whole KB from contiguous memory straight
// into LDS (global_load_lds_dwordx4). A workgroup of eight wavefronts owns 256 x 256 outputs (a wavefront 64 x 128, three
// stages of one block) where tiles are many, 128 x 256 (64 x 64, four stages) where they are few: 8 KB of fragments
// from LDS per 16 MFMAs against 12. One barrier a block; a sub-tile's MFMAs are issued with the FMAs of the sub-tile before.
// The barrier is in a block's middle and fragments are read up to a block ahead. With it between blocks, both wavefronts of a SIMD waited
// behind it for all eight's fragments, 96 or 128 KB at 256 bytes a cycle: 512 x 14336 x 4096 159 us a call, now 153; 2048 x 14336 x 4096 458, now 451; 4096 x 14336 x
// 4096 874, now 843. (FMAs set between the MFMAs one by one, which alone in a loop take a tenth less: 158, 465, 864.)
// Where even those leave units idle, K is cut into shares whose sums a third launch adds.
//
// Several matrices by the same x (q, k and v; gate and up, SwiGLU included) are one product: Parts.
//
// Reference semantics: the float32 product with the dequantized weights (io/mim/dtype.go:118-123).
#include "device_util.h"
#include "kernels.h"
#include "q4_act.h"
#include "q4_halves.h"

namespace mimir {

namespace {

constexpr int kMinRows = 256;     // fewer rows of one matrix stay with the int8 form,
constexpr int kMinPartRows = 9;    // of several together with the other kernels

// Thread t takes elements 4t..4t+3 of row blockIdx.y; a block's eight threads are consecutive lanes.
__global__ __launch_bounds__(256) void fx16_digits_kernel(const float* __restrict__ x, int64_t x_row_stride, int K, uint16_t* __restrict__ X16,
                                                          float* __restrict__ XS, int2* __restrict__ RS) {
    const int nb = K >> 5;
    if (blockIdx.x == 0 && threadIdx.x == 0) RS[blockIdx.y] = make_int2(0, kDigitPairs);
    const float* xr = x + (int64_t)blockIdx.y * x_row_stride;
    uint16_t* strip = X16 + strip_at((int)blockIdx.y, nb);
    const bool lanes = in_lanes(gridDim.y);
    float* xscale = XS + (int64_t)blockIdx.y * nb;
    const int nq = K >> 2;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nq; t += gridDim.x * blockDim.x) {
        f32x4 v;
        __builtin_memcpy(&v, xr + 4 * (int64_t)t, 16);
        float amax = 0.f;
        bool finite = true;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float a = __builtin_fabsf(v[k]);
            finite = finite && a < __builtin_inff();  // false for NaN too
            amax = fmaxf(amax, a);
        }
        amax = group8_max(amax);
        float bad = group8_max(finite ? 0.f : 1.f);
        float scale, inv;
        if (bad != 0.f) {  // a NaN or an infinity in the block: its products are NaN
            scale = __builtin_nanf("");
            inv = 0.f;
            v = f32x4{0.f, 0.f, 0.f, 0.f};
        } else if (amax < 0x1p-100f) {
            scale = 0.f;
            inv = 0.f;
        } else {
            scale = amax / (float)kFixMax;
            inv = (float)kFixMax / amax;
        }
        _Float16 lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            int a = (int)__builtin_rintf(v[k] * inv);
            a = a > kFixMax ? kFixMax : a < -kFixMax ? -kFixMax : a;
            const int d0 = ((a + 2048) & 4095) - 2048;  // balanced: -2048..2047
            const int d1 = (a - d0) >> 12;              // -2048..2048
            lo[k] = (_Float16)(float)(t & 8 ? -d0 : d0);  // odd blocks with their sign turned (tile_body)
            hi[k] = (_Float16)(float)(t & 8 ? -d1 : d1);
        }
        uint16_t* at = strip + (int64_t)(t >> 3) * kGranuleX;
        const int piece = (t & 7) >> 1, within = 4 * (t & 1);
        __builtin_memcpy(at + piece_at((int)blockIdx.y, piece, lanes) + within, lo, 8);
        __builtin_memcpy(at + piece_at((int)blockIdx.y, 4 + piece, lanes) + within, hi, 8);
        if ((t & 7) == 0) xscale[t >> 3] = scale;
    }
}

// In the order of lanes a line of 128 bytes has a piece each of eight rows: eight rows a die (every eighth workgroup), whose cache puts the line together, the eights
// on the dies in turn. Whole calls, against a row a workgroup as rows come (up to 128 of them; more, a strip a die): 128 x 9536 x 4544 55.0 -> 53.7 us, 108 x 4480 x 13056 63.6 -> 62.4,
// 77 x 5120 x 5120 30.0 -> 29.3, 200 x 3136 x 11968 70.0 -> 69.5.
constexpr int kDies = 8, kLineRows = 8;
__device__ inline int row_of_die(int block) { return kLineRows * ((block & (kDies - 1)) + kDies * (block / (kDies * kLineRows))) + block / kDies % kLineRows; }

// A workgroup converts a row of x into halves: x 2^-e = h0 + h1, h0 the binary16 next to it and h1 the binary16 next to
// what that leaves. An element is held to 2^-23 of itself (of float32's 24 bits the last may go: 2^14 + 8 - 2^-9 leaves 8 - 2^-9, which h1 rounds by
// 2^-9). e makes the row's largest element lie in [2^14, 2^15), where h1's smallest step, 2^-24, is below that bound down to
// 2^-2, and holds what is smaller to 2^-25: to 2^-24 of its block's largest as long as that is no less than 2^-15 of the row's. The fixed point
// holds every element to 2^-23.9 of its block's largest, that is most of them to less: its error over normal x is twice the pairs'. A row that has a
// smaller block (zeros aside) takes an exponent a block instead.
// With NORM the row is normalized first (rmsnorm_kernel's operations, one by one): x over its root mean square, times w.
// Memory bounds it: 8 bytes an element. ITEMS: eights of elements a thread holds between the row's maximum and its halves, so that x
// is read once (4096 rows of 14336: 105 us, 156 reading it twice and storing eight bytes a thread); 0: rows of more than 16384, read twice.
template <int ITEMS, bool NORM, bool LANES>
__global__ __launch_bounds__(256) void fx16_halves_kernel(const float* __restrict__ x, const float* __restrict__ w, int64_t x_row_stride, int K,
                                                          uint16_t* __restrict__ X16, float* __restrict__ XS, int2* __restrict__ RS, int M, float inv_k, float eps) {
    constexpr int kHeld = ITEMS ? ITEMS : 1;
    const int nb = K >> 5, n8 = K >> 3, tid = threadIdx.x;
    const int m = LANES ? row_of_die((int)blockIdx.x) : (int)blockIdx.x;
    if (LANES && m >= M) return;
    const float* xr = x + (int64_t)m * x_row_stride;
    uint16_t* strip = X16 + strip_at(m, nb);
    float* xscale = XS + (int64_t)m * nb;
    __shared__ uint32_t part[2][4];
    float scale = 1.f;
    if (NORM) {
        const float ss = wave_sum(strided_sum_squares(xr, K, tid));
        if ((tid & 63) == 0) part[0][tid >> 6] = __builtin_bit_cast(uint32_t, ss);
        __syncthreads();
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) p[i] = __builtin_bit_cast(float, part[0][i]);
        const float total = (p[0] + p[1]) + (p[2] + p[3]);
        const float ms = total * inv_k;
        scale = 1.0f / __builtin_sqrtf(ms + eps);
        __syncthreads();
    }
    auto load = [&](int t, float v[8]) {
        __builtin_memcpy(v, xr + 8 * (int64_t)t, 32);
        if (NORM) {
            float g[8];
            __builtin_memcpy(g, w + 8 * (int64_t)t, 32);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float n = v[k] * scale;
                v[k] = n * g[k];
            }
        }
    };
    // the largest magnitude of the block that this thread and three neighbours hold, as the integer of its bits: the order is the
    // same, a NaN or an infinity is the largest
    auto block_top = [&](const float v[8]) {
        uint32_t top = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t a = __builtin_bit_cast(uint32_t, v[k]) & 0x7fffffffu;
            top = a > top ? a : top;
        }
        uint32_t other = __builtin_bit_cast(uint32_t, dpp_f32<0xb1>(__builtin_bit_cast(float, top)));
        top = other > top ? other : top;
        other = __builtin_bit_cast(uint32_t, dpp_f32<0x4e>(__builtin_bit_cast(float, top)));
        return other > top ? other : top;
    };
    uint32_t most = 0, least = 0x7f800000u;
    float v[kHeld][8];
    auto see = [&](int t, float u[8]) {
        load(t, u);
        const uint32_t top = block_top(u);
        most = top > most ? top : most;
        if (top != 0 && top < least) least = top;
    };
    if (ITEMS) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (tid + 256 * i < n8) see(tid + 256 * i, v[i]);
    } else {
        for (int t = tid; t < n8; t += 256) see(t, v[0]);
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t a = (uint32_t)__shfl_xor((int)most, d), b = (uint32_t)__shfl_xor((int)least, d);
        most = a > most ? a : most;
        least = b < least ? b : least;
    }
    if ((tid & 63) == 0) {
        part[0][tid >> 6] = most;
        part[1][tid >> 6] = least;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        most = part[0][i] > most ? part[0][i] : most;
        least = part[1][i] < least ? part[1][i] : least;
    }
    const bool finite = most < 0x7f800000u;
    const float amax = __builtin_bit_cast(float, most), amin = __builtin_bit_cast(float, least);
    auto exponent = [](float a) { return a > 0.f ? __builtin_amdgcn_frexp_expf(a) - 15 : 0; };  // a 2^-e in [2^14, 2^15)
    const int e_row = finite ? exponent(amax) : 0;
    const int form = finite && amin < amax * 0x1p-15f ? kBlockHalves : kHalves;
    if (tid == 0) RS[m] = make_int2(finite ? e_row : INT32_MAX, form);
    auto convert = [&](int t, const float u[8]) {
        const int e = form == kBlockHalves ? exponent(__builtin_bit_cast(float, block_top(u))) : e_row;
        const bool odd = t & 4;  // odd blocks with their sign turned (tile_body)
        f16x8 h0, h1;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float a = finite ? __builtin_ldexpf(odd ? -u[k] : u[k], -e) : 0.f;
            h0[k] = (_Float16)a;
            h1[k] = (_Float16)(a - (float)h0[k]);
        }
        uint16_t* at = strip + (int64_t)(t >> 2) * kGranuleX;
        *(f16x8*)(at + piece_at(m, t & 3, LANES)) = h0;
        *(f16x8*)(at + piece_at(m, 4 + (t & 3), LANES)) = h1;
        if ((t & 3) == 0) xscale[t >> 2] = finite ? __builtin_ldexpf(1.f, e) : __builtin_nanf("");
    };
    if (ITEMS) {
#pragma unroll
        for (int i = 0; i < kHeld; i++)
            if (tid + 256 * i < n8) convert(tid + 256 * i, v[i]);
    } else {
        for (int t = tid; t < n8; t += 256) {
            load(t, v[0]);
            convert(t, v[0]);
        }
    }
}

// W's integers n - 8 as binary16 and its scales as float32, in granules; an odd block's scale is negative (tile_body says why). A
// wavefront takes a strip's block: lane r + 32 q the eight bytes q of row r, whose low nibbles are piece q of the block's
// first half and whose high nibbles of its second.
__global__ __launch_bounds__(256) void fx16_panel_kernel(Parts parts, uint16_t* __restrict__ P, float* __restrict__ SW, int nb) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, q = lane >> 5;
    const int groups = (nb + 31) >> 5, strip = (int)blockIdx.x / groups, first = ((int)blockIdx.x - strip * groups) * 32 + 8 * wave;  // of blocks
    const int part = parts.swiglu ? strip & 1 : strip >= parts.begin[2] ? 2 : strip >= parts.begin[1] ? 1 : 0;
    const int n = (parts.swiglu ? strip >> 1 : strip - parts.begin[part]) * 32 + r, N = parts.N[part];
    const uint8_t* row = parts.W[part] + (int64_t)(n < N ? n : N - 1) * nb * 18;  // past the matrix: its last row again
    const bool aligned = ((uintptr_t)parts.W[part] & 3) == 0;
    PairBytes pair[4];  // nb is even
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (first + 2 * i < nb) pair[i] = load_pair(row + (first + 2 * i) * 18, q, aligned);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int b = first + i;
        if (b >= nb) return;
        uint16_t* out = P + ((int64_t)strip * nb + b) * kGranuleP + lane * 8;
#pragma unroll
        for (int half = 0; half < 2; half++) *(f16x8*)(out + 512 * half) = nibbles_to_f16(pair[i / 2].lo[i & 1], pair[i / 2].hi[i & 1], half);
        if (q == 0) SW[((int64_t)strip * scale_blocks(nb) + b) * kGranuleS + r] = f16_bits_to_f32((uint16_t)(pair[i / 2].scale[i & 1] ^ ((b & 1) << 15)));
    }
}

// A workgroup's tile of y: WM x (8 / WM) wavefronts of (32 MT) x (32 NT) each, over STAGES stages of one block.
template <int WM, int MT_, int NT_, int STAGES_>
struct Shape {
    static constexpr int WN = 8 / WM, MT = MT_, NT = NT_, STAGES = STAGES_;
    static constexpr int BM = WM * 32 * MT, BN = WN * 32 * NT;
    static constexpr int kChunksX = BM / 32 * 4, kChunksP = BN / 32 * 2;  // KB of a stage
    static constexpr int kX = kChunksX / 8, kLoads = kX + kChunksP / 8;   // a wavefront issues a stage: kX of x, then P's
    static constexpr int stage = (kChunksX + kChunksP) * 1024;
    static constexpr int sw = STAGES * stage;                // float [2 groups][BN / 32][kGroup][32]
    static constexpr int sw_group = BN / 32 * 1024;
    static constexpr int sx = sw + 2 * sw_group;             // float [2][BM]: x's scales of two blocks, where they differ by block
    static constexpr int total = sx + 2 * BM * 4;
    static_assert(kChunksX % 8 == 0 && kChunksP % 8 == 0 && kLoads <= MT * NT && BN <= 256 && BM <= 512, "as many loads a wavefront, one with a sub-tile");
};
using Low = Shape<2, 2, 2, 4>;   // 128 x 256
using Wide = Shape<4, 2, 4, 3>;  // 256 x 256
constexpr int kLdsBytes = Low::total > Wide::total - 2 * 256 * 4 ? Low::total : Wide::total - 2 * 256 * 4;  // Wide has no scales of x

// One tile: rows m0 .. m0 + BM of x by columns n0 .. n0 + BN, blocks b0 .. b0 + count of K (b0 a multiple of a group), of rows of
// x that are all of one form, or halves of either kind (kBlockHalves).
//
// An MFMA rounds its float32 sums downwards more often than upwards, and over the hundreds of blocks of a row that bias
// adds up (4096 x 14336 by normal x: 3.97e-7 of the result, where exact sums of blocks give 3.945e-7). So odd blocks are multiplied with
// their sign turned, x's halves and W's scales both: the bias cancels, 3.84e-7.
template <class S, int FORM>
__device__ __forceinline__ void tile_body(const Operands& o, int m0, int n0, int b0, int count, float* sums, char* lds) {
    constexpr int MT = S::MT, NT = S::NT;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::WN, wn = wave % S::WN;
    const int M = o.M, nb = o.nb;

    // This wavefront's loads: KB kX wave + j of x's granules, then as many of P's. Strips past the matrix re-read its last
    // strip (their results are not stored).
    const char* from[S::kLoads];
    uint32_t into[S::kLoads];
#pragma unroll
    for (int j = 0; j < S::kLoads; j++) {
        const bool of_x = j < S::kX;
        const int c = of_x ? S::kX * wave + j : (S::kLoads - S::kX) * wave + j - S::kX;
        const int strip = of_x ? m0 / 32 + c / 4 : n0 / 32 + c / 2, last = of_x ? (M - 1) / 32 : o.parts.strips - 1;
        const int64_t at = (int64_t)(strip < last ? strip : last) * nb + b0;
        from[j] = of_x ? (const char*)(o.X16 + at * kGranuleX) + (c & 3) * 1024 : (const char*)(o.P + at * kGranuleP) + (c & 1) * 1024;
        into[j] = (of_x ? c : c + S::kChunksX) * 1024;
    }
    const uint32_t lane16 = lane * 16;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    // W's scales: wavefront w brings strip w of the tile's, a group of blocks at a time
    const bool has_sw = wave < S::BN / 32;
    const char* sw_from;
    {
        const int strip = n0 / 32 + (has_sw ? wave : 0), last = o.parts.strips - 1;
        sw_from = (const char*)(o.SW + ((int64_t)(strip < last ? strip : last) * scale_blocks(nb) + b0) * kGranuleS);
    }
    const uint32_t sw_into = lds0 + S::sw + wave * 1024;
    // x's, where they differ by block: one a thread below BM
    const float* xscale = o.XS + (int64_t)(m0 + (tid & (S::BM - 1)) < M ? m0 + (tid & (S::BM - 1)) : M - 1) * nb + b0;

    const int r32 = lane & 31, hi = lane >> 5;
    int piece_off[4];  // of pieces 2 p + hi: half p % 2 of part p / 2
#pragma unroll
    for (int p = 0; p < 4; p++) piece_off[p] = wm * MT * 4096 + piece_at(r32, 2 * p + hi, in_lanes(M)) * 2;
    const int b_off = S::kChunksX * 1024 + wn * NT * 2048 + lane * 16;

    f32x16 acc[MT][NT], zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = zero;

    auto load_stage = [&](int j, uint32_t slot, int step) {
        load_to_lds(from[j], lane16, lds0 + slot + into[j]);
        from[j] += (j < S::kX ? kGranuleX * 2 : kGranuleP * 2) * step;
    };
    if (has_sw) load_to_lds(sw_from, lane16, sw_into);
    auto next_scales = [&](int i) {  // in block i: the next group of W's scales, over the one before this
        if (has_sw && (i & (kGroup - 1)) == 0 && i + kGroup < count) {
            sw_from += 1024;
            load_to_lds(sw_from, lane16, sw_into + ((i / kGroup + 1) & 1) * S::sw_group);
        }
    };
    f32x16 c[2];  // kHalves: the sums of a sub-tile, finished with the next one's products
    c[1] = zero;
    float dlast = 0.f;
    // No branches around the loads: past the end the last block is requested again, into a stage that is not read any more.
    if constexpr (FORM == kHalves) {
        // Fragments are in registers before they are wanted, x's a sub-tile row and W's a block ahead, so that no product waits behind the barrier while
        // every wavefront reads at once. The barrier is in a block's middle: by then its stage has been read, and is filled anew.
        static_assert(MT == 2, "two rows of sub-tiles a block");
        f16x8 a[MT][2][2], b[NT][2];  // a[mt][part][half], b[nt][half]
        auto read_a = [&](int mt, const char* st) {
#pragma unroll
            for (int p = 0; p < 4; p++) a[mt][p >> 1][p & 1] = *(const f16x8*)(st + mt * 4096 + piece_off[p]);
        };
        auto read_b = [&](int nt, const char* st) {
#pragma unroll
            for (int h = 0; h < 2; h++) b[nt][h] = *(const f16x8*)(st + b_off + nt * 2048 + h * 1024);
        };
        for (int i = 0; i < S::STAGES; i++)
#pragma unroll
            for (int j = 0; j < S::kLoads; j++) load_stage(j, i * S::stage, i + 1 < count ? 1 : 0);
        wait_loads<S::kLoads*(S::STAGES - 1)>();
        lds_barrier();
        read_a(0, lds);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) read_b(nt, lds);
        float dw[NT];
        // A sub-tile's products are issued with the FMAs of the one before it, so that the vector unit works while the
        // matrix cores do. What h0 leaves first: the smaller terms.
        auto sub_tile = [&](int sub) {
            const int mt = sub / NT, nt = sub % NT, was = (sub + MT * NT - 1) % (MT * NT);
#pragma unroll
            for (int p = 0; p < 4; p++)
                c[sub & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][1 - (p >> 1)][p & 1], b[nt][p & 1], p == 0 ? zero : c[sub & 1], 0, 0, 0);
            const float d = sub == 0 ? dlast : dw[was % NT];
#pragma unroll
            for (int e = 0; e < 16; e++) acc[was / NT][was % NT][e] = fmaf(d, c[(sub + 1) & 1][e], acc[was / NT][was % NT][e]);
        };
        uint32_t use = 0;  // the stage that is multiplied
        for (int i = 0; i < count; i++) {
            const uint32_t next = use + S::stage == S::sw ? 0 : use + S::stage;
            const int step = i + S::STAGES + 1 < count ? 1 : 0;
            next_scales(i);
            read_a(1, lds + use);
            const char* sw = lds + S::sw + (i / kGroup & 1) * S::sw_group + wn * NT * 1024 + (i & (kGroup - 1)) * 128;
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                sub_tile(nt);
                if (nt == 0)
#pragma unroll
                    for (int t = 0; t < NT; t++) dw[t] = *(const float*)(sw + t * 1024 + r32 * 4);
                __builtin_amdgcn_sched_barrier(0);
            }
            wait_loads<S::kLoads*(S::STAGES - 2)>();  // this wavefront's part of block i + 1 has landed, and W's scales
            lds_barrier();                             // everyone's has, and everyone has read block i for the last time
            read_a(0, lds + next);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
#pragma unroll
                for (int j = nt * S::kLoads / NT; j < (nt + 1) * S::kLoads / NT; j++) load_stage(j, use, step);
                sub_tile(NT + nt);
                read_b(nt, lds + next);
                __builtin_amdgcn_sched_barrier(0);
            }
            dlast = dw[NT - 1];
            use = next;
        }
    } else {
        uint32_t fill = 0;  // the stage that is loaded next
        for (int i = 0; i < S::STAGES - 1; i++) {
#pragma unroll
            for (int j = 0; j < S::kLoads; j++) load_stage(j, fill, i + 1 < count ? 1 : 0);
            fill += S::stage;
        }
        if (tid < S::BM) ((float*)(lds + S::sx))[tid] = *xscale;
        uint32_t use = 0;  // the stage that is multiplied
        for (int i = 0; i < count; i++) {
            wait_loads<S::kLoads*(S::STAGES - 2)>();  // this wavefront's part of block i has landed, and W's scales
            lds_barrier();                             // everyone's has, and everyone has read the block before for the last time
            const int step = i + S::STAGES < count ? 1 : 0;
            const char* st = lds + use;
            next_scales(i);
            xscale += i + 1 < count ? 1 : 0;
            const float next_dx = *xscale;
            f16x8 a[MT][2][2], b[2][2];  // a[mt][part][half], b[nt][half]
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
#pragma unroll
                for (int h = 0; h < 2; h++) b[nt][h] = *(const f16x8*)(st + b_off + nt * 2048 + h * 1024);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int p = 0; p < 4; p++) a[mt][p >> 1][p & 1] = *(const f16x8*)(st + mt * 4096 + piece_off[p]);
            const char* sw = lds + S::sw + (i / kGroup & 1) * S::sw_group + wn * NT * 1024 + (i & (kGroup - 1)) * 128;
#pragma unroll
            for (int j = 0; j < S::kLoads; j++) load_stage(j, fill, step);
            // The products of the two scales, dw dx, are an outer product: v_mfma_f32_32x32x1_2b_f32 makes two (one exact product
            // an output, nothing added: the rounding of a multiplication), its first 32 lanes giving x's rows and W's rows
            // of the first, the other 32 of the second; here the 32 rows of x of sub-tiles (mt, 0) and (mt, 1), and the 64
            // rows of W of both (a lane each).
            const float dw = *(const float*)(sw + hi * 1024 + r32 * 4);
            float dx[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) dx[mt] = ((const float*)(lds + S::sx))[(i & 1) * S::BM + (wm * MT + mt) * 32 + r32];
            f32x32 w, none;
#pragma unroll
            for (int e = 0; e < 32; e++) none[e] = 0.f;
#pragma unroll
            for (int sub = 0; sub < MT * NT; sub++) {  // NT is 2 here: both of b are there
                const int mt = sub / NT, nt = sub % NT;
                f32x16 c0, c1;
                if (FORM == kDigitPairs) {
                    c0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][0][0], b[nt][0], zero, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][1][0], b[nt][0], zero, 0, 0, 0);
                    c0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][0][1], b[nt][1], c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][1][1], b[nt][1], c1, 0, 0, 0);
                } else {
                    c0 = zero;
#pragma unroll
                    for (int p = 0; p < 4; p++) c0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt][1 - (p >> 1)][p & 1], b[nt][p & 1], c0, 0, 0, 0);
                }
                if (nt == 0) w = __builtin_amdgcn_mfma_f32_32x32x1f32(dx[mt], dw, none, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float sum = FORM == kDigitPairs ? fmaf(c1[e], 4096.f, c0[e]) : c0[e];  // digits: the exact integer, rounded once
                    acc[mt][nt][e] = fmaf(w[16 * nt + e], sum, acc[mt][nt][e]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // the next block's scales, at the end: by now their loads have landed with everything requested before them
            __builtin_amdgcn_sched_barrier(0);
            if (tid < S::BM) ((float*)(lds + S::sx))[((i + 1) & 1) * S::BM + tid] = next_dx;
            use = use + S::stage == S::sw ? 0 : use + S::stage;
            fill = fill + S::stage == S::sw ? 0 : fill + S::stage;
        }
    }
    if (FORM == kHalves) {
#pragma unroll
        for (int e = 0; e < 16; e++) acc[MT - 1][NT - 1][e] = fmaf(dlast, c[1][e], acc[MT - 1][NT - 1][e]);
    }
    wait_loads<0>();  // nothing of this tile's is on its way into LDS any more

    // An MFMA leaves a lane one column of y and four consecutive rows per group of four registers; a 4 x 4
    // transposition within each quad of lanes turns that into one row and four consecutive columns a lane.
    const float* resid = sums ? nullptr : o.resid;
    const bool gated = o.parts.swiglu && !sums;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        // this strip's columns: where they go, and which they are there
        const int strip = n0 / 32 + wn * NT + nt;
        if (strip >= o.parts.strips) break;
        if (gated && (nt & 1)) continue;  // taken with the gate's
        int n0s;
        const int part = part_of(o.parts, strip, &n0s);
        float* y = sums ? sums : o.parts.y[part];
        const int N = sums ? o.parts.strips * 32 : o.parts.N[part], n = (sums ? strip * 32 : n0s) + (r32 & ~3);
        const bool wide_ok = (N & 3) == 0 && ((uintptr_t)y & 15) == 0 && (!resid || ((uintptr_t)resid & 15) == 0);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int m = m0 + (wm * MT + mt) * 32 + q * 8 + hi * 4 + (lane & 3);
                const int e_row = FORM == kHalves ? o.RS[m < M ? m : M - 1].x : 0;
                auto row_of = [&](int col, float v[4]) {
#pragma unroll
                    for (int k = 0; k < 4; k++) v[k] = acc[mt][col][4 * q + k];
                    quad_transpose(v, lane);
                    if (FORM == kHalves) under_exponent(v, e_row);
                };
                float v[4];
                row_of(nt, v);
                if (gated) {
                    float u[4];
                    row_of((nt + 1) % NT, u);
#pragma unroll
                    for (int k = 0; k < 4; k++) v[k] = silu_times(v[k], u[k]);
                }
                if (m < M && n < N) store_four(y, resid, m, N, n, v, wide_ok);
            }
    }
}

// Whether one of rows m0 .. m0 + rows has an exponent a block: then all are read by block.
__device__ __forceinline__ bool by_block(const Operands& o, int m0, int rows) {
    bool any = false;
    for (int r = threadIdx.x & 63; r < rows; r += 64) any |= o.RS[m0 + r < o.M ? m0 + r : o.M - 1].y == kBlockHalves;
    return __ballot(any) != 0;
}

// How the product is cut: the first wide_cols columns of 256 into wide tiles, the others into low ones, every tile's K into shares.
struct Cut {
    int wide_m, wide_cols, low_m, low_cols;  // tiles along M, columns of tiles
    int shares, share_blocks;                // the last share may be shorter
};

template <bool DIGITS>
__device__ __forceinline__ void product(const Operands& o, const Cut& cut, char* lds) {
    static_assert(Wide::BN == Low::BN && Wide::BM == 2 * Low::BM, "a wide tile is two low ones");
    const int wide_tiles = cut.wide_m * cut.wide_cols, wide_wgs = ((wide_tiles * cut.shares + 7) >> 3) << 3;
    const bool wide = (int)blockIdx.x < wide_wgs;
    const int tiles = wide ? wide_tiles : cut.low_m * cut.low_cols;
    const int t = tile_of((int)blockIdx.x - (wide ? 0 : wide_wgs), tiles * cut.shares);
    if (t >= tiles * cut.shares) return;  // the whole workgroup
    const int share = t / tiles, tile = t % tiles, tiles_m = wide ? cut.wide_m : cut.low_m;
    const int bm = wide ? Wide::BM : Low::BM, n0 = ((wide ? 0 : cut.wide_cols) + tile / tiles_m) * Low::BN;
    const int b0 = share * cut.share_blocks, count = o.nb - b0 < cut.share_blocks ? o.nb - b0 : cut.share_blocks;
    float* sums = o.sums ? o.sums + (int64_t)share * o.M * o.parts.strips * 32 : nullptr;
    int m0 = tile % tiles_m * bm;
    if (DIGITS) {
        tile_body<Low, kDigitPairs>(o, m0, n0, b0, count, sums, lds);
    } else if (!by_block(o, m0, bm)) {
        if (wide) tile_body<Wide, kHalves>(o, m0, n0, b0, count, sums, lds);
        else tile_body<Low, kHalves>(o, m0, n0, b0, count, sums, lds);
    } else {
        for (const int end = m0 + bm < o.M ? m0 + bm : o.M; m0 < end; m0 += Low::BM) {
            tile_body<Low, kBlockHalves>(o, m0, n0, b0, count, sums, lds);
            lds_barrier();  // the next one fills the stages anew
        }
    }
}

__global__ __launch_bounds__(512) void qgemm_q4_0_fx16_kernel(Operands o, Cut cut) {
    extern __shared__ __align__(1024) char lds[];
    product<false>(o, cut, lds);
}

__global__ __launch_bounds__(512) void qgemm_q4_0_fx16_digits_kernel(Operands o, Cut cut) {
    extern __shared__ __align__(1024) char lds[];
    product<true>(o, cut, lds);
}

// Four columns a thread.
__global__ __launch_bounds__(256) void fx16_sum_kernel(Operands o, int shares) {
    const int64_t ld = (int64_t)o.parts.strips * 32, quads = o.M * ld / 4, step = o.M * ld;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < quads; t += (int64_t)gridDim.x * 256) {
        const int64_t m = 4 * t / ld;
        const int at = (int)(4 * t - m * ld), strip = at >> 5;
        if (o.parts.swiglu && (strip & 1)) continue;
        auto total = [&](const float* from) {
            f32x4 v = *(const f32x4*)from;
            for (int i = 1; i < shares; i++) {
                const f32x4 w = *(const f32x4*)(from + i * step);
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = v[k] + w[k];
            }
            return v;
        };
        f32x4 v = total(o.sums + 4 * t);
        if (o.parts.swiglu) {
            const f32x4 u = total(o.sums + 4 * t + 32);
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = silu_times(v[k], u[k]);
        }
        int n;
        const int part = part_of(o.parts, strip, &n), N = o.parts.N[part];
        n += at & 31;
        const bool wide_ok = (N & 3) == 0 && ((uintptr_t)o.parts.y[part] & 15) == 0 && ((uintptr_t)o.resid & 15) == 0;
        const float out[4] = {v[0], v[1], v[2], v[3]};
        if (n < N) store_four(o.parts.y[part], o.resid, m, N, n, out, wide_ok);
    }
}

// measurement aid: 0 keeps every product on the int8 form, 2 takes the digits' form whatever the shape, 3 the halves'
std::atomic<int> g_fx16{1};

// Microseconds of a product, the pass over W and the shares' sums included, and its cut. A compute unit takes a tile at a
// time; the time of a tile's block grows with how many units are at work, as the clock falls: 0.72 + 0.32 of them for a
// tile of 128 x 256, 1.25 + 0.5 of them for one of 256 x 256 (measured at 32 to 1792 tiles of 4096 and 14336 of K). Shares of K are for
// products whose tiles leave units idle: their sums are written and read at about 4.5 TB/s, the panel at 4.4.
double plan(int64_t M, int64_t strips, int64_t K, int64_t min_share_blocks, size_t sums_bytes, Cut* cut) {
    const int64_t nb = K / 32, cols = (strips + 7) / 8;
    const int64_t tm = (M + Wide::BM - 1) / Wide::BM, tl = (M + Low::BM - 1) / Low::BM;
    const double panel_us = (double)strips * 32 * (double)K * (18.0 / 32.0 + 2.0) / 4.4e6;
    double best = 1e30;
    auto consider = [&](int64_t wide_cols, int64_t shares) {
        const int64_t blocks = (nb + shares * kGroup - 1) / (shares * kGroup) * kGroup, used = (nb + blocks - 1) / blocks;
        if (used != shares) return;
        const int64_t wide = tm * wide_cols * shares, low = tl * (cols - wide_cols) * shares;
        const size_t sums = (size_t)shares * (size_t)M * (size_t)strips * 128;
        if (shares > 1 && (blocks < min_share_blocks || sums > sums_bytes)) return;
        // whole rounds of wide tiles; what is left of the last one is filled with low ones
        double us = 0, idle = 256;
        if (wide) {
            const int64_t rounds = (wide + 255) / 256;
            us += (double)rounds * (double)blocks * (1.25 + 0.5 * (double)wide / (double)(rounds * 256));
            idle = (double)(rounds * 256 - wide);
        }
        if (low) {
            const int64_t beside = wide ? (int64_t)(2 * idle) : 0, left = low > beside ? low - beside : 0, rounds = (left + 255) / 256;
            if (rounds) us += (double)rounds * (double)blocks * (0.72 + 0.32 * (double)left / (double)(rounds * 256));
        }
        if (shares > 1) us += 3.0 + (double)sums * (1.0 + 1.0 / (double)shares) / 4.5e6;
        if (us + panel_us < best) {
            best = us + panel_us;
            *cut = Cut{(int)tm, (int)wide_cols, (int)tl, (int)(cols - wide_cols), (int)shares, (int)blocks};
        }
    };
    for (int64_t shares = 1; shares <= 16; shares++) {
        if (shares > 1 && tl * cols * shares > 1024) break;
        consider(0, shares);
        consider(cols, shares);
        if (shares == 1)
            for (int64_t rounds = 1; rounds * 256 < tm * cols; rounds++)  // whole rounds of wide tiles, then low ones
                if (rounds * 256 / tm > 0) consider(rounds * 256 / tm, 1);
    }
    return best;
}

bool fits(int64_t M, int64_t strips, int64_t K) {
    return M > 0 && strips > 0 && K > 0 && K % 64 == 0 && M < (1 << 30) && K <= (1 << 20) && strips < (1 << 22) && (M + 127) / 128 * ((strips + 7) / 8) < ((int64_t)1 << 24);
}

}  // namespace

void set_q4_0_fx16(int v) { g_fx16 = v; }

hipError_t sum_shares(const Operands& o, int shares, hipStream_t st) {
    const int64_t groups = ((int64_t)o.M * o.parts.strips * 8 + 255) / 256;
    hipLaunchKernelGGL(fx16_sum_kernel, dim3((unsigned)(groups < 16384 ? groups : 16384)), dim3(256), 0, st, o, shares);
    return hipGetLastError();
}

// Whether the product is the faster here than in the int8 form (qgemm_q4_0_fx_cost_us). mi355x_qgemv cuts K into shares of
// no less than 96 blocks: 512 x 4096 x 4096 stays with the int8 form there (88 us, in one pass here 114; 512 x 14336 x 4096 comes here: 151 us, 217
// in the int8 form). That line is one of results and not of time: up to there a product of float32 x has the int8 form's bits, which
// tests/test_gpu_qgemm_fx.py names; in shares of 16 blocks, as the decoder has it, 512 x 4096 x 4096 takes some 65 us.
constexpr int64_t kMinShareBlocks = 96;

double qgemm_q4_0_fx16_cost_us(int64_t M, int64_t N, int64_t K) {
    Cut cut;
    return M < kMinRows || N <= 0 || !fits(M, strips_of(N), K) ? 1e30 : plan(M, strips_of(N), K, kMinShareBlocks, (size_t)-1, &cut);
}

bool qgemm_q4_0_fx16_pays(int64_t M, int64_t N, int64_t K) {
    if (g_fx16 == 0 || N <= 0 || !fits(M, strips_of(N), K)) return false;
    return g_fx16 >= 2 || qgemm_q4_0_fx16_cost_us(M, N, K) < qgemm_q4_0_fx_cost_us(M, N, K);
}

// The same for digits: 2.85 us a step of 64 of K and round of tiles of 128 x 256 (256 x 32768 x 1024, two rounds).
bool qgemm_q4_0_fx16_digits_pay(int64_t M, int64_t N, int64_t K) {
    if (!qgemm_q4_0_fx16_pays(M, N, K)) return false;
    const int64_t tiles = ((M + Low::BM - 1) / Low::BM) * ((N + Low::BN - 1) / Low::BN);
    return (double)N * (double)K * (18.0 / 32.0 + 2.0) / 4.4e6 + (double)((tiles + 255) / 256) * (double)(K / 64) * 2.85 < qgemm_q4_0_fx_cost_us(M, N, K);
}

bool qgemm_q4_0_fx16_forced(Fx16* form) {
    const int v = g_fx16;
    if (v >= 2) *form = v == 2 ? Fx16::Digits : Fx16::Pairs;
    return v >= 2;
}

// X16 in granules, then RS [M] int2, then XS [M, K / 32] float32.
size_t q4_0_fx16_act_bytes(int64_t M, int64_t K) {
    return (size_t)strips_of(M) * (size_t)(K / 32) * kGranuleX * 2 + ((size_t)M * 8 + (size_t)M * (size_t)(K / 32) * 4 + 15) / 16 * 16;
}

template <bool NORM>
static void launch_halves(const float* x, const float* w, double eps, int64_t M, int64_t K, int64_t x_row_stride, void* act, hipStream_t st) {
    uint16_t* X16 = (uint16_t*)act;
    int2* RS = (int2*)(X16 + strips_of(M) * (K / 32) * kGranuleX);
    float* XS = (float*)(RS + M);
    const auto rows = K <= 4096 ? fx16_halves_kernel<2, NORM, false> : K <= 16384 ? fx16_halves_kernel<8, NORM, false> : fx16_halves_kernel<0, NORM, false>;
    const auto by_lanes = K <= 4096 ? fx16_halves_kernel<2, NORM, true> : K <= 16384 ? fx16_halves_kernel<8, NORM, true> : fx16_halves_kernel<0, NORM, true>;
    const auto kernel = in_lanes(M) ? by_lanes : rows;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(in_lanes(M) ? (M + kDies * kLineRows - 1) / (kDies * kLineRows) * (kDies * kLineRows) : M)), dim3(256), 0, st, x, w, x_row_stride, (int)K, X16, XS, RS, (int)M, (float)(1.0 / (double)K), (float)eps);
}

hipError_t q4_0_fx16_convert_act(const float* x, int64_t M, int64_t K, int64_t x_row_stride, void* act, Fx16 form, hipStream_t st) {
    if (form == Fx16::Digits) {
        uint16_t* X16 = (uint16_t*)act;
        int2* RS = (int2*)(X16 + strips_of(M) * (K / 32) * kGranuleX);
        const int gx = (int)((K / 4 + 255) / 256);
        hipLaunchKernelGGL(fx16_digits_kernel, dim3((unsigned)gx, (unsigned)M), dim3(256), 0, st, x, x_row_stride, (int)K, X16, (float*)(RS + M), RS);
    } else {
        launch_halves<false>(x, nullptr, 0, M, K, x_row_stride, act, st);
    }
    return hipGetLastError();
}

// rmsnorm's result converted, for qgemm_q4_0_fx16_parts: x [M, K], 16-byte aligned like w, K a multiple of 32.
hipError_t rmsnorm_fx16(const float* x, const float* w, void* act, int64_t M, int64_t K, double eps, hipStream_t st) {
    launch_halves<true>(x, w, eps, M, K, K, act, st);
    return hipGetLastError();
}

// The most that the shares' sums of a product of up to M rows take (plan): K's pieces of min_share_blocks, and no more than 1024 tiles of
// 128 x 256. It never falls as M grows, where the sums of the one cut of M rows do: 512 rows by 4096 x 14336 take four shares, 2048 none.
static size_t sums_bound(int64_t M, int64_t strips, int64_t K, int64_t min_share_blocks) {
    const int64_t nb = K / 32;
    int64_t shares = 1;
    for (int64_t s = 2; s <= 16; s++)
        if ((nb + s * kGroup - 1) / (s * kGroup) * kGroup >= min_share_blocks) shares = s;
    const size_t by_rows = (size_t)shares * (size_t)M * (size_t)strips * 128, by_tiles = (size_t)1024 * Low::BM * Low::BN * 4;
    return shares == 1 ? 0 : by_rows < by_tiles ? by_rows : by_tiles;
}

// The panel in granules, W's scales, the shares' sums.
static size_t panel_bytes(int64_t strips, int64_t K) { return (size_t)strips * (size_t)(K / 32) * kGranuleP * 2; }
static size_t scales_bytes(int64_t strips, int64_t K) { return (size_t)strips * (size_t)scale_blocks((int)(K / 32)) * kGranuleS * 4; }

size_t qgemm_q4_0_fx16_ws_bytes(int64_t M, int64_t N, int64_t K) {
    return panel_bytes(strips_of(N), K) + scales_bytes(strips_of(N), K) + sums_bound(M, strips_of(N), K, kMinShareBlocks);
}

// x's part of the operands.
static Operands operands(const Parts& parts, const void* act, const float* resid, int64_t M, int64_t K) {
    const int nb = (int)(K / 32);
    const uint16_t* X16 = (const uint16_t*)act;
    const int2* RS = (const int2*)(X16 + strips_of(M) * nb * kGranuleX);
    return Operands{nullptr, nullptr, X16, (const float*)(RS + M), RS, resid, nullptr, (int)M, nb, parts};
}

static hipError_t in_place(const Parts& parts, const void* act, const float* resid, int64_t M, int64_t K, void* ws, size_t ws_bytes, hipStream_t st) {
    Operands o = operands(parts, act, resid, M, K);
    o.sums = (float*)ws;
    return qgemm_q4_0_direct(o, ws_bytes, st);
}

static hipError_t multiply(const Parts& parts, const void* act, const float* resid, int64_t M, int64_t K, int64_t min_share_blocks, void* ws, size_t ws_bytes,
                           Fx16 form, hipStream_t st) {
    const int64_t strips = parts.strips;
    const size_t fixed = panel_bytes(strips, K) + scales_bytes(strips, K);
    if (!ws || ((uintptr_t)ws & 15) != 0 || ((uintptr_t)act & 15) != 0 || !fits(M, strips, K) || ws_bytes < fixed) return hipErrorInvalidValue;
    for (int i = 0; i < 3; i++)
        if (((uintptr_t)parts.W[i] & 1) != 0) return hipErrorInvalidValue;
    static LdsLimit limit, digits_limit;
    if (hipError_t e = limit.raise(kLdsBytes, {(const void*)qgemm_q4_0_fx16_kernel})) return e;
    if (hipError_t e = digits_limit.raise(Low::total, {(const void*)qgemm_q4_0_fx16_digits_kernel})) return e;
    const int nb = (int)(K / 32);
    const bool digits = form == Fx16::Digits;
    Cut cut{0, 0, (int)((M + Low::BM - 1) / Low::BM), (int)((strips + 7) / 8), 1, nb};
    if (!digits) plan(M, strips, K, min_share_blocks, ws_bytes - fixed, &cut);
    uint16_t* P = (uint16_t*)ws;
    float* SW = (float*)((char*)ws + panel_bytes(strips, K));
    Operands o = operands(parts, act, resid, M, K);
    o.P = P;
    o.SW = SW;
    if (cut.shares > 1) o.sums = (float*)((char*)ws + fixed);
    const int64_t wide = (int64_t)cut.wide_m * cut.wide_cols * cut.shares, low = (int64_t)cut.low_m * cut.low_cols * cut.shares;
    hipLaunchKernelGGL(fx16_panel_kernel, dim3((unsigned)((nb + 31) / 32 * strips)), dim3(256), 0, st, parts, P, SW, nb);
    const dim3 grid((unsigned)((wide + 7) / 8 * 8 + (low + 7) / 8 * 8));
    if (digits) hipLaunchKernelGGL(qgemm_q4_0_fx16_digits_kernel, grid, dim3(512), Low::total, st, o, cut);
    else hipLaunchKernelGGL(qgemm_q4_0_fx16_kernel, grid, dim3(512), kLdsBytes, st, o, cut);
    if (cut.shares > 1)
        if (hipError_t e = sum_shares(o, cut.shares, st)) return e;
    char shares[40] = "", beside[60] = "";
    if (cut.shares > 1) snprintf(shares, sizeof shares, ", %d shares of K", cut.shares);
    if (cut.wide_cols && cut.low_cols) snprintf(beside, sizeof beside, ", %d x %d tiles of 128 x 256", cut.low_m, cut.low_cols);
    note_kernel("qgemm_q4_0_fx16_kernel: %d x %d tiles of %s%s%s", cut.wide_cols ? cut.wide_m : cut.low_m, cut.wide_cols ? cut.wide_cols : cut.low_cols,
                cut.wide_cols ? "256 x 256" : "128 x 256", beside, shares);
    return hipGetLastError();
}

// Several matrices by the same rows of x in one product, or gate and up with silu(gate) up as their result: the tiles of
// all of them fill the device together (512 rows by 4096 of K: q, k and v of 4096, 1024 and 1024 rows take 84 us, one by one in
// the int8 form 190; gate and up of 14336 rows 290, one by one 2 x 150). K is cut into shares of 16 blocks and up.
constexpr int64_t kMinPartShareBlocks = 16;
constexpr size_t kMostSums = (size_t)96 << 20;

static bool parts_of(const Fx16Part* part, int n, bool swiglu, int64_t K, Parts* out) {
    if (n < 1 || n > 3 || (swiglu && (n != 2 || part[0].N != part[1].N))) return false;
    *out = Parts{};
    int64_t strips = 0;
    for (int i = 0; i < n; i++) {
        if (part[i].N <= 0 || part[i].N >= (1 << 27) || ((uintptr_t)part[i].W & 1) != 0) return false;
        out->W[i] = (const uint8_t*)part[i].W;
        out->y[i] = part[i].y;
        out->N[i] = (int)part[i].N;
        out->begin[i] = (int)strips;
        strips += strips_of(part[i].N);
    }
    for (int i = n; i < 3; i++) out->begin[i] = (int)strips;
    out->strips = (int)strips;
    out->swiglu = swiglu;
    return fits(1, strips, K);
}

// What qgemm_q4_0_fx16_parts can use of a workspace, for up to M rows.
size_t qgemm_q4_0_fx16_parts_ws_bytes(const Fx16Part* part, int n, int64_t K) {
    Parts p;
    return parts_of(part, n, false, K, &p) ? panel_bytes(p.strips, K) + scales_bytes(p.strips, K) + kMostSums : 0;
}

// Microseconds here, the cheaper way: with the pass over W first, or W read where it lies; and what it uses of the workspace.
static double parts_cost_us(const Parts& p, int64_t M, int64_t K, size_t ws_bytes, bool* direct, size_t* used = nullptr) {
    Cut cut{};
    size_t sums = 0;
    const size_t fixed = panel_bytes(p.strips, K) + scales_bytes(p.strips, K);
    const double panel = fits(M, p.strips, K) && ws_bytes >= fixed ? plan(M, p.strips, K, kMinPartShareBlocks, ws_bytes - fixed, &cut) : 1e30;
    const bool aligned = (((uintptr_t)p.W[0] | (uintptr_t)p.W[1] | (uintptr_t)p.W[2]) & 3) == 0;
    const double in_place = aligned ? qgemm_q4_0_direct_cost_us(M, p.strips, K, ws_bytes, &sums) : 1e30;
    *direct = in_place < panel;
    if (used) *used = *direct ? sums : fixed + (cut.shares > 1 ? (size_t)cut.shares * (size_t)M * (size_t)p.strips * 128 : 0);
    return *direct ? in_place : panel;
}

// Microseconds of the products one by one, on the int8 form or the row kernels.
static double apart_us(const Fx16Part* part, int n, int64_t M, int64_t K) {
    double apart = 0;
    for (int i = 0; i < n; i++) {
        const double rows_us = (double)M * ((double)part[i].N * (double)(K / 32) * 18.0) / 8.7e6, fx = qgemm_q4_0_fx_cost_us(M, part[i].N, K);
        apart += fx < rows_us ? fx : rows_us;
    }
    return apart;
}

// Whether they are the faster together here, in a workspace of ws_bytes, than each on the int8 form or the row kernels.
bool qgemm_q4_0_fx16_parts_pay(const Fx16Part* part, int n, bool swiglu, int64_t M, int64_t K, size_t ws_bytes) {
    Parts p;
    bool direct;
    if (g_fx16 == 0 || M < kMinPartRows || !parts_of(part, n, swiglu, K, &p)) return false;
    // digits, where the int8 form would be taken: one matrix at a time, by a panel
    if (g_fx16 == 2) return n == 1 && qgemm_q4_0_fx_pays(part[0].W, M, part[0].N, K) && fits(M, p.strips, K) && ws_bytes >= panel_bytes(p.strips, K) + scales_bytes(p.strips, K);
    const double us = parts_cost_us(p, M, K, ws_bytes, &direct);
    return us < 1e30 && (g_fx16 >= 3 || us < apart_us(part, n, M, K));
}

// What products of 9 rows up to max_rows use of a workspace of ws_bytes: in one of that size they run as in the larger one.
size_t qgemm_q4_0_fx16_parts_uses(const Fx16Part* part, int n, int64_t K, int64_t max_rows, size_t ws_bytes) {
    Parts p;
    size_t most = 0;
    if (!parts_of(part, n, false, K, &p)) return 0;
    for (int64_t M = kMinPartRows; M <= max_rows; M++) {
        bool direct;
        size_t used;
        if (parts_cost_us(p, M, K, ws_bytes, &direct, &used) < apart_us(part, n, M, K) && used > most) most = used;
    }
    return most;
}

// act: q4_0_fx16_convert_act's for these M rows; ws: ws_bytes, 16-byte aligned. Each part's y = x . W^T; one part alone: + resid, which
// may be y itself; swiglu: part 0's y = silu(x . W0^T) (x . W1^T).
hipError_t qgemm_q4_0_fx16_parts(const Fx16Part* part, int n, bool swiglu, const void* act, const float* resid, int64_t M, int64_t K, void* ws, size_t ws_bytes,
                                 hipStream_t st) {
    Parts p;
    bool direct;
    if (!parts_of(part, n, swiglu, K, &p) || (resid && n != 1) || !ws || ((uintptr_t)ws & 15) != 0) return hipErrorInvalidValue;
    Fx16 form = Fx16::Pairs;
    if (qgemm_q4_0_fx16_forced(&form) && form == Fx16::Digits) return multiply(p, act, resid, M, K, kMinPartShareBlocks, ws, ws_bytes, form, st);
    parts_cost_us(p, M, K, ws_bytes, &direct);
    if (direct) return in_place(p, act, resid, M, K, ws, ws_bytes, st);
    return multiply(p, act, resid, M, K, kMinPartShareBlocks, ws, ws_bytes, form, st);
}

// act: q4_0_fx16_convert_act's for these M rows; ws: qgemm_q4_0_fx16_ws_bytes(M, N, K) bytes, 16-byte aligned.
// y = x . W^T (+ resid, which may be y itself).
hipError_t qgemm_q4_0_fx16(const void* W, const void* act, float* y, const float* resid, int64_t M, int64_t N, int64_t K, void* ws, Fx16 form, hipStream_t st) {
    if (N <= 0 || N >= (1 << 27) || !fits(M, strips_of(N), K)) return hipErrorInvalidValue;
    const int n = (int)strips_of(N);
    const Parts parts{{(const uint8_t*)W, nullptr, nullptr}, {y, nullptr, nullptr}, {(int)N, 0, 0}, {0, n, n}, n, 0};
    return multiply(parts, act, resid, M, K, kMinShareBlocks, ws, qgemm_q4_0_fx16_ws_bytes(M, N, K), form, st);
}

// y = x . W^T, W read where it lies: ws 16-byte aligned.
hipError_t qgemm_q4_0_in_place(const void* W, const void* act, float* y, int64_t M, int64_t N, int64_t K, void* ws, size_t ws_bytes, hipStream_t st) {
    Parts p;
    const Fx16Part alone{W, y, N};
    if (!parts_of(&alone, 1, false, K, &p) || !ws || ((uintptr_t)ws & 15) != 0 || ((uintptr_t)act & 15) != 0) return hipErrorInvalidValue;
    return in_place(p, act, nullptr, M, K, ws, ws_bytes, st);
}

bool qgemm_q4_0_in_place_ok(const void* W, int64_t N, int64_t K) {
    return g_fx16 != 0 && g_fx16 != 2 && N > 0 && N < (1 << 25) && K > 0 && K % 64 == 0 && K <= (1 << 20) && ((uintptr_t)W & 3) == 0;
}

// 16 MiB: one round of workgroups, 256 of 128 rows by 128 columns. (With 64, single products of 200000 x 8192 and longer would take a twentieth less.)
size_t qgemm_q4_0_in_place_sums_bytes(int64_t M, int64_t N, int64_t K) {
    const int64_t pieces = (K / 32 + 7) / 8, shares = pieces < 32 ? pieces : 32, rows = M < kInPlaceRows ? M : kInPlaceRows;
    const size_t all = (size_t)shares * (size_t)rows * (size_t)strips_of(N) * 128, most = (size_t)16 << 20;
    return shares == 1 ? 0 : all < most ? all : most;
}

double qgemm_q4_0_in_place_cost_us(int64_t M, int64_t N, int64_t K) {
    return qgemm_q4_0_direct_cost_us(M, strips_of(N), K, qgemm_q4_0_in_place_sums_bytes(M, N, K));
}

}  // namespace mimir
