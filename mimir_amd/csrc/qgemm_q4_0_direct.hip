// The Q4_0 product of some rows of float32 x (about 16 to 256: short prompts, large batches) by rows of W of up to 2048, and of up to 24
// rows by longer ones (more of these: qgemm_q4_0_parts.hip), x as pairs of binary16 as in
// qgemm_q4_0_fx16.hip and with its arithmetic, W read where it lies: the pass that writes W's integers out costs as much as the
// whole product at these sizes, and the kernel for up to eight rows a group (qgemv_q4_0_rows.hip) reads and unpacks W once
// a group.
//
// A wavefront takes a strip of 32 rows of W and all (up to 128) rows of x of its tile, block by block: sixteen bytes of W a lane,
// some blocks ahead, unpacked into the two halves of the MFMAs' second operand (some 25 instructions a block, beside
// 16 FMAs and 128 cycles of MFMA per 32 rows of x). x's granules pass through LDS, two blocks ahead in registers: read by every wavefront from
// memory they cost more than the products (12 KB a block and wavefront at 77 rows: 77 x 14336 x 4096 took 80 us, now 44). A
// workgroup has four strips by two halves of its share of K, which meet in LDS; the shares' sums are added by a launch of their own.
//
// What bounds it: a step of a wavefront (a block) takes 0.5 us with one strip of x and 1.35 with four, twice its MFMAs and FMAs: the
// wait for the step's barrier and, with few strips, the loads of W (32 lines a request; as one load of 16 bytes off a
// 4-byte boundary a block they cost a tenth more). Whole calls, the row kernel or the int8 form before and this:
//   77 x 5120 x 5120   39 -> 31.6 us     128 x 14336 x 4096   80 -> 57     256 x 4096 x 14336  219 -> 94
//   64 x 14336 x 4096  60 -> 38          77 x 4096 x 14336    77 -> 49     200 x 14336 x 4096  153 -> 85
// (shapes that have since gone to qgemm_q4_0_parts.hip, with its times) and from 24 rows down the row kernel is seldom slower. Blocks' sums are those of qgemm_q4_0_fx16.hip; with K in shares and halves the error
// against 64 bits is 1.05e-7 of the result at 77 x 5120 x 5120 where it was 1.63e-7.
//
// Rows held with an exponent a block (q4_halves.h: Form) take their scales through LDS beside x: four reads and a multiplication an output more a
// block. One such row in the call, against one strip of x at a time with its rows' scales from memory, before, and against the
// forms that this kernel took the place of: 77 x 5120 x 5120 53 -> 34 us (41), 128 x 14336 x 4096 127 -> 66 (84), 256 x 14336 x 4096 217 -> 100 (162).
#include "kernels.h"
#include "q4_halves.h"

namespace mimir {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kTileStrips = 4;  // of x, at most
constexpr int kColStrips = 4;   // of W a workgroup
constexpr int kWaves = 8;

struct Direct {
    int groups, tiles_m;       // of column strips, of rows
    int shares, share_blocks;  // of K; the last share may be shorter, all are even
};

// LDS: [2 halves][2][MS] granules of x, in whose place the halves' sums meet; then where rows have scales a block [2 halves][2][MS 32] of these.
template <int MS>
constexpr int kLdsBytes = 4 * MS * kGranuleX * 2 + 4 * MS * 32 * 4;

// MS strips of x from row m0 on. BY_BLOCK: where a row of them has an exponent a block, all are taken as if they had. A thread brings one
// row's scales through LDS, and a lane reads those of its results' rows from there, four a read, the same for the half's lanes.
template <int MS, bool BY_BLOCK>
__device__ __forceinline__ void direct_tile(const Operands& o, const Direct& d, int m0, int group, int share, float* lds) {
    constexpr int kPairs = 3;  // pairs of blocks of W in registers, this one among them
    const int lane = threadIdx.x & 63, r32 = lane & 31, q = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int col = wave & (kColStrips - 1), second = wave / kColStrips;
    const int M = o.M, nb = o.nb;
    const int strip_at = group * kColStrips + col, strip = strip_at < o.parts.strips ? strip_at : o.parts.strips - 1;  // past the last: not stored
    const int b_share = share * d.share_blocks, in_share = nb - b_share < d.share_blocks ? nb - b_share : d.share_blocks;
    const int first_half = (in_share / 2 + 1) & ~1;  // both even: a share is
    const int b0 = b_share + (second ? first_half : 0), count = second ? in_share - first_half : first_half;

    const int part = o.parts.swiglu ? strip & 1 : strip >= o.parts.begin[2] ? 2 : strip >= o.parts.begin[1] ? 1 : 0;
    const int n = (o.parts.swiglu ? strip >> 1 : strip - o.parts.begin[part]) * 32 + r32, N = o.parts.N[part];
    const uint8_t* w = o.parts.W[part] + ((int64_t)(n < N ? n : N - 1) * nb + b0) * 18 + 8 * q;
    // x's granules, which the half's four wavefronts bring into LDS together: KB `col` of each
    const uint16_t* xg[MS];
    int piece[4];
#pragma unroll
    for (int mt = 0; mt < MS; mt++) {
        const int s = m0 / 32 + mt, last = (M - 1) / 32;
        xg[mt] = o.X16 + ((int64_t)(s < last ? s : last) * nb + b0) * kGranuleX + col * 512 + lane * 8;
    }
#pragma unroll
    for (int p = 0; p < 4; p++) piece[p] = piece_at(r32, 2 * p + q, true);
    uint16_t* stage = (uint16_t*)lds + second * 2 * MS * kGranuleX;  // [2][MS] granules of this half
    // a thread's row of scales: of those that have one exponent, that one
    float* scales = lds + MS * kGranuleX * 2 + second * 2 * MS * 32;  // [2][MS 32] of this half
    const int srow = col * 64 + lane;
    const float* row_scales = nullptr;
    f32x2 scale[2] = {{0.f, 0.f}, {0.f, 0.f}};  // of this pair of blocks and the next
    if (BY_BLOCK && srow < MS * 32) {
        const int m = m0 + srow < M ? m0 + srow : M - 1;
        const int2 info = o.RS[m];
        if (info.y == kBlockHalves) {
            row_scales = o.XS + (int64_t)m * nb + b0;
        } else {
            const float one = info.x == INT32_MAX ? __builtin_nanf("") : __builtin_ldexpf(1.f, info.x);
            scale[0] = scale[1] = f32x2{one, one};
        }
    }

    f32x16 acc[MS], zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MS; mt++) acc[mt] = zero;

    // A pair of blocks is 36 bytes on a 4-byte boundary. Lane half q takes bytes 8 q .. + 12, in which the even block's eights of
    // nibbles q lie two bytes in (q = 0: behind the scale), and 16 + 8 q .. + 12, the odd one's in the last eight.
    u32x3 raw[kPairs][2];
    u32x4 held[2][MS];
    auto load_w = [&](int b, u32x3 to[2]) {
        const uint8_t* from = w + (int64_t)(b < count ? b : count - 2) * 18;
        __builtin_memcpy(&to[0], __builtin_assume_aligned(from, 4), 12);
        __builtin_memcpy(&to[1], __builtin_assume_aligned(from + 16, 4), 12);
    };
    auto load_x = [&](int b, u32x4 to[MS]) {
#pragma unroll
        for (int mt = 0; mt < MS; mt++) to[mt] = *(const u32x4*)(xg[mt] + (int64_t)(b < count ? b : count - 1) * kGranuleX);
    };
    auto store_x = [&](int b, const u32x4 from[MS]) {
#pragma unroll
        for (int mt = 0; mt < MS; mt++) *(u32x4*)(stage + ((b & 1) * MS + mt) * kGranuleX + col * 512 + lane * 8) = from[mt];
    };
    auto load_scales = [&](int b, f32x2& to) {  // b even; a row's blocks are an even number, so a pair lies on 8 bytes
        if (BY_BLOCK && row_scales) to = *(const f32x2*)(row_scales + (b < count ? b : count - 2));
    };
    auto store_scale = [&](int b, float s) {
        if (BY_BLOCK && srow < MS * 32) scales[(b & 1) * MS * 32 + srow] = s;
    };
    auto block = [&](int b, const u32x3& raw_b, bool odd) {
        const uint32_t lo = odd ? raw_b[1] : __builtin_amdgcn_alignbyte(raw_b[1], raw_b[0], 2);
        const uint32_t hi = odd ? raw_b[2] : __builtin_amdgcn_alignbyte(raw_b[2], raw_b[1], 2);
        const auto both = __builtin_amdgcn_permlane32_swap(raw_b[0], raw_b[0], false, false);  // the lower lanes' scales to all
        const uint32_t bits = both[0];
        // odd blocks with their sign turned: b0 is even
        const float dw = f16_bits_to_f32((uint16_t)(odd ? (bits >> 16) ^ 0x8000u : bits & 0xffffu));
        const f16x8 w0 = nibbles_to_f16(lo, hi, 0), w1 = nibbles_to_f16(lo, hi, 1);
        // a strip's products are issued with the FMAs of the one before it
        f32x16 c[2];
        f32x4 dx[2][4];  // x's scales of this block, of the 16 rows that this lane has results of
        auto finish = [&](int mt) {
#pragma unroll
            for (int e = 0; e < 16; e++) acc[mt][e] = fmaf(BY_BLOCK ? dw * dx[mt & 1][e >> 2][e & 3] : dw, c[mt & 1][e], acc[mt][e]);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int mt = 0; mt < MS; mt++) {
            const uint16_t* x = stage + ((b & 1) * MS + mt) * kGranuleX;
            auto part = [&](int p) { return *(const f16x8*)(x + piece[p]); };
            if (BY_BLOCK)
#pragma unroll
                for (int g = 0; g < 4; g++) dx[mt & 1][g] = *(const f32x4*)(scales + ((b & 1) * MS + mt) * 32 + 8 * g + 4 * q);
            f32x16& s = c[mt & 1];
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(part(2), w0, zero, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(part(3), w1, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(part(0), w0, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(part(1), w1, s, 0, 0, 0);
            if (mt > 0) finish(mt - 1);
        }
        finish(MS - 1);
    };
    if (count > 0) {  // past the end the last pair, and the last block of x, is requested again and not used
#pragma unroll
        for (int i = 0; i < kPairs - 1; i++) load_w(2 * i, raw[i]);
        load_x(0, held[0]);
        load_x(1, held[1]);
        store_x(0, held[0]);
        load_x(2, held[0]);
        load_scales(0, scale[0]);
        load_scales(2, scale[1]);
        store_scale(0, scale[0][0]);
    }
    __syncthreads();
    for (int b = 0; b < first_half; b += 2 * kPairs) {
#pragma unroll
        for (int u = 0; u < 2 * kPairs; u++) {
            if (b + u >= first_half) break;
            if (b + u < count) {
                if ((u & 1) == 0) load_w(b + u + 2 * kPairs - 2, raw[(u / 2 + kPairs - 1) % kPairs]);
                store_x(b + u + 1, held[(u + 1) & 1]);
                load_x(b + u + 3, held[(u + 1) & 1]);
                store_scale(b + u + 1, u & 1 ? scale[1][0] : scale[0][1]);
                if (BY_BLOCK && (u & 1)) {
                    scale[0] = scale[1];
                    load_scales(b + u + 3, scale[1]);
                }
                __builtin_amdgcn_sched_barrier(0);
                block(b + u, raw[u / 2][u & 1], u & 1);
            }
            __syncthreads();
        }
    }

    // the second half of the share's blocks to the first's wavefronts
    float* mine = lds + (size_t)col * MS * 16 * 64 + lane;
    if (second) {
#pragma unroll
        for (int mt = 0; mt < MS; mt++)
#pragma unroll
            for (int e = 0; e < 16; e++) mine[(mt * 16 + e) * 64] = acc[mt][e];
    }
    __syncthreads();
    if (!second) {
#pragma unroll
        for (int mt = 0; mt < MS; mt++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[mt][e] = acc[mt][e] + mine[(mt * 16 + e) * 64];
    }
    float* sums = o.sums ? o.sums + (int64_t)share * M * o.parts.strips * 32 : nullptr;
    const bool gated = o.parts.swiglu && !sums;
    if (gated) {  // up's sums to the wavefront that has gate's
        if (!second && (col & 1))
#pragma unroll
            for (int mt = 0; mt < MS; mt++)
#pragma unroll
                for (int e = 0; e < 16; e++) mine[(mt * 16 + e) * 64] = acc[mt][e];
        __syncthreads();
    }
    if (second || strip_at >= o.parts.strips || (gated && (col & 1))) return;
    int n0s;
    const int to = part_of(o.parts, strip, &n0s);
    float* y = sums ? sums : o.parts.y[to];
    const float* resid = sums ? nullptr : o.resid;
    const int cols = sums ? o.parts.strips * 32 : o.parts.N[to], n4 = (sums ? strip * 32 : n0s) + (r32 & ~3);
    const bool wide_ok = (cols & 3) == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)resid & 15) == 0;
    const float* up = mine + (size_t)MS * 16 * 64;
#pragma unroll
    for (int mt = 0; mt < MS; mt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int m = m0 + mt * 32 + g * 8 + q * 4 + (lane & 3), e_row = BY_BLOCK ? 0 : o.RS[m < M ? m : M - 1].x;
            float v[4] = {acc[mt][4 * g], acc[mt][4 * g + 1], acc[mt][4 * g + 2], acc[mt][4 * g + 3]};
            quad_transpose(v, lane);
            if (!BY_BLOCK) under_exponent(v, e_row);
            if (gated) {
                float u[4];
#pragma unroll
                for (int k = 0; k < 4; k++) u[k] = up[(mt * 16 + 4 * g + k) * 64];
                quad_transpose(u, lane);
                if (!BY_BLOCK) under_exponent(u, e_row);
#pragma unroll
                for (int k = 0; k < 4; k++) v[k] = silu_times(v[k], u[k]);
            }
            if (m < M && n4 < cols) store_four(y, resid, m, cols, n4, v, wide_ok);
        }
}

template <int MS>
__global__ __launch_bounds__(64 * kWaves) void qgemm_q4_0_direct_kernel(Operands o, Direct d) {
    extern __shared__ __align__(16) float lds[];
    int t = (int)blockIdx.x;
    const int group = __builtin_amdgcn_readfirstlane(t % d.groups);
    t /= d.groups;
    const int m0 = __builtin_amdgcn_readfirstlane(t % d.tiles_m) * kTileStrips * 32, share = __builtin_amdgcn_readfirstlane(t / d.tiles_m);
    bool by_block = false;
    for (int r = threadIdx.x & 63; r < MS * 32; r += 64) by_block |= o.RS[m0 + r < o.M ? m0 + r : o.M - 1].y == kBlockHalves;
    if (__ballot(by_block) == 0) direct_tile<MS, false>(o, d, m0, group, share, lds);
    else direct_tile<MS, true>(o, d, m0, group, share, lds);
}

template <int MS>
hipError_t launch(const Operands& o, const Direct& d, hipStream_t st) {
    if (kLdsBytes<MS> > 64 * 1024) {
        static LdsLimit limit;
        if (hipError_t e = limit.raise(kLdsBytes<MS>, {(const void*)qgemm_q4_0_direct_kernel<MS>})) return e;
    }
    hipLaunchKernelGGL(qgemm_q4_0_direct_kernel<MS>, dim3((unsigned)(d.groups * d.tiles_m * d.shares)), dim3(64 * kWaves), kLdsBytes<MS>, st, o, d);
    return hipGetLastError();
}

// Microseconds of a product and its cut into shares of K. A compute unit takes a workgroup at a time; one takes 2 us and, for
// every pair of blocks of its share (a block for each half), 0.22 and 0.28 for each strip of x (measured at 24 to 200 rows by
// 14336 x 4096 and 4096 x 14336). Shares: a launch more, and their sums at 4.5 TB/s there and back.
double plan(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, Direct* out) {
    const int64_t nb = K / 32, groups = (strips + kColStrips - 1) / kColStrips, tiles = (M + 32 * kTileStrips - 1) / (32 * kTileStrips);
    const int ms = tiles > 1 ? kTileStrips : (int)strips_of(M);
    const double step_us = 0.22 + 0.28 * ms;
    double best = 1e30;
    for (int64_t shares = 1; shares <= 32; shares++) {
        const int64_t blocks = (nb + 4 * shares - 1) / (4 * shares) * 4, used = (nb + blocks - 1) / blocks;
        if (used != shares) continue;
        const size_t sums = (size_t)shares * (size_t)M * (size_t)strips * 128;
        if (shares > 1 && (blocks < 8 || sums > sums_bytes)) break;
        double us = (double)((groups * tiles * shares + 255) / 256) * (2.0 + (double)(blocks / 2) * step_us);
        if (shares > 1) us += 5.0 + (double)sums * 2 / 4.5e6;
        if (us < best) {
            best = us;
            *out = Direct{(int)groups, (int)tiles, (int)shares, (int)blocks};
        }
    }
    return best;
}

bool fits(int64_t M, int64_t strips, int64_t K) {
    return M > 0 && M <= kInPlaceRows && strips > 0 && strips < (1 << 20) && K > 0 && K % 64 == 0 && K <= (1 << 20);
}

}  // namespace

// What qgemm_q4_0_parts.hip takes instead: the faster by both models and by a tenth, which is how far they may be off: here | there 128 x 9536 x 4544 51.2 us | 55.8 (by the models 45.7 and
// 44.1), 108 x 4480 x 13056 61.7 | 67.2 (53.2, 51.9), 205 x 2240 x 8448 48.5 | 50.4 (39.5, 37.0), 256 x 5120 x 5120 54.4 | 58.2 (51.5, 49.3); of 780 shapes it is behind by more than 3 % at
// three within the tenth (128 x 6208 x 8960 57.6 | 60.0). Nor up to 32 rows by more than 8192 long ones: 29 x 11136 x 11328 54.0 | 60.5, 31 x 12480 x 8960 46.9 | 51.2, but 28 x 8128 x 13376 54.2 | 48.7.
static bool by_parts(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, double us) {
    return qgemm_q4_0_parts_ok(M, strips, K) && !(M <= 32 && strips > 256 && K > 8192) && qgemm_q4_0_parts_cost_us(M, strips, K, sums_bytes, nullptr) <= 0.9 * us;
}

double qgemm_q4_0_direct_cost_us(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, size_t* used) {
    Direct d{};
    if (sums_bytes > kDirectMostSums) sums_bytes = kDirectMostSums;
    const double us = fits(M, strips, K) ? plan(M, strips, K, sums_bytes, &d) : 1e30;
    if (by_parts(M, strips, K, sums_bytes, us)) return qgemm_q4_0_parts_cost_us(M, strips, K, sums_bytes, used);
    if (used) *used = d.shares > 1 ? (size_t)d.shares * (size_t)M * (size_t)strips * 128 : 0;
    return us;
}

// o: the parts, x's halves and their scales, sums: sums_bytes of workspace.
hipError_t qgemm_q4_0_direct(Operands o, size_t sums_bytes, hipStream_t st) {
    const int64_t K = (int64_t)o.nb * 32;
    Direct d;
    if (sums_bytes > kDirectMostSums) sums_bytes = kDirectMostSums;
    if (!fits(o.M, o.parts.strips, K)) return hipErrorInvalidValue;
    const double us = plan(o.M, o.parts.strips, K, sums_bytes, &d);
    if (us >= 1e30) return hipErrorInvalidValue;
    if (by_parts(o.M, o.parts.strips, K, sums_bytes, us)) return qgemm_q4_0_parts(o, sums_bytes, st);
    for (int i = 0; i < 3; i++)
        if (((uintptr_t)o.parts.W[i] & 3) != 0) return hipErrorInvalidValue;
    if (d.shares == 1) o.sums = nullptr;
    const int ms = d.tiles_m > 1 ? kTileStrips : (int)strips_of(o.M);
    if (hipError_t e = ms == 1 ? launch<1>(o, d, st) : ms == 2 ? launch<2>(o, d, st) : ms == 3 ? launch<3>(o, d, st) : launch<4>(o, d, st)) return e;
    if (d.shares > 1)
        if (hipError_t e = sum_shares(o, d.shares, st)) return e;
    note_kernel("qgemm_q4_0_direct_kernel<%d>: %d x %d tiles, %d shares of K", ms, d.tiles_m, d.groups, d.shares);
    return hipGetLastError();
}

}  // namespace mimir
