// Products of many rows of x with Q4_K and Q6_K weights on the matrix cores of
// gfx950: y[M, N] = x[M, K] . W[N, K]^T with x already rounded to int8 per
// super-block of 256 (kq_convert_act), computing what the reference's CPU tiles
// compute (backend/cpu/qtile.go:124-271), which is what its dot products
// compute (qdotQ4KGo and qdotQ6KGo, backend/cpu/qmatmul.go:148-200): per
// super-block an integer sum, one float32 product of the two scales, one
// multiply and one add, the super-blocks of a row taken in order. Every output
// here goes through the same float32 operations in the same order, so the
// results are the CPU's bit for bit.
//
// The integer sum of a super-block is sum_i s(i) q_i x_i with a 6-bit scale and
// a 4-bit quant (Q4_K) or an int8 scale and a 6-bit quant less 32 (Q6_K). The
// scaled weight s q has 10 or 14 bits, too many for the int8 matrix
// instruction, so it is split into two planes: Q4_K's by its scale, s = 8 s1 + s0, a = s1 q and
// b = s0 q (at most 105 each, so that a pair of 16-bit multiplies makes four of them), Q6_K's by
// its bytes, s q = 256 a + b. Either sum is that of two planes of
// v_mfma_i32_32x32x32_i8 against the same fragment of x. Integer sums are
// exact, so the split changes nothing. Q4_K's second sum, the mins against the
// sums of x, is sum over the sixteen 16-element groups of m(g / 2) S(g): one
// v_mfma_f32_32x32x16_f16 per tile and super-block, exact because S (at most
// 16 * 127) and m (at most 63) are integers binary16 holds and the products
// and their sum stay below 2^24.
//
// A workgroup of eight wavefronts owns a tile of 256 or 128 rows of x by 64 rows
// of W and walks K a super-block a step. Its wavefronts are two groups of four, each with half of the rows of x; a group splits half of the next
// super-block's W into LDS (planes in two buffers), multiplies, and turns its integer sums into float32 as above. x goes from memory
// straight into LDS (global_load_lds_dwordx4). LDS has room for 256 rows of a super-block once, so the groups of a tall tile are half a step apart: one
// multiplies, brings in the other's rows and splits W while the other is at its float32 sums, and the other way round. Of 128 rows there are two buffers; a group
// brings in its own rows a step ahead, both are in step, and one barrier a step is enough. Rows of LDS are 256 bytes with their
// 16-byte pieces turned by the row, which makes the 128-bit fragment reads conflict-free.
//
// What bounds it: the MFMAs (of 32 cycles each; 1088 a wavefront and super-block, 64 x 32 outputs, of Q4_K and 1024 of Q6_K) and the vector instructions, which do not overlap with
// them on this device: of Q4_K 256 a wavefront for the float32 operations (eight an output, fixed by the CPU's order), 80 for the split, 423 in all by the counters; of Q6_K, which has no
// mins, 357. At 2048 x 14336 x 4096 that is 92 % of the SIMDs' cycles by Q4_K and 77 % by Q6_K, whose wavefronts wait longer for loads off 2-byte boundaries, at a clock of 1.85 to 1.9 GHz.
// Before (both groups in step, halves of a super-block, split by 24-bit multiplies, tiles of 256 x 64 only where they filled the device) and now, us with x's
// conversion, Q4_K | Q6_K: 655 x 4096 x 14336 244 -> 157 | 238 -> 166, 655 x 14336 x 4096 185 -> 155 | 177 -> 158, 2048 x 14336 x 4096 434 -> 360 (668 TFLOP/s; of bfloat16 x, copies of W in turn, 388) | 419 -> 362,
// 1000 x 5120 x 5120 160 -> 109 | 148 -> 107, 128 x 14336 x 4096 42.1 -> 36.9 | 41.1 -> 39.1, 300 x 2048 x 8192 74 -> 61 | 70 -> 62.
//
// Both matrix instructions take, per lane, the
// bytes or halves k = 16 or 8 (lane / 32).. of row (lane % 32); the result holds
// column (lane % 32) and rows 8 (i / 4) + 4 (lane / 32) + i % 4 in register i.
#include "device_util.h"
#include "kernels.h"
#include "tile_plan.h"

namespace mimir {

#pragma clang fp contract(off)

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

constexpr int kTN = 64;          // rows of W per workgroup
constexpr int kThreads = 512;
constexpr int kSb = 256;         // K per step (a super-block), and bytes per LDS row of int8

// LDS: the rows of x of the super-block under way, two buffers of W's planes, and twice what the end of a super-block needs (scales
// and sums of x, scales and mins of W).
template <int TM>
struct Layout {
    static constexpr int x = 0;
    static constexpr int xbufs = TM == 128 ? 2 : 1;      // buffers of a group's rows of x
    static constexpr int planes = xbufs * TM * kSb;      // [2] of: plane A [kTN][kSb], plane B the same
    static constexpr int plane = kTN * kSb;
    static constexpr int xside = planes + 4 * plane;     // [2] of:
    static constexpr int xsum = 0;                       // binary16[TM][16]
    static constexpr int dx = TM * 32;                   // float[TM]
    static constexpr int xside_bytes = TM * 36;
    static constexpr int wside = xside + 2 * xside_bytes;  // [2] of:
    static constexpr int mins = 0;                       // binary16[kTN][16]
    static constexpr int dw = kTN * 32;                  // float[kTN][2]: d, dmin
    static constexpr int wside_bytes = kTN * 40;
    static constexpr int total = wside + 2 * wside_bytes;
};
static_assert(Layout<256>::total <= 160 * 1024, "a compute unit's LDS");

// Where 16-byte piece `piece` of row `row` sits: the 16 pieces of a row turned by the row, so that 16 rows' equal piece falls on all banks.
__device__ __forceinline__ int piece_at(int row, int piece) { return row * kSb + 16 * (piece ^ (row & 15)); }

__device__ __forceinline__ void phase_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// 16 bytes a lane from base + offset into LDS at lds_base + 16 lane (load_to_lds of gemm_nt_tile.h, a wavefront's address and a lane's offset).
__device__ __forceinline__ void load_to_lds(const uint8_t* base, uint32_t offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(offset), "s"(base) : "memory");
}

// Two 16-bit products a lane, their low halves.
__device__ __forceinline__ uint32_t mul_pairs(uint32_t a, uint32_t b) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b));
}

// Four quants in the bytes of q (each below 64) times the int8 scale s, less 32 s each, split into the digits of 256 a + b, both int8:
// q s + (128 - 32 s) in 16 bits has a in its upper byte and b + 128 in its lower. s and bias: the two numbers in both halves.
__device__ __forceinline__ void split_q6k(uint32_t q, uint32_t s, uint32_t bias, uint32_t& a, uint32_t& b) {
    const s16x2 sc = __builtin_bit_cast(s16x2, s), c = __builtin_bit_cast(s16x2, bias);
    const uint32_t even = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, q, 0x0c020c00u)) * sc + c);
    const uint32_t odd = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, __builtin_amdgcn_perm(0u, q, 0x0c030c01u)) * sc + c);
    a = __builtin_amdgcn_perm(odd, even, 0x07030501u);
    b = __builtin_amdgcn_perm(odd, even, 0x06020400u) ^ 0x80808080u;
}

// scale_min_k4 (backend/cpu/quant.go:129-134) on the twelve scale bytes held as three dwords.
__device__ __forceinline__ uint32_t q4k_min(uint32_t s1, uint32_t s2, int j) {
    const int sh = 8 * (j & 3);
    return j < 4 ? (s1 >> sh) & 63 : ((s2 >> (sh + 4)) & 0xf) | (((s1 >> (sh + 6)) & 3) << 4);
}

// What a thread holds between the loads and the LDS stores of its part of a super-block.
struct FetchedW {
    u32x4 hdr;      // Q4_K: d, dmin and the scales. Q6_K: x, y = the 8 scales of the half, z = d
    u32x4 q;        // 16 bytes of nibbles
    u32x4 qh;       // Q6_K: the 16 bytes of upper bits that go with them
};
struct FetchedX {
    u32x4 sums;     // Q4_K: eight int16 sums of a row of x
    float dx;       // the scale of a row of x
};

// One tile: rows [m0, m0 + 128 MT) of x by rows [n0, n0 + 64) of W.
template <int DT, int MT, bool OUT_BF16>
__device__ __forceinline__ void tile(const uint8_t* __restrict__ W, const uint8_t* __restrict__ act, void* yv, int M, int N, int nsb,
                                     const float* resid, int64_t act_row_bytes, int m0, int n0, uint8_t* smem) {
    constexpr int TM = 128 * MT;      // a wavefront's tile: 32 MT rows of x by 32 of W
    constexpr int GM = TM / 2;        // rows of x a group
    constexpr int NX = GM / 16;       // 1 KB loads of x a wavefront and super-block: four rows each
    constexpr int BB = DT == kQ4_K ? 144 : 210;
    typedef Layout<TM> L;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave >> 2, gw = wave & 3, gt = tid & 255;
    const int wm = gw & 1, wn = gw >> 1, l32 = lane & 31, lh = lane >> 5;

    const int g0 = group * GM;        // this group's first row in the tile

    // This thread's part of W: 16 bytes of nibbles of row wrow_i, piece c4 of half `group` of the super-block. Of the row's index
    // the two bits that tell the rows of sixteen lanes apart are those that turn their pieces away from each other.
    const int c4 = gt & 3, r4 = gt >> 4, j4 = (gt >> 2) & 3;
    const int wrow_i = DT == kQ4_K ? (r4 >> 2) * 16 + (r4 & 1) + 2 * (r4 & 2) + 2 * (j4 & 1) + 4 * (j4 & 2) : (r4 >> 2) * 16 + (r4 & 3) + 4 * j4;
    const int last_n = N - 1 - n0, last_m = M - 1 - m0;
    const uint8_t* w_t = W + (int64_t)n0 * nsb * BB;
    const uint32_t woff = (uint32_t)(wrow_i < last_n ? wrow_i : last_n) * (uint32_t)(nsb * BB);
    const uint8_t* act_t = act + (int64_t)m0 * act_row_bytes;
    // Its parts of x: a lane's piece of the wavefront's loads, and the sums of half a row with the row's scale (two threads a row; with 64 rows a
    // group two threads have the same part: branch-free, and the same bytes to the same place).
    const int gx = L::xbufs == 2 ? g0 : GM - g0;
    uint32_t xoff[NX];
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int r = gx + 4 * (NX * gw + j) + (lane >> 4);
        xoff[j] = (uint32_t)(r < last_m ? r : last_m) * (uint32_t)act_row_bytes + 16 * ((lane & 15) ^ (r & 15));
    }
    const int srow = g0 + ((gt >> 1) & (GM - 1));
    const uint32_t soff = (uint32_t)(srow < last_m ? srow : last_m) * (uint32_t)act_row_bytes;
    const uint8_t* sums_t = act_t + (int64_t)nsb * 256 + 16 * (tid & 1);
    const uint8_t* dx_t = act_t + (int64_t)nsb * 288;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    FetchedW fw;
    FetchedX fx;
    FetchedW fw0;  // the first super-block's, requested together with the second's
    FetchedX fx0;
    auto clamped = [&](int sb) { return sb < nsb ? sb : nsb - 1; };  // past the last super-block: it again, into buffers nobody reads
    auto fetch = [&](FetchedW& fw, FetchedX& fx, int sb) {
        const uint8_t* wb = w_t + (int64_t)sb * BB + woff;
        if (DT == kQ4_K) {
            fw.hdr = *(const u32x4*)wb;
            fw.q = *(const u32x4*)(wb + 16 + 64 * group + 16 * c4);
            fx.sums = *(const u32x4*)(sums_t + (int64_t)sb * 32 + soff);
        } else {
            fw.q = load_u32x4_unaligned(wb + 64 * group + 16 * c4);
            fw.qh = load_u32x4_unaligned(wb + 128 + 32 * group + 16 * (c4 & 1));
            u32x2 sc;
            __builtin_memcpy(&sc, wb + 192 + 8 * group, 8);
            fw.hdr[0] = sc[0], fw.hdr[1] = sc[1];
            fw.hdr[2] = load_u16(wb + 208);
        }
        fx.dx = *(const float*)(dx_t + (int64_t)sb * 4 + soff);
    };
    auto load_x = [&](int sb, int j) {
        load_to_lds(act_t + (int64_t)sb * 256, xoff[j], __builtin_amdgcn_readfirstlane(lds0 + L::x + ((sb & (L::xbufs - 1)) * TM + gx + 4 * (NX * gw + j)) * kSb));
    };
    auto stage = [&](const FetchedW& fw, const FetchedX& fx, int sb) {  // this thread's part of W's planes of super-block sb and of its sums and scales of x; its scales and mins by group 1
        u32x4 alo, blo, ahi, bhi;
        int plo, phi;  // the pieces of the low and the high nibbles' weights
        uint8_t* wside = smem + L::wside + (sb & 1) * L::wside_bytes;
        if (DT == kQ4_K) {
            const int j = 2 * (c4 >> 1);  // sub-blocks 4 group + j (low nibbles) and j + 1 (high) of this thread's bytes
            const int sh0 = 8 * (j & 3);
            uint32_t sl, sh;
            if (group == 0) {
                sl = (fw.hdr[1] >> sh0) & 63, sh = (fw.hdr[1] >> (sh0 + 8)) & 63;
            } else {
                sl = ((fw.hdr[3] >> sh0) & 0xf) | (((fw.hdr[1] >> (sh0 + 6)) & 3) << 4);
                sh = ((fw.hdr[3] >> (sh0 + 8)) & 0xf) | (((fw.hdr[1] >> (sh0 + 14)) & 3) << 4);
            }
            const uint32_t sl1 = (sl >> 3) * 0x00010001u, sl0 = (sl & 7) * 0x00010001u, sh1 = (sh >> 3) * 0x00010001u, shl = (sh & 7) * 0x00010001u;
#pragma unroll
            for (int d = 0; d < 4; d++) {  // a byte's product is at most 15 x 7: four of them in a pair of 16-bit multiplies
                const uint32_t lo = fw.q[d] & 0x0F0F0F0Fu, hi = (fw.q[d] >> 4) & 0x0F0F0F0Fu;
                alo[d] = mul_pairs(lo, sl1), blo[d] = mul_pairs(lo, sl0);
                ahi[d] = mul_pairs(hi, sh1), bhi[d] = mul_pairs(hi, shl);
            }
            plo = 8 * group + 4 * (c4 >> 1) + (c4 & 1);
            phi = plo + 2;
            if (group == 1) {
                float* dw = (float*)(wside + L::dw) + 2 * wrow_i;  // the row's four threads store the same two values
                dw[0] = f16_bits_to_f32((uint16_t)fw.hdr[0]);
                dw[1] = f16_bits_to_f32((uint16_t)(fw.hdr[0] >> 16));
                // the mins of sub-blocks 2 c4 and 2 c4 + 1, each once for its two groups of 16
                u32x2 pairs;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const _Float16 mn = (_Float16)(uint16_t)q4k_min(fw.hdr[2], fw.hdr[3], 2 * c4 + k);
                    pairs[k] = (uint32_t)__builtin_bit_cast(uint16_t, mn) * 0x00010001u;
                }
                *(u32x2*)(wside + L::mins + wrow_i * 32 + 8 * c4) = pairs;
            }
        } else {
            const int shl = c4 >= 2 ? 2 : 0;
            const uint32_t sl = (uint32_t)(int)(int8_t)(fw.hdr[0] >> (8 * c4)), sh = (uint32_t)(int)(int8_t)(fw.hdr[1] >> (8 * c4));
            const uint32_t sl2 = (sl & 0xffffu) * 0x00010001u, sh2 = (sh & 0xffffu) * 0x00010001u;
            const uint32_t cl = ((128u - 32u * sl) & 0xffffu) * 0x00010001u, ch = ((128u - 32u * sh) & 0xffffu) * 0x00010001u;
#pragma unroll
            for (int d = 0; d < 4; d++) {
                const uint32_t a = fw.q[d], b = fw.qh[d] >> shl;
                uint32_t a0, b0, a1, b1;
                split_q6k((a & 0x0F0F0F0Fu) | ((b & 0x03030303u) << 4), sl2, cl, a0, b0);
                split_q6k(((a >> 4) & 0x0F0F0F0Fu) | (b & 0x30303030u), sh2, ch, a1, b1);
                alo[d] = a0, blo[d] = b0, ahi[d] = a1, bhi[d] = b1;
            }
            plo = 8 * group + c4;
            phi = plo + 4;
            if (group == 1) ((float*)(wside + L::dw))[2 * wrow_i] = f16_bits_to_f32((uint16_t)fw.hdr[2]);
        }
        uint8_t* pa = smem + L::planes + (sb & 1) * 2 * L::plane;
        const int at_lo = piece_at(wrow_i, plo), at_hi = piece_at(wrow_i, phi);
        *(u32x4*)(pa + at_lo) = alo;
        *(u32x4*)(pa + at_hi) = ahi;
        *(u32x4*)(pa + L::plane + at_lo) = blo;
        *(u32x4*)(pa + L::plane + at_hi) = bhi;
        uint8_t* xside = smem + L::xside + (sb & 1) * L::xside_bytes;
        if (DT == kQ4_K) {
            const s16x8 s = __builtin_bit_cast(s16x8, fx.sums);
            *(f16x8*)(xside + L::xsum + srow * 32 + 16 * (tid & 1)) = __builtin_convertvector(s, f16x8);
        }
        ((float*)(xside + L::dx))[srow] = fx.dx;
    };

    i32x16 acc_a[MT], acc_b[MT];
    f32x16 acc[MT], accm[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[mt][i] = accm[mt][i] = 0.f;

    const int at0 = piece_at(l32, lh);  // this lane's first piece of a row; the next is 32 bytes on, turned
    auto multiply = [&](int sb, int sbx, bool more) {
        const uint8_t* xa = smem + L::x + ((sb & (L::xbufs - 1)) * TM + g0 + wm * 32 * MT) * kSb;
        const uint8_t* pa = smem + L::planes + (sb & 1) * 2 * L::plane + wn * 32 * kSb;
        i32x4 wa[2], wb[2], x[2][MT];
        auto read = [&](int s) {
            const int at = at0 ^ (32 * s), c = s & 1;
            wa[c] = *(const i32x4*)(pa + at), wb[c] = *(const i32x4*)(pa + L::plane + at);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) x[c][mt] = *(const i32x4*)(xa + mt * 32 * kSb + at);
        };
        read(0);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int c = s & 1;
            if (s + 1 < 8) read(s + 1);
            if (more && s < 4) {
#pragma unroll
                for (int j = s * NX / 4; j < (s + 1) * NX / 4; j++) load_x(sbx, j);
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                if (s == 0) {  // a super-block's first products start its sums from the constant zero
                    i32x16 zero;
#pragma unroll
                    for (int i = 0; i < 16; i++) zero[i] = 0;
                    acc_a[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[c][mt], wa[c], zero, 0, 0, 0);
                    acc_b[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[c][mt], wb[c], zero, 0, 0, 0);
                } else {
                    acc_a[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[c][mt], wa[c], acc_a[mt], 0, 0, 0);
                    acc_b[mt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(x[c][mt], wb[c], acc_b[mt], 0, 0, 0);
                }
            }
        }
    };
    // The end of a super-block: its integer sums into the float32 sums, as the CPU does it.
    auto finish = [&](int sb) {
        const uint8_t* xside = smem + L::xside + (sb & 1) * L::xside_bytes;
        const uint8_t* wside = smem + L::wside + (sb & 1) * L::wside_bytes;
        const float* dwp = (const float*)(wside + L::dw) + 2 * (wn * 32 + l32);
        const float dw = dwp[0], dmin = DT == kQ4_K ? dwp[1] : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int r0 = g0 + wm * 32 * MT + 32 * mt;
            f32x16 summ;
            if (DT == kQ4_K) {
                const f16x8 xs = *(const f16x8*)(xside + L::xsum + (r0 + l32) * 32 + 16 * lh);
                const f16x8 mn = *(const f16x8*)(wside + L::mins + (wn * 32 + l32) * 32 + 16 * lh);
                f32x16 zero;
#pragma unroll
                for (int i = 0; i < 16; i++) zero[i] = 0.f;
                summ = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs, mn, zero, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const f32x4 dx = *(const f32x4*)(xside + L::dx + 4 * (r0 + 8 * j + 4 * lh));
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int i = 4 * j + k;
                    const int sumi = (acc_a[mt][i] << (DT == kQ4_K ? 3 : 8)) + acc_b[mt][i];
                    const float dd = dw * dx[k];
                    const float tt = dd * (float)sumi;
                    acc[mt][i] = acc[mt][i] + tt;
                    if (DT == kQ4_K) {
                        const float dm = dmin * dx[k];
                        const float u = dm * summ[i];
                        accm[mt][i] = accm[mt][i] + u;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // one tile at a time: interleaving them costs registers the kernel lacks
        }
    };

    if (L::xbufs == 2 || group == 1) {
#pragma unroll
        for (int j = 0; j < NX; j++) load_x(0, j);
    }
    fetch(fw0, fx0, 0);
    fetch(fw, fx, clamped(1));
    stage(fw0, fx0, 0);
    wait_loads();
    phase_barrier();
    if (L::xbufs == 1 && group == 1) phase_barrier();
    for (int sb = 0; sb < nsb; sb++) {
        if (L::xbufs == 2) {
            if (sb + 1 < nsb) {
                stage(fw, fx, sb + 1);
                fetch(fw, fx, clamped(sb + 2));
            }
            multiply(sb, sb + 1, sb + 1 < nsb);
            __builtin_amdgcn_sched_barrier(0);
            finish(sb);
            wait_loads();
        } else {
            multiply(sb, sb + group, sb + group < nsb);
            if (sb + 1 < nsb) {
                stage(fw, fx, sb + 1);
                wait_loads();
                fetch(fw, fx, clamped(sb + 2));
            } else {
                wait_loads();
            }
            phase_barrier();
            __builtin_amdgcn_s_setprio(0);
            finish(sb);
            __builtin_amdgcn_s_setprio(1);
        }
        phase_barrier();
    }
    if (L::xbufs == 1 && group == 0) phase_barrier();

    const int n = n0 + wn * 32 + l32;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = m0 + g0 + wm * 32 * MT + 32 * mt + 8 * (i >> 2) + 4 * lh + (i & 3);
            if (m < M && n < N) {
                float v = DT == kQ4_K ? acc[mt][i] - accm[mt][i] : acc[mt][i];
                if (!OUT_BF16 && resid) v = v + resid[(int64_t)m * N + n];
                if (OUT_BF16) ((uint16_t*)yv)[(int64_t)m * N + n] = f32_to_bf16_bits(v);
                else ((float*)yv)[(int64_t)m * N + n] = v;
            }
        }
}

// How the result is cut: 64 tall_cols columns in tiles of 256 rows, handed out first, the rest in tiles of 128.
struct Cut {
    int tall_m, short_m, tall_cols, cols;
};

template <int DT, bool OUT_BF16>
__global__ __launch_bounds__(kThreads, 2) void qgemm_kquant_kernel(const uint8_t* __restrict__ W, const uint8_t* __restrict__ act,
                                                                   void* yv, const float* resid, int M, int N, int nsb, int64_t act_row_bytes, Cut cut) {  // resid may be yv
    extern __shared__ __align__(16) uint8_t smem[];
    // A die's workgroups (every eighth) take a contiguous range of the tiles, those that share rows of W next to each other, so that
    // the second and later ones find W in that die's L2.
    const int tall = cut.tall_m * cut.tall_cols, tall_die = (tall + 7) >> 3;
    int b = blockIdx.x;
    if (b < 8 * tall_die) {
        const int t = (b & 7) * tall_die + (b >> 3);
        if (t < tall) tile<DT, 2, OUT_BF16>(W, act, yv, M, N, nsb, resid, act_row_bytes, (t % cut.tall_m) * 256, (t / cut.tall_m) * kTN, smem);
        return;
    }
    b -= 8 * tall_die;
    const int low = cut.short_m * (cut.cols - cut.tall_cols), low_die = (low + 7) >> 3;
    const int t = (b & 7) * low_die + (b >> 3);
    if (t < low) tile<DT, 1, OUT_BF16>(W, act, yv, M, N, nsb, resid, act_row_bytes, (t % cut.short_m) * 128, (cut.tall_cols + t / cut.short_m) * kTN, smem);
}

// A short tile takes this part of a tall one's time: 0.55 on a device half empty (1.5 us a super-block for 2.7), 0.75 on a full one.
constexpr double kShortCost = 0.66;

// Tall tiles for as many whole rounds of the device as end earliest, short ones for the rest, which a round of tall tiles would leave
// partly empty; returns the end in tall tiles' time.
double plan(int64_t M, int64_t N, Cut* out) {
    const int tall_m = (int)((M + 255) / 256), short_m = (int)((M + 127) / 128), cols = (int)((N + kTN - 1) / kTN);
    *out = Cut{tall_m, short_m, 0, cols};
    double best = makespan(short_m * cols, kShortCost, 0, 0.0);
    const int64_t rounds = (int64_t)tall_m * cols / kUnits;
    for (int64_t round = rounds > 1 ? rounds - 1 : 1; round <= rounds + 1; round++) {
        const int64_t c = round * kUnits / tall_m;
        const int tall = (int)(c < cols ? c : cols);
        const double end = makespan(tall_m * tall, 1.0, short_m * (cols - tall), kShortCost);
        if (end < best - 1e-9) {
            best = end;
            *out = Cut{tall_m, short_m, tall, cols};
        }
    }
    return best;
}

template <int DT, bool OUT_BF16>
hipError_t launch(const QGemvArgs& a, int nsb, hipStream_t st) {
    constexpr int kLds = Layout<256>::total > Layout<128>::total ? Layout<256>::total : Layout<128>::total;
    static LdsLimit limit;
    if (hipError_t e = limit.raise(kLds, {(const void*)qgemm_kquant_kernel<DT, OUT_BF16>})) return e;
    Cut cut;
    plan(a.M, a.N, &cut);
    const int grid = 8 * ((cut.tall_m * cut.tall_cols + 7) / 8 + (cut.short_m * (cut.cols - cut.tall_cols) + 7) / 8);
    note_kernel("qgemm_kquant_kernel: %d x %d tiles of 256 x 64, %d x %d of 128 x 64", cut.tall_m, cut.tall_cols, cut.short_m, cut.cols - cut.tall_cols);
    hipLaunchKernelGGL((qgemm_kquant_kernel<DT, OUT_BF16>), dim3((unsigned)grid), dim3(kThreads), kLds, st,
                       (const uint8_t*)a.W, (const uint8_t*)a.act, (void*)a.y, a.resid, (int)a.M, (int)a.N, nsb, (int64_t)kq_act_bytes(a.K), cut);
    return hipGetLastError();
}

}  // namespace

bool qgemm_kquant_ok(int dt, const QGemvArgs& a) {
    // Q4_K's blocks are read with aligned loads (144 bytes keep a 16-byte aligned W aligned); Q6_K's 2-byte aligned.
    return (dt == kQ4_K || dt == kQ6_K) && a.K % 256 == 0 && a.K > 0 && ((uintptr_t)a.W & (dt == kQ4_K ? 15 : 1)) == 0 &&
           ((uintptr_t)a.act & 15) == 0 && a.M * ((a.N + kTN - 1) / kTN) < ((int64_t)1 << 30) && a.K <= (1 << 20);
}

// What a product takes by this kernel, us, Q4_K and Q6_K alike. Fitted to 950 products of 9 to 600 rows by 512 to 32768 rows of W of 4 to 56 super-blocks (6 % off in the mean).
double qgemm_kquant_us(int64_t M, int64_t N, int64_t K) {
    Cut cut;
    return 4 + (double)(K / 256) * (2.8 * plan(M, N, &cut) - 0.4);
}

// Against the row-by-row kernels, which read W once per row of x, at about 5.8 TB/s (Q4_K) or 5.1 TB/s (Q6_K) while it sits in
// the caches. Measured on 4096 x 4096, 4096 x 14336 and 14336 x 4096 weights, 2 to 64 rows (at 14336 x 4096 and
// eight rows: 49 and 79 us by rows, 35 and 39 us here).
bool qgemm_kquant_pays(int dt, const QGemvArgs& a) {
    if (a.M < 4 || !qgemm_kquant_ok(dt, a)) return false;
    const double rows_us = (double)a.M * (double)a.N * (double)(a.K / 256) * (dt == kQ4_K ? 144 : 210) / (dt == kQ4_K ? 5.8e6 : 5.1e6);
    return qgemm_kquant_us(a.M, a.N, a.K) < rows_us;
}

hipError_t qgemm_kquant(int dt, const QGemvArgs& a, hipStream_t st, bool out_bf16) {
    const int nsb = (int)(a.K / 256);
    if (dt == kQ4_K) return out_bf16 ? launch<kQ4_K, true>(a, nsb, st) : launch<kQ4_K, false>(a, nsb, st);
    return out_bf16 ? launch<kQ6_K, true>(a, nsb, st) : launch<kQ6_K, false>(a, nsb, st);
}

}  // namespace mimir
