// Attention for many query positions at once (a prompt) on the matrix cores of gfx950: the semantics of
// attention.hip (softmax(scale * q.k^T) . v per query row, the query scaled first, p = exp(s - max), the result
// (sum p v) * (1 / sum p), the logsumexp max + log(sum p), a row that sees no key zeros and -Inf, key j hidden from
// query i when causal and j > i + causal_offset; backend/cpu/attention.go:268-292, 437-535), for the calls that kernel
// serves one query row a workgroup, re-reading every key and value for every row.
//
// Two kernels: one on float32 operands, described here, and one for binary16 keys and values, described where it stands.
// A wavefront owns 32 query rows of one head and walks the keys in tiles of 32 with a running maximum and sum per
// row (a row's result is rescaled when its maximum grows), and both products of a tile are MFMAs on float32 operands
// (v_mfma_f32_32x32x2_f32), so that nothing is rounded that the other kernel does not round. Both are computed
// transposed, so that everything a row owns lives in one lane (and its partner 32 lanes on): scores^T = K . Q^T over the
// features, the tile's keys as the first operand from LDS and the lane's own row of Q (scaled, in registers for the
// whole walk, 64 a lane at 128 features) as the second, which leaves a lane 16 of its row's 32 scores in registers (the
// partner holds the other 16): maximum and sum are chains over those registers and one exchange with the partner; then
// result^T = V^T . P^T over the tile's keys, taken in the order the scores' registers hold them, so that p goes from the
// exponential straight into the MFMA's second operand, and the lane ends with 16 features of every 32 of its row. A
// workgroup is four wavefronts with consecutive rows of one head, which share the tile of keys and values in LDS
// (the next tile's rows requested while this one is used; K's rows padded by a float so that 32 keys' equal feature falls on 32 banks).
//
// What differs from the other kernel is the order of the float32 sums (features and keys in pairs as the MFMA takes
// them, keys in tiles of 32 with rescaling), so results agree to float32 rounding, not bit for bit.
#include "device_util.h"
#include "kernels.h"

namespace mimir {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kRows = 32;       // query rows a wavefront
// wavefronts a workgroup (WAVES below, float32): four, 128 consecutive rows of one head, or two where four would leave the device short of workgroups
constexpr int kTile = 32;       // keys a tile

struct PromptParams {
    int64_t q_b, q_h, q_i, k_b, k_h, k_p, v_b, v_h, v_p, o_b, o_h, o_i;
    int B, H, HK, Q, K;
    float scale;
    int causal;
    int64_t causal_offset;
};

// Element e of a row part held as raw 32-bit words.
template <typename KV>
__device__ __forceinline__ float element(const uint32_t* raw, int e);
template <>
__device__ __forceinline__ float element<float>(const uint32_t* raw, int e) { return __builtin_bit_cast(float, raw[e]); }
template <>
__device__ __forceinline__ float element<uint16_t>(const uint32_t* raw, int e) { return f16_bits_to_f32((uint16_t)(raw[e >> 1] >> (16 * (e & 1)))); }

// The two values of a packed pair of bfloat16.
__device__ __forceinline__ float bf16_lo(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); }

// The other half's value: lane ^ 32.
__device__ __forceinline__ float other_half(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, v)));
}

template <int D>
struct Float32Lds {
    static constexpr int KS = D + 1;     // floats between rows of the keys' tile
    float ks[kTile * KS];
    __align__(16) float vs[kTile * D];
    int vbad[2];                         // whether a tile's values hold a NaN or an infinity, for tiles of either parity
};

// Rows [first, first + ROWS) of head h of sequence b.
template <typename KV, int D, int WAVES, int ROWS>
__device__ __forceinline__ void rows_by_float32(const float* __restrict__ q, const KV* __restrict__ k, const KV* __restrict__ v, float* __restrict__ out,
                                                float* __restrict__ lse, const PromptParams& p, int b, int h, int first, float* ks, float* vs, int* vbad) {
    constexpr int KS = Float32Lds<D>::KS;
    constexpr int NT = D / 32;           // 32-feature tiles of the result
    constexpr int PER = D / 8;           // elements of a key (value) row a thread loads: eight threads a row
    constexpr int RP = 8 * WAVES;        // rows of a tile the workgroup loads at once
    constexpr int NP = kTile / RP;       // and how often
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r32 = lane & 31, hi = lane >> 5;
    const int hk = h / (p.H / p.HK);
    const int i0 = ROWS == WAVES * kRows || wave * kRows < ROWS ? first + wave * kRows : p.Q;  // this wavefront's first row, or none
    const int64_t Kt = p.K;
    auto seen_of = [&](int i) -> int {  // keys row i sees
        int64_t s = Kt;
        if (p.causal) {
            s = (int64_t)i + p.causal_offset + 1;
            s = s < 0 ? 0 : s > Kt ? Kt : s;
        }
        return (int)s;
    };
    const int last_row_wg = first + ROWS - 1 < p.Q ? first + ROWS - 1 : p.Q - 1;
    const int last_row_wave = i0 + kRows - 1 < p.Q ? i0 + kRows - 1 : p.Q - 1;
    const int seen_wg = p.causal ? seen_of(last_row_wg) : (int)Kt;
    const int seen_wave = i0 < p.Q ? (p.causal ? seen_of(last_row_wave) : (int)Kt) : 0;

    // this lane's row, scaled, as the MFMA's second operand: lane (feature 2 s + hi, column r32) for s = 0 .. D / 2
    const int row = i0 + r32;
    float qreg[D / 2];
    {
        const int i = row < p.Q ? row : p.Q - 1;
        const float* qr = q + b * p.q_b + (int64_t)h * p.q_h + (int64_t)i * p.q_i + hi;
#pragma unroll
        for (int s = 0; s < D / 2; s++) qreg[s] = qr[2 * s] * p.scale;
    }
    const int seen = row < p.Q ? seen_of(row) : 0;
    float m = -__builtin_inff(), l = 0.f;  // the row's maximum so far; the sum over the keys this half of the lanes holds
    f32x16 o[NT];                          // the row's result, transposed: register e of tile t is feature 32 t + 8 (e / 4) + 4 hi + e % 4
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[t][e] = 0.f;

    // a thread's part of a tile's keys and values: rows tid / 8 + RP n, elements [PER (tid % 8), + PER)
    const int lrow = tid >> 3, lpart = tid & 7;
    const KV* kbase = k + b * p.k_b + (int64_t)hk * p.k_h + PER * lpart;
    const KV* vbase = v + b * p.v_b + (int64_t)hk * p.v_h + PER * lpart;
    constexpr int VEC = PER * (int)sizeof(KV) / 16;  // 16-byte pieces of a thread's part (the host checks their alignment)
    uint32_t kreg[NP][4 * VEC], vreg[NP][4 * VEC];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int n = 0; n < NP; n++) {
            int64_t j = j0 + lrow + RP * n;
            j = j < Kt ? j : Kt - 1;  // rows past the last key: never seen, loaded from the last one
#pragma unroll
            for (int c = 0; c < VEC; c++) {
                const u32x4 kw = ((const u32x4*)(kbase + j * p.k_p))[c], vw = ((const u32x4*)(vbase + j * p.v_p))[c];
#pragma unroll
                for (int w = 0; w < 4; w++) kreg[n][4 * c + w] = kw[w], vreg[n][4 * c + w] = vw[w];
            }
        }
    };
    auto stage = [&](int parity) {
        float chk = 0.f;  // 0 * value summed: NaN as soon as a value is a NaN or an infinity
#pragma unroll
        for (int n = 0; n < NP; n++) {
            const int r = lrow + RP * n;
#pragma unroll
            for (int e = 0; e < PER; e++) ks[r * KS + PER * lpart + e] = element<KV>(kreg[n], e);
#pragma unroll
            for (int e = 0; e < PER; e += 4) {
                const f32x4 f = {element<KV>(vreg[n], e), element<KV>(vreg[n], e + 1), element<KV>(vreg[n], e + 2), element<KV>(vreg[n], e + 3)};
                *(f32x4*)(vs + r * D + PER * lpart + e) = f;
#pragma unroll
                for (int c = 0; c < 4; c++) chk = __builtin_fmaf(f[c], 0.f, chk);
            }
        }
        if (__builtin_amdgcn_ballot_w64(chk != chk) != 0 && lane == 0) vbad[parity] = 1;
    };

    // The matrix cores multiply a whole tile of values by the rows' weights, zero for the keys a row does not see: fine
    // unless such a value is a NaN or an infinity, which the reference never reads for that row. A tile that holds one and
    // is not seen whole by every row of the wavefront takes the vector units for its second product instead, key by
    // key and only for the rows that see the key.
    const int seen_first = i0 < p.Q ? seen_of(i0) : 0;  // the fewest keys a row of this wavefront sees
    if (tid < 2) vbad[tid] = 0;
    if (seen_wg > 0) fetch(0);
    for (int j0 = 0; j0 < seen_wg; j0 += kTile) {
        const int parity = (j0 / kTile) & 1;
        __syncthreads();  // everyone has read the tile before
        stage(parity);
        __syncthreads();
        if (tid == 0) vbad[parity ^ 1] = 0;  // read last before the first barrier above, set next behind it a tile on
        if (j0 + kTile < seen_wg) fetch(j0 + kTile);
        if (j0 >= seen_wave) continue;  // nothing of this tile is seen by this wavefront's rows (uniform)
        const bool by_key = vbad[parity] != 0 && j0 + kTile > seen_first;

        // scores, transposed (K . Q^T): register e is key j0 + 8 (e / 4) + 4 hi + e % 4 against this lane's row
        f32x16 s;
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = 0.f;
#pragma unroll
        for (int f = 0; f < D / 2; f++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(ks[r32 * KS + 2 * f + hi], qreg[f], s, 0, 0, 0);
        float mx = -__builtin_inff();
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int j = j0 + 8 * (e >> 2) + 4 * hi + (e & 3);
            s[e] = j < seen ? s[e] : -__builtin_inff();
            mx = fmaxf(mx, s[e]);
        }
        mx = fmaxf(mx, other_half(mx, lane));
        const float mn = fmaxf(m, mx);
        float al = 1.f, sum = 0.f;
        if (mn > -__builtin_inff()) {  // the row has seen a key by now
            al = __builtin_expf(m - mn);
#pragma unroll
            for (int e = 0; e < 16; e++) {
                s[e] = __builtin_expf(s[e] - mn);
                sum += s[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] = 0.f;
        }
        l = l * al + sum;
        m = mn;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[t][e] = o[t][e] * al;
        // result, transposed (V^T . P^T) over the tile's keys in the order the scores' registers hold them: step f takes
        // key 8 (f / 4) + 4 hi + f % 4 from each half, whose weight for this lane's row is register f
        if (!by_key) {
#pragma unroll
            for (int f = 0; f < kTile / 2; f++) {
                const int key = 8 * (f >> 2) + 4 * hi + (f & 3);
#pragma unroll
                for (int t = 0; t < NT; t++) o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vs[key * D + 32 * t + r32], s[f], o[t], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const float theirs = other_half(s[e], lane);
#pragma unroll
                for (int hk = 0; hk < 2; hk++) {  // the key that register e holds in the lanes of half hk
                    const int key = 8 * (e >> 2) + 4 * hk + (e & 3);
                    const float pk = hi == hk ? s[e] : theirs;
                    if (j0 + key < seen) {
#pragma unroll
                        for (int t = 0; t < NT; t++)
#pragma unroll
                            for (int g = 0; g < 4; g++) {
                                const f32x4 vv = *(const f32x4*)(vs + key * D + 32 * t + 8 * g + 4 * hi);
#pragma unroll
                                for (int c = 0; c < 4; c++) o[t][4 * g + c] = __builtin_fmaf(pk, vv[c], o[t][4 * g + c]);
                            }
                    }
                }
            }
        }
    }

    l += other_half(l, lane);
    if (row >= p.Q) return;
    float* orow = out + b * p.o_b + (int64_t)h * p.o_h + (int64_t)row * p.o_i;
    const float inv = l == 0.f ? 0.f : 1.0f / l;
    const bool wide = (((uintptr_t)orow) & 15) == 0;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4 r;
#pragma unroll
            for (int c = 0; c < 4; c++) r[c] = l == 0.f ? 0.f : o[t][4 * g + c] * inv;
            float* dst = orow + 32 * t + 8 * g + 4 * hi;
            if (wide) *(f32x4*)dst = r;
            else
#pragma unroll
                for (int c = 0; c < 4; c++) dst[c] = r[c];
        }
    if (lse && hi == 0) lse[((int64_t)b * p.H + h) * p.Q + row] = l == 0.f ? -__builtin_inff() : m + __builtin_logf(l);
}

template <typename KV, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES, (sizeof(KV) == 4 && D == 128 && WAVES == 2) ? 1 : 2) void attn_prompt_kernel(const float* __restrict__ q, const KV* __restrict__ k,
                                                                                                                     const KV* __restrict__ v, float* __restrict__ out,
                                                                                                                     float* __restrict__ lse, PromptParams p) {
    __shared__ float ks[kTile * Float32Lds<D>::KS];
    __shared__ __align__(16) float vs[kTile * D];
    __shared__ int vbad[2];
    // the grid is (head, sequence, block of rows), the last rows first: under causality they see the most keys, and
    // workgroups are handed out in this order
    rows_by_float32<KV, D, WAVES, WAVES * kRows>(q, k, v, out, lse, p, blockIdx.y, blockIdx.x, (int)(gridDim.z - 1 - blockIdx.z) * WAVES * kRows, ks, vs, vbad);
}

// The same for keys and values in binary16, whose products it makes of bfloat16 parts that add up to their factors, exactly, on instructions sixteen times
// as fast as the float32 one. A key or a value is two (its 11 bits), an element of a row of Q and a weight three (24 bits), and a product is the six of
// theirs: what differs is the order of the float32 sums. Keys are not taken as the binary16 they are: an MFMA cuts its sums off by the exponents of their
// terms, and counts a subnormal's as 2^-14, which is up to 2^-15 of a score of subnormal keys.
//   - scores: a row of Q is scaled by a power of two that takes its largest element to [2^14, 2^15); the products of the upper parts have a sum of their own.
//   - result: weights are 2^64 times what they are, so that the parts of all that a float32 holds are normal numbers.
// A workgroup that finds a NaN or an infinity among its keys and values, or a row of Q with an element other than zero below 2^-114 of its largest, or with a
// largest beyond 2^100 or below 2^-100, starts anew with rows_by_float32 (a layer of 512 rows then takes 98 us, or 126 with an infinity in the last key, for 89 with
// float32 operands alone; of 2048 rows 451, or 580, for 450).
// Against 64 bits the results' error is 0.4 to 0.65 of what it is with float32 operands (1.5e-7 for 3.4e-7 over 512 normal keys, 2.9e-7 for 4.6e-7
// over 2048, 5.2e-7 for 1.2e-6 with scores four times as far apart).
//
// LDS holds a tile's keys row by row, sixteen-byte pieces turned by the row so that 32 rows' equal piece falls on all banks, and its values
// transposed, a feature's 32 keys in the order in which a lane holds its scores (keys 16 u + 8 a + 4 hi + c at 16 u + 8 hi +
// 4 a + c), so that a lane's weights go from the exponential into the second operand; two neighbouring keys' values
// meet in one dword on the way in. The third parts of Q are there too.
//
// What bounds it is a wavefront's chain: some 750 vector instructions a tile (exponentials, masks, parts, staging: 3000 cycles) and the
// 96 MFMAs' 3072 (those on float32 operands would be 8192), and a causal call ends with the rows that walk all keys. So a workgroup is four
// wavefronts of 32 rows each only where there are many (KS = 1), and otherwise (KS = 2) two pairs of wavefronts, 32 rows a pair, that
// take a step's two tiles of keys, one each, and join their maxima, sums and results through LDS at the end: half the chain.
// One layer of 32 heads of 128 features over 8 key heads, us:
//   rows, keys            float32 operands   KS = 1   KS = 2
//   512                         91             65       45
//   2048                       455            276      272
//   5 prompts of 131            35             32       27
//   8 prompts of 512           200            132      159
//   8 heads, 512 of 2048       326            218      137

constexpr float kLog2e = 1.4426950408889634f, kLog2eLow = (float)(1.4426950408889634074 - (double)kLog2e), kLn2 = 0.6931471805599453f;

// 2^up e^x for x <= 0, and for NaN: 2^t with t the float32 next to x / ln 2, times 1 + ln 2 (x / ln 2 - t). Ten instructions where
// the general function, which has overflow to care for, takes fifteen. Not for t below -126, whose 2^t is no normal number.
template <int UP>
__device__ __forceinline__ float exp_down(float x) {
    const float t = x * kLog2e, y = __builtin_ldexpf(__builtin_amdgcn_exp2f(t), UP);
    const float held = fmaxf(x, -128.f), th = held * kLog2e;  // an infinity leaves nothing to mend
    const float rest = __builtin_fmaf(held, kLog2eLow, __builtin_fmaf(held, kLog2e, -th));
    return __builtin_fmaf(y, rest * kLn2, y);
}

// The same for UP = 64 and any x down to where 2^64 e^x is no normal number any more.
__device__ __forceinline__ float exp_far_down(float x) {
    const float t = x * kLog2e, lift = t < -64.f ? 64.f : 0.f, y = __builtin_ldexpf(__builtin_amdgcn_exp2f(t + lift), 64 - (int)lift);  // t + 64 is exact there
    const float held = fmaxf(x, -128.f), th = held * kLog2e;
    const float rest = __builtin_fmaf(held, kLog2eLow, __builtin_fmaf(held, kLog2e, -th));
    return __builtin_fmaf(y, rest * kLn2, y);
}

constexpr float kFar = -80.f;  // e^x of an x above is far from subnormal

template <int D, int KS>
__global__ __launch_bounds__(256, 2) void attn_prompt_half_kernel(const float* __restrict__ q, const uint16_t* __restrict__ k, const uint16_t* __restrict__ v,
                                                                         float* __restrict__ out, float* __restrict__ lse, PromptParams p) {
    constexpr int NT = D / 32;                 // 32-feature tiles of the result
    constexpr int NS = D / 16;                 // steps of the scores' product
    constexpr int PER = D / 8, PD = PER / 2;   // elements, dwords of a key (value) row a thread loads: eight threads a row, a row of each tile
    constexpr int G = 4 / KS;                  // groups of 32 query rows a workgroup
    constexpr int kStep = kTile * KS;          // keys a step
    constexpr int kOwn = KS > 1 && D == 128 ? 1 : 0;  // steps whose third part of Q stays in registers: the LDS has no room for it
    __shared__ union Lds {
        struct {
            uint16_t kv[4][KS][kTile * D];     // upper and lower parts of the step's keys and of its values
            bf16x8 q2[G][NS - kOwn][64];       // the third part of a group's rows, a lane's eight features of each step of the scores' product
        };
        struct {
            float results[KS > 1 ? G : 1][16 * NT * 64];
            float ml[KS > 1 ? G : 1][2][64];   // maximum and sum of the rows' second half of the keys
        };
        Float32Lds<D> by_float32;
    } lds;
    static_assert(sizeof(Lds) + 64 <= 80 * 1024, "two workgroups a compute unit");
    __shared__ int odd;                        // whether the products of float32 operands are to be taken
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r32 = lane & 31, hi = lane >> 5, half = wave % KS;
    const int b = blockIdx.y, h = blockIdx.x, hk = h / (p.H / p.HK), bx = (int)(gridDim.z - 1 - blockIdx.z);  // the last rows first
    const int i0 = (bx * G + wave / KS) * kRows;
    const int64_t Kt = p.K;
    auto seen_of = [&](int i) -> int {  // keys row i sees
        int64_t s = Kt;
        if (p.causal) {
            s = (int64_t)i + p.causal_offset + 1;
            s = s < 0 ? 0 : s > Kt ? Kt : s;
        }
        return (int)s;
    };
    const int last_row_wg = (bx + 1) * G * kRows - 1 < p.Q ? (bx + 1) * G * kRows - 1 : p.Q - 1;
    const int last_row_wave = i0 + kRows - 1 < p.Q ? i0 + kRows - 1 : p.Q - 1;
    const int seen_wg = p.causal ? seen_of(last_row_wg) : (int)Kt;
    const int seen_wave = i0 < p.Q ? (p.causal ? seen_of(last_row_wave) : (int)Kt) : 0;
    const int seen_first = i0 < p.Q ? seen_of(i0) : 0;  // the fewest keys a row of this wavefront sees
    const int row = i0 + r32;
    const int seen = row < p.Q ? seen_of(row) : 0;
    if (tid == 0) odd = 0;
    __syncthreads();

    // this lane's row, scaled: features 16 s + 8 hi .. + 8 of step s as the second operand's parts
    bf16x8 q0[NS], q1[NS], q2_own[kOwn ? kOwn : 1];
    float up = 1.f;  // 2^e
    {
        const float* qr = q + b * p.q_b + (int64_t)h * p.q_h + (int64_t)(row < p.Q ? row : p.Q - 1) * p.q_i + 8 * hi;
        float amax = 0.f;
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int c = 0; c < 8; c++) amax = fmaxf(amax, __builtin_fabsf(qr[16 * s + c] * p.scale));
        amax = fmaxf(amax, other_half(amax, lane));
        bool odd_row = amax != 0.f && !(amax > 0x1p-100f && amax < 0x1p100f);
        asm volatile("" ::: "memory");  // the row is read again, not kept
        const int e = odd_row || amax == 0.f ? 0 : __builtin_amdgcn_frexp_expf(amax) - 15;
        up = __builtin_ldexpf(1.f, e);
#pragma unroll
        for (int s = 0; s < NS; s++) {
            u32x4 part[3];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float a[2];
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float x = qr[16 * s + 2 * i + j] * p.scale;
                    a[j] = __builtin_ldexpf(x, -e);
                    odd_row |= !(x == 0.f || __builtin_fabsf(a[j]) >= 0x1p-100f);
                }
#pragma unroll
                for (int n = 0; n < 3; n++) {
                    part[n][i] = pack_bf16(a[0], a[1]);
                    a[0] -= bf16_lo(part[n][i]);
                    a[1] -= bf16_hi(part[n][i]);
                }
            }
            q0[s] = __builtin_bit_cast(bf16x8, part[0]);
            q1[s] = __builtin_bit_cast(bf16x8, part[1]);
            if (s < kOwn) q2_own[s] = __builtin_bit_cast(bf16x8, part[2]);
            else if (KS == 1 || half == 0) lds.q2[wave / KS][s - kOwn][lane] = __builtin_bit_cast(bf16x8, part[2]);  // the pair's rows are the same
        }
        if (__builtin_amdgcn_ballot_w64(odd_row) != 0 && lane == 0) odd = 1;
    }
    float m = -__builtin_inff(), l = 0.f;  // the row's maximum so far; the sum over the keys this half of the lanes holds
    f32x16 o[NT], zero;                    // the row's result, transposed: register e of tile t is feature 32 t + 8 (e / 4) + 4 hi + e % 4
#pragma unroll
    for (int e = 0; e < 16; e++) zero[e] = 0.f;
#pragma unroll
    for (int t = 0; t < NT; t++) o[t] = zero;

    // a thread's part of a tile's keys and values: rows tid / 8 + 32 n, elements [PER (tid % 8), + PER)
    const int lrow = tid >> 3, lpart = tid & 7;
    const uint16_t* kbase = k + b * p.k_b + (int64_t)hk * p.k_h + PER * lpart;
    const uint16_t* vbase = v + b * p.v_b + (int64_t)hk * p.v_h + PER * lpart;
    u32x4 kreg[KS][PD / 4], vreg[KS][PD / 4];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int n = 0; n < KS; n++) {
            int64_t j = j0 + lrow + kTile * n;
            j = j < Kt ? j : Kt - 1;  // rows past the last key: never seen, loaded from the last one
#pragma unroll
            for (int c = 0; c < PD / 4; c++) {
                kreg[n][c] = ((const u32x4*)(kbase + j * p.k_p))[c];
                vreg[n][c] = ((const u32x4*)(vbase + j * p.v_p))[c];
            }
        }
    };
    auto key_piece = [](int r, int piece) { return D == 128 ? piece ^ (r & 15) : piece ^ ((r >> 1) & 7); };
    auto value_at = [](int f, int slot) { return f * kTile + ((((slot >> 3) ^ ((f >> 2) & 3)) << 3) | (slot & 7)); };
    auto slot_of = [](int key) { return (key & 16) | (key & 4) << 1 | (key & 8) >> 1 | (key & 3); };
    auto stage = [&]() {
        const f16x2 none = {(_Float16)0.f, (_Float16)0.f};
        f16x2 chk = none;  // 0 * each summed: NaN as soon as one is a NaN or an infinity
#pragma unroll
        for (int n = 0; n < KS; n++) {
            uint16_t *kh = lds.kv[0][n], *kl = lds.kv[1][n], *vh = lds.kv[2][n], *vl = lds.kv[3][n];
            const int r = lrow;
#pragma unroll
            for (int c = 0; c < PD / 4; c++) {
                u32x4 upper, lower;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const f16x2 two = as_f16x2(kreg[n][c][i]);
                    const float f0 = (float)two[0], f1 = (float)two[1];
                    upper[i] = pack_bf16(f0, f1);
                    lower[i] = pack_bf16(f0 - bf16_lo(upper[i]), f1 - bf16_hi(upper[i]));
                }
                const int at = r * D + key_piece(r, lpart * (PD / 4) + c) * 8;
                *(u32x4*)(kh + at) = upper;
                *(u32x4*)(kl + at) = lower;
            }
            // the thread eight lanes on has the neighbouring key's same features: of two features, the even key's thread stores the first's two keys
            const int odd = r & 1, slot = slot_of(r & ~1);
#pragma unroll
            for (int w = 0; w < PD; w++) {
                const uint32_t mine = vreg[n][w >> 2][w & 3];
                const uint32_t theirs = __builtin_bit_cast(uint32_t, dpp_f32<0x128>(__builtin_bit_cast(float, mine)));  // row_ror:8
                const uint32_t two = odd ? __builtin_amdgcn_perm(mine, theirs, 0x07060302u) : __builtin_amdgcn_perm(theirs, mine, 0x05040100u);
                const float f0 = (float)as_f16x2(two)[0], f1 = (float)as_f16x2(two)[1];
                const uint32_t upper = pack_bf16(f0, f1), lower = pack_bf16(f0 - bf16_lo(upper), f1 - bf16_hi(upper));
                const int at = value_at(PER * lpart + 2 * w + odd, slot);
                *(uint32_t*)(vh + at) = upper;
                *(uint32_t*)(vl + at) = lower;
                chk = __builtin_bit_cast(f16x2, mine) * none + chk;
                const uint32_t key = kreg[n][w >> 2][w & 3];
                chk = __builtin_bit_cast(f16x2, key) * none + chk;
            }
        }
        const float bad = (float)chk[0] + (float)chk[1];
        if (__builtin_amdgcn_ballot_w64(bad != bad) != 0 && lane == 0) odd = 1;
    };

    const bf16x8* q2 = &lds.q2[wave / KS][0][lane];
    const uint16_t *kh = lds.kv[0][half], *kl = lds.kv[1][half], *vh = lds.kv[2][half], *vl = lds.kv[3][half];
    if (seen_wg > 0) fetch(0);
    bool by_float32 = false;
    for (int jw = 0; jw < seen_wg; jw += kStep) {
        const int j0 = jw + kTile * half;
        __syncthreads();  // everyone has read the tiles before
        stage();
        __syncthreads();
        if (odd != 0) {  // the same for all: it is set before the barrier above or behind the next one
            by_float32 = true;
            break;
        }
        if (jw + kStep < seen_wg) fetch(jw + kStep);
        if (j0 >= seen_wave) continue;  // nothing of this tile is seen by this wavefront's rows (uniform)
        const bool whole = j0 + kTile <= seen_first;

        // scores, transposed (K . Q^T): register e is 2^-e of key j0 + 8 (e / 4) + 4 hi + e % 4 against this lane's row
        f32x16 s = zero, s1 = zero;  // of the upper parts, of the five others
        int k0 = r32 * D + key_piece(r32, hi) * 8;
        asm volatile("" : "+v"(k0));  // eight addresses worked out again for each tile instead of eight registers
#pragma unroll
        for (int f = 0; f < NS; f++) {
            const bf16x8 h8 = *(const bf16x8*)(kh + (k0 ^ 16 * f)), l8 = *(const bf16x8*)(kl + (k0 ^ 16 * f)), q2f = f < kOwn ? q2_own[f < kOwn ? f : 0] : q2[(f - kOwn) * 64];
            s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l8, q2f, s1, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l8, q1[f], s1, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, q2f, s1, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l8, q0[f], s1, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, q1[f], s1, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, q0[f], s, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = s[e] + s1[e];
        float mx = -__builtin_inff(), least = s[0];
#pragma unroll
        for (int e = 1; e < 16; e++) least = fminf(least, s[e]);
        if (!whole) {
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] = 8 * (e >> 2) + (e & 3) < seen - j0 - 4 * hi ? s[e] : -__builtin_inff();
        }
#pragma unroll
        for (int e = 0; e < 16; e++) mx = fmaxf(mx, s[e]);
        mx = fmaxf(mx, other_half(mx, lane)) * up;
        const float mn = fmaxf(m, mx);
        const bool any = mn > -__builtin_inff();  // the row has seen a key by now
        float sum = 0.f;
        if (__builtin_amdgcn_ballot_w64(any && __builtin_fmaf(least, up, -mn) < kFar) == 0) {
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] = exp_down<64>(__builtin_fmaf(s[e], up, -mn));
        } else {  // seldom
#pragma unroll
            for (int e = 0; e < 16; e++) s[e] = exp_far_down(__builtin_fmaf(s[e], up, -mn));
        }
        if (!any) s = zero;
#pragma unroll
        for (int e = 0; e < 16; e++) sum += s[e];
        // in two factors where the first maximum is far below
        const float down = any ? m - mn : 0.f, down0 = fmaxf(down, kFar), down1 = down - down0;
        const float al = exp_down<0>(down0);
        m = mn;
        l = l * al;
        if (__builtin_amdgcn_ballot_w64(al != 1.f) != 0) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[t][e] = o[t][e] * al;
            if (__builtin_amdgcn_ballot_w64(down1 != 0.f) != 0) {
                const float al1 = exp_down<0>(fmaxf(down1, kFar));
                l = l * al1;
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int e = 0; e < 16; e++) o[t][e] = o[t][e] * al1;
            }
        }
        l = l + sum;
        bf16x8 p0[2], p1[2], p2[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            u32x4 a, b, c;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float x = s[8 * u + 2 * i], y = s[8 * u + 2 * i + 1];
                a[i] = pack_bf16(x, y);
                const float x1 = x - bf16_lo(a[i]), y1 = y - bf16_hi(a[i]);
                b[i] = pack_bf16(x1, y1);
                c[i] = pack_bf16(x1 - bf16_lo(b[i]), y1 - bf16_hi(b[i]));
            }
            __builtin_amdgcn_sched_barrier(0);
            p0[u] = __builtin_bit_cast(bf16x8, a), p1[u] = __builtin_bit_cast(bf16x8, b), p2[u] = __builtin_bit_cast(bf16x8, c);
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int at = value_at(32 * t + r32, 16 * u + 8 * hi);
                const bf16x8 h8 = *(const bf16x8*)(vh + at), l8 = *(const bf16x8*)(vl + at);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l8, p2[u], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l8, p1[u], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, p2[u], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l8, p0[u], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, p1[u], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, p0[u], o[t], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (by_float32) {
        __syncthreads();
        rows_by_float32<uint16_t, D, 4, G * kRows>(q, k, v, out, lse, p, b, h, bx * G * kRows, lds.by_float32.ks, lds.by_float32.vs, lds.by_float32.vbad);
        return;
    }

    l += other_half(l, lane);
    if (KS > 1) {  // the second wavefront's half of the keys joins the first's
        float* theirs = lds.results[wave / KS] + lane;
        __syncthreads();
        if (half == 1) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) theirs[64 * (16 * t + e)] = o[t][e];
            lds.ml[wave / KS][0][lane] = m;
            lds.ml[wave / KS][1][lane] = l;
        }
        __syncthreads();
        if (half == 1) return;
        const float m1 = lds.ml[wave / KS][0][lane], l1 = lds.ml[wave / KS][1][lane], mn = fmaxf(m, m1);
        const float d0 = m == mn ? 0.f : m - mn, d1 = m1 == mn ? 0.f : m1 - mn, a0 = exp_down<0>(fmaxf(d0, kFar)), a1 = exp_down<0>(fmaxf(d1, kFar));
        const float b0 = exp_down<0>(fmaxf(d0 - fmaxf(d0, kFar), kFar)), b1 = exp_down<0>(fmaxf(d1 - fmaxf(d1, kFar), kFar));
        l = l * a0 * b0 + l1 * a1 * b1;
        m = mn;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[t][e] = o[t][e] * a0 * b0 + theirs[64 * (16 * t + e)] * a1 * b1;
    }
    if (row >= p.Q) return;
    float* orow = out + b * p.o_b + (int64_t)h * p.o_h + (int64_t)row * p.o_i;
    const float inv = l == 0.f ? 0.f : 1.0f / l;
    const bool wide = (((uintptr_t)orow) & 15) == 0;
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            f32x4 r;
#pragma unroll
            for (int c = 0; c < 4; c++) r[c] = l == 0.f ? 0.f : o[t][4 * g + c] * inv;
            float* dst = orow + 32 * t + 8 * g + 4 * hi;
            if (wide) *(f32x4*)dst = r;
            else
#pragma unroll
                for (int c = 0; c < 4; c++) dst[c] = r[c];
        }
    if (lse && hi == 0) lse[((int64_t)b * p.H + h) * p.Q + row] = l == 0.f ? -__builtin_inff() : m + __builtin_logf(__builtin_ldexpf(l, -64));
}

std::atomic<int> g_prompt{1};  // measurement aid: 0 keeps every call on the kernel that takes a query row a workgroup, 2 those over binary16 on float32 operands

template <typename KV, int WAVES>
hipError_t launch_f32(const AttnArgs& a, const PromptParams& p, hipStream_t st) {
    const dim3 grid((unsigned)a.H, (unsigned)a.B, (unsigned)((a.Q + WAVES * kRows - 1) / (WAVES * kRows))), block(64 * WAVES);
    const KV *k = (const KV*)a.k, *v = (const KV*)a.v;
    if (a.D == 128) hipLaunchKernelGGL((attn_prompt_kernel<KV, 128, WAVES>), grid, block, 0, st, a.q, k, v, a.out, a.lse, p);
    else hipLaunchKernelGGL((attn_prompt_kernel<KV, 64, WAVES>), grid, block, 0, st, a.q, k, v, a.out, a.lse, p);
    return hipGetLastError();
}

template <int KS>
hipError_t launch_f16(const AttnArgs& a, const PromptParams& p, hipStream_t st) {
    constexpr int kWg = 4 / KS * kRows;
    const dim3 grid((unsigned)a.H, (unsigned)a.B, (unsigned)((a.Q + kWg - 1) / kWg)), block(256);
    const uint16_t *k = (const uint16_t*)a.k, *v = (const uint16_t*)a.v;
    if (a.D == 128) hipLaunchKernelGGL((attn_prompt_half_kernel<128, KS>), grid, block, 0, st, a.q, k, v, a.out, a.lse, p);
    else hipLaunchKernelGGL((attn_prompt_half_kernel<64, KS>), grid, block, 0, st, a.q, k, v, a.out, a.lse, p);
    return hipGetLastError();
}

}  // namespace

void set_attention_prompt(int v) { g_prompt = v; }

// Calls this kernel takes: at least 64 query positions, keys and values of 64 or 128 features in float32 or binary16
// whose rows start on 16 bytes (a thread loads an eighth of a row), no additive mask, no device-side key count.
bool attention_prompt_ok(const AttnArgs& a) {
    const int DV = a.DV > 0 ? a.DV : a.D;
    const int esz = a.kv_dtype == kF16 ? 2 : 4;
    if (g_prompt == 0 || a.mask || a.dyn_k || a.Q < 64 || a.K < 1 || DV != a.D || (a.D != 64 && a.D != 128) || (a.kv_dtype != kF16 && a.kv_dtype != kF32) ||
        a.HK <= 0 || a.H % a.HK != 0 || a.B <= 0 || a.B > 65535 || a.H > 65535 || a.Q > (1 << 22) || a.K > (1 << 30))
        return false;
    for (int s = 0; s < 3; s++)
        if ((a.k_strides[s] * esz) % 16 != 0 || (a.v_strides[s] * esz) % 16 != 0) return false;
    return ((uintptr_t)a.k & 15) == 0 && ((uintptr_t)a.v & 15) == 0;
}

hipError_t attention_prompt(const AttnArgs& a, hipStream_t st) {
    PromptParams p;
    p.q_b = a.q_strides[0]; p.q_h = a.q_strides[1]; p.q_i = a.q_strides[2];
    p.k_b = a.k_strides[0]; p.k_h = a.k_strides[1]; p.k_p = a.k_strides[2];
    p.v_b = a.v_strides[0]; p.v_h = a.v_strides[1]; p.v_p = a.v_strides[2];
    p.o_b = a.o_strides[0]; p.o_h = a.o_strides[1]; p.o_i = a.o_strides[2];
    p.B = (int)a.B; p.H = a.H; p.HK = a.HK; p.Q = (int)a.Q; p.K = (int)a.K;
    p.scale = (float)a.scale;
    p.causal = a.causal;
    p.causal_offset = a.causal_offset;
    // where workgroups of 128 rows would be fewer than the device holds at two a compute unit: two wavefronts a workgroup (float32), or
    // two wavefronts on the same rows (binary16; at 512 workgroups the two are level, see the figures there)
    const bool few = a.B * a.H * ((a.Q + 4 * kRows - 1) / (4 * kRows)) < 512;
    note_kernel("attn_prompt_kernel");
    if (a.kv_dtype == kF16 && (a.float32_operands || g_prompt == 2)) return few ? launch_f32<uint16_t, 2>(a, p, st) : launch_f32<uint16_t, 4>(a, p, st);
    if (a.kv_dtype == kF16) return few ? launch_f16<2>(a, p, st) : launch_f16<1>(a, p, st);
    return few ? launch_f32<float, 2>(a, p, st) : launch_f32<float, 4>(a, p, st);
}

}  // namespace mimir
