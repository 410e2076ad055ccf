// Products of a few rows of x with Q4_K or Q6_K weights on the int8 matrix cores
// of gfx950, W read once per eight rows of x: the decoding step of a batch of
// sequences for models with K-quant linears. The arithmetic is qdotQ4KGo's and
// qdotQ6KGo's (backend/cpu/qmatmul.go:148-172, 180-200), operation for operation,
// so the results are the CPU's bits like those of the other K-quant kernels
// (qgemv_kquant.hip, qgemm_kquant.hip). Q4_K: per super-block of 256 the integer sums
//   sumi = sum_j sc_j (sub-block j's quants . x),  summ = sum_j m_j (sum of x over sub-block j)
// with the 6-bit scales and mins of scale_min_k4, then in float32
//   dd = d_w d_x, dm = dmin_w d_x, acc += dd float(sumi), accm += dm float(summ)
// over the super-blocks in order, and acc - accm at the end.
//
// x comes rounded to int8 per super-block (kq_convert_act: quants, sums of 16, scale).
//
// What bounds it is W's way into the matrix core's operands. Neighbouring lanes hold neighbouring rows there, and a load whose
// lanes touch a line each costs the cache 64 lookups (x and W loaded so, 4096 x 14336: 16 us), so both come as rows, 16 bytes a lane, and change
// lanes in LDS that is the wavefront's own: no barrier but the one before the sums. A workgroup owns sixteen rows of W, so that a
// matrix of 4096 rows has one for every compute unit, in up to sixteen wavefronts, which take the super-blocks round robin and have all or
// most of theirs under way from the start: with one ahead every second super-block cost a trip to memory. Matrices of up to twice as many
// rows take two tiles of sixteen a workgroup, which share the operand of x, larger ones several workgroups of four wavefronts a compute unit (launch_shape).
//
// The operands are sixteen rows wide: column n of the second is row n of W, row 8 c + m of the first is row m of x with everything but
// group c of the weights zeroed, c = 0 or 1 (those lanes read zeros kept in LDS), so that one instruction keeps two groups of
// weights with scales of their own apart. A lane then has one group's sums for its row of W and four rows of x, times its
// scale; two exchanges between the wavefront's halves add the groups and leave a lane two rows' integer sums. The float32
// terms of all super-blocks meet in LDS, and one thread per output adds them in the super-blocks' order, which is the CPU's.
//
// Measured, us a call on rows already converted, eight rows of x, the form before it (32 rows of W a workgroup in four or eight wavefronts, one
// super-block ahead) and this one: Q4_K 4096 x 14336 20.2 12.2 (loads alone 9.6), 2048 x 8192 10.4 6.4, 6144 x 4096 8.5 6.8, 4096 x 4096 7.0 4.9,
// 28672 x 4096 22.6 20.9-23.5 (66 MB: 3.0 TB/s); Q6_K 4096 x 14336 26.6 14.7 (48 MB: 3.3 TB/s), 2048 x 8192 16.7 9.0, 4096 x 4096
// 11.0 6.1, 28672 x 4096 31.5 27.5.
#include "device_util.h"
#include "kernels.h"
#include "rope_tail.h"

namespace mimir {

#pragma clang fp contract(off)

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 8;    // rows of x a group holds
constexpr uint32_t kBeyond = 1u << 30;  // an offset, or a bit of one, past every buffer's end: the load gives zeros and touches no memory

// The sums of lanes 32 apart: lanes of the lower half get v[0] and v[1] of both, lanes of the upper half v[2] and v[3].
__device__ __forceinline__ void add_halves(const int v[4], int out[2]) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)v[i], (uint32_t)v[i + 2], false, false);
        const uint32_t a = r[0], b = r[1];
        out[i] = (int)(a + b);
    }
}

// Lane numbers: r = lane % 16 is a lane's row of W (and of the first operand: row r % 8 of x, group r / 8), g = lane / 16 its
// quarter of an instruction's K, and of the result rows 4 g..4 g + 3.
//
// A super-block of x in a wavefront's LDS: 256 bytes of zeros (where the lanes of the other group read), quants [8][256] with rows 288
// bytes apart (72 dwords: the eight rows that the lanes of a quarter read fall on different banks), sums [8][16] int16.
constexpr int kXRow = 288, kXq = 256, kXs = kXq + 8 * kXRow, kXBytes = kXs + 256;

// WBlock<DT> says how a row's super-block is cut into 16-byte pieces; operands() reads x's part of the products from LDS, terms() makes the
// float32 terms of row r of W (wl: its super-block in LDS) with rows 4 (g % 2) + 2 (g / 2) and the one after it of x, whose scales are xd.
template <int DT> struct WBlock;

// A 144-byte block is d, dmin, twelve bytes of scales (scale_min_k4, backend/cpu/quant.go:129-134), then four groups of 32 bytes whose
// low nibbles are sub-block 2 p and high nibbles sub-block 2 p + 1. An instruction takes the low (or the high) nibbles of
// two groups, 2 pp and 2 pp + 1: sixteen bytes a lane, 64 in a row of W. The mins' sum m_j (sums of 16) is one
// v_mfma_f32_16x16x16_f16 over the sixteen sums: integers below 2^11 and 2^6, exact, as is their sum.
template <> struct WBlock<kQ4_K> {
    static constexpr int kBytes = 144, kTerms = 2;
    static constexpr int kPieces = 9, kStride = 144;  // rows 36 dwords apart: the 16 lanes of a quarter fall on all 64 banks
    __device__ __forceinline__ static int piece_offset(int c) { return 16 * c; }
    i32x4 x[2][2];
    f16x4 sums;
    __device__ __forceinline__ void operands(const uint8_t* xl, uint32_t r, uint32_t g) {
        const uint8_t* xa = (g >> 1) == (r >> 3) ? xl + kXq + (r & 7) * kXRow + 64 * (g >> 1) + 16 * (g & 1) : xl;
#pragma unroll
        for (int pp = 0; pp < 2; pp++)
#pragma unroll
            for (int hi = 0; hi < 2; hi++) x[pp][hi] = *(const i32x4*)(xa + 128 * pp + 32 * hi);
        const u32x2 sv = *(const u32x2*)(xl + kXs + (r & 7) * 32 + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = sv[i >> 1];
            sums[i] = (_Float16)(int16_t)(v >> (16 * (i & 1)));
        }
    }
    // t[0] = d_w d_x float(sumi), t[1] = dmin_w d_x float(summ)
    __device__ __forceinline__ void terms(const uint8_t* wl, const float xd[2], uint32_t g, float t[kTerms][2]) const {
        const u32x4 hdr = *(const u32x4*)wl;
        u32x4 q[2];
#pragma unroll
        for (int pp = 0; pp < 2; pp++) q[pp] = *(const u32x4*)(wl + 16 + 64 * pp + 16 * g);
        const uint32_t s0 = hdr[1], s1 = hdr[2], s2 = hdr[3];
        // scales and mins 0..3 and 4..7, a byte each
        const uint32_t sc0 = s0 & 0x3f3f3f3fu, sc1 = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
        const uint32_t mn0 = s1 & 0x3f3f3f3fu, mn1 = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
        int sumi[4] = {0, 0, 0, 0};
#pragma unroll
        for (int pp = 0; pp < 2; pp++) {
            const uint32_t sc = (pp ? sc1 : sc0) >> (16 * (g >> 1));  // sub-blocks 4 pp + 2 c and the one after it, c = g / 2
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                i32x4 w;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t qv = q[pp][i];
                    w[i] = (int)((hi ? qv >> 4 : qv) & 0x0F0F0F0Fu);
                }
                const i32x4 c = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[pp][hi], w, i32x4{0, 0, 0, 0}, 0, 0, 0);
                const int s = (int)((sc >> (8 * hi)) & 0xff);
#pragma unroll
                for (int i = 0; i < 4; i++) sumi[i] += __mul24(s, c[i]);  // 24-bit multiplies: |sum| <= 32 * 15 * 127
            }
        }
        // mins 2 g and 2 g + 1 as binary16: the sums of 16 number 4 g.. are theirs
        const uint32_t mn = (g & 2 ? mn1 : mn0) >> (16 * (g & 1));
        f16x4 b;
        b[0] = b[1] = (_Float16)(uint16_t)(mn & 0xff);
        b[2] = b[3] = (_Float16)(uint16_t)((mn >> 8) & 0xff);
        const f32x4 cm = __builtin_amdgcn_mfma_f32_16x16x16f16(sums, b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        int two[2];
        add_halves(sumi, two);
        const uint32_t dd = hdr[0];
        const float dw = f16_bits_to_f32((uint16_t)dd), dmin = f16_bits_to_f32((uint16_t)(dd >> 16));
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float d = dw * xd[i], dm = dmin * xd[i];
            t[0][i] = d * (float)two[i];
            t[1][i] = dm * (g & 2 ? cm[2 + i] : cm[i]);
        }
    }
};

// Q6_K (qdotQ6KGo, backend/cpu/qmatmul.go:180-200): 210-byte blocks, so a row's blocks start on even addresses only and the
// 16-byte loads are unaligned ones: thirteen pieces from the block's start and a fourteenth over its last 16 bytes (194..209), which
// lands behind them in the slab (bytes 208..223 of the row there: the scale d at 222). Half h2 of a super-block (128 weights) is 64
// bytes of ql and 32 of qh: slab s = 0..3 of the half (32 weights) has its low four bits in the low (s < 2) or high nibbles of
// ql[64 h2 + 32 (s & 1) ..] and its upper two at bit 2 s of qh[32 h2 ..]; a scale per chunk of 16, a zero point of 32. An instruction
// takes a slab, eight weights a lane, its two chunks as the two groups. The operand is 4 (q - 32), an int8 (the zero point is a bit
// turned, the shift by two an alignment of the two fields), so the sums of 16 are not needed; the integer sum is shifted
// back at the end, exactly.
template <> struct WBlock<kQ6_K> {
    static constexpr int kBytes = 210, kTerms = 1;
    static constexpr int kPieces = 14, kStride = 240;  // 60 dwords: as above
    __device__ __forceinline__ static int piece_offset(int c) { return c < 13 ? 16 * c : 194; }
    u32x2 x[2][4];
    __device__ __forceinline__ void operands(const uint8_t* xl, uint32_t r, uint32_t g) {
        const uint8_t* xa = (g >> 1) == (r >> 3) ? xl + kXq + (r & 7) * kXRow + 8 * g : xl;
#pragma unroll
        for (int h2 = 0; h2 < 2; h2++)
#pragma unroll
            for (int s = 0; s < 4; s++) x[h2][s] = *(const u32x2*)(xa + 128 * h2 + 32 * s);
    }
    // t[0] = d_w d_x float(sum over the chunks of sc (q - 32) . x)
    __device__ __forceinline__ void terms(const uint8_t* wl, const float xd[2], uint32_t g, float t[kTerms][2]) const {
        const u32x4 sc = *(const u32x4*)(wl + 192);
        int sumi[4] = {0, 0, 0, 0};
#pragma unroll
        for (int h2 = 0; h2 < 2; h2++) {
            const u32x2 ql[2] = {*(const u32x2*)(wl + 64 * h2 + 8 * g), *(const u32x2*)(wl + 64 * h2 + 32 + 8 * g)};
            const u32x2 qh = *(const u32x2*)(wl + 128 + 32 * h2 + 8 * g);
            uint32_t up[2];
#pragma unroll
            for (int i = 0; i < 2; i++) up[i] = qh[i] ^ 0xAAAAAAAAu;  // bit 5 of every weight turned: q - 32
#pragma unroll
            for (int s = 0; s < 4; s++) {
                uint32_t w[2], xa[2];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t lo = ql[s & 1][i];
                    w[i] = ((s < 2 ? lo << 2 : lo >> 2) & 0x3C3C3C3Cu) | ((s < 3 ? up[i] << (6 - 2 * s) : up[i]) & 0xC0C0C0C0u);
                    xa[i] = x[h2][s][i];
                }
                const i32x4 c = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)(((uint64_t)xa[1] << 32) | xa[0]), (long)(((uint64_t)w[1] << 32) | w[0]),
                                                                      i32x4{0, 0, 0, 0}, 0, 0, 0);
                // the scale of chunk 8 h2 + 2 s + c, c = g / 2
                const uint32_t sd = sc[2 * h2 + (s >> 1)] >> (8 * (g >> 1));
                const int scale = (int)(int8_t)(sd >> (16 * (s & 1)));
#pragma unroll
                for (int i = 0; i < 4; i++) sumi[i] += __mul24(scale, c[i]);  // |c| <= 16 * 128 * 127, times 128, sixteen times: below 2^30
            }
        }
        int two[2];
        add_halves(sumi, two);
        const float dw = f16_bits_to_f32(*(const uint16_t*)(wl + 222));
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float dd = dw * xd[i];
            t[0][i] = dd * (float)(two[i] >> 2);
        }
    }
};

// What a lane fetches of a super-block: its pieces of W, and of x for the wavefront's LDS.
template <int LOADS> struct Stage {
    u32x4 w[LOADS];
    u32x4 xq[2];  // two 16-byte pieces of the eight rows' quants
    u32x4 xs;     // a piece of their sums (lanes 0..15 store theirs; Q4_K)
    float xd[2];  // the scales of the rows whose terms this lane makes
};

// kTiles: tiles of sixteen rows of W that share the operand of x. kDepth: super-blocks a wavefront has under way. kRounds: how many
// times that many it takes at most (0: any number; the last requests of a loop of unknown length are for nothing).
// ROPE: W is q | k | v of a decoding step; the rotation and the cache writes ride on the results (rope_kv's arithmetic, interleaved
// pairs), y gets the rotated queries only.
template <int DT, int kTiles, int kWaves, int kDepth, int kRounds, bool ROPE>
__global__ __launch_bounds__(64 * kWaves) void qgemv_kq_rows_kernel(const uint8_t* __restrict__ W, const uint8_t* act, float* y, const float* resid,
                                                                    int M_all, int N, int nsb, int64_t act_row_bytes, int y_bf16, const Q4RopeTail rope) {
    typedef WBlock<DT> WB;
    constexpr int kT = WB::kTerms, kCols = 16 * kTiles, kAll = kCols * WB::kPieces, kLoads = (kAll + 63) / 64, kSlab = kCols * WB::kStride;
    typedef Stage<kLoads> St;
    extern __shared__ __align__(16) uint8_t smem[];  // per wavefront x and the slab of W, then the terms [nsb][kT][8 rows of x][kCols]
    float* terms = (float*)(smem + kWaves * (kXBytes + kSlab));
    const int tid = threadIdx.x;
    const uint32_t lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blockIdx.z: the group of eight rows of x
    const int64_t row0 = (int64_t)kRows * blockIdx.z;
    const int M = M_all - (int)row0 < kRows ? M_all - (int)row0 : kRows;
    const int n0 = blockIdx.x * kCols, left = N - n0 < kCols ? N - n0 : kCols;
    uint8_t* xl = smem + wave * (kXBytes + kSlab);
    uint8_t* slab = xl + kXBytes;
    *(uint32_t*)(xl + 4 * lane) = 0;

    // piece p = 64 i + lane of a super-block of the rows: row p / kPieces, piece p % kPieces of it; rows beyond N repeat the last one
    const uint8_t* wbase = W + (int64_t)n0 * nsb * WB::kBytes;
    uint32_t goff[kLoads], loff[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        int p = 64 * i + lane;
        p = p < kAll ? p : kAll - 1;  // a last load that is not full repeats the last piece in its upper lanes
        const int row = p / WB::kPieces, c = p - WB::kPieces * row;
        goff[i] = (uint32_t)(row < left ? row : left - 1) * (uint32_t)(nsb * WB::kBytes) + WB::piece_offset(c);
        loff[i] = row * WB::kStride + 16 * c;
    }
    // x: rows from M on lie past the buffer's end and read as zeros, as does every super-block past the last one
    const uint32_t xbytes = (uint32_t)act_row_bytes, m0 = 4 * (g & 1) + 2 * (g >> 1);  // m0: the rows of x whose terms this lane makes
    const __amdgpu_buffer_rsrc_t wr = buffer_of(wbase, (uint32_t)(nsb * WB::kBytes) * left), xr = buffer_of(act + row0 * act_row_bytes, xbytes * M);
    const uint32_t xo = (lane >> 4) * xbytes + 16 * r, so = lane < 16 ? (lane >> 1) * xbytes + 16 * (lane & 1) : kBeyond, dof = m0 * xbytes;

    // (every fetch has the same number of loads, and none lies under a branch: the compiler counts those that may still be out)
    auto fetch = [&](St& f, int sb) {
        const uint32_t past = sb < nsb ? 0 : kBeyond;
        const int at = sb < nsb ? sb : nsb - 1;
        const uint8_t* wb = wbase + (int64_t)at * WB::kBytes;
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            if (DT == kQ4_K) f.w[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, goff[i] | past, at * WB::kBytes, 0);
            else __builtin_memcpy(&f.w[i], __builtin_assume_aligned(wb + goff[i], 2), 16);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) f.xq[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, (xo + 4 * i * xbytes) | past, at * 256, 0);
        if (kT == 2) f.xs = __builtin_amdgcn_raw_buffer_load_b128(xr, so | past, nsb * 256 + at * 32, 0);
#pragma unroll
        for (int i = 0; i < 2; i++) f.xd[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, (dof + i * xbytes) | past, nsb * 288 + at * 4, 0));
    };
    auto work = [&](const St& f, int sb) {
        // W and x of the super-block into this wavefront's LDS (its own: a wavefront's LDS operations complete in order)
#pragma unroll
        for (int i = 0; i < kLoads; i++)
            if (64 * (i + 1) <= kAll || (int)lane < kAll - 64 * i) *(u32x4*)(slab + loff[i]) = f.w[i];
#pragma unroll
        for (int i = 0; i < 2; i++) *(u32x4*)(xl + kXq + (4 * i + (lane >> 4)) * kXRow + 16 * r) = f.xq[i];
        if (kT == 2 && lane < 16) *(u32x4*)(xl + kXs + 16 * lane) = f.xs;
        WB b;
        b.operands(xl, r, g);
#pragma unroll
        for (int tile = 0; tile < kTiles; tile++) {
            float t[kT][2];
            b.terms(slab + (16 * tile + r) * WB::kStride, f.xd, g, t);
            float* at = terms + ((sb * kTiles + tile) * 64 + lane) * 2 * kT;
            if constexpr (kT == 2) *(f32x4*)at = f32x4{t[0][0], t[1][0], t[0][1], t[1][1]};
            else *(f32x2*)at = f32x2{t[0][0], t[0][1]};
        }
    };
    // up to a multiple of eight super-blocks with zeros: a sum from zero is never a negative zero, so they change no bit of it
    for (int i = tid; i < (((nsb + 7) & ~7) - nsb) * kTiles * 128 * kT; i += 64 * kWaves) terms[nsb * kTiles * 128 * kT + i] = 0.f;
    St f[kDepth];
#pragma unroll
    for (int u = 0; u < kDepth; u++) {
        fetch(f[u], wave + u * kWaves);
        __builtin_amdgcn_sched_barrier(0);  // in this order: what is requested first returns first
    }
    auto round = [&](int sb0, bool more) {
#pragma unroll
        for (int u = 0; u < kDepth; u++) {
            const int sb = sb0 + u * kWaves;
            if (sb < nsb) work(f[u], sb);       // the same for the whole wavefront
            __builtin_amdgcn_sched_barrier(0);  // one super-block at a time: interleaved they would not fit the registers
            if (more) fetch(f[u], sb + kDepth * kWaves);
        }
    };
    if constexpr (kRounds > 0) {
#pragma unroll
        for (int i = 0; i < kRounds; i++) round(wave + i * kDepth * kWaves, i + 1 < kRounds);
    } else {
        for (int sb0 = wave; sb0 < nsb; sb0 += kDepth * kWaves) round(sb0, true);
    }
    __syncthreads();
    if (tid >= kRows * kCols) return;
    // one thread an output: the CPU's order; the next eight super-blocks' terms are requested before these are added
    float acc[kT], t[2][8][kT];
#pragma unroll
    for (int i = 0; i < kT; i++) acc[i] = 0.f;
    auto request = [&](float (*to)[kT], int sb0) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float* at = terms + ((sb0 + j) * kTiles * 128 + tid) * kT;
            if constexpr (kT == 2) {
                const f32x2 v = *(const f32x2*)at;
                to[j][0] = v[0];
                to[j][1] = v[1];
            } else to[j][0] = *at;
        }
    };
    auto add = [&](const float (*from)[kT]) {
#pragma unroll
        for (int j = 0; j < 8; j++)
#pragma unroll
            for (int i = 0; i < kT; i++) acc[i] = acc[i] + from[j][i];
    };
    request(t[0], 0);
    for (int sb0 = 0;;) {
        if ((sb0 += 8) < nsb) request(t[1], sb0);
        add(t[0]);
        if (sb0 >= nsb) break;
        if ((sb0 += 8) < nsb) request(t[0], sb0);
        add(t[1]);
        if (sb0 >= nsb) break;
    }
    const float v = kT == 2 ? acc[0] - acc[kT - 1] : acc[0];
    // thread 128 tile + 2 lane + j has row m0 + j of x (see terms)
    const int of = (tid & 127) >> 1, m = 4 * ((of >> 4) & 1) + 2 * (of >> 5) + (tid & 1), n = n0 + 16 * (tid >> 7) + (of & 15);
    if constexpr (ROPE) {
        // rows (n, n + 1), n even, are a pair of features: the even row's lane takes its neighbour's result and stores both
        const float other = dpp_f32<0x4e>(v);  // quad_perm [2,3,0,1]
        const int seq = (int)row0 + m;
        if ((n & 1) == 0 && n < N && m < M) q4_rope_store(rope, *rope.pos, seq, n, v, other, y + (int64_t)seq * N);
        return;
    }
    if (n < N && m < M) {
        const int64_t at = (row0 + m) * N + n;
        const float out = resid ? v + resid[at] : v;
        if (y_bf16) ((uint16_t*)y)[at] = f32_to_bf16_bits(out);
        else y[at] = out;
    }
}

}  // namespace

static std::atomic<int> g_kq_rows{0};  // measurement aid: 1 = never, 2 = for any number of rows the kernel takes
void set_kquant_rows(int v) { g_kq_rows = v; }
bool kquant_rows_by_rule() { return g_kq_rows == 0; }

static std::atomic<int> g_kq_rows_waves{0};  // measurement aid: 4, 8 or 16 wavefronts to a workgroup where there is a form of that many
void set_kquant_rows_waves(int v) { g_kq_rows_waves = v == 4 || v == 8 || v == 16 ? v : 0; }

// LDS of a workgroup: per wavefront a super-block of x and the slab of W, and the terms.
static size_t rows_lds(int dt, int64_t nsb, int tiles, int waves) {
    return (size_t)waves * (kXBytes + 16 * tiles * (dt == kQ4_K ? WBlock<kQ4_K>::kStride : WBlock<kQ6_K>::kStride)) +
           (size_t)((nsb + 7) & ~7) * (dt == kQ4_K ? 2 : 1) * kRows * 16 * tiles * sizeof(float);
}

// Rows of x, converted (kq_convert_act); the terms of sixteen rows of W in LDS; Q4_K's W 16-byte aligned, Q6_K's on an even address.
bool qgemv_kquant_rows_ok(int dt, const QGemvArgs& a) {
    const int64_t nsb = a.K / 256;
    return (dt == kQ4_K || dt == kQ6_K) && g_kq_rows != 1 && a.M >= 1 && a.M <= 8 * 65535 && a.act && a.K % 256 == 0 && nsb > 0 &&
           ((uintptr_t)a.W & (dt == kQ4_K ? 15 : 1)) == 0 && ((uintptr_t)a.act & 15) == 0 && a.N > 0 && a.N <= (1ll << 30) &&
           rows_lds(dt, nsb, 1, 4) <= 160 * 1024;
}

// One converted row of bfloat16 x (of float32 x they are qgemv_kquant_stream.hip's): the kernels that give a row of W to a wavefront (qgemv_kquant.hip) have little to read a wavefront where rows are short and many. us, there | here,
// Q4_K: 8192 x 256 5.5 | 4.2, 8192 x 2048 6.2 | 5.5, 12288 x 2048 8.0 | 6.8, 32768 x 2048 17.3 | 13.0, 128256 x 2048 56 | 36; Q6_K: 8192 x 2048 6.0 | 5.9, 12288 x 2048 9.3 | 8.7,
// 32768 x 2048 20.4 | 18.0; but Q6_K 9216 x 2048 7.2 | 7.6, 10240 x 1536 6.8 | 7.0, and of longer rows Q4_K 16384 x 3072 11.2 | 11.9, 4096 x 14336 11.5 | 11.7,
// 4096 x 20480 14.2 | 16.6; Q6_K 4096 x 14336 15.8 | 17.1.
static bool one_row_pays(int dt, const QGemvArgs& a) {
    const int64_t nsb = a.K / 256;
    return nsb <= 8 && a.N >= 8192 && (dt == kQ4_K || nsb <= 5 || a.N == 8192 || a.N >= 11264);
}

// Where it is the faster choice. Two to eight rows always; beyond, by what both kernels take: here 3 us and 0.42 ns (Q4_K; of rows of up to eight super-blocks 0.38) or 0.56 ns
// (Q6_K) per super-block of sixteen rows of W and group of eight rows of x, half of those counted that the last of a workgroup's four wavefronts have less, and a tenth more where
// rows of more than 32 super-blocks leave LDS room for fewer workgroups; the tiled kernel qgemm_kquant_us. On 950 products of 9 to 512 rows, 512 x 1024 to 32768 x 8192
// and 14336 x 14336, the choice takes 0.04 % longer than the faster kernel in the mean, 11 % at most. us, here | there: Q4_K 79 x 5248 x 1024 9.1 | 10.9, 58 x 4160 x 8960 48 | 55, 300 x 1152 x 4096 22.6 | 27,
// 83 x 5632 x 13312 103 | 85, 205 x 2688 x 2560 22.3 | 19.2; Q6_K 25 x 22272 x 2048 25.5 | 31.2, 64 x 5184 x 2048 16.3 | 17.4, 41 x 10432 x 1792 21.0 | 16.0, 98 x 3520 x 3072 21.0 | 23.2.
static double rows_us(int dt, int64_t M, int64_t N, int64_t nsb) {
    const int64_t sixteens = (N + 15) / 16 * ((M + kRows - 1) / kRows);
    const double each = (double)nsb + 0.5 * (double)(-nsb & 3), ns = dt == kQ4_K ? (nsb <= 8 ? 0.378 : 0.42) : 0.56;
    return 3 + (double)sixteens * each * ns * 1e-3 * (nsb > 32 ? 1.1 : 1);
}
bool qgemv_kquant_rows_pays(int dt, const QGemvArgs& a) {
    if (!qgemv_kquant_rows_ok(dt, a)) return false;
    if (a.M == 1) return one_row_pays(dt, a);
    if (g_kq_rows == 2 || a.M <= 8) return true;
    if (a.M > 512) return false;
    const double us = rows_us(dt, a.M, a.N, a.K / 256);
    return us < 3 + 1.4 * (double)(a.K / 256) || us < qgemm_kquant_us(a.M, a.N, a.K);  // no product takes less than one round of short tiles
}
// What 9 to 512 rows take by the one of these two.
double qgemv_kquant_us(int dt, int64_t M, int64_t N, int64_t K) {
    const double us = rows_us(dt, M, N, K / 256);
    return us < 3 + 1.4 * (double)(K / 256) ? us : std::min(us, qgemm_kquant_us(M, N, K));
}

template <int DT, int TILES, int WAVES, int DEPTH, int ROUNDS, bool ROPE>
static hipError_t launch_kq_rows(const QGemvArgs& a, hipStream_t st, bool bf16, const Q4RopeTail* rope) {
    const int nsb = (int)(a.K / 256);
    const auto kernel = qgemv_kq_rows_kernel<DT, TILES, WAVES, DEPTH, ROUNDS, ROPE>;
    static LdsLimit limit;
    if (hipError_t e = limit.raise(160 * 1024, {(const void*)kernel})) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((a.N + 16 * TILES - 1) / (16 * TILES)), 1, (unsigned)((a.M + kRows - 1) / kRows)),
                       dim3(64 * WAVES), rows_lds(DT, nsb, TILES, WAVES), st, (const uint8_t*)a.W, (const uint8_t*)a.act, a.y, a.resid, (int)a.M,
                       (int)a.N, nsb, (int64_t)kq_act_bytes(a.K), bf16 ? 1 : 0, rope ? *rope : Q4RopeTail{});
    return hipGetLastError();
}

// By the super-blocks that a wavefront takes: as many under way as it takes in one round or two, sixteen wavefronts hold two within their 128 registers,
// fewer four. (Three of three: with four asked for, 4 x 12480 x 2304 Q4_K took 10.1 us, so 8.5; four for six, 25 x 12288 x 4608 34.6, three in two rounds 32.0.)
// Two tiles in sixteen or eight wavefronts fit LDS, or are taken, for so few super-blocks that a wavefront has no more than are here.
template <int DT, int TILES, int WAVES, bool ROPE>
static hipError_t launch_depth(const QGemvArgs& a, hipStream_t st, bool bf16, const Q4RopeTail* rope) {
    const int64_t each = (a.K / 256 + WAVES - 1) / WAVES;
    if (each <= 1) return launch_kq_rows<DT, TILES, WAVES, 1, 1, ROPE>(a, st, bf16, rope);
    if constexpr (TILES == 2 && WAVES == 16) return hipErrorInvalidValue;
    else {
        if (each <= 2) return launch_kq_rows<DT, TILES, WAVES, 2, 1, ROPE>(a, st, bf16, rope);
        if constexpr (WAVES == 16) {
            if (each <= 4) return launch_kq_rows<DT, TILES, WAVES, 2, 2, ROPE>(a, st, bf16, rope);
            return launch_kq_rows<DT, TILES, WAVES, 2, 0, ROPE>(a, st, bf16, rope);
        } else {
            if (each == 3) return launch_kq_rows<DT, TILES, WAVES, 3, 1, ROPE>(a, st, bf16, rope);
            if (each == 4) return launch_kq_rows<DT, TILES, WAVES, 4, 1, ROPE>(a, st, bf16, rope);
            if constexpr (WAVES == 4 || DT == kQ4_K)
                if (each <= 6) return launch_kq_rows<DT, TILES, WAVES, 3, 2, ROPE>(a, st, bf16, rope);
            if constexpr (TILES == 1)
                if (each <= 8) return launch_kq_rows<DT, TILES, WAVES, 4, 2, ROPE>(a, st, bf16, rope);
            if constexpr (WAVES == 4) return launch_kq_rows<DT, TILES, WAVES, 4, 0, ROPE>(a, st, bf16, rope);
            else return hipErrorInvalidValue;
        }
    }
}

// By the sixteens of rows of W, times groups of x, and the super-blocks of a row. us a call on converted rows, tiles x wavefronts (a product not named 8 rows):
//   up to 256 sixteens, one workgroup a compute unit: 1 x 16 | 1 x 8 | 1 x 4, 4096 x 14336 Q4_K 12.1 | 13.6 | 13.4, Q6_K 14.7 | 17.3 | 15.9
//   up to 512, two tiles: Q4_K 2 x 16 while it fits (16 super-blocks), 6144 x 4096 6.9, 2 x 8 7.4; then 2 x 8: 2 x 6912 x 4608 9.0, 2 x 4 10.7, 1 x 4 9.4; of more
//     than 48 super-blocks 2 x 4: 4 x 7296 x 13824 20.0, 1 x 4 20.5. Q6_K 2 x 8 to 32 super-blocks: 8 x 8192 x 7168 17.4, 2 x 4 18.5; then 2 x 4: 4 x 4352 x 12544 21.8, 1 x 4 24.9
//   beyond, one tile, so that three to five workgroups share a unit: 1 x 4 | 2 x 4, Q4_K 16 x 13568 x 7424 32.2 | 44.7, 88 x 4032 x 7936 43.1 | 66.1, 8 x 12032 x 4096
//     11.7 | 13.3; Q6_K 4 x 8512 x 6400 20.1 | 23.5, 72 x 3776 x 7936 44.2 | 53.3. Two tiles where the operand of x that they share is what counts: short rows by many groups (Q4_K 188
//     x 960 x 1536 1 x 4 9.0 | 2 x 4 8.5, 61 x 2688 x 1536 7.6 | 7.1; 45 x 4480 x 1280 8.0 | 8.8) or
//     of up to four super-blocks (1 x 65536 x 1024 15.0 | 14.2) or of sixteen, four to each wavefront (32 x 28672 x 4096 60.4 | 58.2, 64 x 4096 x 4096 17.8 | 16.9), short rows of Q6_K from 1200 sixteens on (1 x 20480 x 2048 12.7 | 12.4, 159 x 10560 x 1792 60.7 | 55.3; 30 x 4416 x 1536, 1104 of them,
//     8.9 | 10.0); and where one tile a workgroup is a second round and two are not: LDS has room for five of a unit of up to eight super-blocks (Q4_K 1 x 24576 x 1024
//     7.2 | 6.5) and for three of 17 to 24 (Q4_K 162 x 704 x 5120 14.8 | 14.3) or more than 32 (Q6_K 22 x 5120 x 9216 36.6 | 35.1).
template <int DT, bool ROPE>
static hipError_t launch_shape(const QGemvArgs& a, hipStream_t st, bool bf16, const Q4RopeTail* rope) {
    const int64_t nsb = a.K / 256, wgs = (a.N + 15) / 16 * ((a.M + kRows - 1) / kRows);
    const int fixed = g_kq_rows_waves;
    auto fits = [&](int tiles, int waves) { return rows_lds(DT, nsb, tiles, waves) <= 160 * 1024 && (fixed == 0 || fixed == waves); };
    if (wgs <= 256 && fits(1, 16)) return launch_depth<DT, 1, 16, ROPE>(a, st, bf16, rope);
    if constexpr (DT == kQ4_K) {
        if (wgs <= 512 && fits(2, 16)) return launch_depth<DT, 2, 16, ROPE>(a, st, bf16, rope);
        if (wgs <= 512 && fits(2, 8)) return launch_depth<DT, 2, 8, ROPE>(a, st, bf16, rope);
        const bool short_rows = nsb <= 8 && ((wgs > 1024 && a.M > 48) || (wgs > 1280 && wgs <= 1536) || (wgs > 2560 && nsb <= 4));
        const bool even = nsb == 16 && wgs >= 1024 && a.M > 24;
        if ((wgs <= 512 || short_rows || even || (wgs > 768 && wgs <= 1024 && nsb > 16 && nsb <= 24)) && fits(2, 4)) return launch_depth<DT, 2, 4, ROPE>(a, st, bf16, rope);
    } else {
        if (wgs <= 512 && nsb <= 32 && fits(2, 8)) return launch_depth<DT, 2, 8, ROPE>(a, st, bf16, rope);
        if ((wgs <= 512 || (wgs > 1200 && nsb <= 8) || (wgs > 768 && wgs <= 1024 && nsb > 32)) && fits(2, 4)) return launch_depth<DT, 2, 4, ROPE>(a, st, bf16, rope);
    }
    return launch_depth<DT, 1, 4, ROPE>(a, st, bf16, rope);
}

// The q | k | v product of a decoding step with the rotation and the cache writes as its tail (see Q4RopeTail; interleaved pairs,
// even widths).
bool qgemv_kquant_rows_rope_ok(int dt, const QGemvArgs& a) { return qgemv_kquant_rows_ok(dt, a) && !a.resid && a.N % 2 == 0; }

hipError_t qgemv_kquant_rows_rope(int dt, const QGemvArgs& a, const Q4RopeTail& rope, hipStream_t st) {
    return dt == kQ4_K ? launch_shape<kQ4_K, true>(a, st, false, &rope) : launch_shape<kQ6_K, true>(a, st, false, &rope);
}

// y_bf16: a.y holds bfloat16, rounded as the results are stored.
hipError_t qgemv_kquant_rows(int dt, const QGemvArgs& a, hipStream_t st, bool y_bf16) {
    return dt == kQ4_K ? launch_shape<kQ4_K, false>(a, st, y_bf16, nullptr) : launch_shape<kQ6_K, false>(a, st, y_bf16, nullptr);
}

}  // namespace mimir
