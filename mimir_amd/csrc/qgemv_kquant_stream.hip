// One to three rows of x by Q4_K or Q6_K weights with a workgroup per compute unit, for
// gfx950: the arithmetic of qgemv_kquant.hip (the CPU's bits: integers exact, a
// row's super-blocks added in their order; backend/cpu/qmatmul.go:141-254), what
// differs is the launch. A lane keeps its part of x in registers for all rows of W
// that its wavefront takes, DEPTH rows of W are under way, and nothing in the loop
// over rows waits for anything but W: a super-block's term goes to LDS, and the
// terms of all of a workgroup's rows are added at the end, a lane a row, where the
// kernel of short workgroups adds a row's one after the other with one lane at work.
// Converted x, us there and here: Q4_K 28672 x 4096 18.9, 14.4 (4.6 TB/s; a large copy 5.1), 14336 x 4096 11.3, 9.1; Q6_K 28672 x 4096 26.7, 21.8. Of a short
// product's 4.5 us 1.5 are any dependent launch's, 1 the trip to memory for x, 0.5 its rounding, 0.5 the sums at the end.
//
// Sixteen lanes (Q4_K) or eight (Q6_K) super-blocks make a load of a wavefront; rows
// of W of more are cut over wavefronts, shorter ones are several rows a load.
//
// So few workgroups can also do for themselves, while their first rows of W are under
// way, what was a launch before the product: the RMSNorm and the rounding of x
// (kHeadNorm), or the rounding alone (kHeadRound). Sixteen lanes round a super-block, so
// that the divisions and the sums over lanes are done for four at once: 56 super-blocks
// by a wavefront each would take a compute unit 2.8 us. As tails they have the residual,
// the rotation with the cache writes, or SiLU(gate) up.
#include <algorithm>

#include "device_util.h"
#include "kernels.h"
#include "kq_act.h"
#include "rope_tail.h"

namespace mimir {

#pragma clang fp contract(off)

namespace {

constexpr int kMostWaves = 16, kFewWaves = 8;  // a workgroup, with one row of x and with more
constexpr int kMostRows = 3;
constexpr int kStride = 256 + 16;    // a super-block's quants of x in LDS
constexpr uint32_t kPast = 1u << 31; // an offset past every buffer: the load is not made
constexpr int kMaxLds = 160 * 1024;
constexpr int64_t kMaxBytes = 1ll << 30;  // from a workgroup's first row of W to its last

enum { kHeadAct = 0, kHeadRound = 1, kHeadNorm = 2 };
enum { kTailPlain = 0, kTailRope = 1, kTailSwiglu = 2 };

struct Job {
    const uint8_t* W;
    const uint8_t* x;      // a converted row, or float32 values; rows x_row bytes apart
    const float* norm_w;
    float* y;
    const float* resid;
    int64_t x_row;
    int N, nsb;            // results; super-blocks of a row
    int rows;              // results a workgroup
    int cuts, each;        // wavefronts a row of W, super-blocks of each
    int packed;            // rows of W a load
    int waves;             // a workgroup
    float inv_d, eps;
    Q4RopeTail rope;
};

template <int DT>
struct Raw;
template <>
struct Raw<kQ4_K> {
    u32x4 hdr, q[2];  // d, dmin and the 12 scale bytes; bytes 16 j .. and 64 + 16 j .. of the nibbles
};
template <>
struct Raw<kQ6_K> {
    u32x4 ql, qh;     // bytes off 4-byte boundaries as the aligned dwords that hold them
    uint32_t ql_top, qh_top, sc[3], d;
};
// A lane's part of x: the chunks of sixteen that its weights of a block are multiplied by, their sums and the scale.
template <int DT>
struct X {
    static constexpr int kChunks = DT == kQ4_K ? 4 : 2;
    u32x4 q[kChunks];
    int s[kChunks];
    float d;
};

// The terms of a row in LDS, a multiple of 16 bytes and that odd, so that lanes that read a row each meet different banks.
template <int DT>
__host__ __device__ constexpr int term_row(int nsb) {
    return 16 * (((DT == kQ4_K ? 8 : 4) * nsb + 15) / 16 | 1);
}

__device__ __forceinline__ uint32_t max16(uint32_t v) {  // over rows of sixteen lanes
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true));
}

// kq_round_superblock's results by sixteen lanes: lane l holds values 64 i + 4 l .. + 3 of the super-block in v[i]. Into LDS.
__device__ __forceinline__ void round_by_sixteen(const f32x4 v[4], int l, uint8_t* q, uint16_t* sums, float* d_out) {
    uint32_t top = 0;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float value = v[i][k];  // a cast of the vector's element in place reads the first of them
            top = max(top, __builtin_bit_cast(uint32_t, value) & 0x7fffffffu);
        }
    top = max16(top);
    const bool finite = top < 0x7f800000u, some = finite && top != 0;
    const float amax = __builtin_bit_cast(float, top);
    const float d = amax / 127.0f, id = 127.0f / amax;
    uint32_t packed[4];
    if (!__any(some && id == __builtin_inff())) {
        // |v id| rounds to at most 127: the sum with 1.5 x 2^23 is the nearest whole number, ties to even, in the lowest bits
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t r[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float t = v[i][k] * id;
                r[k] = __builtin_bit_cast(uint32_t, t + 12582912.0f);
            }
            packed[i] = __builtin_amdgcn_perm(r[1], r[0], 0x0c0c0400u) | __builtin_amdgcn_perm(r[3], r[2], 0x04000c0cu);
        }
    } else {  // a largest value below 127 / (the largest float32): as kq_round_superblock
#pragma unroll
        for (int i = 0; i < 4; i++) {
            packed[i] = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                int r = (int)__builtin_rintf(v[i][k] * id);
                r = r > 127 ? 127 : r < -127 ? -127 : r;
                packed[i] |= (uint32_t)(r & 0xff) << (8 * k);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t p = some ? packed[i] : 0;
        *(uint32_t*)(q + 64 * i + 4 * l) = p;
        const int s16 = dpp_i32_quad_sum(__builtin_amdgcn_sdot4((int)p, 0x01010101, 0, false));
        if ((l & 3) == 0) sums[4 * i + (l >> 2)] = (uint16_t)(int16_t)s16;
    }
    if (l == 0) *d_out = !finite ? __builtin_nanf("") : some ? d : 0.f;
}

// Of the block at `at` from the buffer's start. j: the lane's place among those of a super-block.
__device__ __forceinline__ void fetch(Raw<kQ4_K>& f, __amdgpu_buffer_rsrc_t w, uint32_t at, int j) {
    f.hdr = __builtin_amdgcn_raw_buffer_load_b128(w, at, 0, 0);
    const uint32_t q = at + 16 * j;
    f.q[0] = __builtin_amdgcn_raw_buffer_load_b128(w, q + 16, 0, 0);
    f.q[1] = __builtin_amdgcn_raw_buffer_load_b128(w, q + 80, 0, 0);
}
__device__ __forceinline__ void fetch(Raw<kQ6_K>& f, __amdgpu_buffer_rsrc_t w, uint32_t at, int j) {
    const int n = j >> 2, c = j & 3;
    const uint32_t from = at & ~3u, ql = from + 64 * n + 16 * c, qh = from + 128 + 32 * n + 16 * (c & 1), sc = from + 192 + 8 * n;
    f.ql = __builtin_amdgcn_raw_buffer_load_b128(w, ql, 0, 0);
    f.ql_top = __builtin_amdgcn_raw_buffer_load_b32(w, ql + 16, 0, 0);
    f.qh = __builtin_amdgcn_raw_buffer_load_b128(w, qh, 0, 0);
    f.qh_top = __builtin_amdgcn_raw_buffer_load_b32(w, qh + 16, 0, 0);
#pragma unroll
    for (int i = 0; i < 3; i++) f.sc[i] = __builtin_amdgcn_raw_buffer_load_b32(w, sc + 4 * i, 0, 0);
    f.d = __builtin_amdgcn_raw_buffer_load_b32(w, from + 208, 0, 0);
}

// qdotQ4KGo's integers (qmatmul.go:148-172). Lane j of a super-block: sub-blocks 2 g, 2 g + 1, 2 g + 4, 2 g + 5, g = j / 2, their chunk h = j % 2.
template <int ROWS>
__device__ __forceinline__ void dot(const Raw<kQ4_K>& f, const X<kQ4_K> (&x)[ROWS], uint32_t, int j, int (&sumi)[ROWS], int (&summ)[ROWS]) {
    const int sh = 16 * (j >> 1);
    const uint32_t s0 = f.hdr[1] >> sh, s1 = f.hdr[2] >> sh, s2 = f.hdr[3] >> sh;
    // scale_min_k4 (backend/cpu/quant.go:129-134)
    const int sc_a = s0 & 63, sc_b = (s0 >> 8) & 63, m_a = s1 & 63, m_b = (s1 >> 8) & 63;
    const int sc_c = (s2 & 0xf) | ((s0 >> 2) & 0x30), sc_e = ((s2 >> 8) & 0xf) | ((s0 >> 10) & 0x30);
    const int m_c = ((s2 >> 4) & 0xf) | ((s1 >> 2) & 0x30), m_e = ((s2 >> 12) & 0xf) | ((s1 >> 10) & 0x30);
    int w[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t w0 = f.q[0][i], w1 = f.q[1][i];
        w[0][i] = (int)(w0 & 0x0F0F0F0Fu);
        w[1][i] = (int)((w0 >> 4) & 0x0F0F0F0Fu);
        w[2][i] = (int)(w1 & 0x0F0F0F0Fu);
        w[3][i] = (int)((w1 >> 4) & 0x0F0F0F0Fu);
    }
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        int q[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) q[c] = __builtin_amdgcn_sdot4(w[c][i], (int)x[r].q[c][i], q[c], false);
        // 24-bit multiplies: scales and mins below 64, sums within 16 x 15 x 127
        sumi[r] = dpp_i32_quad_sum(__mul24(sc_a, q[0]) + __mul24(sc_b, q[1]) + __mul24(sc_c, q[2]) + __mul24(sc_e, q[3]));
        summ[r] = dpp_i32_quad_sum(__mul24(m_a, x[r].s[0]) + __mul24(m_b, x[r].s[1]) + __mul24(m_c, x[r].s[2]) + __mul24(m_e, x[r].s[3]));
    }
}
// qdotQ6KGo's (qmatmul.go:180-200). Lane j = 4 n + c: chunks 8 n + c and 8 n + c + 4.
template <int ROWS>
__device__ __forceinline__ void dot(const Raw<kQ6_K>& f, const X<kQ6_K> (&x)[ROWS], uint32_t at, int j, int (&sumi)[ROWS], int (&)[ROWS]) {
    const uint32_t mis = at & 3;
    const int c = j & 3, shl = c & 2;
    int w[2][4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t a = __builtin_amdgcn_alignbyte(i == 3 ? f.ql_top : f.ql[i < 3 ? i + 1 : 3], f.ql[i], mis);
        const uint32_t b = __builtin_amdgcn_alignbyte(i == 3 ? f.qh_top : f.qh[i < 3 ? i + 1 : 3], f.qh[i], mis) >> shl;
        w[0][i] = (int)((a & 0x0F0F0F0Fu) | ((b & 0x03030303u) << 4));  // 0..63 a byte
        w[1][i] = (int)(((a >> 4) & 0x0F0F0F0Fu) | (b & 0x30303030u));
    }
    const uint32_t low = __builtin_amdgcn_alignbyte(f.sc[1], f.sc[0], mis), high = __builtin_amdgcn_alignbyte(f.sc[2], f.sc[1], mis);
    const int sc_l = (int)(int8_t)(low >> (8 * c)), sc_h = (int)(int8_t)(high >> (8 * c));
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
        int dl = 0, dh = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            dl = __builtin_amdgcn_sdot4(w[0][i], (int)x[r].q[0][i], dl, false);
            dh = __builtin_amdgcn_sdot4(w[1][i], (int)x[r].q[1][i], dh, false);
        }
        const int sum = dpp_i32_quad_sum(__mul24(sc_l, dl - 32 * x[r].s[0]) + __mul24(sc_h, dh - 32 * x[r].s[1]));
        sumi[r] = sum + __builtin_amdgcn_update_dpp(0, sum, 0x141, 0xf, 0xf, true);
    }
}

// The lane's part of x of super-block sb, from LDS.
template <int DT>
__device__ __forceinline__ void read_x(X<DT>& x, const uint8_t* q, const uint8_t* sums, const uint8_t* d, int sb, int j) {
    const int first = DT == kQ4_K ? 4 * (j >> 1) + (j & 1) : 8 * (j >> 2) + (j & 3);
    constexpr int kOff[4] = {0, DT == kQ4_K ? 2 : 4, 8, 10};
#pragma unroll
    for (int i = 0; i < X<DT>::kChunks; i++) {
        x.q[i] = *(const u32x4*)(q + sb * kStride + 16 * (first + kOff[i]));
        x.s[i] = ((const int16_t*)sums)[16 * sb + first + kOff[i]];
    }
    x.d = ((const float*)d)[sb];
}

// A row's sum over its super-blocks, in order.
template <int DT>
__device__ __forceinline__ float add_row(const uint8_t* terms, int nsb) {
    constexpr int kBatch = 4, kEach = DT == kQ4_K ? 2 : 4;  // 16-byte reads under way, super-blocks of each
    float acc = 0.f, under = 0.f;
    for (int sb0 = 0; sb0 < nsb; sb0 += kBatch * kEach) {
        f32x4 t[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            const int last = (nsb - 1) / kEach, at = sb0 / kEach + i;
            t[i] = *(const f32x4*)(terms + 16 * (at < last ? at : last));
        }
#pragma unroll
        for (int i = 0; i < kBatch; i++)
#pragma unroll
            for (int k = 0; k < kEach; k++) {
                if (sb0 + i * kEach + k >= nsb) continue;
                if constexpr (DT == kQ4_K) {
                    acc = acc + t[i][2 * k];
                    under = under + t[i][2 * k + 1];
                } else {
                    acc = acc + t[i][k];
                }
            }
    }
    return DT == kQ4_K ? acc - under : acc;
}

constexpr int kDepth = 2;  // rows of W, or packs of them, under way a wavefront

// x's rows converted, end to end in LDS, the terms behind them.
__host__ __device__ __forceinline__ int x_bytes(int nsb) { return (nsb * (kStride + 36) + 15) / 16 * 16; }

template <int DT, int ROWS, int HEAD, int TAIL>
__global__ __launch_bounds__(64 * (ROWS > 1 ? kFewWaves : kMostWaves)) void qgemv_kquant_stream_kernel(Job a) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int BB = DT == kQ4_K ? 144 : 210, kLanes = DT == kQ4_K ? 4 : 8;  // bytes and lanes of a super-block
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), m0 = blockIdx.y;  // several of x only with ROWS 1
    const int nsb = a.nsb, R = a.rows, first = blockIdx.x * R, threads = 64 * a.waves, xb = x_bytes(nsb);
    const int live = a.N - first < R ? a.N - first : R;  // results of a row of x
    const uint8_t* xr = a.x + (int64_t)m0 * a.x_row;
    uint8_t* terms = smem + ROWS * xb;
    const int stride = term_row<DT>(nsb);
    const int local = TAIL == kTailSwiglu ? 2 * R : R;  // rows of W

    // What does not depend on W is requested first: loads come back in order.
    int pos = 0;
    if (TAIL == kTailRope) pos = *a.rope.pos;
    float res = 0.f;  // of the first result that this thread puts together
    const int my_row = ROWS > 1 ? tid / R : 0, my_result = tid - my_row * R;
    if (TAIL == kTailPlain && a.resid && (ROWS > 1 ? my_row < ROWS : tid < R) && my_result < live) res = a.resid[(int64_t)(m0 + my_row) * a.N + first + my_result];
    // Four super-blocks are a wavefront's task. The norm's sums are a row of x for every 256 threads, its tasks from the last wavefront down.
    constexpr int kTurns = HEAD == kHeadNorm ? (ROWS + 1) / 2 : 1;
    const int tasks = (nsb + 3) / 4, l16 = lane & 15;
    const int squares = a.waves / 4, square0 = wave / 4;
    const int sides = HEAD == kHeadNorm ? a.waves / tasks : 1;
    const int task0 = HEAD == kHeadNorm ? (a.waves - 1 - wave) % tasks : wave, side = HEAD == kHeadNorm ? (a.waves - 1 - wave) / tasks : 0;
    f32x4 v[kTurns][4], nw[4];
    float sq[kTurns][16];
    u32x4 xq[ROWS];
    uint32_t xt[ROWS];
    auto request = [&](int task, f32x4 to[4], const float* from) {
        const int sb = 4 * task + (lane >> 4) < nsb ? 4 * task + (lane >> 4) : nsb - 1;
#pragma unroll
        for (int i = 0; i < 4; i++) to[i] = *(const f32x4*)(from + 256 * sb + 64 * i + 4 * l16);
    };
    if constexpr (HEAD == kHeadAct) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            if (tid < 16 * nsb) xq[r] = ((const u32x4*)(xr + r * a.x_row))[tid];
            if (tid < 9 * nsb) xt[r] = ((const uint32_t*)(xr + r * a.x_row + nsb * 256))[tid];
        }
    } else if constexpr (HEAD == kHeadNorm) {
#pragma unroll
        for (int u = 0; u < kTurns; u++)
            if (square0 < squares && square0 + u * squares < ROWS) {
                const float* row = (const float*)(xr + (square0 + u * squares) * a.x_row);
                const int t = tid & 255;
#pragma unroll
                for (int i = 0; i < 16; i++) sq[u][i] = row[t + 256 * i < 256 * nsb ? t + 256 * i : 0];
            }
#pragma unroll
        for (int u = 0; u < kTurns; u++)
            if (side + u * sides < ROWS) request(task0, v[u], (const float*)(xr + (side + u * sides) * a.x_row));
        if (side < ROWS) request(task0, nw, a.norm_w);
    } else if (task0 < tasks) {
        request(task0, v[0], (const float*)xr);
    }

    // This wavefront's rows of W: packs of `packed` rows, every groups-th; this lane's super-block of them
    const int groups = a.waves / a.cuts, group = wave / a.cuts, cut = wave - group * a.cuts;
    const int j = lane & (kLanes - 1), unit = lane / kLanes, in_pack = unit / a.each, sb = cut * a.each + unit - in_pack * a.each;
    const int packs = (local + a.packed - 1) / a.packed;
    const int turns = group < groups ? (packs - group + groups - 1) / groups : 0;
    const bool mine = in_pack < a.packed && sb < nsb;
    const int sbx = sb < nsb ? sb : nsb - 1;
    const uint32_t row_bytes = (uint32_t)(nsb * BB);
    const uint8_t* base = a.W + (int64_t)first * row_bytes;
    const uint32_t lead = DT == kQ4_K ? 0 : (uint32_t)(uintptr_t)base & 3;
    const int64_t left = ((int64_t)(TAIL == kTailSwiglu ? 2 * a.N : a.N) - first) * row_bytes + lead;
    const __amdgpu_buffer_rsrc_t w = buffer_of(base - lead, (uint32_t)(((left < kMaxBytes ? left : kMaxBytes) + 3) & ~3));
    auto place = [&](int turn, int& row) -> uint32_t {  // of this lane's super-block of a turn; row: among the workgroup's
        row = (group + turn * groups) * a.packed + in_pack;
        const bool upper = TAIL == kTailSwiglu && row >= R;
        const int result = upper ? row - R : row;
        const bool there = mine && turn < turns && row < local && result < live;
        const uint32_t at = lead + __umul24((uint32_t)(upper ? a.N + result : result), row_bytes) + (uint32_t)(sb * BB);
        return there ? at : kPast;
    };
    Raw<DT> slot[kDepth];
    int row;
#pragma unroll
    for (int d = 0; d < kDepth; d++) fetch(slot[d], w, place(d, row), j);
    __builtin_amdgcn_sched_barrier(0);

    if constexpr (HEAD == kHeadAct) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const uint8_t* from = xr + r * a.x_row;
            uint8_t* to = smem + r * xb;
            for (int c = tid; c < 16 * nsb; c += threads) *(u32x4*)(to + (c >> 4) * kStride + (c & 15) * 16) = c == tid ? xq[r] : ((const u32x4*)from)[c];
            for (int c = tid; c < 9 * nsb; c += threads) ((uint32_t*)(to + nsb * kStride))[c] = c == tid ? xt[r] : ((const uint32_t*)(from + nsb * 256))[c];
        }
    } else if constexpr (HEAD == kHeadNorm) {  // rmsnorm_kernel's arithmetic (nn/transformer.go:50-61)
        float* part = (float*)terms;
#pragma unroll
        for (int u = 0; u < kTurns; u++)
            if (square0 < squares && square0 + u * squares < ROWS) {
                float ss = 0.f;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float s = sq[u][i] * sq[u][i];
                    ss = ss + ((tid & 255) + 256 * i < 256 * nsb ? s : 0.f);
                }
                ss = wave_sum(ss);
                if (lane == 0) part[4 * (square0 + u * squares) + (wave & 3)] = ss;
            }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int to = 4 * task0 + (lane >> 4);
#pragma unroll
        for (int u = 0; u < kTurns; u++) {
            const int r = side + u * sides;
            if (r >= ROWS) break;
            const float total = (part[4 * r] + part[4 * r + 1]) + (part[4 * r + 2] + part[4 * r + 3]);
            const float ms = total * a.inv_d;
            const float scale = 1.0f / __builtin_sqrtf(ms + a.eps);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float t = v[u][i][k] * scale;
                    v[u][i][k] = t * nw[i][k];
                }
            uint8_t* x = smem + r * xb;
            if (to < nsb) round_by_sixteen(v[u], l16, x + to * kStride, (uint16_t*)(x + nsb * kStride) + 16 * to, (float*)(x + nsb * (kStride + 32)) + to);
        }
    } else {
        for (int task = task0; task < tasks; task += a.waves) {
            if (task != task0) request(task, v[0], (const float*)xr);
            const int to = 4 * task + (lane >> 4);
            if (to < nsb) round_by_sixteen(v[0], l16, smem + to * kStride, (uint16_t*)(smem + nsb * kStride) + 16 * to, (float*)(smem + nsb * (kStride + 32)) + to);
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    X<DT> x[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; r++) read_x<DT>(x[r], smem + r * xb, smem + r * xb + nsb * kStride, smem + r * xb + nsb * (kStride + 32), sbx, j);
    const int pairs = R >> 1;
    float cosine = 1.f, sine = 0.f;
    bool rotates = false;
    const int my_pair = TAIL == kTailRope ? tid % pairs : 0;
    if (TAIL == kTailRope && tid < ROWS * pairs && 2 * my_pair < live) rotates = q4_rope_coeffs(a.rope, pos, first + 2 * my_pair, &cosine, &sine);

    auto multiply = [&](const Raw<DT>& f, int turn) {
        const uint32_t at = place(turn, row);
        int sumi[ROWS], summ[ROWS];
        dot<ROWS>(f, x, at, j, sumi, summ);
        uint32_t dw;
        if constexpr (DT == kQ4_K) dw = f.hdr[0];
        else dw = f.d >> (8 * (at & 3));
        if (j == 0 && at != kPast) {
            uint8_t* to = terms + row * stride + sb * (DT == kQ4_K ? 8 : 4);
#pragma unroll
            for (int r = 0; r < ROWS; r++, to += local * stride) {
                const float dd = f16_bits_to_f32((uint16_t)dw) * x[r].d;
                *(float*)to = dd * (float)sumi[r];
                if (DT == kQ4_K) {
                    const float dm = f16_bits_to_f32((uint16_t)(dw >> 16)) * x[r].d;
                    *(float*)(to + 4) = dm * (float)summ[r];
                }
            }
        }
    };
    // Whole rounds without a branch, so that each wait counts the loads that may still be out; the rest asks for nothing more.
    int t0 = 0;
    for (; t0 + kDepth <= turns; t0 += kDepth) {
#pragma unroll
        for (int d = 0; d < kDepth; d++) {
            multiply(slot[d], t0 + d);
            int ahead;
            fetch(slot[d], w, place(t0 + d + kDepth, ahead), j);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < kDepth - 1; d++) {
        if (t0 + d >= turns) break;
        multiply(slot[d], t0 + d);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (TAIL == kTailRope) {  // pairs of rows
        for (int t = tid; t < ROWS * pairs; t += threads) {
            const int r = t / pairs, pair = t - r * pairs;
            if (2 * pair >= live) continue;
            if (t != tid) rotates = q4_rope_coeffs(a.rope, pos, first + 2 * pair, &cosine, &sine);
            const uint8_t* from = terms + (r * local + 2 * pair) * stride;
            const float p = add_row<DT>(from, nsb), q = add_row<DT>(from + stride, nsb);
            q4_rope_store_with(a.rope, pos, m0 + r, first + 2 * pair, p, q, rotates, cosine, sine, a.y + (int64_t)(m0 + r) * a.N);
        }
        return;
    }
    for (int t = tid; t < ROWS * R; t += threads) {
        const int r = ROWS > 1 ? t / R : 0, result = t - r * R;
        if (result >= live) continue;
        const uint8_t* from = terms + (r * local + result) * stride;
        const int64_t at = (int64_t)(m0 + r) * a.N + first + result;
        float out = add_row<DT>(from, nsb);
        if (TAIL == kTailSwiglu) {
            out = silu_times(out, add_row<DT>(from + R * stride, nsb));
        } else if (a.resid) {
            out = out + (t == tid ? res : a.resid[at]);
        }
        a.y[at] = out;
    }
}

// How a product is laid out: a workgroup a compute unit, more where its rows are more than kMaxRows.
constexpr int kMaxRows = 128, kUnits = 256;
int results_of(int64_t N, bool swiglu) {
    const int64_t turns = (N + (int64_t)kUnits * kMaxRows / (swiglu ? 2 : 1) - 1) / ((int64_t)kUnits * kMaxRows / (swiglu ? 2 : 1));
    const int64_t r = (N + kUnits * turns - 1) / (kUnits * turns);
    return (int)((r + 1) & ~1);
}
int lds_of(int dt, int64_t nsb, int x_rows, int rows) {
    const int64_t terms = dt == kQ4_K ? term_row<kQ4_K>((int)nsb) : term_row<kQ6_K>((int)nsb);
    return (int)std::min<int64_t>(x_rows * (x_bytes((int)nsb) + rows * terms), 1 << 30);
}

template <int DT, int ROWS, int HEAD, int TAIL>
hipError_t launch(const Job& j, int64_t M, hipStream_t st) {
    const auto kernel = qgemv_kquant_stream_kernel<DT, ROWS, HEAD, TAIL>;
    static LdsLimit limit;
    const int lds = lds_of(DT, j.nsb, ROWS, TAIL == kTailSwiglu ? 2 * j.rows : j.rows);
    if (lds > 48 * 1024)
        if (hipError_t e = limit.raise(kMaxLds, {(const void*)kernel})) return e;
    note_kernel("qgemv_kquant_stream_kernel<%d>", ROWS);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((j.N + j.rows - 1) / j.rows), (unsigned)(ROWS > 1 ? 1 : M)), dim3(64 * (unsigned)j.waves), lds, st, j);
    return hipGetLastError();
}
template <int ROWS, int HEAD, int TAIL>
hipError_t launch(int dt, const Job& j, int64_t M, hipStream_t st) {
    return dt == kQ4_K ? launch<kQ4_K, ROWS, HEAD, TAIL>(j, M, st) : launch<kQ6_K, ROWS, HEAD, TAIL>(j, M, st);
}
template <int HEAD, int TAIL>
hipError_t launch_rows(int dt, const Job& j, int64_t M, int x_rows, hipStream_t st) {
    switch (x_rows) {
    case 1: return launch<1, HEAD, TAIL>(dt, j, M, st);
    case 2: return launch<2, HEAD, TAIL>(dt, j, M, st);
    default: return launch<3, HEAD, TAIL>(dt, j, M, st);
    }
}

// The share of the lanes of kFewWaves wavefronts that have a super-block in a turn.
double lanes_used(int dt, int nsb) {
    const int units = dt == kQ4_K ? 16 : 8, cuts = (nsb + units - 1) / units;
    if (cuts == 1) return (double)(units / nsb * nsb) / units;
    return (double)(nsb * (kFewWaves / cuts)) / (units * kFewWaves);
}
int head_of(const QGemvArgs& a, const KqStream& s) { return a.act ? kHeadAct : s.norm_w ? kHeadNorm : kHeadRound; }
// Rows of x a workgroup: all, but for the forms that have one of them a workgroup.
int x_rows_of(const QGemvArgs& a, const KqStream& s) { return a.act && s.rope ? 1 : (int)std::min<int64_t>(a.M, 1 << 16); }

}  // namespace

static std::atomic<int> g_kq_stream{0};  // measurement aid: 1 = never, 4 to 16 = wherever the kernel takes the product, with so many wavefronts a workgroup
void set_kquant_stream(int v) { g_kq_stream = v; }

bool qgemv_kquant_stream_ok(int dt, const QGemvArgs& a, const KqStream& s) {
    if ((dt != kQ4_K && dt != kQ6_K) || a.K <= 0 || a.K % 256 || a.N <= 0 || a.N > (1 << 22) || a.M <= 0 || a.M > 65535) return false;
    const int64_t nsb = a.K / 256, lanes = dt == kQ4_K ? 4 : 8, rows = results_of(a.N, s.swiglu) * (s.swiglu ? 2 : 1);
    const int x_rows = x_rows_of(a, s);
    if (x_rows > kMostRows || (x_rows > 1 && head_of(a, s) == kHeadRound)) return false;
    if (nsb * lanes > 64 * (x_rows > 1 ? kFewWaves : kMostWaves) || ((uintptr_t)a.W & (dt == kQ4_K ? 15 : 1))) return false;
    const int64_t row_bytes = nsb * (dt == kQ4_K ? 144 : 210);
    if ((s.swiglu ? a.N + rows : rows) * row_bytes >= kMaxBytes) return false;
    const int head = head_of(a, s);
    if (head != kHeadAct && (((uintptr_t)a.x & 15) || a.x_row_stride % 4)) return false;
    if (head == kHeadNorm && (nsb > 16 || ((uintptr_t)s.norm_w & 15))) return false;
    if ((s.swiglu && (s.rope || a.resid)) || (head == kHeadRound && s.rope) || (head != kHeadNorm && s.swiglu) || (head == kHeadNorm && !s.swiglu && !s.rope) || (s.rope && a.N % 2)) return false;
    return lds_of(dt, nsb, x_rows, (int)rows) <= kMaxLds;
}

// From a converted row where W has more rows than the kernels of short workgroups can be spread over at once, from float32 x where their rounding of x, by four wavefronts a
// workgroup or a launch of its own, is what takes the time; always where a launch before the product goes with it. us, there | here, converted row: Q4_K 1024 x 4096 3.2 | 3.8,
// 2048 x 2048 3.5 | 3.6, 2500 x 1024 3.9 | 3.4, 4096 x 4096 4.9 | 4.6, 28672 x 4096 18.9 | 14.4, 128256 x 2048 37 | 28; Q6_K 2048 x 4096 4.4 | 4.5, 2048 x 8192 6.8 | 6.4,
// 8192 x 2048 6.0 | 6.0, 28672 x 4096 26.7 | 21.8; float32 x: Q4_K 1024 x 2048 3.45 | 3.60, 512 x 4096 4.1 | 3.8, 2048 x 2048 4.1 | 3.85, 4096 x 14336 13.5 | 10.8;
// Q6_K 2048 x 1024 3.7 | 3.9, 512 x 4096 4.6 | 4.0, 4096 x 14336 16.5 | 14.7. Two and three converted rows where the kernel that reads W once for eight has four wavefronts a workgroup, and where
// enough lanes here have a super-block (K = 4096, 8192 and 14336; of Q4_K as well where W is read by two rows): two rows there | here: Q4_K 8192 x 4096 7.3 | 7.4, 14336 x 4096 12.7 | 10.2, 14336 x
// 14336 35.6 | 26.1, 38912 x 5120 33 | 29, Q6_K 14336 x 4096 16.2 | 13.7, but 20480 x 3072 17.7 | 19.0, 20480 x 5120 27.6 | 30.4; three: Q4_K 14336 x 2048 7.7 | 7.9, 14336 x 4096 12.7 | 11.3, Q6_K
// 14336 x 8192 29.4 | 26.5, but Q4_K 38912 x 5120 33 | 39.3, Q6_K 28672 x 5120 37 | 44; four are level, eight (28672 x 4096 Q4_K 22.4) twice as slow here but with the spills of eight rows in registers.
// A step with its norms here, us, four blocks: two sequences Q4_K of 512, 1024, 2048 and 4096 features 122 | 114, 140 | 126, 163 | 147, 243 | 225, Q6_K 123 | 115, 141 | 131, 189 | 165, 301 | 274; three Q4_K 117 | 115,
// 134 | 128, 163 | 153, 246 | 241, Q6_K 118 | 116, 140 | 132, 174 | 171, 306 | 288, but of 2560 features, whose rows leave three lanes in eight idle, 181 | 185 and 206 | 210; four of 4096 336 | 336.
bool qgemv_kquant_stream_pays(int dt, const QGemvArgs& a, const KqStream& s) {
    if (g_kq_stream == 1 || !kquant_by_rule() || !qgemv_kquant_stream_ok(dt, a, s)) return false;
    if (g_kq_stream) return true;
    const int head = head_of(a, s);
    const double lanes = lanes_used(dt, (int)(a.K / 256));
    if (head == kHeadNorm) return a.M < 3 || lanes >= 0.7;
    if (a.M > 1 && !s.rope) return a.N > 8192 && a.K >= 2048 * (a.M - 1) && (lanes >= 0.8 || (a.M == 2 && (dt == kQ4_K || a.K > 8192)));
    return head == kHeadAct ? a.N > 2048 : a.N * a.K > (2ll << 20) || a.K >= 3072;
}

hipError_t qgemv_kquant_stream(int dt, const QGemvArgs& a, const KqStream& s, hipStream_t st) {
    const int head = head_of(a, s);
    Job j{};
    j.W = (const uint8_t*)a.W;
    j.x = head == kHeadAct ? (const uint8_t*)a.act : (const uint8_t*)a.x;
    j.x_row = head == kHeadAct ? (int64_t)kq_act_bytes(a.K) : a.x_row_stride * 4;
    j.norm_w = s.norm_w;
    j.y = a.y;
    j.resid = a.resid;
    j.N = (int)a.N;
    j.nsb = (int)(a.K / 256);
    j.rows = results_of(a.N, s.swiglu);
    const int units = dt == kQ4_K ? 16 : 8;
    j.cuts = (j.nsb + units - 1) / units;
    j.each = (j.nsb + j.cuts - 1) / j.cuts;
    j.packed = j.cuts == 1 ? units / j.each : 1;
    const int forced = g_kq_stream, x_rows = x_rows_of(a, s);
    // A wavefront for each load of the first turn where they are few. Else eight, which wait for each other less (28672 x 4096 Q4_K 15.0 us, 15.5 with sixteen), but for long rows,
    // whose rounding takes all there are (4096 x 14336 Q4_K 10.8 with sixteen, 11.3 with eight; Q6_K 14.65 with twelve, 14.8, 15.2 with sixteen).
    const int tasks = ((s.swiglu ? 2 : 1) * j.rows + j.packed - 1) / j.packed * j.cuts;
    j.waves = x_rows > 1 ? kFewWaves : forced >= 4 && forced <= kMostWaves ? forced : tasks <= kMostWaves ? std::max(tasks, 8) : j.nsb <= 16 ? 8 : dt == kQ4_K ? kMostWaves : 12;
    j.waves = std::max(j.waves, j.cuts);
    j.inv_d = (float)(1.0 / (double)a.K);
    j.eps = (float)s.eps;
    if (s.rope) j.rope = *s.rope;
    if (s.rope) return head == kHeadAct ? launch<1, kHeadAct, kTailRope>(dt, j, a.M, st) : launch_rows<kHeadNorm, kTailRope>(dt, j, a.M, x_rows, st);
    if (s.swiglu) return launch_rows<kHeadNorm, kTailSwiglu>(dt, j, a.M, x_rows, st);
    return head == kHeadAct ? launch_rows<kHeadAct, kTailPlain>(dt, j, a.M, x_rows, st) : launch<1, kHeadRound, kTailPlain>(dt, j, a.M, st);
}

}  // namespace mimir
