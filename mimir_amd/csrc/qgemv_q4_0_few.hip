// Two to four rows of x by Q4_0 weights with a workgroup per compute unit, for gfx950:
// the integers and a block's float32 operations of one row's kernel (qgemv_q4_0_stream.hip,
// io/mim/dtype.go:118-123 and backend/cpu/gemv.go:73-104) for each row of x, W read once; the blocks'
// sums are within rounding of its (lanes and cuts of a row of W are other ones).
//
// The kernel that reads W once for eight rows (qgemv_q4_0_rows.hip) has 32 rows of W a
// workgroup, so that 4096 rows of W are half the compute units, and works on eight rows of x
// whatever their number. Here eight wavefronts of 256 registers keep the digits of up to four rows
// of x for their pairs of blocks, 50 registers a row, and walk the rows of W, two of them
// under way a wavefront; a row of W costs them some 70 vector instructions a row of
// x, which up to three rows hide behind W's loads. Rows of W longer than 64 pairs of
// blocks are cut over wavefronts. Results meet in LDS; a thread adds a result's cuts in order.
//
// As its first phase it takes the conversion of x, where the rows' digits fit LDS beside each other. For
// a step of two sequences x may come converted, with the residual as tail, or be normalized
// first, with the rotation and the cache writes or SiLU(gate) up as tails: 32 steps of two sequences of four
// blocks of 4096 features 11.4 -> 9.5 ms (of three 11.7 -> 11.3, of 2048 features 7.0 -> 7.4; of four 12.0 -> 13.1).
#include <algorithm>

#include "device_util.h"
#include "kernels.h"
#include "q4_act.h"
#include "q4_job.h"
#include "rope_tail.h"

namespace mimir {

namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves, kDepth = 2, kMostRows = 4;
constexpr int kMaxLds = 160 * 1024;

struct Few {
    const uint8_t* W[3];  // q, k, v; gate, up; or one matrix
    int n[3];
    const uint8_t* x;     // converted rows or float32 ones, x_row bytes apart
    const float* norm_w;
    float* y;
    const float* resid;
    int64_t x_row;
    int N, nb;            // results, blocks of a row
    int rows;             // results a workgroup
    int cuts, each;       // wavefronts a row of W, pairs of blocks of each
    float inv_d, eps;
    Q4RopeTail rope;
};
enum { kTailPlain = 0, kTailRope = 1, kTailSwiglu = 2 };

template <int ROWS, int HEAD, int TAIL>
__global__ __launch_bounds__(kThreads) void qgemv_q4_0_few_kernel(Few a) {
    extern __shared__ u32x4 smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = a.nb, nbp = nb | 1, npairs = nb >> 1, nq = nb * 4, R = a.rows, first = blockIdx.x * R;
    const int live = a.N - first < R ? a.N - first : R, local = TAIL == kTailSwiglu ? 2 * R : R;
    const int x16 = (int)(q4_0_act_row_bytes((int64_t)nb * 32) >> 4);  // 16-byte pieces of a converted row
    float* part = (float*)(smem + (HEAD == kHeadAct ? 0 : ROWS * x16));   // [row of W][cut][row of x]
    const uint32_t row_bytes = (uint32_t)nb * 18;

    // ---- requests, in the order in which they are wanted ----
    int pos = 0;
    if (TAIL == kTailRope) pos = *a.rope.pos;
    float res = 0.f;  // of the result that this thread puts together first
    const int my_row = tid / R, my_result = tid - my_row * R;
    if (TAIL == kTailPlain && a.resid && my_row < ROWS && my_result < live) res = a.resid[(int64_t)my_row * a.N + first + my_result];
    constexpr int kTurns = (ROWS + 1) / 2;  // of the two halves of the workgroup that normalize a row of x each
    const int half = wave >> 2, t256 = tid & 255;
    NormRow norm_row[HEAD == kHeadNorm ? kTurns : 1];
    float squares[kTurns];
    if constexpr (HEAD == kHeadNorm) {
#pragma unroll
        for (int u = 0; u < kTurns; u++)
            if (half + 2 * u < ROWS) squares[u] = norm_load(norm_row[u], (const float*)(a.x + (half + 2 * u) * a.x_row), a.norm_w, nq, t256);
    }
    const int item = tid < nq ? tid : nq - 1;
    f32x4 lo[ROWS], hi[ROWS];
    if constexpr (HEAD == kHeadConvert) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const float* row = (const float*)(a.x + r * a.x_row) + 32 * (item >> 2) + 4 * (item & 3);
            __builtin_memcpy(&lo[r], row, 16);
            __builtin_memcpy(&hi[r], row + 16, 16);
        }
    }
    const int groups = kWaves / a.cuts, group = wave / a.cuts, cut = wave - group * a.cuts;
    const int own = cut * a.each + lane;
    const bool mine = lane < a.each && own < npairs;
    const int p = mine ? own : 0;
    const int turns = group < groups ? (local - group + groups - 1) / groups : 0;
    u32x4 d0[ROWS][kDigits], d1[ROWS][kDigits];
    float s0[ROWS], s1[ROWS];
    auto read_x = [&](int r, const u32x4* plane) {
#pragma unroll
        for (int j = 0; j < kDigits; j++) {
            d0[r][j] = plane[j * nbp + 2 * p];
            d1[r][j] = plane[j * nbp + 2 * p + 1];
        }
        const float* scale = (const float*)(plane + kDigits * nbp);
        s0[r] = scale[2 * p];
        s1[r] = scale[2 * p + 1];
    };
    if constexpr (HEAD == kHeadAct) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) read_x(r, (const u32x4*)(a.x + r * a.x_row));
    }
    auto fetch = [&](PairRegs& t, int turn) {  // past the last turn, or of a result that there is none of, nothing is read
        const int row = group + turn * groups, result = TAIL == kTailSwiglu && row >= R ? row - R : row;
        const bool there = turn < turns && result < live;
        int g = first + (there ? result : 0);
        const uint8_t* W = a.W[0];
        if (TAIL == kTailSwiglu && row >= R) W = a.W[1];
        if (TAIL == kTailRope) {
            if (g >= a.n[0] + a.n[1]) g -= a.n[0] + a.n[1], W = a.W[2];
            else if (g >= a.n[0]) g -= a.n[0], W = a.W[1];
        }
        const __amdgpu_buffer_rsrc_t w = buffer_of(W + (int64_t)g * row_bytes, there ? row_bytes : 0);
        const uint32_t at = mine ? 36u * (uint32_t)p : 1u << 31;
        t.a = __builtin_amdgcn_raw_buffer_load_b128(w, at, 0, 0);
        t.b = __builtin_amdgcn_raw_buffer_load_b128(w, at + 16, 0, 0);
        t.c = __builtin_amdgcn_raw_buffer_load_b32(w, at + 32, 0, 0);
    };
    PairRegs slot[kDepth];
#pragma unroll
    for (int d = 0; d < kDepth; d++) fetch(slot[d], d);
    __builtin_amdgcn_sched_barrier(0);

    // ---- x into LDS in its fixed-point form ----
    if constexpr (HEAD == kHeadNorm) {
#pragma unroll
        for (int u = 0; u < kTurns; u++)
            if (half + 2 * u < ROWS) {
                const float ss = wave_sum(squares[u]);
                if (lane == 0) part[4 * (half + 2 * u) + (wave & 3)] = ss;
            }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int u = 0; u < kTurns; u++) {
            const int r = half + 2 * u;
            if (r < ROWS) norm_convert(norm_row[u], part + 4 * r, nullptr, smem + r * x16, (float*)(smem + r * x16 + kDigits * nbp), nbp, nq, t256, a.inv_d, a.eps);
        }
    } else if constexpr (HEAD == kHeadConvert) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            u32x4* plane = smem + r * x16;
            if (tid < nq) {
                float l[4] = {lo[r][0], lo[r][1], lo[r][2], lo[r][3]}, h[4] = {hi[r][0], hi[r][1], hi[r][2], hi[r][3]};
                q4_convert_item(l, h, plane, (float*)(plane + kDigits * nbp), nbp, tid >> 2, tid & 3);
            }
            for (int t = tid + kThreads; t < nq; t += kThreads) {  // whole blocks: four consecutive items
                const float* row = (const float*)(a.x + r * a.x_row) + 32 * (t >> 2) + 4 * (t & 3);
                f32x4 vl, vh;
                __builtin_memcpy(&vl, row, 16);
                __builtin_memcpy(&vh, row + 16, 16);
                float l[4] = {vl[0], vl[1], vl[2], vl[3]}, h[4] = {vh[0], vh[1], vh[2], vh[3]};
                q4_convert_item(l, h, plane, (float*)(plane + kDigits * nbp), nbp, t >> 2, t & 3);
            }
        }
    }
    if constexpr (HEAD != kHeadAct) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int r = 0; r < ROWS; r++) read_x(r, smem + r * x16);
    }
    const int pairs = R >> 1, my_pair = TAIL == kTailRope ? tid % pairs : 0;
    float cosine = 1.f, sine = 0.f;
    bool rotates = false;
    if (TAIL == kTailRope && tid < ROWS * pairs && 2 * my_pair < live) rotates = q4_rope_coeffs(a.rope, pos, first + 2 * my_pair, &cosine, &sine);

    auto multiply = [&](const PairRegs& t, int turn) {
        const int row = group + turn * groups;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const float sum = wave_sum(pair_term(t, d0[r], d1[r], s0[r], s1[r], mine));
            if (lane == 0) part[(row * a.cuts + cut) * ROWS + r] = sum;
        }
    };
    int t0 = 0;
    for (; t0 + kDepth <= turns; t0 += kDepth) {  // whole rounds, without a branch between the loads
#pragma unroll
        for (int d = 0; d < kDepth; d++) {
            multiply(slot[d], t0 + d);
            fetch(slot[d], t0 + d + kDepth);
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
    auto sum_of = [&](int row, int r) {
        float s = part[row * a.cuts * ROWS + r];
        for (int c = 1; c < a.cuts; c++) s = s + part[(row * a.cuts + c) * ROWS + r];
        return s;
    };
    if constexpr (TAIL == kTailRope) {
        for (int t = tid; t < ROWS * pairs; t += kThreads) {
            const int r = t / pairs, pair = t - r * pairs;
            if (2 * pair >= live) continue;
            if (t != tid) rotates = q4_rope_coeffs(a.rope, pos, first + 2 * pair, &cosine, &sine);
            q4_rope_store_with(a.rope, pos, r, first + 2 * pair, sum_of(2 * pair, r), sum_of(2 * pair + 1, r), rotates, cosine, sine, a.y + (int64_t)r * a.N);
        }
        return;
    }
    for (int t = tid; t < ROWS * R; t += kThreads) {
        const int r = t / R, result = t - r * R;
        if (result >= live) continue;
        const int64_t at = (int64_t)r * a.N + first + result;
        float out = sum_of(result, r);
        if (TAIL == kTailSwiglu) {
            out = silu_times(out, sum_of(R + result, r));
        } else if (a.resid) {
            out = out + (t == tid ? res : a.resid[at]);
        }
        a.y[at] = out;
    }
}

constexpr int kUnits = 256;
int results_of(int64_t N) { return (int)(((N + kUnits - 1) / kUnits + 1) & ~1); }
int64_t lds_of(int64_t K, int rows, int head, int local, int cuts) {
    const int64_t x = head == kHeadAct ? 0 : rows * (int64_t)q4_0_act_row_bytes(K);
    return x + std::max<int64_t>((int64_t)local * cuts * rows * 4, 4 * 4 * rows);
}

template <int ROWS, int HEAD, int TAIL>
hipError_t launch(const Few& f, hipStream_t st) {
    const auto kernel = qgemv_q4_0_few_kernel<ROWS, HEAD, TAIL>;
    static LdsLimit limit;
    const int lds = (int)lds_of((int64_t)f.nb * 32, ROWS, HEAD, TAIL == kTailSwiglu ? 2 * f.rows : f.rows, f.cuts);
    if (lds > 48 * 1024)
        if (hipError_t e = limit.raise(kMaxLds, {(const void*)kernel})) return e;
    note_kernel("qgemv_q4_0_few_kernel<%d>", ROWS);
    hipLaunchKernelGGL(kernel, dim3((unsigned)((f.N + f.rows - 1) / f.rows)), dim3(kThreads), lds, st, f);
    return hipGetLastError();
}
int head_of(const QGemvArgs& a, const Q4Few& q) { return a.act ? kHeadAct : q.norm_w ? kHeadNorm : kHeadConvert; }

}  // namespace

static std::atomic<int> g_few{0};  // measurement aid: 1 = never, 2 = wherever the kernel takes the product
void set_q4_few(int v) { g_few = v; }
bool q4_0_few_on() { return g_few != 1; }

bool qgemv_q4_0_few_ok(const QGemvArgs& a, const Q4Few& q) {
    const int64_t npairs = a.K / 64;
    if (a.M < 2 || a.M > kMostRows || a.K <= 0 || a.K % 64 || npairs > 64 * kWaves || a.N <= 0 || a.N > (1 << 24) || a.K > (1 << 20)) return false;
    const void* W[3] = {a.W, q.W1, q.W2};
    for (const void* w : W)
        if ((uintptr_t)w & 3) return false;
    const int head = head_of(a, q), cuts = (int)((npairs + 63) / 64), R = results_of(a.N);
    if (a.M > 2 && head != kHeadConvert) return false;
    if (head != kHeadAct && (((uintptr_t)a.x & 15) || a.x_row_stride % 4)) return false;
    if (head == kHeadNorm && (!q4_0_norm_head_ok(a.K) || ((uintptr_t)q.norm_w & 15))) return false;
    if (q.rope && (a.N % 2 || q.n0 % 2 || q.n1 % 2)) return false;
    if ((q.rope || q.swiglu) != (head == kHeadNorm) || ((q.rope || q.swiglu) && a.resid)) return false;
    return lds_of(a.K, (int)a.M, head, q.swiglu ? 2 * R : R, cuts) <= kMaxLds;
}
// float32 x. A turn of a workgroup's wavefronts takes as long however many of their lanes have a pair of blocks, and a row of x more as much again, where the kernel for eight rows takes
// what W's bytes take: here where that share of the lanes is large, or the rows of W are few. us, there | here, of all lanes (K = 4096, 8192 of them): two rows 4096 x 4096 9.6 | 5.6, 14336 x
// 4096 16.6 | 10.3; three 8192 x 4096 12.2 | 9.3, 28672 x 8192 44 | 36; four 4096 x 4096 9.7 | 8.7, but 38912 x 4096 31.3 | 31.9, 14336 x 8192 26.3 | 29.5. Of less than half of them, two
// rows 5120 x 256 5.4 | 5.2, 11008 x 1024 10.0 | 8.8, 14336 x 1536 10.1 | 9.4, but 8192 x 256 5.5 | 6.8, 28672 x 1024 12.0 | 16.6; three 2048 x 256 5.3 | 5.1, 4096 x 1024 6.5 | 6.5, 6144 x 2048 8.1 | 7.5, but
// 28672 x 2048 15.9 | 17.6; four 1024 x 512 5.6 | 5.3, 4096 x 2048 7.9 | 7.7. Of 0.63 to 0.75 (K = 5120, 6144, 11008): two rows 14336 x 5120 19.2 | 16.9; three 3072 x 5120 10.5 | 9.8, but 14336 x 5120
// 19.2 | 22.1, 38912 x 11008 75 | 90; four 1024 x 11008 13.0 | 11.8, but 3072 x 11008 15.8 | 19.5. K = 3072, whose rows fit a wavefront: three 14336 x 3072 13.3 | 12.6, four 4096 x 3072 8.8 | 8.7, but 128256 x 3072 71 | 94.
// All that where K is a multiple of 256, whole runs of that kernel; else it takes up to twice as long: two 32704 x 640 17.7 | 18.5, 22528 x 11072 66 | 32; three 18688 x 448 17.4 | 14.0, 16640 x 14528 104 | 49,
// but 15962 x 640 14.6 | 18.2; four 2688 x 384 7.7 | 6.6, 25280 x 6592 78 | 46, 11098 x 1728 13.8 | 12.8, but 4608 x 320 7.6 | 8.7, 20544 x 1152 16 | 20.
bool qgemv_q4_0_few_pays(const QGemvArgs& a, const Q4Few& q) {
    if (g_few == 1 || !qgemv_q4_0_few_ok(a, q)) return false;
    if (g_few == 2) return true;
    const int64_t pairs = a.K / 64, cuts = (pairs + 63) / 64;
    const double lanes = (double)(pairs * (kWaves / cuts)) / (64 * kWaves);  // that work, in the workgroup
    const bool runs = a.K % 256 == 0;
    if (a.M == 2) return !runs || lanes >= 0.5 || (double)a.N <= 4096 + 28000 * lanes;
    if (a.M == 3) {
        if (!runs) return lanes >= 0.25 || a.N <= 12288;
        if (lanes >= (cuts == 1 ? 0.75 : 0.85)) return true;
        return cuts == 1 ? (double)a.N <= 1536 + 10500 * lanes : a.N <= (lanes >= 0.75 ? 4096 : 3072);
    }
    if (!runs) return a.K > 1536 || a.N <= 3072;
    if (lanes >= 1) return a.N <= (cuts == 1 ? 28672 : 2048);
    return cuts == 1 ? (double)a.N <= std::min(4096.0, 600 + 7000 * lanes) : a.N <= (lanes >= 0.75 ? 2048 : 1024);
}

hipError_t qgemv_q4_0_few(const QGemvArgs& a, const Q4Few& q, hipStream_t st) {
    const int head = head_of(a, q), npairs = (int)(a.K / 64);
    Few f{};
    f.W[0] = (const uint8_t*)a.W;
    f.W[1] = (const uint8_t*)q.W1;
    f.W[2] = (const uint8_t*)q.W2;
    f.n[0] = (int)q.n0;
    f.n[1] = (int)q.n1;
    f.x = head == kHeadAct ? (const uint8_t*)a.act : (const uint8_t*)a.x;
    f.x_row = head == kHeadAct ? (int64_t)q4_0_act_bytes(a.K) : a.x_row_stride * 4;
    f.norm_w = q.norm_w;
    f.y = a.y;
    f.resid = a.resid;
    f.N = (int)a.N;
    f.nb = (int)(a.K / 32);
    f.rows = results_of(a.N);
    f.cuts = (npairs + 63) / 64;
    f.each = (npairs + f.cuts - 1) / f.cuts;
    f.inv_d = (float)(1.0 / (double)a.K);
    f.eps = (float)q.eps;
    if (q.rope) f.rope = *q.rope;
    if (q.rope) return launch<2, kHeadNorm, kTailRope>(f, st);
    if (q.swiglu) return launch<2, kHeadNorm, kTailSwiglu>(f, st);
    if (head == kHeadAct) return launch<2, kHeadAct, kTailPlain>(f, st);
    return a.M == 2 ? launch<2, kHeadConvert, kTailPlain>(f, st) : a.M == 3 ? launch<3, kHeadConvert, kTailPlain>(f, st) : launch<4, kHeadConvert, kTailPlain>(f, st);
}

}  // namespace mimir
