// The Q4_0 product of 25 to 256 rows of float32 x by rows of W of more than 2048: x as pairs of binary16, W read where it lies and the
// arithmetic as in qgemm_q4_0_direct.hip, without that kernel's barrier a block. Each of a workgroup's wavefronts has a part of its share of K to itself: up to
// 80 rows of x by 64 of W, in sixteens (v_mfma_f32_16x16x32_f16: a block and half of x an instruction), two sides of 64 by four parts or one by eight.
//
// A wavefront's W comes as whole lines, eight blocks of its 64 rows at a time, straight into LDS of its own, the next eight under way (a lane a row took
// 32 lines a request); x's operands from memory into registers, each asked for again for the next block when it has been read: they lie in
// the order of lanes, 1 KB a load (piece_at). No wait in the loop is for another wavefront, so that the two of a SIMD multiply and unpack in
// turn. The parts' sums meet in LDS at the end, in a loop: as straight code, run once a launch, this took 3 us to fetch.
//
// What bounds it, 77 x 14336 x 4096, 31 us: 5 to 11 us until a wavefront's first 18 KB of W are asked for and there, then 0.65 us a block and SIMD,
// twice its MFMAs (640 cycles) and as much as these and its 140 VALU instructions together; 3.5 us for sums and stores. Whole calls, qgemm_q4_0_direct_kernel and this:
//   32 x 14336 x 4096   32.4 -> 24.4 us   64 x 14336 x 4096  39.7 -> 31.5   77 x 14336 x 4096  46.6 -> 35.3   128 x 14336 x 4096  57.6 -> 50.3
//   77 x 5120 x 5120    32.0 -> 27.8     128 x 5120 x 5120   38.1 -> 35.0  160 x 5120 x 5120   51.6 -> 38.2   96 x 4096 x 4096    29.3 -> 22.3
//   77 x 4096 x 14336   49.3 -> 42.8     160 x 4096 x 14336  88.8 -> 62.2  256 x 4096 x 4096   41.0 -> 32.0
// Error against 64 bits, of the result: 9.6e-8 at 77 x 5120 x 5120 where it was 1.05e-7, 9.4e-8 to 1.25e-7 at the others (9.9e-8 to 1.57e-7).
// Touching x's lines ahead of their loads cost 3 us; six sixteens of rows a wavefront do not fit its registers (96 x 14336 x 4096: 66 us, as two of three 42).
#include "kernels.h"
#include "q4_halves.h"

namespace mimir {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kMostTiles = 5;    // sixteens of rows of x, at most
constexpr int kCols = 4;         // sixteens of rows of W a wavefront: two strips
constexpr int kWaves = 8;        // of a workgroup: one or two sides of two strips by eight or four parts of its share of K
constexpr int kChunk = 8;        // blocks of W that come into LDS together: of a row 144 bytes, nine pieces of sixteen
constexpr int kRowBytes = kChunk * 18, kPieces = kRowBytes / 16, kChunkBytes = 64 * kRowBytes;

struct Plan {
    int sides, groups;         // of two strips of W, of as many sides
    int tiles_m, mt;           // of mt sixteens of rows: 128 rows are one, more than five sixteens of them two of half
    int shares, share_blocks;  // of K; the last share may be shorter, all are even
};

// LDS: a wavefront's two chunks of W, in whose place the parts' sums meet, and x's scales of a pair of blocks where rows have them a block.
constexpr int kScaleFloats = 2 * kMostTiles * 16;
constexpr int kWaveBytes = 2 * kChunkBytes + kScaleFloats * 4;
constexpr int kLdsBytes = kWaves * kWaveBytes;
static_assert(kLdsBytes <= 160 * 1024 && kWaves / 2 * kMostTiles * kCols * 4 * 64 * 4 + kMostTiles * 64 <= kLdsBytes, "LDS of a compute unit");

// A wavefront's sixteen bytes a lane from `from` to lds_base + 16 lane, as load_to_lds with an address a lane.
__device__ __forceinline__ void load_piece(const uint8_t* from, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(from) : "memory");
}

// x's granules as a buffer, so that an address is a lane's offset and a scalar one: 2 VALU instructions a load fewer.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t x_resource(const Operands& o) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)o.X16, 0, ((o.M + 31) / 32) * o.nb * (kGranuleX * 2), 0x00020000);
}

template <int MT>
struct Tile {
    const Operands& o;
    uint8_t* chunks;     // this wavefront's [2][64 rows][144 bytes]
    uint32_t chunks_at;  // its address
    float* scales;       // [2 blocks][16 MT rows]
    int lane, r16, q, m0, b0, count;
    const uint8_t* rows[2];  // the two strips' first rows of W
    int last_row[2];         // of the strip, where the matrix ends in it
    __amdgpu_buffer_rsrc_t x16;
    int x_at;                // where a lane's piece of a granule's binary16 lies; of what they left, 2 KB away
    u32x4 x[MT][2];          // pieces of x of the block to come: binary16 and what it left

    __device__ __forceinline__ int chunk_start(int c) const {  // in blocks of the row: the last chunk reaches back where the row ends in it
        const int at = b0 + kChunk * c, last = o.nb - kChunk;
        return at < last ? at : last;
    }
    __device__ __forceinline__ void load_chunk(int c) const {
        const int at = chunk_start(c);
        int own = lane;
        asm volatile("" : "+v"(own));  // the addresses anew for each chunk: kept, they are eighteen registers
        const int row0 = own / kPieces, piece0 = own - row0 * kPieces;
#pragma unroll 1
        for (int i = 0; i < kPieces; i++) {  // 64 pieces on: seven rows and a piece
            const bool wraps = piece0 + i >= kPieces;
            const int row = row0 + 7 * i + (wraps ? 1 : 0), piece = piece0 + i - (wraps ? kPieces : 0), r = row & 31;
            const uint8_t* base = row & 32 ? rows[1] : rows[0];
            const int last = row & 32 ? last_row[1] : last_row[0];
            load_piece(base + (uint32_t)((r < last ? r : last) * o.nb + at) * 18u + piece * 16, chunks_at + (c & 1) * kChunkBytes + i * 1024);
        }
    }
    // Where tile mt of x's block b lies: past the last strip that one again, not stored. Up to eight strips by 2^15 blocks: 2^30 bytes.
    __device__ __forceinline__ int granule(int mt, int b) const {
        const int g = m0 / 16 + mt, last = (o.M - 1) / 32, s = (g >> 1) < last ? g >> 1 : last;
        return (s * o.nb + b0 + b) * (kGranuleX * 2) + (g & 1) * 256;
    }
    __device__ __forceinline__ void load_x(int mt, int b) {
        const int base = granule(mt, b);
        x[mt][0] = __builtin_amdgcn_raw_buffer_load_b128(x16, x_at, base, 0);
        x[mt][1] = __builtin_amdgcn_raw_buffer_load_b128(x16, x_at + 2048, base, 0);
    }
    template <bool BY_BLOCK>
    __device__ __forceinline__ void run(int nchunks, f32x4 (&acc)[MT][kCols]);
};

// What a lane takes of a block: its column's eight bytes q & 1 of nibbles, the low or the high ones of them, and its scale.
struct RawBlock { uint32_t lo, hi, more, scale; };

template <int MT>
template <bool BY_BLOCK>
__device__ __forceinline__ void Tile<MT>::run(int nchunks, f32x4 (&acc)[MT][kCols]) {
    const int h = q & 1, shift = 4 * (q >> 1);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // rows' scales: a lane brings those of rows lane and lane + 64, a pair of blocks at a time; of rows with one exponent, that one
    constexpr int kOwn = (MT * 16 + 63) / 64;
    const float* row_scales[kOwn];
    f32x2 scale[kOwn];
    auto load_scales = [&](int b) {  // b even; a row's blocks are an even number, so a pair lies on 8 bytes
#pragma unroll
        for (int i = 0; i < kOwn; i++)
            if (BY_BLOCK && row_scales[i]) scale[i] = *(const f32x2*)(row_scales[i] + (b < count ? b : count - 2));
    };
    if (BY_BLOCK) {
#pragma unroll
        for (int i = 0; i < kOwn; i++) {
            const int m = m0 + lane + 64 * i < o.M ? m0 + lane + 64 * i : o.M - 1;
            const int2 info = o.RS[m];
            row_scales[i] = info.y == kBlockHalves ? o.XS + (int64_t)m * o.nb + b0 : nullptr;
            const float one = info.x == INT32_MAX ? __builtin_nanf("") : __builtin_ldexpf(1.f, info.x);
            scale[i] = f32x2{one, one};
        }
        load_scales(0);
    }
    RawBlock raw[kCols];
    auto read_raw = [&](const uint8_t* pair, bool odd) {  // pair: where this lane's column has the pair of blocks in LDS
#pragma unroll
        for (int t = 0; t < kCols; t++) {
            const uint32_t* w = (const uint32_t*)(pair + t * 16 * kRowBytes);
            if (odd) {
                raw[t].scale = w[4];
                raw[t].lo = w[5 + 2 * h];
                raw[t].hi = w[6 + 2 * h];
            } else {
                raw[t].scale = w[0];
                raw[t].lo = w[2 * h];
                raw[t].hi = w[2 * h + 1];
                raw[t].more = w[2 * h + 2];
            }
        }
    };
    auto block = [&](int b, bool odd, const uint8_t* next_pair) {
        f16x8 w[kCols];
        float dw[kCols];
#pragma unroll
        for (int t = 0; t < kCols; t++) {
            const uint32_t lo = odd ? raw[t].lo : __builtin_amdgcn_alignbyte(raw[t].hi, raw[t].lo, 2);
            const uint32_t hi = odd ? raw[t].hi : __builtin_amdgcn_alignbyte(raw[t].more, raw[t].hi, 2);
            w[t] = nibbles_to_f16(lo >> shift, hi >> shift, 0);
            // odd blocks with their sign turned: b0 is even
            dw[t] = f16_bits_to_f32((uint16_t)(odd ? (raw[t].scale >> 16) ^ 0x8000u : raw[t].scale & 0xffffu));
        }
        read_raw(next_pair, !odd);  // behind a chunk's last pair: not used
        f32x4 c[2][kCols], dx[2];
        auto finish = [&](int mt) {
#pragma unroll
            for (int t = 0; t < kCols; t++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[mt][t][e] = fmaf(BY_BLOCK ? dw[t] * dx[mt & 1][e] : dw[t], c[mt & 1][t][e], acc[mt][t][e]);
        };
        const int next = b + 1 < count ? b + 1 : b;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            if (BY_BLOCK) dx[mt & 1] = *(const f32x4*)(scales + (odd ? MT * 16 : 0) + mt * 16 + 4 * q);
#pragma unroll
            for (int t = 0; t < kCols; t++) c[mt & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[mt][1]), w[t], zero, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < kCols; t++) c[mt & 1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[mt][0]), w[t], c[mt & 1][t], 0, 0, 0);
            if (mt > 0) finish(mt - 1);
            __builtin_amdgcn_sched_barrier(0x6);  // the tile's registers are read: but for VALU and SALU nothing crosses
            load_x(mt, next);
            __builtin_amdgcn_sched_barrier(0);
        }
        finish(MT - 1);
    };
    for (int c = 0; c < nchunks; c++) {
        // chunk c has been asked for before at least the 2 MT loads of x that are the newest now; the first of two, before nine of the second
        if (c > 0) {
            wait_loads<2 * MT>();
            if (c + 1 < nchunks) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // what is still read of the chunk before
                load_chunk(c + 1);
            }
        } else if (nchunks > 1) {
            wait_loads<kPieces>();
        } else {
            wait_loads<0>();
        }
        const int first = kChunk * c, blocks = count - first < kChunk ? count - first : kChunk;
        const uint8_t* pair = chunks + (c & 1) * kChunkBytes + r16 * kRowBytes + (b0 + first - chunk_start(c)) * 18;
        read_raw(pair, false);
        for (int b = 0; b < blocks; b += 2) {
            if (BY_BLOCK) {
#pragma unroll
                for (int i = 0; i < kOwn; i++)
                    if (lane + 64 * i < MT * 16) {
                        scales[lane + 64 * i] = scale[i][0];
                        scales[MT * 16 + lane + 64 * i] = scale[i][1];
                    }
                load_scales(first + b + 2);
                __builtin_amdgcn_wave_barrier();
            }
            block(first + b, false, pair);
            pair += 36;
            block(first + b + 1, true, pair);
        }
    }
}

template <int MT>
__global__ __launch_bounds__(64 * kWaves) void qgemm_q4_0_parts_kernel(Operands o, Plan d) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int t = (int)blockIdx.x;
    const int group = __builtin_amdgcn_readfirstlane(t % d.groups);
    t /= d.groups;
    const int m0 = __builtin_amdgcn_readfirstlane(t % d.tiles_m) * MT * 16, share = __builtin_amdgcn_readfirstlane(t / d.tiles_m);
    const int M = o.M, lane = threadIdx.x & 63, side = wave & (d.sides - 1), part = wave / d.sides, parts = kWaves / d.sides;
    int2 info[(MT * 16 + 63) / 64];
#pragma unroll
    for (int i = 0; i < (MT * 16 + 63) / 64; i++) info[i] = o.RS[m0 + lane + 64 * i < M ? m0 + lane + 64 * i : M - 1];

    const int b_share = share * d.share_blocks, in_share = o.nb - b_share < d.share_blocks ? o.nb - b_share : d.share_blocks;
    const int from = in_share / 2 * part / parts * 2, to = in_share / 2 * (part + 1) / parts * 2;
    Tile<MT> tile{o, lds + wave * kWaveBytes, 0, nullptr, lane, lane & 15, lane >> 4, m0, b_share + from, to - from, {}, {}, x_resource(o), 0, {}};
    tile.x_at = piece_at(tile.r16, tile.q, true) * 2;
    tile.chunks_at = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)tile.chunks);
    tile.scales = (float*)(tile.chunks + 2 * kChunkBytes);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int at = (group * d.sides + side) * 2 + i, strip = at < o.parts.strips ? at : o.parts.strips - 1;  // past the last: not stored
        const int p = o.parts.swiglu ? strip & 1 : strip >= o.parts.begin[2] ? 2 : strip >= o.parts.begin[1] ? 1 : 0;
        const int n = (o.parts.swiglu ? strip >> 1 : strip - o.parts.begin[p]) * 32;
        tile.rows[i] = o.parts.W[p] + (int64_t)n * o.nb * 18;
        tile.last_row[i] = o.parts.N[p] - 1 - n;
    }
    f32x4 acc[MT][kCols];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int c = 0; c < kCols; c++) acc[mt][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int nchunks = (tile.count + kChunk - 1) / kChunk;
    if (nchunks > 0) {
        tile.load_chunk(0);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) tile.load_x(mt, 0);
        if (nchunks > 1) tile.load_chunk(1);
    }
    bool by_block = false;
#pragma unroll
    for (int i = 0; i < (MT * 16 + 63) / 64; i++) by_block |= info[i].y == kBlockHalves;
    by_block = __ballot(by_block) != 0;
    if (nchunks > 0) {  // a share of fewer pairs of blocks than parts leaves some without: nothing of x's is theirs to read
        if (by_block) tile.template run<true>(nchunks, acc);
        else tile.template run<false>(nchunks, acc);
    }

    // The parts' sums: the upper two's to the lower two, these two's to whichever wavefront stores them. A loop over tiles, not their
    // code one after the other: run once a launch, it would be fetched as slowly as it is long.
    constexpr int kTiles = MT * kCols;
    f32x4* slots = (f32x4*)lds;  // [kWaves / 2][kTiles][lane]
    f32x4* mine = slots + (wave & (kWaves / 2 - 1)) * kTiles * 64 + lane;
    int* exponents = (int*)(lds + kLdsBytes) - kMostTiles * 16;
    __syncthreads();
    if (wave >= kWaves / 2) {
#pragma unroll
        for (int t = 0; t < kTiles; t++) mine[t * 64] = acc[t / kCols][t % kCols];
    }
    if (wave == 0) {
#pragma unroll
        for (int i = 0; i < (MT * 16 + 63) / 64; i++)
            if (lane + 64 * i < MT * 16) exponents[lane + 64 * i] = by_block ? 0 : info[i].x;
    }
    __syncthreads();
    if (wave < kWaves / 2) {
#pragma unroll
        for (int t = 0; t < kTiles; t++) {
            const f32x4 other = mine[t * 64];
            f32x4& a = acc[t / kCols][t % kCols];
#pragma unroll
            for (int e = 0; e < 4; e++) a[e] = a[e] + other[e];
            mine[t * 64] = a;
        }
    }
    __syncthreads();

    float* sums = o.sums ? o.sums + (int64_t)share * M * o.parts.strips * 32 : nullptr;
    const bool gated = o.parts.swiglu && !sums;
    const int each = gated ? 2 : kCols;  // sixteens of columns with results: gated, the second strip is up's, of the first one's columns
#pragma unroll 1
    for (int i = wave; i < d.sides * MT * each; i += kWaves) {
        const int c = i % each, mt = i / each % MT, of = i / each / MT;
        const int strip = (group * d.sides + of) * 2 + (c >> 1);
        if (strip >= o.parts.strips) continue;
        auto value = [&](int t, float v[4]) {
            f32x4 a = slots[(of * kTiles + t) * 64 + lane];
            for (int s = of + d.sides; s < kWaves / 2; s += d.sides) {
                const f32x4 b = slots[(s * kTiles + t) * 64 + lane];
#pragma unroll
                for (int k = 0; k < 4; k++) a[k] = a[k] + b[k];
            }
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = a[k];
            quad_transpose(v, lane);
        };
        const int row = mt * 16 + 4 * (lane >> 4) + (lane & 3), m = m0 + row, e_row = exponents[row];
        float v[4];
        value(mt * kCols + c, v);
        if (!by_block) under_exponent(v, e_row);
        if (gated) {
            float u[4];
            value(mt * kCols + c + 2, u);
            if (!by_block) under_exponent(u, e_row);
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = silu_times(v[k], u[k]);
        }
        int n;
        const int p = part_of(o.parts, strip, &n);
        float* y = sums ? sums : o.parts.y[p];
        const float* resid = sums ? nullptr : o.resid;
        const int cols = sums ? o.parts.strips * 32 : o.parts.N[p], n4 = (sums ? strip * 32 : n) + (c & 1) * 16 + (lane & 12);
        const bool wide_ok = (cols & 3) == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)resid & 15) == 0;
        if (m < M && n4 < cols) store_four(y, resid, m, cols, n4, v, wide_ok);
    }
}

template <int MT>
hipError_t launch(const Operands& o, const Plan& d, hipStream_t st) {
    static LdsLimit limit;
    if (hipError_t e = limit.raise(kLdsBytes, {(const void*)qgemm_q4_0_parts_kernel<MT>})) return e;
    hipLaunchKernelGGL(qgemm_q4_0_parts_kernel<MT>, dim3((unsigned)(d.groups * d.tiles_m * d.shares)), dim3(64 * kWaves), kLdsBytes, st, o, d);
    return hipGetLastError();
}

// Microseconds of a product and its cut: how many columns a workgroup has, and shares of K. A compute unit takes a workgroup at a time: 6.6 us, and a
// block of a wavefront 0.16 + 0.2 a sixteen of rows, and up to 0.33 more with as many workgroups as units, all of which read W and x (the
// clock falls, too). Shares: a launch, and 1.1 us a MB of their sums. Fitted to 45 shapes of 25 to 256 rows, each with all its cuts (2048 x 2560 to
// 14336 x 4096 and 4096 x 14336): of them the model takes the fastest but for four, where it is 3 % off. 4 us of all are a launch, which the
// callers count.
double plan(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, Plan* out) {
    const int64_t nb = K / 32, of_tile = (M + 127) / 128;
    const int sixteens = (int)((M + 16 * of_tile - 1) / (16 * of_tile)), halves = sixteens > kMostTiles ? 2 : 1, mt = (sixteens + halves - 1) / halves;
    const int64_t tiles = of_tile * halves;
    double best = 1e30;
    for (int sides = 1; sides <= 2; sides++) {
        const int64_t groups = (strips + 2 * sides - 1) / (2 * sides), parts = kWaves / sides;
        for (int64_t shares = 1; shares <= 32; shares++) {
            const int64_t blocks = (nb + 4 * shares - 1) / (4 * shares) * 4, used = (nb + blocks - 1) / blocks;
            if (used != shares) continue;
            const size_t sums = (size_t)shares * (size_t)M * (size_t)strips * 128;
            if (shares > 1 && (blocks < 8 || sums > sums_bytes)) break;
            const int64_t groups_all = groups * tiles * shares;
            const double a_part = (double)((blocks / 2 + parts - 1) / parts * 2);
            double us = (double)((groups_all + 255) / 256) * (6.6 + a_part * (0.16 + 0.2 * mt)) + a_part * 0.33 * (double)groups_all / 256.0;
            if (shares > 1) us += 1.1 + (double)sums * 1.1e-6;
            if (us < best) {
                best = us;
                *out = Plan{sides, (int)groups, (int)tiles, mt, (int)shares, (int)blocks};
            }
        }
    }
    return best - 4.0;
}

}  // namespace

// More rows than the row kernels are seldom slower at, and rows of W that give every part of K work. By up to 64 blocks (K 2048) the
// workgroups of qgemm_q4_0_direct_kernel are as fast (32768 x 1024: 96 rows 29.4 us there and 29.6 here, 128 rows 35.0 and 36.0).
bool qgemm_q4_0_parts_ok(int64_t M, int64_t strips, int64_t K) {
    return M > 24 && M <= kInPlaceRows && strips > 0 && strips < (1 << 20) && K > 2048 && K % 64 == 0 && K <= (1 << 20);
}

double qgemm_q4_0_parts_cost_us(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, size_t* used) {
    Plan d{};
    const double us = plan(M, strips, K, sums_bytes < kDirectMostSums ? sums_bytes : kDirectMostSums, &d);
    if (used) *used = d.shares > 1 ? (size_t)d.shares * (size_t)M * (size_t)strips * 128 : 0;
    return us;
}

// o: as for qgemm_q4_0_direct, of a shape that is ok.
hipError_t qgemm_q4_0_parts(Operands o, size_t sums_bytes, hipStream_t st) {
    for (int i = 0; i < 3; i++)
        if (((uintptr_t)o.parts.W[i] & 3) != 0) return hipErrorInvalidValue;
    Plan d;
    plan(o.M, o.parts.strips, (int64_t)o.nb * 32, sums_bytes < kDirectMostSums ? sums_bytes : kDirectMostSums, &d);
    if (d.shares == 1) o.sums = nullptr;
    const hipError_t e = d.mt == 1 ? launch<1>(o, d, st) : d.mt == 2 ? launch<2>(o, d, st) : d.mt == 3 ? launch<3>(o, d, st)
                       : d.mt == 4 ? launch<4>(o, d, st) : launch<5>(o, d, st);
    if (e) return e;
    if (d.shares > 1)
        if (hipError_t e = sum_shares(o, d.shares, st)) return e;
    note_kernel("qgemm_q4_0_parts_kernel<%d>: %d x %d tiles of %d x %d, %d shares of K", d.mt, d.tiles_m, d.groups, 16 * d.mt, 64 * d.sides, d.shares);
    return hipGetLastError();
}

}  // namespace mimir
