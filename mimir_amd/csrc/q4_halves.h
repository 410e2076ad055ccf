// What the kernels share that multiply many rows by Q4_0 weights: x as pairs of binary16 (qgemm_q4_0_fx16.hip, qgemm_q4_0_direct.hip) or
// bfloat16 as it is (qgemm_q4_0_blocks.hip).
#pragma once
#include "device_util.h"
#include "kernels.h"

namespace mimir {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef float f32x32 __attribute__((ext_vector_type(32)));

// Operands lie in memory as the product reads them, so that every load is a whole KB: granules of 32 rows by one block
// of 32 of K, the granules of a strip of 32 rows one after the other.
constexpr int kGranuleX = 2048;   // binary16 of a granule of x: 32 rows of 128 bytes, eight pieces of 16 (piece_at)
constexpr int kGranuleP = 1024;   // of W: two halves of the block, each in the order of lanes of an MFMA's operand
constexpr int kGranuleS = 32;     // float32 scales of W
constexpr int kGroup = 8;         // blocks whose scales come into LDS together: a KB a strip

// x: row m's pieces 4 part + 2 half + hi of a block, hi which eight of the half's sixteen. Of up to kInPlaceRows rows they lie in the order of
// an operand's lanes, piece by piece of the 32 rows: a load of an operand is whole lines (with a row's pieces beside one another the
// product that reads them from memory took 35 cycles a load of 1 KB: 80 x 14336 x 4096 39.0 us, now 35.6). Of more rows a row's block
// is one line for the kernels that write it, and its pieces lie at piece ^ turn, so that the 32 rows of a read from LDS fall on all banks.
__host__ __device__ inline int64_t strip_at(int m, int nb) { return (int64_t)(m >> 5) * nb * kGranuleX; }
__host__ __device__ inline int turn_of(int m) { return (m >> 1) & 7; }
__host__ __device__ inline bool in_lanes(int64_t M) { return M <= kInPlaceRows; }
__host__ __device__ inline int piece_at(int m, int piece, bool lanes) { return lanes ? piece * 256 + (m & 31) * 8 : (m & 31) * 64 + ((piece ^ turn_of(m)) << 3); }

// How a row of x is held. The row's information is {exponent, form}.
enum Form { kHalves = 0, kBlockHalves = 1, kDigitPairs = 2 };

__host__ __device__ inline int scale_blocks(int nb) { return (nb + kGroup - 1) / kGroup * kGroup; }  // of a strip: whole groups

// What is multiplied by the same x: up to three matrices, or gate and up, whose strips then lie in turn.
struct Parts {
    const uint8_t* W[3];
    float* y[3];
    int N[3];      // rows of W
    int begin[3];  // first strip; those of parts that are not there lie past the last
    int strips;    // of all
    int swiglu;    // W[0] and W[1] are gate and up: y[0] gets silu(gate) up
};

struct Operands {
    const uint16_t* P;
    const float* SW;
    const uint16_t* X16;
    const float* XS;
    const int2* RS;
    const float* resid;  // may be y; added to what one part's y gets
    float* sums;         // where K is cut into shares: [share][M][32 strips] float32, finished by fx16_sum_kernel
    int M, nb;
    Parts parts;
};

// Where column 0 of a strip goes: its part, and the column it is there. SwiGLU: of both gate's and up's strips, the result's.
__device__ __forceinline__ int part_of(const Parts& p, int strip, int* n) {
    const int part = p.swiglu ? 0 : strip >= p.begin[2] ? 2 : strip >= p.begin[1] ? 1 : 0;
    *n = (p.swiglu ? strip >> 1 : strip - p.begin[part]) * 32;
    return part;
}

// Up to four neighbouring columns n.. of row m of y [.., N] (+ resid): in one store where they are whole and aligned.
__device__ __forceinline__ void store_four(float* y, const float* resid, int64_t m, int N, int n, const float v[4], bool wide_ok) {
    if (wide_ok && n + 3 < N) {
        f32x4 out = {v[0], v[1], v[2], v[3]};
        if (resid) {
            const f32x4 r = *(const f32x4*)(resid + m * N + n);
#pragma unroll
            for (int k = 0; k < 4; k++) out[k] = out[k] + r[k];
        }
        *(f32x4*)(y + m * N + n) = out;
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (n + k >= N) continue;
            float out = v[k];
            if (resid) out = out + resid[m * N + n + k];
            y[m * N + n + k] = out;
        }
    }
}

// A row's results under its exponent; INT32_MAX: a row with a NaN or an infinity.
__device__ __forceinline__ void under_exponent(float v[4], int e) {
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = e == INT32_MAX ? __builtin_nanf("") : __builtin_ldexpf(v[k], e);
}

// What lane half q takes of a pair of blocks: of each its eight bytes q of nibbles, and, q = 0, its scale's bits.
struct PairBytes { uint32_t lo[2], hi[2], scale[2]; };

// 36 bytes at `pair`, as two loads of twelve where they are on a 4-byte boundary: bytes 8 q .. + 12 have the even block's eight two
// bytes in (q = 0: behind the scale), 16 + 8 q .. + 12 the odd one's last (q = 0: behind the scale and two bytes). Five loads of two bytes a
// block, which is all that blocks' own alignment allows, took the pass over W a little longer.
__device__ __forceinline__ PairBytes load_pair(const uint8_t* pair, int q, bool aligned) {
    PairBytes p;
    if (aligned) {
        u32x3 a, b;
        __builtin_memcpy(&a, __builtin_assume_aligned(pair + 8 * q, 4), 12);
        __builtin_memcpy(&b, __builtin_assume_aligned(pair + 16 + 8 * q, 4), 12);
        p.lo[0] = __builtin_amdgcn_alignbyte(a[1], a[0], 2);
        p.hi[0] = __builtin_amdgcn_alignbyte(a[2], a[1], 2);
        p.lo[1] = b[1];
        p.hi[1] = b[2];
        p.scale[0] = a[0] & 0xffffu;
        p.scale[1] = b[0] >> 16;
    } else {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint16_t* src = (const uint16_t*)(pair + 18 * i + 2 + 8 * q);
            p.lo[i] = (uint32_t)src[0] | (uint32_t)src[1] << 16;
            p.hi[i] = (uint32_t)src[2] | (uint32_t)src[3] << 16;
            p.scale[i] = load_u16(pair + 18 * i);
        }
    }
    return p;
}

// Eight nibbles (the low or the high ones of two dwords) as the binary16 integers n - 8: the nibble into the mantissa of binary16's
// 1024, minus 1032.
__device__ __forceinline__ f16x8 nibbles_to_f16(uint32_t lo, uint32_t hi, int half) {
    const f16x2 off = {(_Float16)1032.f, (_Float16)1032.f};
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t nib = ((i ? hi : lo) >> (4 * half)) & 0x0f0f0f0fu;
        const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, nib, 0x04010400u);
        const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, nib, 0x04030402u);
        v[2 * i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, p0) - off);
        v[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, p1) - off);
    }
    return __builtin_bit_cast(f16x8, v);
}

// A KB from global memory into LDS: lane l's 16 bytes from base + 16 l to lds_base + 16 l. Written out because the
// compiler, given the builtin, waits for every load under way before any LDS access; these loads are counted by hand
// (the compiler does not see them, so its own waits for the register loads of the scales can only be longer than
// needed, never shorter: loads return in order). The instruction takes its LDS base from M0, which an asm statement
// cannot name as clobbered: nothing else in these kernels uses M0, and it is set anew before every load (s_nop: gemm_nt_tile.h).
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t lane16, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(lane16), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A die's workgroups (every eighth, round-robin) take a contiguous range of the tiles, the tile's rows of x varying
// fastest: those that run together share few column panels of P through the die's L2.
__device__ __forceinline__ int tile_of(int b, int ntiles) {
    const int per_die = (ntiles + 7) >> 3;
    return (b & 7) * per_die + (b >> 3);
}

// The shares' sums of K, in their order: y = ((s0 + s1) + ..) (+ resid), or silu(gate) up of them.
hipError_t sum_shares(const Operands& o, int shares, hipStream_t st);

// The product with W read where it lies (qgemm_q4_0_direct.hip): up to kInPlaceRows rows.
constexpr size_t kDirectMostSums = (size_t)64 << 20;
double qgemm_q4_0_direct_cost_us(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, size_t* used = nullptr);  // of sums_bytes
hipError_t qgemm_q4_0_direct(Operands o, size_t sums_bytes, hipStream_t st);

// The same by a wavefront a part of K (qgemm_q4_0_parts.hip), which the two above pass on to where it is the faster.
bool qgemm_q4_0_parts_ok(int64_t M, int64_t strips, int64_t K);
double qgemm_q4_0_parts_cost_us(int64_t M, int64_t strips, int64_t K, size_t sums_bytes, size_t* used);
hipError_t qgemm_q4_0_parts(Operands o, size_t sums_bytes, hipStream_t st);

inline int64_t strips_of(int64_t rows) { return (rows + 31) / 32; }

}  // namespace mimir
