// Packed GEMMs on CDNA4 matrix cores (gfx950), FP32 accumulate:
//   hi-only   C = A_hi B_hi                      (tomos_gemm, tier DEFAULT)
//   split     C ~= A_hi B_hi + A_hi B_lo + A_lo B_hi
//             (tomos_gemm_split with both operands packed; tomos_gemm, tier
//             MATERIALIZE, with FP32 B).
// The hi-only form is the reference's 16-bit tensor-core GEMM on wh
// (mm_fp32_bf16_pure_bf16_gemm_direct_fastk_precomp2_serp,
// mm_cuda_kernels.cu:35372; mm_fp32_16_pure_half_wide_bigreg_sq_*, :37826);
// the split has no reference counterpart.
//
// Two steps:
//  1. stage: each operand is written as 16-bit planes in a K-contiguous
//     layout (A as [M][K], B as [N][K]) so every MFMA operand is one 16-byte
//     load.  Hi-only: A's hi word as the 16-bit tiers decode it (FP32_BF16:
//     bf16 as stored; FP32_16: fp32_16_half_only, fp16) and FP32 B rounded
//     to nearest-even bf16 / fp16.  Split: the exact value a, hi = rn16(a),
//     lo = rn16(a - hi); FP32_16 uses fp16 planes with a power-of-two scale
//     2^s per operand, chosen from the operand's largest magnitude, so the hi
//     and lo terms stay clear of fp16 overflow and underflow (C is rescaled
//     by 2^-(sA+sB) in the epilogue); FP32_BF16 uses bf16 planes.
//     The planes are stored as the LDS images the GEMM reads: blocks of 128
//     rows x 32 k, so a K slice of a tile is one contiguous run per operand.
//  2. gemm: 256 x 256 (or 128 x 128) C tiles, K slices through two LDS
//     stages by DMA, 1 (hi-only) or 3 (split) MFMA 32x32x16 per tile and
//     16-wide k step into one FP32 accumulator; splits of K where the tiles
//     leave the chip idle.
#include <algorithm>
#include <type_traits>

#include "codec.hpp"
#include "common.hpp"
#include "tomos_hip.h"

namespace tomos_hip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kPadRows = 256;   // operand rows are padded to the larger tile
constexpr int kBlockRows = 128, kBlockK = 32;
constexpr int kBlockElems = kBlockRows * kBlockK;  // one plane's block: 8 KB

// Element offset of the 8-element chunk (row r, k .. k+7) of a staged
// operand of nk slices.  A slice holds two blocks of every 128-row group, one
// after the other: the hi and the lo plane of 32 k (TERMS == 3), or the hi
// plane of two times 32 k (TERMS == 1, `second` = k / 32 % 2).  Inside a block
// a row is 64 bytes; its four 16-byte chunks are permuted by the row so that
// the 16 lanes that a 16-byte LDS read serves together touch all banks.
__host__ __device__ __forceinline__ int64_t chunk_offset(int64_t r, int64_t slice, int second, int64_t nk, int c) {
    const int row = static_cast<int>(r % kBlockRows);
    return ((r / kBlockRows * nk + slice) * 2 + second) * kBlockElems + row * kBlockK + ((c ^ ((row >> 2) & 3)) * 8);
}

// ---------------------------------------------------------------- operands
// A GEMM operand as the prep kernels read it: X column-major with leading
// dimension ld, either packed planes (wh/wr of FP32_16 or FP32_BF16) or a
// plain FP32 array (f != nullptr).
struct Src {
    int fmt;                 // TOMOS_FP32_16 | TOMOS_FP32_BF16 (packed); ignored for FP32
    const uint16_t* wh;
    const uint16_t* wr;
    const float* f;
    int64_t ld;
};

__device__ __forceinline__ float decode_exact(int fmt, uint32_t h, uint32_t r) {
    return fmt == TOMOS_FP32_16 ? codec::fp32_16_decode_exact(h, r) : __uint_as_float((h << 16) | r);
}

__device__ __forceinline__ uint16_t bf16_rn(float v) {
    return static_cast<uint16_t>(codec::f32_to_bf16_bits(v));
}
__device__ __forceinline__ uint16_t f16_rn(float v) {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
}
__device__ __forceinline__ float bf16_val(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

__device__ __forceinline__ int fp16_scale_exp(bool f16, const unsigned* absmax_bits) {
    // power-of-two scale bringing max |x| to about 2^13 (fp16 max is 65504)
    if (!f16) return 0;
    const float mx = __uint_as_float(*absmax_bits);
    int e = 0;
    frexpf(mx > 0.0f ? mx : 1.0f, &e);
    return 13 - e;
}

// alpha times 2^-(sA + sB): what the staged scales of both operands leave to
// undo (absA == nullptr: none).
__device__ __forceinline__ double unscaled_alpha(double alpha, const unsigned* absA, const unsigned* absB) {
    return absA ? ldexp(alpha, -(fp16_scale_exp(true, absA) + fp16_scale_exp(true, absB))) : alpha;
}

__device__ __forceinline__ void split16(bool f16, float v, int sc, uint16_t& h16, uint16_t& l16) {
    if (f16) {
        const float x = ldexpf(v, sc);
        const _Float16 h = static_cast<_Float16>(x);
        const _Float16 l = static_cast<_Float16>(x - static_cast<float>(h));
        h16 = __builtin_bit_cast(uint16_t, h);
        l16 = __builtin_bit_cast(uint16_t, l);
    } else {
        h16 = bf16_rn(v);
        l16 = bf16_rn(v - bf16_val(h16));
    }
}

enum { PREP_HI = 1, PREP_SPLIT = 3 };

typedef u32x4 u32x4_u __attribute__((aligned(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_u __attribute__((aligned(4)));

// The words of elements idx .. idx+7 of a packed plane, of which the first
// `count` exist (the others are zero words): one 16-byte load at element
// alignment for a whole run.
__device__ __forceinline__ u32x4 words8(const uint16_t* __restrict__ p, int64_t idx, int64_t count) {
    if (count >= 8) return *reinterpret_cast<const u32x4_u*>(p + idx);
    u32x4 w = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 7; ++e)
        if (e < count) w[e / 2] |= static_cast<uint32_t>(p[idx + e]) << (16 * (e & 1));
    return w;
}

// Exact values of elements idx .. idx+7, zero beyond `count`.
__device__ __forceinline__ void values8(const Src& s, int64_t idx, int64_t count, float (&v)[8]) {
    if (s.f) {
        if (count >= 8) {
            const f32x4 v0 = *reinterpret_cast<const f32x4_u*>(s.f + idx);
            const f32x4 v1 = *reinterpret_cast<const f32x4_u*>(s.f + idx + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] = v0[e]; v[4 + e] = v1[e]; }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = e < count ? s.f[idx + e] : 0.0f;
        }
        return;
    }
    const u32x4 wh = words8(s.wh, idx, count), wr = words8(s.wr, idx, count);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int b = 16 * (e & 1);
        const float x = decode_exact(s.fmt, (wh[e / 2] >> b) & 0xFFFFu, (wr[e / 2] >> b) & 0xFFFFu);
        v[e] = e < count ? x : 0.0f;
    }
}

// hi (and, for PREP_SPLIT, lo) bits of elements idx .. idx+7, zero beyond `count`.
template <int MODE>
__device__ __forceinline__ void prep8(const Src& s, int64_t idx, int64_t count, bool f16, int sc, uint16_t (&h)[8],
                                      uint16_t (&l)[8]) {
    if (MODE == PREP_HI && !s.f) {
        const u32x4 wh = words8(s.wh, idx, count);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // zero words stay zero in both formats' hi decode
            const uint32_t hb = s.fmt == TOMOS_FP32_16 ? codec::fp32_16_half_bits2(wh[q]) : wh[q];
            h[2 * q] = static_cast<uint16_t>(hb);
            h[2 * q + 1] = static_cast<uint16_t>(hb >> 16);
        }
        return;
    }
    float v[8];
    values8(s, idx, count, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if constexpr (MODE == PREP_HI) h[e] = f16 ? f16_rn(v[e]) : bf16_rn(v[e]);
        else split16(f16, v[e], sc, h[e], l[e]);
    }
}

__global__ void absmax_clear_kernel(unsigned* out) { out[threadIdx.x] = 0; }

// max |x| over an operand (exact values), for the fp16 split scale: runs of 8
// rows a thread, columns strided over blockIdx.y.
__global__ __launch_bounds__(256) void absmax_kernel(Src s, int64_t rows, int64_t cols,
                                                     unsigned* __restrict__ out_bits) {
    float mx = 0.0f;
    const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
    if (i < rows)
        for (int64_t j = blockIdx.y; j < cols; j += gridDim.y) {
            float v[8];
            values8(s, i + j * s.ld, rows - i, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float a = fabsf(v[e]);
                if (a <= 3.0e38f) mx = fmaxf(mx, a);  // ignore Inf/NaN
            }
        }
    for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((threadIdx.x & 63) == 0) atomicMax(out_bits, __float_as_uint(mx));
}

__device__ __forceinline__ u32x4 pack8(const uint16_t (&h)[8]) {
    u32x4 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = static_cast<uint32_t>(h[2 * q]) | (static_cast<uint32_t>(h[2 * q + 1]) << 16);
    return v;
}

// Stores the chunk of k .. k+7 (k a multiple of 8) of row r.
template <int MODE>
__device__ __forceinline__ void store_chunk(uint16_t* __restrict__ out, int64_t r, int64_t k, int64_t nk, u32x4 h,
                                            u32x4 l) {
    const int c = static_cast<int>(k % kBlockK) / 8;
    if constexpr (MODE == PREP_HI) {
        const int second = static_cast<int>(k / kBlockK % 2);
        *reinterpret_cast<u32x4*>(out + chunk_offset(r, k / (2 * kBlockK), second, nk, c)) = h;
    } else {
        *reinterpret_cast<u32x4*>(out + chunk_offset(r, k / kBlockK, 0, nk, c)) = h;
        *reinterpret_cast<u32x4*>(out + chunk_offset(r, k / kBlockK, 1, nk, c)) = l;
    }
}

// K-contiguous operand (X is K x R column-major): row r of the operand is
// X's column r.  A block takes 32 rows x 64 k: 128 contiguous bytes (or more)
// of every column in, 64-byte rows out.  grid = (ceil(Kp / 64), pad_r / 32).
template <int MODE>
__global__ __launch_bounds__(256) void prep_k_kernel(Src s, int64_t rows, int64_t cols, int64_t pad_r, int64_t nk,
                                                     int64_t Kp, uint16_t* __restrict__ out,
                                                     const unsigned* __restrict__ absmax_bits, bool f16) {
    const int sc = MODE == PREP_SPLIT ? fp16_scale_exp(f16, absmax_bits) : 0;
    const int64_t k = static_cast<int64_t>(blockIdx.x) * 64 + threadIdx.x % 8 * 8;
    if (k >= Kp) return;
    for (int64_t r = static_cast<int64_t>(blockIdx.y) * 32 + threadIdx.x / 8; r < pad_r;
         r += static_cast<int64_t>(gridDim.y) * 32) {
        uint16_t h[8], l[8];
        prep8<MODE>(s, k + r * s.ld, r < cols ? rows - k : 0, f16, sc, h, l);
        store_chunk<MODE>(out, r, k, nk, pack8(h), pack8(l));
    }
}

// R-contiguous operand (X is R x K column-major): row r of the operand is
// X's row r, so 64 x 64 tiles are transposed through LDS.  A thread loads 8
// rows of two adjacent columns and writes their pairs as 32-bit words; rows
// of 33 words spread both the writes and the reads over the banks.
// grid = (ceil(Kp / 64), pad_r / 64).
template <int MODE>
__global__ __launch_bounds__(256) void prep_t_kernel(Src s, int64_t rows, int64_t cols, int64_t nk, int64_t Kp,
                                                     uint16_t* __restrict__ out,
                                                     const unsigned* __restrict__ absmax_bits, bool f16) {
    constexpr int kPlanes = MODE == PREP_SPLIT ? 2 : 1;
    __shared__ uint32_t tile[kPlanes][64][33];  // [row][k pair]
    const int sc = MODE == PREP_SPLIT ? fp16_scale_exp(f16, absmax_bits) : 0;
    const int64_t k0 = static_cast<int64_t>(blockIdx.x) * 64, r0 = static_cast<int64_t>(blockIdx.y) * 64;
    {
        const int rv = threadIdx.x % 8 * 8, kp = threadIdx.x / 8;  // 8 rows, one k pair
        uint16_t h[2][8], l[2][8];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int64_t k = k0 + 2 * kp + b;
            prep8<MODE>(s, r0 + rv + k * s.ld, k < cols ? rows - (r0 + rv) : 0, f16, sc, h[b], l[b]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            tile[0][rv + e][kp] = static_cast<uint32_t>(h[0][e]) | (static_cast<uint32_t>(h[1][e]) << 16);
            if constexpr (MODE == PREP_SPLIT)
                tile[kPlanes - 1][rv + e][kp] = static_cast<uint32_t>(l[0][e]) | (static_cast<uint32_t>(l[1][e]) << 16);
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int idx = threadIdx.x + it * 256, c = idx % 8, i = idx / 8;  // chunk of 8 k, row
        if (k0 + 8 * c >= Kp) continue;
        u32x4 h, l = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            h[q] = tile[0][i][4 * c + q];
            if constexpr (MODE == PREP_SPLIT) l[q] = tile[kPlanes - 1][i][4 * c + q];
        }
        store_chunk<MODE>(out, r0 + i, k0 + 8 * c, nk, h, l);
    }
}

// ------------------------------------------------------------------- gemm
template <bool F16>
__device__ __forceinline__ void mfma32(const u32x4& a, const u32x4& b, f32x16& c) {
    if constexpr (F16) {
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    } else {
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
}

// C tile -> (tm, tn).  Block ids go round-robin over the 8 XCDs; the remap
// gives each XCD a contiguous run of ids, and inside a run the tiles are
// ordered in groups of kGroupN tile columns walked down M, so the ~32 blocks
// an XCD holds at once cover an 8 x 4 patch of C (8 A row panels and 4 B
// column panels in that XCD's L2) instead of one whole tile column.
constexpr int kGroupN = 4;
__device__ __forceinline__ void tile_of(int64_t bid, int64_t tiles_m, int64_t tiles_n, int64_t& tm, int64_t& tn) {
    const int64_t nb = tiles_m * tiles_n;
    if (nb % 8 == 0) bid = (bid % 8) * (nb / 8) + bid / 8;
    const int64_t per_group = tiles_m * kGroupN;
    const int64_t g = bid / per_group, w = bid - g * per_group;
    const int64_t gn = min(static_cast<int64_t>(kGroupN), tiles_n - g * kGroupN);
    tn = g * kGroupN + w % gn;
    tm = w / gn;
}

// 16 bytes a lane from base + voff into LDS at lds + 16 * lane, without a
// register in between.  As assembly, so that the compiler does not order
// every later LDS read behind the DMA (it cannot tell the stages apart): the
// kernel waits itself, with wait_stage().  No other instruction here uses M0.
__device__ __forceinline__ void dma16(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base)
                 : "memory");
}
// This wave's DMA but the last `LATER` has landed and its LDS reads have
// returned; then all waves meet.
template <int LATER>
__device__ __forceinline__ void wait_stage() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LATER) : "memory");
}

// A, B: staged operands (chunk_offset).  WM x WN waves, a wave owns MT x NT
// MFMA 32x32x16 tiles.  The B fragment is the MFMA's first operand, so the
// accumulator is C^T per tile and each lane holds C rows (lane % 32): the
// column-major stores of a 32-lane half are 128 contiguous bytes.
//
// A K slice (two blocks per 128 rows of A and B) goes to one of two LDS
// stages by DMA; a slice is two phases, split by k (TERMS == 3: 16 k, hi and
// lo; TERMS == 1: 32 k).  The second phase's fragments are read during the
// first phase's MFMAs and the next slice's first phase during the second's;
// the one barrier of a slice stands between the two, where this slice's
// reads are done (its stage is refilled right away, one slice ahead) and the
// next slice has landed.
// Bound by the matrix pipes: 8192^3 split, bf16, 3.1 -> 2.33 ms (1.42 PFLOP/s
// of MFMA work; a plain bf16 library product of that size runs at 1.15).
// Before, the slices went through registers into padded LDS rows, between two
// barriers a slice, and the tiles were 256 x 256 whatever their number.
template <bool F16, int TERMS, int WM, int WN, int MT, int NT>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mfma_kernel(
    int64_t M, int64_t N, int64_t nk, int64_t slices, const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
    double alpha, double beta, float* __restrict__ C, int64_t ldc, const unsigned* __restrict__ absA,
    const unsigned* __restrict__ absB, float* __restrict__ partial) {
    static_assert(TERMS == 1 || TERMS == 3, "hi-only or 3-term split");
    constexpr int BM = 32 * WM * MT, BN = 32 * WN * NT;
    constexpr int kThreads = 64 * WM * WN;
    constexpr int GA = BM / kBlockRows, GB = BN / kBlockRows;  // 128-row groups
    constexpr uint32_t kGroup = 2 * kBlockElems * 2;           // bytes of a group's slice
    constexpr uint32_t kStage = (GA + GB) * kGroup;
    constexpr uint32_t kStep = kThreads * 16;                  // bytes per DMA of the block
    constexpr int kLoads = kStage / kStep;                     // DMAs per thread and slice
    extern __shared__ __attribute__((aligned(1024))) char gemm_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int64_t split = blockIdx.x / (tiles_m * tiles_n);
    int64_t tm, tn;
    tile_of(blockIdx.x - split * tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;
    const int64_t s0 = split * slices, s1 = min(nk, s0 + slices);

    f32x16 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.0f;

    const char* ga = reinterpret_cast<const char*>(A) + tm * GA * nk * kGroup;
    const char* gb = reinterpret_cast<const char*>(B) + tn * GB * nk * kGroup;
    const uint32_t lds0 = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)gemm_lds));
    const uint32_t voff = tid * 16, wave_lds = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);
    auto load_slice = [&](int64_t s, uint32_t stage) {
#pragma unroll
        for (int g = 0; g < GA; ++g)
#pragma unroll
            for (uint32_t x = 0; x < kGroup; x += kStep)
                dma16(ga + (g * nk + s) * kGroup + x, voff, stage + g * kGroup + x + wave_lds);
#pragma unroll
        for (int g = 0; g < GB; ++g)
#pragma unroll
            for (uint32_t x = 0; x < kGroup; x += kStep)
                dma16(gb + (g * nk + s) * kGroup + x, voff, stage + (GA + g) * kGroup + x + wave_lds);
    };
    // fragment addresses: row lane % 32 of the wave's first tile, the chunk of
    // k 8 (lane / 32), permuted as stored; the other chunk of a block is at ^ 32
    const int sw = (lane >> 2) & 3, row = lane & 31;
    const uint32_t chunk = (((lane >> 5) ^ sw) * 16);
    const int am = wm * MT * 32, bn = wn * NT * 32;
    const uint32_t fa = (am / kBlockRows) * kGroup + (am % kBlockRows + row) * 64 + chunk;
    const uint32_t fb = (GA + bn / kBlockRows) * kGroup + (bn % kBlockRows + row) * 64 + chunk;
    // a[x][i], b[x][j]: x = hi / lo plane (split) or the two k steps of the phase
    struct Frag {
        u32x4 a[2][MT], b[2][NT];
    };
    auto read_phase = [&](Frag& f, uint32_t stage, int phase) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const uint32_t block = (TERMS == 3 ? x : phase) * (kBlockElems * 2);
            const uint32_t flip = (TERMS == 3 ? phase : x) * 32;
#pragma unroll
            for (int i = 0; i < MT; ++i)
                f.a[x][i] = *reinterpret_cast<const u32x4*>(gemm_lds + stage + ((fa ^ flip) + block + i * 2048));
#pragma unroll
            for (int j = 0; j < NT; ++j)
                f.b[x][j] = *reinterpret_cast<const u32x4*>(gemm_lds + stage + ((fb ^ flip) + block + j * 2048));
        }
    };
    auto multiply = [&](const Frag& f) {
        if constexpr (TERMS == 3) {  // lo*hi, hi*lo, hi*hi
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
                        mfma32<F16>(f.b[t == 1 ? 1 : 0][j], f.a[t == 0 ? 1 : 0][i], acc[j][i]);
        } else {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i) mfma32<F16>(f.b[x][j], f.a[x][i], acc[j][i]);
        }
    };

    Frag f0, f1;
    uint32_t stage = 0;
    load_slice(s0, 0);
    if (s0 + 1 < s1) {
        load_slice(s0 + 1, kStage);
        wait_stage<kLoads>();
    } else {
        wait_stage<0>();
    }
    read_phase(f0, 0, 0);
    for (int64_t s = s0; s < s1; ++s) {
        read_phase(f1, stage, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f0);
        __builtin_amdgcn_sched_barrier(0);
        wait_stage<0>();
        if (s + 2 < s1) load_slice(s + 2, stage);
        stage ^= kStage;
        if (s + 1 < s1) read_phase(f0, stage, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f1);
        __builtin_amdgcn_sched_barrier(0);
    }
    // epilogue: acc[j][i][v] is C(row, col) with row = m tile i, lane % 32 and
    // col = n tile j, 8 (v / 4) + 4 (lane / 32) + v % 4
    const double scale = F16 ? unscaled_alpha(alpha, absA, absB) : alpha;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int64_t r = m0 + am + i * 32 + row;
        if (r >= M) continue;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int64_t col = n0 + bn + j * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
                if (col < N) {
                    if (partial) {
                        partial[(split * N + col) * M + r] = acc[j][i][v];
                        continue;
                    }
                    float* p = C + r + col * ldc;
                    double t = scale * static_cast<double>(acc[j][i][v]);
                    if (beta != 0.0) t += beta * static_cast<double>(*p);
                    *p = static_cast<float>(t);
                }
            }
    }
}

// C = scale * (sum of the K splits' partial products, in FP64) + beta C
__global__ __launch_bounds__(256) void gemm_split_sum_kernel(int64_t M, int64_t N, int splits,
                                                             const float* __restrict__ partial, double alpha,
                                                             double beta, float* __restrict__ C, int64_t ldc,
                                                             const unsigned* __restrict__ absA,
                                                             const unsigned* __restrict__ absB) {
    const double scale = unscaled_alpha(alpha, absA, absB);
    const int64_t total = M * N;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; t < total;
         t += static_cast<int64_t>(gridDim.x) * 256) {
        double v = 0.0;
        for (int q = 0; q < splits; ++q) v += static_cast<double>(partial[q * total + t]);
        float* p = C + t % M + t / M * ldc;
        v *= scale;
        if (beta != 0.0) v += beta * static_cast<double>(*p);
        *p = static_cast<float>(v);
    }
}

// Staged operands: absmax words, A, B, then the partial products of K splits.
struct Planes {
    int64_t Mp, Np, Kp, nk;  // padded sizes, K slices
    unsigned* absmax;
    uint16_t *A, *B;
    float* partial;
};

int64_t slice_k(int terms) { return terms == 3 ? kBlockK : 2 * kBlockK; }

Planes planes_of(int terms, int64_t M, int64_t N, int64_t K, void* base_ptr) {
    Planes p;
    p.Mp = ceil_div(M, kPadRows) * kPadRows;
    p.Np = ceil_div(N, kPadRows) * kPadRows;
    p.nk = std::max<int64_t>(ceil_div(K, slice_k(terms)), 1);
    p.Kp = p.nk * slice_k(terms);
    // the planes start on 16 bytes, which their stores and the DMA take, at any
    // alignment of the scratch: up to 15 of the 256 bytes ahead of them go
    const uintptr_t base = reinterpret_cast<uintptr_t>(base_ptr);
    p.absmax = reinterpret_cast<unsigned*>((base + 15) & ~uintptr_t(15));
    p.A = reinterpret_cast<uint16_t*>((base + 256) & ~uintptr_t(15));
    p.B = p.A + p.Mp * p.nk * 2 * kBlockK;
    p.partial = reinterpret_cast<float*>(p.B + p.Np * p.nk * 2 * kBlockK);
    return p;
}

// Launch shape.  256 x 256 tiles (8 waves) read the LDS least per MFMA and
// are taken where they about fill the chip; below that 128 x 128 (4 waves,
// two blocks a CU), and K is split while the tiles are under half the 512
// blocks the chip holds, as long as a split keeps kMinSlices slices.
// Measured (hi-only whole call, us, before / now / with 256-wide tiles and
// splits): 712 x 83 x 5473 178 / 27 / 38; 2451 x 337 x 2714 107 / 36 / 45;
// 2000^3 88 / 47 / 58; 3001 x 1501 x 6001 223 / 117 / 118; 4096^3 (256 tiles)
// 173 / 142 / 143.  Splitting for 768 or 1024 blocks: 4950 x 397 x 4895 75 -> 87.
struct Shape {
    bool large;
    int64_t tiles, slices;  // C tiles, K slices per split
    int splits;
};
constexpr int64_t kMinSlices = 8, kLargeTiles = 192, kSplitBlocks = 512;
Shape shape_of(int64_t M, int64_t N, int64_t nk) {
    Shape h;
    const int64_t big = ceil_div(M, 256) * ceil_div(N, 256), small = ceil_div(M, 128) * ceil_div(N, 128);
    h.large = big >= kLargeTiles;
    h.tiles = h.large ? big : small;
    int64_t splits = h.large ? 1 : std::max<int64_t>(1, kSplitBlocks / small);
    splits = std::max<int64_t>(1, std::min<int64_t>(splits, nk / kMinSlices));
    h.slices = ceil_div(nk, splits);
    h.splits = static_cast<int>(ceil_div(nk, h.slices));
    return h;
}

// Stage one operand: X is rows x cols column-major; kcontig means the GEMM's
// K runs down X's columns (X is K x R), otherwise along its rows (X is R x K).
void stage(int mode, bool f16, const Src& x, bool kcontig, int64_t rows, int64_t cols, int64_t pad_r, int64_t nk,
           int64_t Kp, uint16_t* out, const unsigned* absmax, hipStream_t s) {
    require(kcontig || pad_r / 64 < 65536, "gemm: operand too large");
    const dim3 grid(static_cast<unsigned>(ceil_div(Kp, 64)),
                    static_cast<unsigned>(kcontig ? std::min<int64_t>(pad_r / 32, 65535) : pad_r / 64));
    if (kcontig) {
        if (mode == PREP_HI)
            prep_k_kernel<PREP_HI><<<grid, 256, 0, s>>>(x, rows, cols, pad_r, nk, Kp, out, absmax, f16);
        else
            prep_k_kernel<PREP_SPLIT><<<grid, 256, 0, s>>>(x, rows, cols, pad_r, nk, Kp, out, absmax, f16);
    } else {
        if (mode == PREP_HI)
            prep_t_kernel<PREP_HI><<<grid, 256, 0, s>>>(x, rows, cols, nk, Kp, out, absmax, f16);
        else
            prep_t_kernel<PREP_SPLIT><<<grid, 256, 0, s>>>(x, rows, cols, nk, Kp, out, absmax, f16);
    }
    TOMOS_LAUNCH_CHECK("gemm operand staging");
}

}  // namespace

// Staged planes only (the least a call needs), and with the K splits' partials.
size_t gemm_planes_bytes(int terms, int64_t M, int64_t N, int64_t K) {
    const Planes p = planes_of(terms, M, N, K, nullptr);
    return static_cast<size_t>((p.Mp + p.Np) * p.nk * 2 * kBlockK) * 2 + 256;
}
size_t gemm_mfma_scratch_bytes(int terms, int64_t M, int64_t N, int64_t K) {
    const Planes p = planes_of(terms, M, N, K, nullptr);
    const Shape h = shape_of(M, N, p.nk);
    return gemm_planes_bytes(terms, M, N, K) + (h.splits > 1 ? static_cast<size_t>(h.splits) * M * N * 4 : 0);
}

size_t gemm_split_scratch_bytes(int64_t M, int64_t N, int64_t K) { return gemm_mfma_scratch_bytes(3, M, N, K); }

// C = alpha op(A) op(B) + beta C on 16-bit MFMA with FP32 accumulation:
// terms == 1 multiplies the hi words (A's packed hi word as the 16-bit
// tiers decode it, B rounded to nearest-even bf16/fp16), terms == 3 the
// split A_hi B_hi + A_hi B_lo + A_lo B_hi of the exact values.  f16 picks
// fp16 planes (FP32_16) over bf16 ones (FP32_BF16).  A is M x K (a_kcontig:
// stored K x M, i.e. transposed), B is K x N (b_kcontig: stored K x N, the
// plain layout; otherwise stored N x K).
void gemm_mfma(int terms, bool f16, const Src& a, bool a_kcontig, const Src& b, bool b_kcontig, int64_t M,
               int64_t N, int64_t K, double alpha, double beta, float* c, int64_t ldc, void* scratch,
               size_t scratch_bytes, hipStream_t s) {
    require(terms == 1 || terms == 3, "gemm_mfma: terms must be 1 or 3");
    if (M == 0 || N == 0) return;
    const size_t least = gemm_planes_bytes(terms, M, N, K), need = gemm_mfma_scratch_bytes(terms, M, N, K);
    if (!scratch) {
        scratch = fallback_scratch(need);
        scratch_bytes = need;
    }
    require(scratch_bytes >= least, "gemm: scratch too small (need " + std::to_string(least) + " bytes)");
    const Planes p = planes_of(terms, M, N, K, scratch);
    const int mode = terms == 3 ? PREP_SPLIT : PREP_HI;
    const bool scaled = terms == 3 && f16;
    if (scaled) {
        absmax_clear_kernel<<<1, 2, 0, s>>>(p.absmax);
        if (K > 0) {
            auto absmax = [&](const Src& x, int64_t rows, int64_t cols, unsigned* out) {
                const int64_t bx = ceil_div(rows, 2048);  // about 2048 blocks in all
                const dim3 grid(static_cast<unsigned>(bx),
                                static_cast<unsigned>(std::min(cols, std::max<int64_t>(2048 / bx, 1))));
                absmax_kernel<<<grid, 256, 0, s>>>(x, rows, cols, out);
            };
            absmax(a, a_kcontig ? K : M, a_kcontig ? M : K, p.absmax);
            absmax(b, b_kcontig ? K : N, b_kcontig ? N : K, p.absmax + 1);
            TOMOS_LAUNCH_CHECK("absmax_kernel");
        }
    }
    stage(mode, f16, a, a_kcontig, a_kcontig ? K : M, a_kcontig ? M : K, p.Mp, p.nk, p.Kp, p.A, p.absmax, s);
    stage(mode, f16, b, b_kcontig, b_kcontig ? K : N, b_kcontig ? N : K, p.Np, p.nk, p.Kp, p.B, p.absmax + 1, s);
    Shape h = shape_of(M, N, p.nk);
    if (scratch_bytes < need) {  // a scratch of the planes alone: no K splits
        h.splits = 1;
        h.slices = p.nk;
    }
    const int64_t nblocks = h.tiles * h.splits;
    require(nblocks < (int64_t(1) << 31), "gemm: grid too large");
    const unsigned* absA = scaled ? p.absmax : nullptr;
    const unsigned* absB = scaled ? p.absmax + 1 : nullptr;
    float* partial = h.splits > 1 ? p.partial : nullptr;
    auto launch = [&](auto* k, int threads, int tile) {
        const int lds = 2 * 2 * (tile / kBlockRows) * 2 * kBlockElems * 2;  // two stages of A and B slices
        TOMOS_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        k<<<static_cast<unsigned>(nblocks), threads, lds, s>>>(M, N, p.nk, h.slices, p.A, p.B, alpha, beta, c, ldc, absA,
                                                               absB, partial);
    };
    auto run = [&](auto f16_, auto terms_) {
        if (h.large) launch(gemm_mfma_kernel<f16_, terms_, 2, 4, 4, 2>, 512, 256);
        else launch(gemm_mfma_kernel<f16_, terms_, 2, 2, 2, 2>, 256, 128);
    };
    using one = std::integral_constant<int, 1>;
    using three = std::integral_constant<int, 3>;
    if (f16) {
        if (terms == 3) run(std::true_type{}, three{});
        else run(std::true_type{}, one{});
    } else {
        if (terms == 3) run(std::false_type{}, three{});
        else run(std::false_type{}, one{});
    }
    TOMOS_LAUNCH_CHECK("gemm_mfma_kernel");
    if (h.splits > 1) {
        const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(ceil_div(M * N, 256), 16384));
        gemm_split_sum_kernel<<<blocks, 256, 0, s>>>(M, N, h.splits, partial, alpha, beta, c, ldc, absA, absB);
        TOMOS_LAUNCH_CHECK("gemm_split_sum_kernel");
    }
}

void gemm_split(int a_type, int64_t M, int64_t N, int64_t K, double alpha, const uint16_t* awh,
                const uint16_t* awr, int64_t lda, const uint16_t* bwh, const uint16_t* bwr, int64_t ldb,
                double beta, float* c, int64_t ldc, void* scratch, size_t scratch_bytes, hipStream_t s) {
    require(a_type == TOMOS_FP32_16 || a_type == TOMOS_FP32_BF16, "gemm_split: packed operands only");
    require(M >= 0 && N >= 0 && K >= 0, "gemm_split: negative size");
    require(lda >= std::max<int64_t>(M, 1) && ldb >= std::max<int64_t>(K, 1) && ldc >= std::max<int64_t>(M, 1),
            "gemm_split: bad leading dimension");
    if (M == 0 || N == 0) return;
    require(c != nullptr && (K == 0 || (awh && awr && bwh && bwr)), "gemm_split: null pointer");
    const Src a{a_type, awh, awr, nullptr, lda}, b{a_type, bwh, bwr, nullptr, ldb};
    gemm_mfma(3, a_type == TOMOS_FP32_16, a, false, b, true, M, N, K, alpha, beta, c, ldc, scratch, scratch_bytes,
              s);
}

// tomos_gemm's packed-A tiers on matrix cores: DEFAULT (hi words) and
// MATERIALIZE (3-term split of the exact values), FP32 B.
void gemm_packed_mfma(int a_type, int tier, bool ta, bool tb, double alpha, int64_t M, int64_t N, int64_t K,
                      const uint16_t* wh, const uint16_t* wr, int64_t lda, const float* b, int64_t ldb,
                      double beta, float* c, int64_t ldc, hipStream_t s) {
    const int terms = tier == TOMOS_TIER_MATERIALIZE ? 3 : 1;
    const Src a{a_type, wh, wr, nullptr, lda}, bs{a_type, nullptr, nullptr, b, ldb};
    gemm_mfma(terms, a_type == TOMOS_FP32_16, a, ta, bs, !tb, M, N, K, alpha, beta, c, ldc, nullptr, 0, s);
}

}  // namespace tomos_hip

using namespace tomos_hip;

extern "C" {

size_t tomos_gemm_split_scratch_size(int64_t M, int64_t N, int64_t K) {
    if (M < 0 || N < 0 || K < 0) return 0;
    return gemm_split_scratch_bytes(M, N, K);
}

int tomos_gemm_split(int a_type, int64_t M, int64_t N, int64_t K, double alpha, const uint16_t* a_wh,
                     const uint16_t* a_wr, int64_t lda, const uint16_t* b_wh, const uint16_t* b_wr,
                     int64_t ldb, double beta, float* c, int64_t ldc, void* scratch,
                     size_t scratch_bytes, tomos_stream_t s) {
    return guarded([&] {
        gemm_split(a_type, M, N, K, alpha, a_wh, a_wr, lda, b_wh, b_wr, ldb, beta, c, ldc, scratch,
                   scratch_bytes, s);
    });
}

}  // extern "C"
