// Dense GEMV on plain and packed column-major matrices, for gfx950.
//
// Storage formats: F32, F64, FP32_16 and FP32_BF16 (planar wh/wr uint16
// planes).  Tiers (see tomos_hip.h): DEFAULT decodes wh only and
// accumulates in FP32; FAST decodes wh only and accumulates in FP64; EXACT
// rebuilds the exact FP32 value from wh+wr and accumulates in FP64.
//
// y = A x   (NO_TRANSPOSE): each thread owns one 16-byte vector of rows
//           (8 packed / 4 fp32 / 2 fp64 rows) and streams every column of
//           its block's column range, 8 columns per batch so 8 independent
//           16-B loads are in flight per lane.  x[j] is wave-uniform and is
//           read through the scalar cache.  When m is too small to fill the
//           chip, the waves of a block split the columns and add their sums
//           through LDS in a fixed order; a wide matrix of few rows is split
//           over the grid too, with partial sums that a second pass adds.
// z = A^T y (TRANSPOSE): a block owns a chunk of rows and a group of CB
//           columns; each lane keeps CB column accumulators in VGPRs and
//           walks the chunk in 16-B row vectors (loads coalesced along the
//           column), the wave reduces the CB accumulators with a transpose
//           butterfly (CB-1 shuffles per lane instead of 6*CB), the four
//           waves combine through LDS, and the per-chunk partials are summed
//           in a fixed order by a second pass.  Short columns are owned whole
//           by a block or a wave, without partials.  No atomics anywhere: results are
//           bit-reproducible run to run.
#include <algorithm>

#include "codec.hpp"
#include "common.hpp"
#include "gemv.hpp"
#include "tomos_hip.h"

namespace tomos_hip {

namespace {

// FMT_PBF with DEC_HI also serves native BF16 storage (the hi plane is a
// bf16 array); FMT_H16 is native IEEE binary16 storage.
enum { FMT_F32 = 0, FMT_F64 = 1, FMT_P16 = 2, FMT_PBF = 3, FMT_H16 = 4 };
enum { DEC_NATIVE = 0, DEC_HI = 1, DEC_EXACT = 2 };

constexpr int kThreads = 256;

template <int FMT>
constexpr int vec_full() {
    return FMT == FMT_F64 ? 2 : (FMT == FMT_F32 ? 4 : 8);
}
template <int FMT>
constexpr bool is16() {
    return FMT == FMT_P16 || FMT == FMT_PBF || FMT == FMT_H16;
}

// Raw (undecoded) bits of VEC consecutive elements.
template <int FMT, int DEC, int VEC>
struct Raw {
    uint32_t h[4];
    uint32_t r[4];
};

// 16-byte vectors are read at element alignment: gfx950 global loads take
// any, so an lda that is no multiple of the vector (an unpadded odd m) costs
// a cache line more per 1 KB wave load, where element-wise loads cost eight
// times the load instructions (131071 x 501 FP32_16 EXACT, odd lda, with the
// pair decode: N 76 -> 51 us, T 118 -> 74 us).
template <bool NTL>
__device__ __forceinline__ uint4 load_vec16(const void* p) {
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4), aligned(2)));
    u32x4 v;
    if constexpr (NTL) v = __builtin_nontemporal_load(static_cast<const u32x4*>(p));
    else v = *static_cast<const u32x4*>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}

template <int FMT, int DEC, int VEC, bool NTL>
__device__ __forceinline__ void load_raw(const void* __restrict__ a,
                                         const uint16_t* __restrict__ wr, int64_t idx,
                                         Raw<FMT, DEC, VEC>& R) {
    if constexpr (is16<FMT>()) {
        const uint16_t* p = static_cast<const uint16_t*>(a) + idx;
        if constexpr (VEC == 8) {
            const uint4 t = load_vec16<NTL>(p);
            R.h[0] = t.x; R.h[1] = t.y; R.h[2] = t.z; R.h[3] = t.w;
            if constexpr (DEC == DEC_EXACT) {
                const uint4 q = load_vec16<NTL>(wr + idx);
                R.r[0] = q.x; R.r[1] = q.y; R.r[2] = q.z; R.r[3] = q.w;
            }
        } else {
            R.h[0] = *p;
            if constexpr (DEC == DEC_EXACT) R.r[0] = wr[idx];
        }
    } else if constexpr (FMT == FMT_F32) {
        const float* p = static_cast<const float*>(a) + idx;
        if constexpr (VEC == 4) {
            const uint4 t = load_vec16<NTL>(p);
            R.h[0] = t.x; R.h[1] = t.y; R.h[2] = t.z; R.h[3] = t.w;
        } else {
            R.h[0] = __float_as_uint(*p);
        }
    } else {
        const double* p = static_cast<const double*>(a) + idx;
        if constexpr (VEC == 2) {
            const uint4 t = load_vec16<NTL>(p);
            R.h[0] = t.x; R.h[1] = t.y; R.h[2] = t.z; R.h[3] = t.w;
        } else {
            const uint2 t = *reinterpret_cast<const uint2*>(p);
            R.h[0] = t.x; R.h[1] = t.y;
        }
    }
}

__device__ __forceinline__ float half_bits_to_float(uint32_t hb) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(hb)));
}

template <int FMT, int DEC>
__device__ __forceinline__ float decode16(uint32_t h, uint32_t r) {
    if constexpr (FMT == FMT_H16) {
        return half_bits_to_float(h);
    } else if constexpr (FMT == FMT_P16) {
        if constexpr (DEC == DEC_EXACT) return codec::fp32_16_decode_exact(h, r);
        else return half_bits_to_float(codec::fp32_16_half_bits(h));
    } else {
        if constexpr (DEC == DEC_EXACT) return __uint_as_float((h << 16) | r);
        else return __uint_as_float(h << 16);
    }
}

// Whether an FP32_16 vector holds a saturated word (the exact pair decode
// leaves those out).
template <int FMT, int DEC>
__device__ __forceinline__ bool saturated(const Raw<FMT, DEC, 8>& R) {
    return (codec::fp32_16_saturated2(R.h[0]) | codec::fp32_16_saturated2(R.h[1]) |
            codec::fp32_16_saturated2(R.h[2]) | codec::fp32_16_saturated2(R.h[3])) != 0;
}

// RARE = false: an exact FP32_16 vector without saturated words.
template <int FMT, int DEC, int VEC, class ACC, bool RARE = true>
__device__ __forceinline__ void decode(const Raw<FMT, DEC, VEC>& R, ACC (&out)[VEC]) {
    if constexpr (is16<FMT>()) {
        if constexpr (VEC == 8) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if constexpr (FMT == FMT_P16) {
                    float v0, v1;
                    if constexpr (DEC == DEC_HI) {
                        const uint32_t hb = codec::fp32_16_half_bits2(R.h[k]);
                        v0 = half_bits_to_float(hb & 0xFFFFu);
                        v1 = half_bits_to_float(hb >> 16);
                    } else {
                        codec::fp32_16_decode_exact2(R.h[k], R.r[k], v0, v1);
                    }
                    out[2 * k] = static_cast<ACC>(v0);
                    out[2 * k + 1] = static_cast<ACC>(v1);
                    continue;
                }
                const uint32_t h = R.h[k];
                const uint32_t r = (DEC == DEC_EXACT) ? R.r[k] : 0u;
                out[2 * k] = static_cast<ACC>(decode16<FMT, DEC>(h & 0xFFFFu, r & 0xFFFFu));
                out[2 * k + 1] = static_cast<ACC>(decode16<FMT, DEC>(h >> 16, r >> 16));
            }
            if constexpr (FMT == FMT_P16 && DEC == DEC_EXACT && RARE) {
                if (saturated(R)) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const int b = 16 * (k & 1);
                        out[k] = static_cast<ACC>(
                            decode16<FMT, DEC>((R.h[k / 2] >> b) & 0xFFFFu, (R.r[k / 2] >> b) & 0xFFFFu));
                    }
                }
            }
        } else {
            out[0] = static_cast<ACC>(decode16<FMT, DEC>(R.h[0], (DEC == DEC_EXACT) ? R.r[0] : 0u));
        }
    } else if constexpr (FMT == FMT_F32) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) out[k] = static_cast<ACC>(__uint_as_float(R.h[k]));
    } else {
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const uint64_t b = (static_cast<uint64_t>(R.h[2 * k + 1]) << 32) | R.h[2 * k];
            out[k] = static_cast<ACC>(__longlong_as_double(static_cast<long long>(b)));
        }
    }
}

__device__ __forceinline__ double read_coef(double host, const double* dev, double mul) {
    return dev ? mul * (*dev) : host;
}

// x[j .. j+U), a wave's U columns.  One branch on the type for all of them,
// so that their scalar loads are in flight together.  LAST: entries at j1 and
// beyond repeat x[j1-1].
template <int U, class ACC, bool LAST>
__device__ __forceinline__ void load_x_cols(const void* __restrict__ x, bool x64, int64_t j, int64_t j1,
                                            ACC (&xs)[U]) {
    if (x64) {
        double t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = static_cast<const double*>(x)[LAST ? min(j + u, j1 - 1) : j + u];
#pragma unroll
        for (int u = 0; u < U; ++u) xs[u] = static_cast<ACC>(t[u]);
    } else {
        float t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = static_cast<const float*>(x)[LAST ? min(j + u, j1 - 1) : j + u];
#pragma unroll
        for (int u = 0; u < U; ++u) xs[u] = static_cast<ACC>(t[u]);
    }
}

// x of a lane's VEC rows starting at i (all in range); the first `lo` are 0.
template <int VEC, class ACC>
__device__ __forceinline__ void load_x_rows(const void* __restrict__ x, bool x64, int64_t i, int lo,
                                            ACC (&xv)[VEC]) {
    if (x64) {
        typedef double vd __attribute__((ext_vector_type(VEC), aligned(8)));
        const vd t = *reinterpret_cast<const vd*>(static_cast<const double*>(x) + i);
#pragma unroll
        for (int v = 0; v < VEC; ++v) xv[v] = static_cast<ACC>(t[v]);
    } else {
        typedef float vf __attribute__((ext_vector_type(VEC), aligned(4)));
        const vf t = *reinterpret_cast<const vf*>(static_cast<const float*>(x) + i);
#pragma unroll
        for (int v = 0; v < VEC; ++v) xv[v] = static_cast<ACC>(t[v]);
    }
#pragma unroll
    for (int v = 0; v < VEC - 1; ++v)
        if (v < lo) xv[v] = ACC(0);
}

// Stores alpha*acc + beta*y (y not read when beta == 0); returns the
// stored value.
__device__ __forceinline__ double store_y(void* __restrict__ y, bool y64, int64_t i, double alpha,
                                          double acc, double beta) {
    if (y64) {
        double* p = static_cast<double*>(y) + i;
        double r = alpha * acc;
        if (beta != 0.0) r += beta * (*p);
        *p = r;
        return r;
    } else {
        float* p = static_cast<float*>(y) + i;
        double r = alpha * acc;
        if (beta != 0.0) r += beta * static_cast<double>(*p);
        const float f = static_cast<float>(r);
        *p = f;
        return static_cast<double>(f);
    }
}

// Block-wide FP64 sum, fixed order; every thread of the block must call it.
__device__ __forceinline__ void block_sumsq_out(double v, double* out) {
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    __shared__ double part[16];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = part[0];
        for (unsigned w = 1; w < blockDim.x / 64; ++w) s += part[w];
        *out = s;
    }
}

// ------------------------------------------------------------ NO_TRANSPOSE
// Columns whose loads are in flight together (EXACT: two planes, and 8 would
// take 256 VGPRs).
template <int DEC>
constexpr int kBatchCols = DEC == DEC_EXACT ? 4 : 8;

// acc += A[i0 .. i0+VEC, j0 .. j1) x[j0 .. j1): U columns' loads in flight.
// The indices of whole batches need no clamping: with it, its scalar
// operations ahead of every batch's loads took 1050000 x 300 bf16 hi from 110
// to 126 us.
template <int FMT, int DEC, int VEC, class ACC, bool NTL>
__device__ __forceinline__ void sweep_columns(const void* __restrict__ a, const uint16_t* __restrict__ wr,
                                              int64_t lda, const void* __restrict__ x, bool x64, int64_t i0,
                                              int64_t j0, int64_t j1, ACC (&acc)[VEC]) {
    constexpr int U = kBatchCols<DEC>;
    int64_t j = j0;
    for (; j + U <= j1; j += U) {
        Raw<FMT, DEC, VEC> R[U];
        ACC xs[U];
#pragma unroll
        for (int u = 0; u < U; ++u) load_raw<FMT, DEC, VEC, NTL>(a, wr, i0 + (j + u) * lda, R[u]);
        load_x_cols<U, ACC, false>(x, x64, j, j1, xs);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ACC av[VEC];
            decode<FMT, DEC, VEC, ACC>(R[u], av);
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] = fma(av[v], xs[u], acc[v]);
        }
    }
    if (j < j1) {  // the last columns, their loads in flight together as well
        Raw<FMT, DEC, VEC> R[U];
        ACC xs[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j + u < j1) load_raw<FMT, DEC, VEC, NTL>(a, wr, i0 + (j + u) * lda, R[u]);
        load_x_cols<U, ACC, true>(x, x64, j, j1, xs);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (j + u < j1) {
                ACC av[VEC];
                decode<FMT, DEC, VEC, ACC>(R[u], av);
#pragma unroll
                for (int v = 0; v < VEC; ++v) acc[v] = fma(av[v], xs[u], acc[v]);
            }
        }
    }
}

// The same sum in FP64 from ACC sums over at most `chain` columns (a multiple
// of the batch) each; FP64 sums throughout when ACC is double.
template <int FMT, int DEC, int VEC, class ACC, bool NTL>
__device__ __forceinline__ void sweep_chains(const void* __restrict__ a, const uint16_t* __restrict__ wr,
                                             int64_t lda, const void* __restrict__ x, bool x64, int64_t i0,
                                             int64_t j0, int64_t j1, int64_t chain, double (&sum)[VEC]) {
    if constexpr (sizeof(ACC) == 8) {
        sweep_columns<FMT, DEC, VEC, ACC, NTL>(a, wr, lda, x, x64, i0, j0, j1, sum);
    } else {
        for (int64_t c0 = j0; c0 < j1; c0 += chain) {
            ACC acc[VEC];
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] = ACC(0);
            sweep_columns<FMT, DEC, VEC, ACC, NTL>(a, wr, lda, x, x64, i0, c0, min(j1, c0 + chain), acc);
#pragma unroll
            for (int v = 0; v < VEC; ++v) sum[v] += static_cast<double>(acc[v]);
        }
    }
}

// First row of a lane's vector: i, or m - VEC where the vector would run
// past the matrix (the lane then reads rows of its neighbour as well and
// uses only its own).
template <int VEC>
__device__ __forceinline__ int64_t first_row(int64_t i, int64_t m) {
    return min(i, m - VEC);
}

// A lane owns VEC rows and all columns.  Bound by HBM when the rows alone
// fill the chip (plan_n).
template <int FMT, int DEC, int VEC, class ACC, bool NTL>
__global__ __launch_bounds__(kThreads) void gemv_n_kernel(
    int64_t m, int64_t n, const void* __restrict__ a, const uint16_t* __restrict__ wr,
    int64_t lda, const void* __restrict__ x, bool x64, void* __restrict__ y, bool y64, Coef coef, int64_t chain) {
    if (coef.skip && *coef.skip) return;
    const int64_t ir = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) * VEC;
    double acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = 0.0;
    const int64_t i0 = first_row<VEC>(ir, m);
    if (ir < m) sweep_chains<FMT, DEC, VEC, ACC, NTL>(a, wr, lda, x, x64, i0, 0, n, chain, acc);
    const double al = read_coef(coef.alpha, coef.dalpha, coef.alpha_mul);
    const double be = read_coef(coef.beta, coef.dbeta, coef.beta_mul);
    double sq = 0.0;
    if (ir < m) {
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            if (i0 + v >= ir) {
                const double r = store_y(y, y64, i0 + v, al, acc[v], be);
                sq += r * r;
            }
    }
    if (coef.sumsq) block_sumsq_out(sq, coef.sumsq + blockIdx.x);
}

// The rows alone do not fill the chip: a block takes RL x VEC rows and its
// column groups (64 / RL in each wave) split the columns; their sums meet in
// lane shuffles and LDS and are added in group order, in FP64.  One launch
// and no partials in memory: 20000 x 200 bf16 hi 5.2 + 4.1 -> 5.5 us,
// 1e6 x 1000 FP32_16 hi 389 + 5 -> 347 us (5.8 TB/s).  RL = 16, 256-byte runs
// of a column, where there are few row blocks.  A wide matrix is split by
// columns over gridDim.y as well, the sums go to partial[split][m] and
// gemv_n_finish adds them (plan_n).
constexpr int kSplitLds = 512;  // VEC * sizeof(ACC) * waves at most
template <int FMT, int DEC, int VEC, class ACC, int RL, bool NTL>
__global__ __launch_bounds__(kSplitLds / VEC / sizeof(ACC) >= 16 ? 1024 : 64 * (kSplitLds / VEC / sizeof(ACC)))
void gemv_n_split_kernel(int64_t m, int64_t n, const void* __restrict__ a, const uint16_t* __restrict__ wr,
                         int64_t lda, const void* __restrict__ x, bool x64, void* __restrict__ y, bool y64,
                         Coef coef, int64_t split_cols, int64_t col_chunk, int64_t chain, ACC* __restrict__ partial) {
    if (coef.skip && *coef.skip) return;
    constexpr int kStride = RL + 1;  // v-major slots, odd stride: reads of consecutive rows spread over the banks
    extern __shared__ double red[];  // [waves][VEC][kStride]
    const int lane = threadIdx.x & 63, rl = lane % RL;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int64_t b0 = static_cast<int64_t>(blockIdx.x) * RL * VEC;
    const int64_t ir = b0 + rl * VEC;
    double acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = 0.0;
    const int64_t i0 = first_row<VEC>(ir, m);
    if (ir < m) {
        const int64_t c0 = blockIdx.y * split_cols, c1 = min(n, c0 + split_cols);
        const int64_t j0 = c0 + (RL == 64 ? wave * col_chunk : (wave * (64 / RL) + lane / RL) * col_chunk);
        sweep_chains<FMT, DEC, VEC, ACC, NTL>(a, wr, lda, x, x64, i0, j0, min(c1, j0 + col_chunk), chain, acc);
    }
#pragma unroll
    for (int o = RL; o < 64; o *= 2)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] += __shfl_xor(acc[v], o);
    if (ir < m && lane < RL) {
        const int sh = static_cast<int>(ir - i0);
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            if (v >= sh) red[(wave * VEC + v - sh) * kStride + rl] = acc[v];
    }
    __syncthreads();
    const double al = read_coef(coef.alpha, coef.dalpha, coef.alpha_mul);
    const double be = read_coef(coef.beta, coef.dbeta, coef.beta_mul);
    double sq = 0.0;
    for (int r = threadIdx.x; r < RL * VEC && b0 + r < m; r += blockDim.x) {
        double s = 0.0;
        for (int w = 0; w < waves; ++w) s += red[(w * VEC + r % VEC) * kStride + r / VEC];
        if (partial) {
            partial[blockIdx.y * m + b0 + r] = static_cast<ACC>(s);
        } else {
            const double t = store_y(y, y64, b0 + r, al, s, be);
            sq += t * t;
        }
    }
    if (coef.sumsq && !partial) block_sumsq_out(sq, coef.sumsq + blockIdx.x);
}

// y from the column splits' partial sums, in split order, FP64.
template <class ACC>
__global__ __launch_bounds__(kThreads) void gemv_n_finish(int64_t m, int splits, const ACC* __restrict__ partial,
                                                          void* __restrict__ y, bool y64, Coef coef) {
    if (coef.skip && *coef.skip) return;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    double sq = 0.0;
    if (i < m) {
        double s = 0.0;
        for (int c = 0; c < splits; c += 8) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[u] = c + u < splits ? static_cast<double>(partial[static_cast<int64_t>(c + u) * m + i]) : 0.0;
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
        const double r = store_y(y, y64, i, read_coef(coef.alpha, coef.dalpha, coef.alpha_mul), s,
                                 read_coef(coef.beta, coef.dbeta, coef.beta_mul));
        sq = r * r;
    }
    if (coef.sumsq) block_sumsq_out(sq, coef.sumsq + blockIdx.x);
}

// --------------------------------------------------------------- TRANSPOSE
// Transpose-reduce across a wave: L values per lane in, after log2(L)
// exchange stages lane l holds the wave sum of column l / (64 / L).
template <int L, int OFF, class T>
struct WaveTR {
    static __device__ __forceinline__ void run(T* v, int lane) {
        const bool upper = (lane & OFF) != 0;
#pragma unroll
        for (int t = 0; t < L / 2; ++t) {
            const T send = upper ? v[t] : v[t + L / 2];
            const T keep = upper ? v[t + L / 2] : v[t];
            v[t] = keep + __shfl_xor(send, OFF);
        }
        WaveTR<L / 2, OFF / 2, T>::run(v, lane);
    }
};
template <int OFF, class T>
struct WaveTR<1, OFF, T> {
    static __device__ __forceinline__ void run(T* v, int) {
#pragma unroll
        for (int o = OFF; o >= 1; o >>= 1) v[0] += __shfl_xor(v[0], o);
    }
};

// Replaces the first `lo` rows of a vector by zero words: their x is zero,
// but they may hold Inf.  On the raw words, so that the decode stays next to
// its FMA (one v_fma_mix for a half).  A zero word is finite in every format
// and not one of FP32_16's saturated words, which would send the last vector
// of every column through dot_rows' slow path (300 x 4000 EXACT: 24 -> 13 us).
template <int FMT, int DEC, int VEC>
__device__ __forceinline__ void clear_rows(Raw<FMT, DEC, VEC>& R, int lo) {
    if (VEC == 1) return;
#pragma unroll
    for (int v = 0; v < VEC - 1; ++v)
        if (v < lo) {
            if constexpr (is16<FMT>()) {
                const uint32_t keep = 0xFFFF0000u >> (16 * (v & 1));
                R.h[v / 2] &= keep;
                if constexpr (DEC == DEC_EXACT) R.r[v / 2] &= keep;
            } else if constexpr (FMT == FMT_F32) {
                R.h[v] = 0;
            } else {
                R.h[2 * v] = R.h[2 * v + 1] = 0;
            }
        }
}

template <int FMT, int DEC, int VEC, class ACC>
__device__ __forceinline__ ACC dot_rows(Raw<FMT, DEC, VEC>& R, const ACC (&xv)[VEC], int lo, bool edge, ACC s) {
    if (edge) clear_rows<FMT, DEC, VEC>(R, lo);  // wave-uniform: skipped but at the last rows
    if constexpr (FMT == FMT_P16 && DEC == DEC_EXACT && VEC == 8) {
        if (__builtin_expect(__any(saturated(R)), 0)) {
            // element by element in a rolled loop that shifts the vector down:
            // unrolled here, a block of columns overflows the instruction cache
            Raw<FMT, DEC, VEC> q = R;
            ACC xs[VEC];
#pragma unroll
            for (int v = 0; v < VEC; ++v) xs[v] = xv[v];
#pragma clang loop unroll(disable)
            for (int e = 0; e < VEC; ++e) {
                s = fma(static_cast<ACC>(decode16<FMT, DEC>(q.h[0] & 0xFFFFu, q.r[0] & 0xFFFFu)), xs[0], s);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    q.h[k] = (q.h[k] >> 16) | (k < 3 ? q.h[(k + 1) & 3] << 16 : 0u);
                    q.r[k] = (q.r[k] >> 16) | (k < 3 ? q.r[(k + 1) & 3] << 16 : 0u);
                }
#pragma unroll
                for (int v = 0; v < VEC - 1; ++v) xs[v] = xs[v + 1];
            }
            return s;
        }
    }
    ACC av[VEC];
    decode<FMT, DEC, VEC, ACC, false>(R, av);
#pragma unroll
    for (int v = 0; v < VEC; ++v) s = fma(av[v], xv[v], s);
    return s;
}

template <int FMT, int DEC, int VEC, class ACC, int CB, bool NTL>
__global__ __launch_bounds__(kThreads) void gemv_t_kernel(
    int64_t m, int64_t n, const void* __restrict__ a, const uint16_t* __restrict__ wr,
    int64_t lda, const void* __restrict__ x, bool x64, int64_t rows_per_chunk, int ncg,
    ACC* __restrict__ partial, const int* __restrict__ skip) {
    if (skip && *skip) return;
    const int bid = blockIdx.x;
    const int chunk = bid / ncg;
    const int cg = bid - chunk * ncg;
    const int64_t r0 = static_cast<int64_t>(chunk) * rows_per_chunk;
    const int64_t r1 = min(m, r0 + rows_per_chunk);
    const int64_t c0 = static_cast<int64_t>(cg) * CB;
    const int ncols = static_cast<int>(min<int64_t>(CB, n - c0));

    ACC acc[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[c] = ACC(0);

    constexpr int UB = DEC == DEC_EXACT ? 4 : 8;
    for (int64_t ir = r0 + static_cast<int64_t>(threadIdx.x) * VEC; ir < r1;
         ir += static_cast<int64_t>(kThreads) * VEC) {
        const int64_t i = first_row<VEC>(ir, m);
        const int lo = static_cast<int>(ir - i);
        ACC xv[VEC];
        load_x_rows<VEC, ACC>(x, x64, i, lo, xv);
        const bool edge = __any(lo != 0);
        const int64_t base = i + c0 * lda;
        // batches of UB columns, the next batch's loads in flight during this
        // one's sums; past the last column the last one again, its sum unused
        Raw<FMT, DEC, VEC> R[2][UB];
#pragma unroll
        for (int u = 0; u < UB; ++u)
            load_raw<FMT, DEC, VEC, NTL>(a, wr, base + min(u, ncols - 1) * lda, R[0][u]);
#pragma unroll
        for (int cb = 0; cb < CB; cb += UB) {
            if (cb < ncols) {
                if (cb + UB < ncols) {
#pragma unroll
                    for (int u = 0; u < UB; ++u)
                        load_raw<FMT, DEC, VEC, NTL>(a, wr, base + min(cb + UB + u, ncols - 1) * lda,
                                                     R[(cb / UB + 1) & 1][u]);
                }
#pragma unroll
                for (int u = 0; u < UB; ++u)
                    acc[cb + u] = dot_rows<FMT, DEC, VEC, ACC>(R[(cb / UB) & 1][u], xv, lo, edge, acc[cb + u]);
            }
        }
    }

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    WaveTR<CB, 32, ACC>::run(acc, lane);
    __shared__ ACC red[kThreads / 64][CB];
    constexpr int kGroup = 64 / CB;
    if ((lane % kGroup) == 0) red[wave][lane / kGroup] = acc[0];
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < ncols) {
        const int c = threadIdx.x;
        const ACC s = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
        partial[static_cast<int64_t>(chunk) * n + c0 + c] = s;
    }
}

// Short columns: a block owns CG whole columns, so there are no chunk
// partials and no second launch.  Each lane walks the rows in steps of the
// block with the loads of four row steps in flight; a vector's VEC products
// are summed in ACC, everything above that in FP64.  `partial` != nullptr:
// the sums go there (one chunk) instead of y.  20000 x 200 bf16 hi:
// 13.4 + 3.5 (chunks and their sum) -> 5.0 us; R^-T v, 300 x 300 FP64: 8.1 -> 4.0.
constexpr int kColThreads = 512;
template <int FMT, int DEC, int VEC, class ACC, int CG, bool NTL>
__global__ __launch_bounds__(kColThreads) void gemv_t_cols_kernel(
    int64_t m, int64_t n, const void* __restrict__ a, const uint16_t* __restrict__ wr, int64_t lda,
    const void* __restrict__ x, bool x64, ACC* __restrict__ partial, void* __restrict__ y, bool y64, Coef coef) {
    if (coef.skip && *coef.skip) return;
    constexpr int U = 4;
    const int64_t c0 = static_cast<int64_t>(blockIdx.x) * CG;
    const int ncols = static_cast<int>(min<int64_t>(CG, n - c0));
    double acc[CG];
#pragma unroll
    for (int c = 0; c < CG; ++c) acc[c] = 0.0;
    constexpr int64_t kStep = static_cast<int64_t>(kColThreads) * VEC;
    for (int64_t ir = static_cast<int64_t>(threadIdx.x) * VEC; ir < m; ir += U * kStep) {
        Raw<FMT, DEC, VEC> R[U][CG];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (ir + u * kStep < m) {
                const int64_t base = first_row<VEC>(ir + u * kStep, m) + c0 * lda;
#pragma unroll
                for (int c = 0; c < CG; ++c)
                    load_raw<FMT, DEC, VEC, NTL>(a, wr, base + min(c, ncols - 1) * lda, R[u][c]);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (ir + u * kStep < m) {
                const int64_t i = first_row<VEC>(ir + u * kStep, m);
                const int lo = static_cast<int>(ir + u * kStep - i);
                ACC xv[VEC];
                load_x_rows<VEC, ACC>(x, x64, i, lo, xv);
                const bool edge = __any(lo != 0);
#pragma unroll
                for (int c = 0; c < CG; ++c)
                    acc[c] += static_cast<double>(dot_rows<FMT, DEC, VEC, ACC>(R[u][c], xv, lo, edge, ACC(0)));
            }
    }
    __shared__ double red[kColThreads / 64][CG];
#pragma unroll
    for (int c = 0; c < CG; ++c) {
        for (int o = 32; o >= 1; o >>= 1) acc[c] += __shfl_xor(acc[c], o);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = acc[c];
    }
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < ncols) {
        const int c = threadIdx.x;
        double s = 0.0;
        for (int w = 0; w < kColThreads / 64; ++w) s += red[w][c];
        if (partial) partial[c0 + c] = static_cast<ACC>(s);
        else
            store_y(y, y64, c0 + c, read_coef(coef.alpha, coef.dalpha, coef.alpha_mul), s,
                    read_coef(coef.beta, coef.dbeta, coef.beta_mul));
    }
}

// Short columns and many of them: a wave owns CG whole columns (a strided
// loop over the column groups bounds the grid), so that lanes without a row
// cost a wave and not a block of 512, and the loads of CG columns are in
// flight together; sums as in gemv_t_cols_kernel.  Bound by HBM: 4000 x
// 60000 bf16 hi 76 us (6.3 TB/s; that kernel 106, row chunks of 64 columns
// 82), 64 x 1000000 62 us (1195, 228).
constexpr int kWaveCols = 8;
constexpr int64_t kWaveBlocks = int64_t(1) << 18;
template <int FMT, int DEC, int VEC, class ACC, int CG, bool NTL>
__global__ __launch_bounds__(kThreads) void gemv_t_wave_kernel(
    int64_t m, int64_t n, const void* __restrict__ a, const uint16_t* __restrict__ wr, int64_t lda,
    const void* __restrict__ x, bool x64, ACC* __restrict__ partial, void* __restrict__ y, bool y64, Coef coef) {
    if (coef.skip && *coef.skip) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * (kThreads / 64);
    for (int64_t c0 = (static_cast<int64_t>(blockIdx.x) * (kThreads / 64) + wave) * CG; c0 < n; c0 += waves * CG) {
        const int ncols = static_cast<int>(min<int64_t>(CG, n - c0));
        double acc[CG];
#pragma unroll
        for (int c = 0; c < CG; ++c) acc[c] = 0.0;
        for (int64_t ir = static_cast<int64_t>(lane) * VEC; ir < m; ir += 64 * VEC) {
            const int64_t i = first_row<VEC>(ir, m);
            const int lo = static_cast<int>(ir - i);
            Raw<FMT, DEC, VEC> R[CG];
#pragma unroll
            for (int c = 0; c < CG; ++c)
                load_raw<FMT, DEC, VEC, NTL>(a, wr, i + (c0 + min(c, ncols - 1)) * lda, R[c]);
            ACC xv[VEC];
            load_x_rows<VEC, ACC>(x, x64, i, lo, xv);
            const bool edge = __any(lo != 0);
#pragma unroll
            for (int c = 0; c < CG; ++c)
                acc[c] += static_cast<double>(dot_rows<FMT, DEC, VEC, ACC>(R[c], xv, lo, edge, ACC(0)));
        }
        WaveTR<CG, 32, double>::run(acc, lane);
        const int c = lane / (64 / CG);
        if (lane % (64 / CG) == 0 && c < ncols) {
            if (partial) partial[c0 + c] = static_cast<ACC>(acc[0]);
            else
                store_y(y, y64, c0 + c, read_coef(coef.alpha, coef.dalpha, coef.alpha_mul), acc[0],
                        read_coef(coef.beta, coef.dbeta, coef.beta_mul));
        }
    }
}

// Adds the chunk partials of 32 columns: 8 chunk slices per column (a slice
// takes every eighth chunk, four loads in flight), added in slice order
// (64 chunks x 501: 7.0 us with a thread per column, 5.1 with the slices).
constexpr int kFinCols = 32, kFinSlices = kThreads / kFinCols;
template <class ACC>
__global__ __launch_bounds__(kThreads) void gemv_t_finish(int64_t n, int chunks,
                                                          const ACC* __restrict__ partial,
                                                          void* __restrict__ y, bool y64,
                                                          Coef coef) {
    if (coef.skip && *coef.skip) return;
    const int col = threadIdx.x % kFinCols, slice = threadIdx.x / kFinCols;
    const int64_t j = static_cast<int64_t>(blockIdx.x) * kFinCols + col;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (j < n)
        for (int c = slice; c < chunks; c += 4 * kFinSlices)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c + q * kFinSlices < chunks)
                    s[q] += static_cast<double>(partial[static_cast<int64_t>(c + q * kFinSlices) * n + j]);
    __shared__ double red[kFinSlices][kFinCols];
    red[slice][col] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (slice != 0 || j >= n) return;
    double t = 0.0;
    for (int q = 0; q < kFinSlices; ++q) t += red[q][col];
    store_y(y, y64, j, read_coef(coef.alpha, coef.dalpha, coef.alpha_mul), t,
            read_coef(coef.beta, coef.dbeta, coef.beta_mul));
}

// ------------------------------------------------------------------ plans
struct Kind {
    int fmt, dec;
    bool acc64;
};

Kind classify(int a_type, int tier) {
    require(tier == TOMOS_TIER_DEFAULT || tier == TOMOS_TIER_FAST || tier == TOMOS_TIER_EXACT,
            "gemv: unknown tier");
    switch (a_type) {
        case TOMOS_F32: return {FMT_F32, DEC_NATIVE, tier != TOMOS_TIER_DEFAULT};
        case TOMOS_F64: return {FMT_F64, DEC_NATIVE, true};
        case TOMOS_FP32_16:
            return {FMT_P16, tier == TOMOS_TIER_EXACT ? DEC_EXACT : DEC_HI, tier != TOMOS_TIER_DEFAULT};
        case TOMOS_FP32_BF16:
            return {FMT_PBF, tier == TOMOS_TIER_EXACT ? DEC_EXACT : DEC_HI, tier != TOMOS_TIER_DEFAULT};
        // native 16-bit storage: the stored value is the exact one, so EXACT
        // (like FAST) decodes it and accumulates in FP64
        case TOMOS_BF16: return {FMT_PBF, DEC_HI, tier != TOMOS_TIER_DEFAULT};
        case TOMOS_F16: return {FMT_H16, DEC_HI, tier != TOMOS_TIER_DEFAULT};
        default:
            throw Error(kErrUnsupported, "gemv: unsupported matrix type " + std::to_string(a_type));
    }
}

int vec_full_of(int fmt) { return fmt == FMT_F64 ? 2 : (fmt == FMT_F32 ? 4 : 8); }
// Bytes of A that an element's product reads.
constexpr int64_t elem_bytes(int fmt, int dec) {
    return fmt == FMT_F64 ? 8 : (fmt == FMT_F32 || dec == DEC_EXACT ? 4 : 2);
}
int cb_of(const Kind& k) { return k.acc64 ? 32 : 64; }
constexpr int64_t kTargetBlocks = 1024;

// Column splits that the scratch of a NO_TRANSPOSE call holds partial sums
// of (0: none).
int n_scratch_splits(const Kind& k, int64_t m, int64_t n) {
    const int64_t bx = ceil_div(m, static_cast<int64_t>(kThreads) * vec_full_of(k.fmt));
    if (bx >= kTargetBlocks / 2 || n <= 16) return 0;
    const int64_t s = std::min(ceil_div(kTargetBlocks, bx), std::min<int64_t>(ceil_div(n, 8), 32));
    const int64_t splits = ceil_div(n, ceil_div(n, s));
    return splits > 1 ? static_cast<int>(splits) : 0;
}

// NO_TRANSPOSE.  waves = 1: a lane's rows to itself (gemv_n_kernel), from
// kTargetWaves / 2 waves of rows up (530000 x 50 F32 23.6 us with two waves a
// block that split the columns, 19.3 without).  Below, the waves of a block
// split the columns (gemv_n_split_kernel) until about kTargetWaves waves
// share the work, two columns a wave at least; blocks of 16 row lanes while
// 64-lane blocks are under a quarter of the wanted waves.  splits > 1: the
// columns are split over the grid as well (split_pays).
struct PlanN {
    int waves, row_lanes, splits;
    int64_t blocks, split_cols, col_chunk, chain;
};
constexpr int64_t kTargetWaves = 4096;
// Whether `bytes` of A in few blocks are read sooner by more of them, at the
// cost of a second launch (10 us with the partial sums).  A block reads 75 GB/s
// of a matrix that the caches hold and 36 (16 row lanes) or 40 of one that
// they do not, FP32_16's decode bounds it to 28 (hi) and 26 or 40 (EXACT); the
// chip reads 5.5, 6.2 and 4.8 TB/s.  us, one launch / two: 300 x 100000 F32
// 390 / 36, 16384 x 10000 bf16 hi 76 / 58, but 16384 x 4000 24 / 32 and 60000 x
// 1000 EXACT 50 / 62 (these two stay at one).
bool split_pays(const Kind& k, int64_t blocks, int row_lanes, double bytes) {
    if (blocks >= 200) return false;
    const bool cached = bytes <= static_cast<double>(kStreamLoadBytes), p16 = k.fmt == FMT_P16;
    const double wide = row_lanes == 64 ? 40e3 : 36e3;  // bytes per us
    const double block = !p16 ? (cached ? 75e3 : wide) : (k.dec == DEC_HI ? 28e3 : row_lanes == 64 ? 40e3 : 26e3);
    const double chip = p16 ? 4.8e6 : (cached ? 5.5e6 : 6.2e6);
    return bytes / std::min(static_cast<double>(blocks) * block, chip) > bytes / chip + 10.0;
}
constexpr int64_t kSplitWork = int64_t(64) << 10;  // bytes of A for a block of a split at least
PlanN plan_n(const Kind& k, int64_t m, int64_t n) {
    PlanN p;
    const int64_t v = m >= vec_full_of(k.fmt) ? vec_full_of(k.fmt) : 1;
    const int64_t row_waves = ceil_div(m, 64 * v);
    const int64_t most = std::min<int64_t>(16, kSplitLds / (v * (k.acc64 ? 8 : 4)));
    int64_t w = 1;
    if (row_waves < kTargetWaves / 2)
        while (w < most && row_waves * w < kTargetWaves && n >= 4 * w) w *= 2;
    p.waves = static_cast<int>(w);
    p.row_lanes = row_waves * w < kTargetWaves / 4 && n >= 4 * w ? 16 : 64;
    p.blocks = w > 1 ? ceil_div(m, p.row_lanes * v) : ceil_div(m, kThreads * v);
    // FP32 sums run over 8 to 64 columns and meet in FP64: the fewer rows, the
    // fewer columns, down to n / 32, what a split of the scratch stands for
    const int64_t parts = n_scratch_splits(k, m, n);
    p.chain = std::min<int64_t>(std::max<int64_t>(n / std::max<int64_t>(parts, 1) / 8 * 8, 8), 64);
    p.splits = 1;
    const int64_t eb = elem_bytes(k.fmt, k.dec);
    if (w > 1 && split_pays(k, p.blocks, p.row_lanes, static_cast<double>(m) * static_cast<double>(n * eb))) {
        if (row_waves * parts >= 512) {  // enough blocks with whole 1 KB runs of a column
            p.row_lanes = 64;
            p.blocks = row_waves;
        }
        const int64_t most_splits = std::min(ceil_div(kTargetBlocks, p.blocks), p.row_lanes * v * n * eb / kSplitWork);
        p.splits = static_cast<int>(std::max<int64_t>(std::min(parts, most_splits), 1));
    }
    p.split_cols = ceil_div(std::max<int64_t>(n, 1), p.splits);
    p.splits = static_cast<int>(ceil_div(std::max<int64_t>(n, 1), p.split_cols));
    p.col_chunk = ceil_div(p.split_cols, w * (64 / p.row_lanes));
    return p;
}

struct PlanT {
    int ncg;
    int64_t rows_per_chunk;
    int chunks;
};
PlanT plan_t(const Kind& k, int64_t m, int64_t n) {
    PlanT p;
    const int64_t cb = cb_of(k);
    p.ncg = static_cast<int>(ceil_div(std::max<int64_t>(n, 1), cb));
    const int64_t step = static_cast<int64_t>(kThreads) * vec_full_of(k.fmt);
    const int64_t row_steps = std::max<int64_t>(ceil_div(m, step), 1);
    const int64_t want_chunks = std::max<int64_t>(1, ceil_div(kTargetBlocks, p.ncg));
    const int64_t kr = std::min<int64_t>(std::max<int64_t>(ceil_div(row_steps, want_chunks), 1), 64);
    p.rows_per_chunk = kr * step;
    p.chunks = static_cast<int>(std::max<int64_t>(ceil_div(m, p.rows_per_chunk), 1));
    return p;
}

// TRANSPOSE: whole columns up to kColBytes bytes each, longer ones are cut
// into row chunks.  A block of 512 threads takes them (gemv_t_cols_kernel),
// or a wave (gemv_t_wave_kernel) where there are enough for every CU: above
// 4096 columns of up to 4 KB, which leave most of a block's lanes without a
// row (1000 x 5000 FP32_16 EXACT 16.8 us by blocks, 9.6 by waves), above 8192
// of up to 24 KB (4000 x 5000 hi 11.9 and 15.1, 4000 x 60000 118 and 81); of
// longer ones a block's loads are as many (16000 x 10000 66 and 78).
constexpr int64_t kColBytes = int64_t(128) << 10;
bool t_waves(int64_t col_bytes, int64_t n) {
    return col_bytes <= (int64_t(24) << 10) && n > (col_bytes <= 4096 ? 4096 : 8192);
}
bool t_cols(const Kind& k, int64_t m) {
    return m * elem_bytes(k.fmt, k.dec) <= kColBytes;
}

// The kind a GEMV runs with: F32 GEMV^T accumulates in FP64 in every tier
// (the FP64-sum kernel streams A faster on gfx950 than the FP32-sum one,
// and it is the more accurate; the reference's tiled FP32 GEMV accumulates
// in FP64 too, mv_cuda_kernels.cu:863-990).
Kind kind_for(int a_type, int tier, int trans) {
    Kind k = classify(a_type, tier);
    if (trans == TOMOS_TRANSPOSE && k.fmt == FMT_F32) k.acc64 = true;
    return k;
}

size_t scratch_for(const Kind& k, int trans, int64_t m, int64_t n) {
    const size_t acc = k.acc64 ? 8 : 4;
    if (trans == TOMOS_NO_TRANSPOSE) {
        return static_cast<size_t>(n_scratch_splits(k, m, n)) * static_cast<size_t>(m) * acc;
    }
    PlanT p = plan_t(k, m, n);
    return static_cast<size_t>(p.chunks) * static_cast<size_t>(n) * acc;
}

// Whether a pass over the matrix uses non-temporal loads: columns on 16-byte
// boundaries only, since a vector that straddles two cache lines wants the
// line kept for its neighbour (131071 x 501 EXACT, odd lda: N 115 us
// non-temporal, 77 us cacheable).
template <int FMT, int DEC>
bool streams(int64_t m, int64_t n, int64_t lda) {
    return lda % vec_full<FMT>() == 0 && stream_loads(m * n * elem_bytes(FMT, DEC));
}

template <int FMT, int DEC, int VEC, class ACC, bool NTL>
int launch_n(int64_t m, int64_t n, const void* a, const uint16_t* wr, int64_t lda, const void* x, bool x64,
             void* y, bool y64, const Coef& coef, ACC* partial, const PlanN& p, hipStream_t s) {
    const unsigned blocks = static_cast<unsigned>(p.blocks);
    if (p.waves == 1) {
        gemv_n_kernel<FMT, DEC, VEC, ACC, NTL><<<blocks, kThreads, 0, s>>>(m, n, a, wr, lda, x, x64, y, y64, coef,
                                                                           p.chain);
        TOMOS_LAUNCH_CHECK("gemv_n_kernel");
        return static_cast<int>(blocks);
    }
    const dim3 grid(blocks, static_cast<unsigned>(p.splits));
    const size_t lds = static_cast<size_t>(p.waves) * VEC * (p.row_lanes + 1) * sizeof(double);
    if (p.row_lanes == 16)
        gemv_n_split_kernel<FMT, DEC, VEC, ACC, 16, NTL><<<grid, 64 * p.waves, lds, s>>>(
            m, n, a, wr, lda, x, x64, y, y64, coef, p.split_cols, p.col_chunk, p.chain, partial);
    else
        gemv_n_split_kernel<FMT, DEC, VEC, ACC, 64, NTL><<<grid, 64 * p.waves, lds, s>>>(
            m, n, a, wr, lda, x, x64, y, y64, coef, p.split_cols, p.col_chunk, p.chain, partial);
    TOMOS_LAUNCH_CHECK("gemv_n_split_kernel");
    if (!partial) return static_cast<int>(blocks);
    const unsigned fb = static_cast<unsigned>(ceil_div(m, kThreads));
    gemv_n_finish<ACC><<<fb, kThreads, 0, s>>>(m, p.splits, partial, y, y64, coef);
    TOMOS_LAUNCH_CHECK("gemv_n_finish");
    return static_cast<int>(fb);
}

template <int FMT, int DEC, class ACC>
int run_n(int64_t m, int64_t n, const void* a, const uint16_t* wr, int64_t lda, const void* x,
          bool x64, void* y, bool y64, const Coef& coef, void* scratch, const PlanN& p, hipStream_t s) {
    constexpr int VF = vec_full<FMT>();
    ACC* part = static_cast<ACC*>(scratch);
    if (m < VF)
        return launch_n<FMT, DEC, 1, ACC, false>(m, n, a, wr, lda, x, x64, y, y64, coef, part, p, s);
    if (streams<FMT, DEC>(m, n, lda))
        return launch_n<FMT, DEC, VF, ACC, true>(m, n, a, wr, lda, x, x64, y, y64, coef, part, p, s);
    return launch_n<FMT, DEC, VF, ACC, false>(m, n, a, wr, lda, x, x64, y, y64, coef, part, p, s);
}

template <int FMT, int DEC, int VEC, class ACC, bool NTL>
void launch_t_cols(int64_t m, int64_t n, const void* a, const uint16_t* wr, int64_t lda, const void* x, bool x64,
                   ACC* part, void* y, bool y64, const Coef& coef, hipStream_t s) {
    // one column a block while that fills the chip about twice, then two, then four
    if (t_waves(m * elem_bytes(FMT, DEC), n))
        gemv_t_wave_kernel<FMT, DEC, VEC, ACC, kWaveCols, NTL>
            <<<static_cast<unsigned>(std::min(ceil_div(n, kWaveCols * (kThreads / 64)), kWaveBlocks)), kThreads, 0, s>>>(
                m, n, a, wr, lda, x, x64, part, y, y64, coef);
    else if (n <= 512)
        gemv_t_cols_kernel<FMT, DEC, VEC, ACC, 1, NTL><<<static_cast<unsigned>(n), kColThreads, 0, s>>>(
            m, n, a, wr, lda, x, x64, part, y, y64, coef);
    else if (n <= 1024)
        gemv_t_cols_kernel<FMT, DEC, VEC, ACC, 2, NTL><<<static_cast<unsigned>(ceil_div(n, 2)), kColThreads, 0, s>>>(
            m, n, a, wr, lda, x, x64, part, y, y64, coef);
    else
        gemv_t_cols_kernel<FMT, DEC, VEC, ACC, 4, NTL><<<static_cast<unsigned>(ceil_div(n, 4)), kColThreads, 0, s>>>(
            m, n, a, wr, lda, x, x64, part, y, y64, coef);
    TOMOS_LAUNCH_CHECK("gemv_t_cols_kernel");
}

// Returns the number of chunk partials written when `finish` is false.
template <int FMT, int DEC, class ACC>
int run_t(int64_t m, int64_t n, const void* a, const uint16_t* wr, int64_t lda, const void* x,
          bool x64, void* y, bool y64, const Coef& coef, void* scratch, bool cols,
          const PlanT& p, hipStream_t s, bool finish = true) {
    constexpr int VF = vec_full<FMT>();
    constexpr int CB = sizeof(ACC) == 8 ? 32 : 64;
    ACC* part = static_cast<ACC*>(scratch);
    if (cols && m > 0) {
        ACC* one = finish ? nullptr : part;
        if (m < VF)
            launch_t_cols<FMT, DEC, 1, ACC, false>(m, n, a, wr, lda, x, x64, one, y, y64, coef, s);
        // non-temporal above what the last-level cache holds (60000 x 2000
        // bf16 hi, 240 MB, again and again: 36 us cacheable, 41 not)
        else if (DEC != DEC_EXACT && m * n * elem_bytes(FMT, DEC) > (int64_t(256) << 20) && streams<FMT, DEC>(m, n, lda))
            launch_t_cols<FMT, DEC, VF, ACC, true>(m, n, a, wr, lda, x, x64, one, y, y64, coef, s);
        else
            launch_t_cols<FMT, DEC, VF, ACC, false>(m, n, a, wr, lda, x, x64, one, y, y64, coef, s);
        return 1;
    }
    const int64_t blocks = static_cast<int64_t>(p.chunks) * p.ncg;
    require(blocks < (int64_t(1) << 31), "gemv: grid too large");
    if (m > 0) {
        const dim3 grid(static_cast<unsigned>(blocks));
        // the EXACT tier reads A with cacheable loads: its non-temporal form
        // needs 256 VGPRs (one wave per SIMD), the cacheable one ~140
        if (DEC != DEC_EXACT && m >= VF && streams<FMT, DEC>(m, n, lda))
            gemv_t_kernel<FMT, DEC, VF, ACC, CB, true><<<grid, kThreads, 0, s>>>(
                m, n, a, wr, lda, x, x64, p.rows_per_chunk, p.ncg, part, coef.skip);
        else if (m >= VF)
            gemv_t_kernel<FMT, DEC, VF, ACC, CB, false><<<grid, kThreads, 0, s>>>(
                m, n, a, wr, lda, x, x64, p.rows_per_chunk, p.ncg, part, coef.skip);
        else  // in place only: otherwise whole columns
            gemv_t_kernel<FMT, DEC, 1, ACC, CB, false><<<grid, kThreads, 0, s>>>(
                m, n, a, wr, lda, x, x64, p.rows_per_chunk, p.ncg, part, coef.skip);
        TOMOS_LAUNCH_CHECK("gemv_t_kernel");
    }
    if (!finish) return p.chunks;
    gemv_t_finish<ACC><<<dim3(static_cast<unsigned>(ceil_div(n, kFinCols))), kThreads, 0, s>>>(
        n, m > 0 ? p.chunks : 0, part, y, y64, coef);
    TOMOS_LAUNCH_CHECK("gemv_t_finish");
    return p.chunks;
}

}  // namespace

// Whether x (nx entries) and y (ny entries) share memory.
static bool overlap(const void* x, int x_type, int64_t nx, const void* y, int y_type, int64_t ny) {
    const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), y0 = reinterpret_cast<uintptr_t>(y);
    return x0 < y0 + static_cast<uintptr_t>(ny) * (y_type == TOMOS_F64 ? 8 : 4) &&
           y0 < x0 + static_cast<uintptr_t>(nx) * (x_type == TOMOS_F64 ? 8 : 4);
}

size_t gemv_scratch_bytes(int a_type, int tier, int trans, int64_t m, int64_t n) {
    return scratch_for(kind_for(a_type, tier, trans), trans, m, n);
}

// 16 rows a block at least; split blocks of 16 row lanes only while there are
// under kTargetWaves / 2 of them, otherwise at least 128 rows (m < VEC: one block).
int64_t gemv_sumsq_blocks_max(int64_t m) {
    m = std::max<int64_t>(m, 1);
    return std::min(ceil_div(m, 16), std::max(ceil_div(m, 128), kTargetWaves / 2));
}

void gemv(int a_type, int tier, int trans, const Coef& coef, int64_t m, int64_t n, const void* a,
          const uint16_t* wr, int64_t lda, int x_type, const void* x, int y_type, void* y,
          void* scratch, size_t scratch_bytes, hipStream_t s, int* sumsq_blocks) {
    require(trans == TOMOS_NO_TRANSPOSE || trans == TOMOS_TRANSPOSE, "gemv: bad trans");
    const Kind k = kind_for(a_type, tier, trans);
    require(m >= 0 && n >= 0, "gemv: negative size");
    require(lda >= std::max<int64_t>(m, 1), "gemv: lda < m");
    require(x_type == TOMOS_F32 || x_type == TOMOS_F64, "gemv: x must be F32 or F64");
    require(y_type == TOMOS_F32 || y_type == TOMOS_F64, "gemv: y must be F32 or F64");
    const int64_t rows_out = trans == TOMOS_NO_TRANSPOSE ? m : n;
    require(coef.sumsq == nullptr || trans == TOMOS_NO_TRANSPOSE, "gemv: sumsq needs NO_TRANSPOSE");
    if (sumsq_blocks) *sumsq_blocks = 0;
    if (rows_out == 0) return;
    require(y != nullptr, "gemv: null y");
    const int64_t inner = trans == TOMOS_NO_TRANSPOSE ? n : m;
    if (inner > 0) require(a != nullptr && x != nullptr, "gemv: null A or x");
    if (k.dec == DEC_EXACT) require(wr != nullptr || inner == 0, "gemv: EXACT tier needs the wr plane");
    const size_t need = scratch_for(k, trans, m, n);
    // y over x: by partial sums, which are complete before y is written
    const bool in_place = overlap(x, x_type, inner, y, y_type, rows_out);
    const bool cols = trans == TOMOS_TRANSPOSE && m > 0 && t_cols(k, m) && !in_place;
    PlanN pn{};
    if (trans == TOMOS_NO_TRANSPOSE) pn = plan_n(k, m, n);
    const bool parts = pn.splits > 1 || (in_place && pn.waves > 1 && need > 0);
    if (need > 0) {
        if (scratch == nullptr) {
            if (trans == TOMOS_TRANSPOSE ? !cols : parts) scratch = fallback_scratch(need);
        } else {
            require(scratch_bytes >= need, "gemv: scratch too small (need " + std::to_string(need) +
                                               " bytes)");
        }
    }
    const bool x64 = x_type == TOMOS_F64, y64 = y_type == TOMOS_F64;

    if (trans == TOMOS_NO_TRANSPOSE) {
        // n == 0 falls through with an empty column range: y = beta*y.
        int nb = 0;
#define RUN_N(F, D, A) nb = run_n<F, D, A>(m, n, a, wr, lda, x, x64, y, y64, coef, parts ? scratch : nullptr, pn, s)
        if (k.fmt == FMT_F32) { if (k.acc64) RUN_N(FMT_F32, DEC_NATIVE, double); else RUN_N(FMT_F32, DEC_NATIVE, float); }
        else if (k.fmt == FMT_F64) RUN_N(FMT_F64, DEC_NATIVE, double);
        else if (k.fmt == FMT_H16) { if (k.acc64) RUN_N(FMT_H16, DEC_HI, double); else RUN_N(FMT_H16, DEC_HI, float); }
        else if (k.fmt == FMT_P16) {
            if (k.dec == DEC_EXACT) RUN_N(FMT_P16, DEC_EXACT, double);
            else if (k.acc64) RUN_N(FMT_P16, DEC_HI, double);
            else RUN_N(FMT_P16, DEC_HI, float);
        } else {
            if (k.dec == DEC_EXACT) RUN_N(FMT_PBF, DEC_EXACT, double);
            else if (k.acc64) RUN_N(FMT_PBF, DEC_HI, double);
            else RUN_N(FMT_PBF, DEC_HI, float);
        }
#undef RUN_N
        if (sumsq_blocks) *sumsq_blocks = nb;
    } else {
        const PlanT p = plan_t(k, m, n);
#define RUN_T(F, D, A) run_t<F, D, A>(m, n, a, wr, lda, x, x64, y, y64, coef, scratch, cols, p, s)
        if (k.fmt == FMT_F32) { if (k.acc64) RUN_T(FMT_F32, DEC_NATIVE, double); else RUN_T(FMT_F32, DEC_NATIVE, float); }
        else if (k.fmt == FMT_F64) RUN_T(FMT_F64, DEC_NATIVE, double);
        else if (k.fmt == FMT_H16) { if (k.acc64) RUN_T(FMT_H16, DEC_HI, double); else RUN_T(FMT_H16, DEC_HI, float); }
        else if (k.fmt == FMT_P16) {
            if (k.dec == DEC_EXACT) RUN_T(FMT_P16, DEC_EXACT, double);
            else if (k.acc64) RUN_T(FMT_P16, DEC_HI, double);
            else RUN_T(FMT_P16, DEC_HI, float);
        } else {
            if (k.dec == DEC_EXACT) RUN_T(FMT_PBF, DEC_EXACT, double);
            else if (k.acc64) RUN_T(FMT_PBF, DEC_HI, double);
            else RUN_T(FMT_PBF, DEC_HI, float);
        }
#undef RUN_T
    }
}

int gemv_t_partials(int a_type, int tier, int64_t m, int64_t n, const void* a, const uint16_t* wr,
                    int64_t lda, int x_type, const void* x, void* scratch, size_t scratch_bytes,
                    const int* skip, hipStream_t s) {
    const Kind k = classify(a_type, tier);
    require(k.acc64, "gemv_t_partials: needs an FP64-accumulating tier");
    require(m >= 1 && n >= 1 && lda >= m, "gemv_t_partials: bad sizes");
    const size_t need = scratch_for(k, TOMOS_TRANSPOSE, m, n);
    require(scratch != nullptr && scratch_bytes >= need, "gemv_t_partials: scratch too small");
    const PlanT p = plan_t(k, m, n);
    const bool x64 = x_type == TOMOS_F64;
    const bool cols = t_cols(k, m);
    Coef c;
    c.skip = skip;
    int chunks = 0;
#define RUN_TP(F, D) \
    chunks = run_t<F, D, double>(m, n, a, wr, lda, x, x64, nullptr, false, c, scratch, cols, p, s, false)
    if (k.fmt == FMT_F32) RUN_TP(FMT_F32, DEC_NATIVE);
    else if (k.fmt == FMT_F64) RUN_TP(FMT_F64, DEC_NATIVE);
    else if (k.fmt == FMT_H16) RUN_TP(FMT_H16, DEC_HI);
    else if (k.fmt == FMT_P16) { if (k.dec == DEC_EXACT) RUN_TP(FMT_P16, DEC_EXACT); else RUN_TP(FMT_P16, DEC_HI); }
    else { if (k.dec == DEC_EXACT) RUN_TP(FMT_PBF, DEC_EXACT); else RUN_TP(FMT_PBF, DEC_HI); }
#undef RUN_TP
    return chunks;
}

}  // namespace tomos_hip

using namespace tomos_hip;

extern "C" {

size_t tomos_gemv_scratch_size(int a_type, int tier, int trans, int64_t m, int64_t n) {
    size_t out = 0;
    int rc = guarded([&] {
        require(m >= 0 && n >= 0, "tomos_gemv_scratch_size: negative size");
        out = gemv_scratch_bytes(a_type, tier, trans, m, n);
    });
    return rc == 0 ? out : 0;
}

int tomos_gemv(int a_type, int tier, int trans, double alpha, int64_t m, int64_t n, const void* a,
               const uint16_t* wr, int64_t lda, int x_type, const void* x, double beta,
               int y_type, void* y, void* scratch, size_t scratch_bytes, tomos_stream_t s) {
    return guarded([&] {
        Coef c;
        c.alpha = alpha;
        c.beta = beta;
        gemv(a_type, tier, trans, c, m, n, a, wr, lda, x_type, x, y_type, y, scratch,
             scratch_bytes, s);
    });
}

}  // extern "C"
