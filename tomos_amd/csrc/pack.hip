// Pack (FP32 -> planar wh/wr) and unpack/decode kernels.
//
// Layout: column-major m x n source with leading dimension ld_src, planar
// uint16 wh/wr destinations with leading dimension ld_dst.  One thread
// handles a run of 8 consecutive rows of one column with 16-byte loads and
// stores (32 B of FP32, 16 B of each plane) at element alignment, which
// gfx950 takes for any leading dimension; the rows past the last whole run
// go one by one.  A matrix without padding on either side is one long
// column.  Grid = (row runs, columns): coalesced along rows, HBM-bound (8 B
// moved per element).  500000 x 301 FP32_16: pack 221 -> 212 us (5.7 TB/s),
// exact unpack 400 (2-byte loads, scalar decode) -> 213 us (5.7 TB/s).
#include <algorithm>

#include "codec.hpp"
#include "common.hpp"
#include "tomos_hip.h"

namespace tomos_hip {

namespace {

template <int VARIANT>
__device__ __forceinline__ void encode(float v, uint16_t& h, uint16_t& r) {
    if constexpr (VARIANT == TOMOS_PACK_FP32_16) codec::fp32_16_encode<0>(v, h, r);
    else if constexpr (VARIANT == TOMOS_PACK_FP32_16_CLAMPED) codec::fp32_16_encode<1>(v, h, r);
    else if constexpr (VARIANT == TOMOS_PACK_FP32_16_TRUNCATED) codec::fp32_16_encode<2>(v, h, r);
    else if constexpr (VARIANT == TOMOS_PACK_FP32_BF16) codec::fp32_bf16_encode<false>(v, h, r);
    else codec::fp32_bf16_encode<true>(v, h, r);
}

constexpr int kRun = 8;  // rows per thread

typedef unsigned int u32x4 __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));

// 16 bytes at element alignment.  Non-temporal loads and stores measured no
// faster (16 GB: pack 2.74 against 2.84 ms, exact unpack 2.98 against 2.87).
template <class V>
__device__ __forceinline__ V load16(const void* p) {
    return *static_cast<const V*>(p);
}
template <class V>
__device__ __forceinline__ void store16(void* p, V v) {
    *static_cast<V*>(p) = v;
}

template <int VARIANT>
__global__ __launch_bounds__(256) void pack_kernel(int64_t m, int64_t n, const float* __restrict__ src,
                                                   int64_t ld_src, uint16_t* __restrict__ wh,
                                                   uint16_t* __restrict__ wr, int64_t ld_dst) {
    const int64_t j = static_cast<int64_t>(blockIdx.y) * blockDim.y + threadIdx.y;
    const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * kRun;
    if (i0 >= m || j >= n) return;
    const float* s = src + j * ld_src + i0;
    uint16_t* h = wh + j * ld_dst + i0;
    uint16_t* r = wr + j * ld_dst + i0;
    if (i0 + kRun <= m) {
        const f32x4 a = load16<f32x4>(s), b = load16<f32x4>(s + 4);
        u32x4 ph, pr;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint16_t h0, h1, r0, r1;
            encode<VARIANT>(k < 2 ? a[2 * k] : b[2 * k - 4], h0, r0);
            encode<VARIANT>(k < 2 ? a[2 * k + 1] : b[2 * k - 3], h1, r1);
            ph[k] = h0 | (uint32_t(h1) << 16);
            pr[k] = r0 | (uint32_t(r1) << 16);
        }
        store16(h, ph);
        store16(r, pr);
    } else {
        const int cnt = static_cast<int>(m - i0);
        for (int k = 0; k < cnt; ++k) encode<VARIANT>(s[k], h[k], r[k]);
    }
}

// Pack of a row-major source (row i at src + i ld_src): tiles of kTileRows x
// kTileCols are read along the rows (256 bytes each), encoded, turned in LDS
// as (h, r) words and written along the columns (256 bytes of each plane).
// HBM-bound like
// pack_kernel, in place of a transposed copy and a pack of it (20 matrices
// up to 200000 x 512, on average: 368 + 39 us so, 68 us here, 3.7 TB/s).
constexpr int kTileRows = 128, kTileCols = 64;
// Odd: the words that a wave stores at a step (one column of each 4, 16 lanes
// a row, 4 rows) hit 64 different banks, those that it loads (every eighth
// row, 16 lanes a column, 4 columns) 32.
constexpr int kTilePitch = kTileRows + 1;
constexpr int64_t kTileBlocks = int64_t(1) << 20;  // further tiles in a loop: 2^32 work items bound a launch

template <int VARIANT>
__global__ __launch_bounds__(256) void pack_rows_kernel(int64_t m, int64_t n, const float* __restrict__ src,
                                                        int64_t ld_src, uint16_t* __restrict__ wh,
                                                        uint16_t* __restrict__ wr, int64_t ld_dst,
                                                        int64_t row_tiles, int64_t col_tiles) {
    __shared__ uint32_t tile[kTileCols * kTilePitch];
    const int t = threadIdx.x;
    for (int64_t g = blockIdx.x; g < row_tiles * col_tiles; g += gridDim.x) {
        const int64_t rt = g / col_tiles;
        const int64_t i0 = rt * kTileRows, j0 = (g - rt * col_tiles) * kTileCols;
        const int c0 = (t & 15) * 4, r = t >> 4;
        const bool whole = j0 + c0 + 4 <= n;
        f32x4 v[kTileRows / 16];
#pragma unroll
        for (int q = 0; q < kTileRows / 16; ++q) {
            const int64_t i = i0 + r + 16 * q;
            v[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (i >= m) continue;
            const float* s = src + i * ld_src + j0 + c0;
            if (whole) {
                v[q] = load16<f32x4>(s);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (j0 + c0 + k < n) v[q][k] = s[k];
            }
        }
        if (g != static_cast<int64_t>(blockIdx.x)) __syncthreads();  // the last tile has been read
#pragma unroll
        for (int q = 0; q < kTileRows / 16; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint16_t h, l;
                encode<VARIANT>(v[q][k], h, l);
                tile[(c0 + k) * kTilePitch + r + 16 * q] = h | (uint32_t(l) << 16);
            }
        __syncthreads();
        const int i = (t & 15) * kRun;
        const int64_t left = m - i0 - i;
        for (int c = t >> 4; c < kTileCols && j0 + c < n && left > 0; c += 16) {
            const uint32_t* w = tile + c * kTilePitch + i;
            uint16_t* h = wh + (j0 + c) * ld_dst + i0 + i;
            uint16_t* l = wr + (j0 + c) * ld_dst + i0 + i;
            if (left >= kRun) {
                u32x4 ph, pl;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    ph[k] = (w[2 * k] & 0xFFFFu) | (w[2 * k + 1] << 16);
                    pl[k] = (w[2 * k] >> 16) | (w[2 * k + 1] & 0xFFFF0000u);
                }
                store16(h, ph);
                store16(l, pl);
            } else {
                for (int k = 0; k < static_cast<int>(left); ++k) {
                    h[k] = static_cast<uint16_t>(w[k] & 0xFFFFu);
                    l[k] = static_cast<uint16_t>(w[k] >> 16);
                }
            }
        }
    }
}

template <int DEC>
__device__ __forceinline__ float decode_f32(uint32_t h, uint32_t r) {
    if constexpr (DEC == TOMOS_DECODE_FP32_16_EXACT) return codec::fp32_16_decode_exact(h, r);
    else if constexpr (DEC == TOMOS_DECODE_FP32_16_HALF)
        return codec::half_bits_to_f32(codec::fp32_16_half_bits(h));
    else if constexpr (DEC == TOMOS_DECODE_FP32_16_HALF_FAST)
        return codec::half_bits_to_f32(codec::fp32_16_half_bits_fast(h));
    else if constexpr (DEC == TOMOS_DECODE_FP32_16_BF16)
        return codec::u2f(codec::fp32_16_bf16_bits(h) << 16);
    else if constexpr (DEC == TOMOS_DECODE_FP32_BF16_EXACT) return codec::fp32_bf16_decode_exact(h, r);
    else if constexpr (DEC == TOMOS_DECODE_FP32_BF16_HI) return codec::fp32_bf16_decode_hi(h);
    else if constexpr (DEC == TOMOS_DECODE_FP32_BF16_EXACT_ROUNDED)
        return codec::fp32_bf16_decode_exact_rounded(h, r);
    else return codec::fp32_16_decode_exact_truncated(h, r);
}

template <int DEC>
constexpr bool needs_wr() {
    return DEC == TOMOS_DECODE_FP32_16_EXACT || DEC == TOMOS_DECODE_FP32_BF16_EXACT ||
           DEC == TOMOS_DECODE_FP32_BF16_EXACT_ROUNDED ||
           DEC == TOMOS_DECODE_FP32_16_EXACT_TRUNCATED;
}

template <int DEC>
__global__ __launch_bounds__(256) void unpack_kernel(int64_t m, int64_t n, const uint16_t* __restrict__ wh,
                                                     const uint16_t* __restrict__ wr,
                                                     int64_t ld_src, float* __restrict__ dst,
                                                     int64_t ld_dst) {
    const int64_t j = static_cast<int64_t>(blockIdx.y) * blockDim.y + threadIdx.y;
    const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * kRun;
    if (i0 >= m || j >= n) return;
    const uint16_t* h = wh + j * ld_src + i0;
    const uint16_t* r = needs_wr<DEC>() ? wr + j * ld_src + i0 : nullptr;
    float* d = dst + j * ld_dst + i0;
    if (i0 + kRun <= m) {
        const u32x4 hv = load16<u32x4>(h);
        u32x4 rv = {0u, 0u, 0u, 0u};
        if constexpr (needs_wr<DEC>()) rv = load16<u32x4>(r);
        float v[kRun];
        bool pairs = false;  // decoded in pairs: an exact FP32_16 run without saturated words
        if constexpr (DEC == TOMOS_DECODE_FP32_16_EXACT) {
            pairs = (codec::fp32_16_saturated2(hv[0]) | codec::fp32_16_saturated2(hv[1]) |
                     codec::fp32_16_saturated2(hv[2]) | codec::fp32_16_saturated2(hv[3])) == 0;
            if (pairs) {
#pragma unroll
                for (int k = 0; k < 4; ++k) codec::fp32_16_decode_exact2(hv[k], rv[k], v[2 * k], v[2 * k + 1]);
            }
        }
        if (!pairs) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[2 * k] = decode_f32<DEC>(hv[k] & 0xFFFFu, rv[k] & 0xFFFFu);
                v[2 * k + 1] = decode_f32<DEC>(hv[k] >> 16, rv[k] >> 16);
            }
        }
        store16(d, f32x4{v[0], v[1], v[2], v[3]});
        store16(d + 4, f32x4{v[4], v[5], v[6], v[7]});
    } else {
        const int cnt = static_cast<int>(m - i0);
        for (int k = 0; k < cnt; ++k) d[k] = decode_f32<DEC>(h[k], needs_wr<DEC>() ? r[k] : 0u);
    }
}

template <int DEC>
__global__ __launch_bounds__(256) void decode_wh_kernel(int64_t count,
                                                        const uint16_t* __restrict__ wh,
                                                        uint16_t* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const uint32_t h = wh[i];
    uint32_t o;
    if constexpr (DEC == TOMOS_DECODE_FP32_16_HALF) o = codec::fp32_16_half_bits(h);
    else if constexpr (DEC == TOMOS_DECODE_FP32_16_HALF_FAST) o = codec::fp32_16_half_bits_fast(h);
    else if constexpr (DEC == TOMOS_DECODE_FP32_16_BF16) o = codec::fp32_16_bf16_bits(h);
    else o = h;  // FP32_BF16 hi-only: wh already is the bf16 pattern
    out[i] = static_cast<uint16_t>(o);
}

// A matrix whose columns follow each other without padding on both sides is
// one column of m * n rows: whole runs throughout and aligned ones if the
// first is.  Not where one launch dimension cannot hold that column: HIP takes
// fewer than 2^32 work items in each (2^35 rows here).
constexpr bool one_column(int64_t m, int64_t n, int64_t ld_src, int64_t ld_dst) {
    return ld_src == m && ld_dst == m && n <= (int64_t(1) << 35) / m &&
           (m * n + 256 * kRun - 1) / (256 * kRun) * 256 < (int64_t(1) << 32);
}
static_assert(one_column(2000000, 1000, 2000000, 2000000) && one_column(1 << 20, (1 << 15) - 1, 1 << 20, 1 << 20) &&
                  !one_column(1 << 20, 1 << 15, 1 << 20, 1 << 20) && !one_column(35000000, 1000, 35000000, 35000000) &&
                  !one_column(int64_t(1) << 40, int64_t(1) << 30, int64_t(1) << 40, int64_t(1) << 40) &&
                  !one_column(8, 3, 9, 8),
              "an unpadded matrix is one column up to 2^35 elements");
void flatten(int64_t& m, int64_t& n, int64_t& ld_src, int64_t& ld_dst) {
    if (one_column(m, n, ld_src, ld_dst)) {
        m *= n;
        n = 1;
        ld_src = ld_dst = m;
    }
}

// A block's 256 threads take runs of one column, or of several where the
// columns are short: padded columns of 100 rows left 243 threads without a
// run (unpack of 100 x 100000, exact FP32_16: 74 -> 24 us).
struct RunShape {
    dim3 grid, block;
};
RunShape run_shape(int64_t m, int64_t n) {
    unsigned tx = 256;
    while (tx > 1 && n > 1 && static_cast<int64_t>(tx / 2) * kRun >= m) tx /= 2;
    const unsigned ty = 256 / tx;
    return {dim3(static_cast<unsigned>(ceil_div(m, tx * kRun)), static_cast<unsigned>(ceil_div(n, ty))), dim3(tx, ty)};
}

template <int VARIANT>
void launch_pack_rows(int64_t m, int64_t n, const float* src, int64_t ld_src, uint16_t* wh, uint16_t* wr,
                      int64_t ld_dst, hipStream_t s) {
    const int64_t ct = ceil_div(n, static_cast<int64_t>(kTileCols)), rt = ceil_div(m, static_cast<int64_t>(kTileRows));
    const unsigned blocks = static_cast<unsigned>(std::min(rt * ct, kTileBlocks));
    pack_rows_kernel<VARIANT><<<blocks, 256, 0, s>>>(m, n, src, ld_src, wh, wr, ld_dst, rt, ct);
    TOMOS_LAUNCH_CHECK("pack_rows_kernel");
}

template <int VARIANT>
void launch_pack(int64_t m, int64_t n, const float* src, int64_t ld_src, uint16_t* wh,
                 uint16_t* wr, int64_t ld_dst, hipStream_t s) {
    flatten(m, n, ld_src, ld_dst);
    const RunShape r = run_shape(m, n);
    pack_kernel<VARIANT><<<r.grid, r.block, 0, s>>>(m, n, src, ld_src, wh, wr, ld_dst);
    TOMOS_LAUNCH_CHECK("pack_kernel");
}

template <int DEC>
void launch_unpack(int64_t m, int64_t n, const uint16_t* wh, const uint16_t* wr, int64_t ld_src,
                   float* dst, int64_t ld_dst, hipStream_t s) {
    flatten(m, n, ld_src, ld_dst);
    const RunShape r = run_shape(m, n);
    unpack_kernel<DEC><<<r.grid, r.block, 0, s>>>(m, n, wh, wr, ld_src, dst, ld_dst);
    TOMOS_LAUNCH_CHECK("unpack_kernel");
}

}  // namespace

}  // namespace tomos_hip

using namespace tomos_hip;

extern "C" {

int tomos_pack_rows(int variant, int64_t m, int64_t n, const float* src, int64_t ld_src, uint16_t* wh,
                    uint16_t* wr, int64_t ld_dst, tomos_stream_t s) {
    return guarded([&] {
        require(m >= 0 && n >= 0, "tomos_pack_rows: negative size");
        require(ld_src >= n && ld_dst >= m, "tomos_pack_rows: leading dimension too small");
        if (m == 0 || n == 0) return;
        require(src && wh && wr, "tomos_pack_rows: null pointer");
        switch (variant) {
            case TOMOS_PACK_FP32_16:
                launch_pack_rows<TOMOS_PACK_FP32_16>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_16_CLAMPED:
                launch_pack_rows<TOMOS_PACK_FP32_16_CLAMPED>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_16_TRUNCATED:
                launch_pack_rows<TOMOS_PACK_FP32_16_TRUNCATED>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_BF16:
                launch_pack_rows<TOMOS_PACK_FP32_BF16>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_BF16_ROUNDED:
                launch_pack_rows<TOMOS_PACK_FP32_BF16_ROUNDED>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            default:
                throw Error(kErrInvalidArgument, "tomos_pack_rows: unknown variant");
        }
    });
}

int tomos_pack(int variant, int64_t m, int64_t n, const float* src, int64_t ld_src, uint16_t* wh,
               uint16_t* wr, int64_t ld_dst, tomos_stream_t s) {
    return guarded([&] {
        require(m >= 0 && n >= 0, "tomos_pack: negative size");
        require(ld_src >= m && ld_dst >= m, "tomos_pack: leading dimension < m");
        require(n <= 2147483647, "tomos_pack: too many columns");
        if (m == 0 || n == 0) return;
        require(src && wh && wr, "tomos_pack: null pointer");
        switch (variant) {
            case TOMOS_PACK_FP32_16:
                launch_pack<TOMOS_PACK_FP32_16>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_16_CLAMPED:
                launch_pack<TOMOS_PACK_FP32_16_CLAMPED>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_16_TRUNCATED:
                launch_pack<TOMOS_PACK_FP32_16_TRUNCATED>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_BF16:
                launch_pack<TOMOS_PACK_FP32_BF16>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            case TOMOS_PACK_FP32_BF16_ROUNDED:
                launch_pack<TOMOS_PACK_FP32_BF16_ROUNDED>(m, n, src, ld_src, wh, wr, ld_dst, s);
                break;
            default:
                throw Error(kErrInvalidArgument, "tomos_pack: unknown variant");
        }
    });
}

int tomos_unpack(int dec, int64_t m, int64_t n, const uint16_t* wh, const uint16_t* wr,
                 int64_t ld_src, float* dst, int64_t ld_dst, tomos_stream_t s) {
    return guarded([&] {
        require(m >= 0 && n >= 0, "tomos_unpack: negative size");
        require(ld_src >= m && ld_dst >= m, "tomos_unpack: leading dimension < m");
        require(n <= 2147483647, "tomos_unpack: too many columns");
        if (m == 0 || n == 0) return;
        require(wh && dst, "tomos_unpack: null pointer");
        const bool exact = dec == TOMOS_DECODE_FP32_16_EXACT || dec == TOMOS_DECODE_FP32_BF16_EXACT ||
                           dec == TOMOS_DECODE_FP32_BF16_EXACT_ROUNDED ||
                           dec == TOMOS_DECODE_FP32_16_EXACT_TRUNCATED;
        require(!exact || wr != nullptr, "tomos_unpack: exact decoders need the wr plane");
        switch (dec) {
#define TOMOS_UNPACK_CASE(D) \
    case D: launch_unpack<D>(m, n, wh, wr, ld_src, dst, ld_dst, s); break;
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_16_EXACT)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_16_HALF)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_16_HALF_FAST)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_16_BF16)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_BF16_EXACT)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_BF16_HI)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_BF16_EXACT_ROUNDED)
            TOMOS_UNPACK_CASE(TOMOS_DECODE_FP32_16_EXACT_TRUNCATED)
#undef TOMOS_UNPACK_CASE
            default:
                throw Error(kErrInvalidArgument, "tomos_unpack: unknown decoder");
        }
    });
}

int tomos_decode_wh(int dec, int64_t count, const uint16_t* wh, uint16_t* out, tomos_stream_t s) {
    return guarded([&] {
        require(count >= 0, "tomos_decode_wh: negative count");
        if (count == 0) return;
        require(wh && out, "tomos_decode_wh: null pointer");
        const dim3 grid(static_cast<unsigned>(ceil_div(count, 256)));
        switch (dec) {
            case TOMOS_DECODE_FP32_16_HALF:
                decode_wh_kernel<TOMOS_DECODE_FP32_16_HALF><<<grid, 256, 0, s>>>(count, wh, out);
                break;
            case TOMOS_DECODE_FP32_16_HALF_FAST:
                decode_wh_kernel<TOMOS_DECODE_FP32_16_HALF_FAST><<<grid, 256, 0, s>>>(count, wh, out);
                break;
            case TOMOS_DECODE_FP32_16_BF16:
                decode_wh_kernel<TOMOS_DECODE_FP32_16_BF16><<<grid, 256, 0, s>>>(count, wh, out);
                break;
            case TOMOS_DECODE_FP32_BF16_HI:
                decode_wh_kernel<TOMOS_DECODE_FP32_BF16_HI><<<grid, 256, 0, s>>>(count, wh, out);
                break;
            default:
                throw Error(kErrInvalidArgument,
                            "tomos_decode_wh: decoder must produce 16-bit values");
        }
        TOMOS_LAUNCH_CHECK("decode_wh_kernel");
    });
}

}  // extern "C"
