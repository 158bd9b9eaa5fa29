// Dense Gaussian sketch: fill an (rows x cols, ld) column-major matrix with
// i.i.d. N(0,1) values (create_gaussian_sketch(Dense&),
// src/dispatch/gaussian_sketch_registries.cpp:16-30,
// src/kernels/cuda/sketch/gaussian_sketch_cuda_kernels.cu:21-45).
//
// The reference seeds its generator from the wall clock, so its sketches
// are not reproducible; this one is counter-based and takes the seed as an
// argument, so a (seed, shape) pair always gives the same matrix, whatever
// ld, stream or launch shape.
//
// Generator.  Entries are produced in pairs: pair p covers rows 2q and
// 2q+1 of column j, p = j * ceil(rows / 2) + q.  Its 64 random bits are
// the p-th output of SplitMix64 started at `seed` (Steele, Lea & Flood,
// "Fast splittable pseudorandom number generators", OOPSLA 2014):
// z = mix(seed + (p + 1) * 0x9e3779b97f4a7c15).  The top 23 bits give
// u1 = (b + 1/2) 2^-23 in (0, 1), bits 8..31 give u2 = b 2^-24 in [0, 1),
// and the Box-Muller transform (Box & Muller 1958) turns them into two
// independent normals r cos(2 pi u2), r sin(2 pi u2), r = sqrt(-2 ln u1).
// The transform runs in FP32 (logarithm, root, sine and cosine of exactly
// these arguments, below), the way the reference computes its values in
// float before the cast.  The output
// type's conversion rounds to nearest even.
//
// Roofline: each entry is written once and nothing is read, so the kernel
// is bounded by HBM writes (sizeof(T) bytes per entry) or by the VALU
// work of the mixer and the transform (about 100 operations per pair).
#include "codec.hpp"
#include "common.hpp"
#include "tomos_hip.h"

namespace tomos_hip {
namespace {

constexpr uint64_t kGolden = 0x9e3779b97f4a7c15ull;
constexpr int kGaussThreads = 256;

__device__ __forceinline__ uint64_t sm64_mix(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

// The transform over exactly the inputs it gets.  The library's logf, sqrtf
// and sincospif spend about half their operations on arguments that cannot
// occur here (subnormals, infinities, angles beyond a turn), and the kernel is
// bound by the VALU: 2000 x 131072 FP32 318 -> 230 us.
__device__ __forceinline__ float2 box_muller(uint64_t z) {
    const uint32_t hi = static_cast<uint32_t>(z >> 32);
    const uint32_t w = static_cast<uint32_t>(z >> 8) & 0xFFFFFFu;  // u2 = w 2^-24
    // b + 1/2 with b < 2^23 is exact in FP32 (with 24-bit b it would round
    // and move u1 near 1, where r is most sensitive to it)
    const float u1 = (static_cast<float>(hi >> 9) + 0.5f) * 0x1p-23f;
    // t = -2 ln u1 = -2 ln 2 log2 u1, the constant in two parts: its rounding
    // and the product's, half of them in r, are as large as what the products
    // below leave.  v_log_f32 keeps its relative accuracy as u1 nears 1 (r <
    // 0.02: r within 1.5e-7, relative; with logf and sqrtf 1.8e-7; over 4e8
    // values errors up to 7.2e-7, 4.5e-8 in the 2-norm, with them 9.0 and 5.1)
    const float lg = __builtin_amdgcn_logf(u1);
    constexpr float kHi = -0x1.62e430p+0f, kLo = 0x1.05c610p-28f;  // -2 ln 2
    const float th = lg * kHi;
    const float t = th + fmaf(lg, kLo, fmaf(lg, kHi, -th));
    // r = sqrt(t) = r0 + r1, t rsqrt(t) and its correction, kept apart so that
    // r is not rounded before the products; t is 0 or above 1e-7
    const float y = __builtin_amdgcn_rsqf(fmaxf(t, 1e-30f));
    const float r0 = t * y;
    const float r1 = fmaf(-r0, r0, t) * (0.5f * y);
    // sin and cos of pi v, v = 2 u2 less its quadrant q / 2: |v| <= 1/4, exact
    const uint32_t q = (w + 0x200000u) >> 22;
    const float v = static_cast<float>(static_cast<int32_t>(w << 10) >> 10) * 0x1p-23f;
    const float x = v * v;
    // least-squares fits over x in [0, 1/16], each coefficient refitted after
    // the ones before it were rounded: relative errors 1.1e-10 and 5e-10
    float ps = fmaf(x, 0x1.465b16p-4f, -0x1.32b458p-1f);
    ps = fmaf(x, ps, 0x1.466b82p+1f);
    ps = fmaf(x, ps, -0x1.4abbcep+2f);
    // pi in two parts: its rounding alone would be half an ulp of the sine
    const float sn = fmaf(v, 0x1.921fb6p+1f, v * fmaf(x, ps, -0x1.777a5cp-24f));
    float pc = fmaf(x, 0x1.d61e28p-3f, -0x1.55b684p+0f);
    pc = fmaf(x, pc, 0x1.03c1b6p+2f);
    pc = fmaf(x, pc, -0x1.3bd3ccp+2f);
    const float cs = fmaf(x, pc, 1.0f);
    // quadrants 0..4: (c, s), (-s, c), (-c, -s), (s, -c), (c, s)
    const bool swap = q & 1u;
    const uint32_t sc = (q << 30) + 0x40000000u, ss = q << 30;  // sign bits
    const float c = codec::u2f(codec::f2u(swap ? sn : cs) ^ (sc & 0x80000000u));
    const float d = codec::u2f(codec::f2u(swap ? cs : sn) ^ (ss & 0x80000000u));
    return make_float2(fmaf(r0, c, r1 * c), fmaf(r0, d, r1 * d));
}

// Two adjacent entries of one column; VEC: the pair is stored with one
// aligned store (base and ld even, checked on the host).
template <int TYPE, bool VEC>
__device__ __forceinline__ void store_pair(void* col, int64_t row, float a, float b, bool two) {
    if constexpr (TYPE == TOMOS_F64) {
        double* p = static_cast<double*>(col) + row;
        if (VEC && two) *reinterpret_cast<double2*>(p) = make_double2(a, b);
        else { p[0] = a; if (two) p[1] = b; }
    } else if constexpr (TYPE == TOMOS_F32) {
        float* p = static_cast<float*>(col) + row;
        if (VEC && two) *reinterpret_cast<float2*>(p) = make_float2(a, b);
        else { p[0] = a; if (two) p[1] = b; }
    } else {
        uint32_t ha, hb;
        if constexpr (TYPE == TOMOS_F16) {
            const _Float16 x = static_cast<_Float16>(a), y = static_cast<_Float16>(b);
            ha = __builtin_bit_cast(uint16_t, x);
            hb = __builtin_bit_cast(uint16_t, y);
        } else {
            ha = codec::f32_to_bf16_bits(a);
            hb = codec::f32_to_bf16_bits(b);
        }
        uint16_t* p = static_cast<uint16_t*>(col) + row;
        if (VEC && two) *reinterpret_cast<uint32_t*>(p) = ha | (hb << 16);
        else { p[0] = static_cast<uint16_t>(ha); if (two) p[1] = static_cast<uint16_t>(hb); }
    }
}

// grid.x covers the row pairs of a column (kGaussThreads per block), grid.y
// strides over the columns: the generator's state moves on by a constant.
// EVEN: every pair has two rows.
template <int TYPE, bool VEC, bool EVEN>
__global__ __launch_bounds__(kGaussThreads) void gaussian_fill_kernel(int64_t rows, int64_t cols,
                                                                      void* out, int64_t ld,
                                                                      uint64_t seed) {
    constexpr int64_t esz = TYPE == TOMOS_F64 ? 8 : TYPE == TOMOS_F32 ? 4 : 2;
    const int64_t half = (rows + 1) >> 1;
    const int64_t q = static_cast<int64_t>(blockIdx.x) * kGaussThreads + threadIdx.x;
    if (q >= half) return;
    const int64_t row = 2 * q;
    const bool two = EVEN || row + 1 < rows;
    const uint64_t p = static_cast<uint64_t>(blockIdx.y) * static_cast<uint64_t>(half) + static_cast<uint64_t>(q);
    uint64_t state = seed + (p + 1) * kGolden;
    const uint64_t step = static_cast<uint64_t>(gridDim.y) * static_cast<uint64_t>(half) * kGolden;
    char* col = static_cast<char*>(out) + blockIdx.y * ld * esz;
#pragma unroll 2
    for (int64_t j = blockIdx.y; j < cols; j += gridDim.y) {
        const float2 g = box_muller(sm64_mix(state));
        store_pair<TYPE, VEC>(col, row, g.x, g.y, two);
        state += step;
        col += gridDim.y * ld * esz;
    }
}

template <int TYPE>
void launch_fill(int64_t rows, int64_t cols, void* out, int64_t ld, uint64_t seed, hipStream_t st) {
    constexpr int64_t esz = TYPE == TOMOS_F64 ? 8 : TYPE == TOMOS_F32 ? 4 : 2;
    const int64_t half = (rows + 1) >> 1;
    const bool vec = (reinterpret_cast<uintptr_t>(out) % (2 * esz) == 0) && (ld % 2 == 0);
    // about 16384 blocks: enough to fill the chip several times over, few
    // enough that a thread's set-up (64-bit products) is spread over many pairs
    const int64_t bx = ceil_div(half, kGaussThreads);
    const int64_t by = std::min<int64_t>(std::min<int64_t>(cols, 65535), std::max<int64_t>(16384 / bx, 1));
    const dim3 grid(static_cast<unsigned>(bx), static_cast<unsigned>(by));
    const bool even = rows % 2 == 0;
#define TOMOS_FILL(V, E) gaussian_fill_kernel<TYPE, V, E><<<grid, kGaussThreads, 0, st>>>(rows, cols, out, ld, seed)
    if (vec) { if (even) TOMOS_FILL(true, true); else TOMOS_FILL(true, false); }
    else { if (even) TOMOS_FILL(false, true); else TOMOS_FILL(false, false); }
#undef TOMOS_FILL
    TOMOS_LAUNCH_CHECK("gaussian_fill_kernel");
}

// One entry per sketch row (the reference's CSR sketches,
// generate_countsketch_csr_idxs, countsketch_kernels.cpp:34-53): row i
// holds column z % cols, z the i-th SplitMix64 output from seed ^ kColSalt;
// kind 0 stores the sign of z's top bit (+-1), kind 1 leaves the values to
// the Gaussian fill.
constexpr uint64_t kColSalt = 0xc2b2ae3d27d4eb4full;

template <class I, int VT>
__global__ void csr_sketch_pattern_kernel(int64_t rows, int64_t cols, uint64_t seed, I* rp, I* ci, void* vals,
                                          bool signs, bool pattern) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i <= rows; i += stride) {
        if (pattern) rp[i] = static_cast<I>(i);
        if (i == rows) break;
        const uint64_t z = sm64_mix((seed ^ kColSalt) + (static_cast<uint64_t>(i) + 1) * kGolden);
        if (pattern) ci[i] = static_cast<I>(z % static_cast<uint64_t>(cols));
        if (signs) {
            const float v = (z >> 63) ? 1.0f : -1.0f;
            if constexpr (VT == TOMOS_F64) static_cast<double*>(vals)[i] = v;
            else if constexpr (VT == TOMOS_F32) static_cast<float*>(vals)[i] = v;
            else if constexpr (VT == TOMOS_F16) static_cast<uint16_t*>(vals)[i] = (z >> 63) ? 0x3C00 : 0xBC00;
            else static_cast<uint16_t*>(vals)[i] = (z >> 63) ? 0x3F80 : 0xBF80;
        }
    }
}

template <class I>
void launch_pattern(int vt, int64_t rows, int64_t cols, uint64_t seed, void* rp, void* ci, void* vals, bool signs,
                    bool pattern, hipStream_t st) {
    const unsigned g = static_cast<unsigned>(std::min<int64_t>(std::max<int64_t>(ceil_div(rows + 1, 256), 1), 8192));
    I* r = static_cast<I*>(rp);
    I* c = static_cast<I*>(ci);
    switch (vt) {
        case TOMOS_F64: csr_sketch_pattern_kernel<I, TOMOS_F64><<<g, 256, 0, st>>>(rows, cols, seed, r, c, vals, signs, pattern); break;
        case TOMOS_F32: csr_sketch_pattern_kernel<I, TOMOS_F32><<<g, 256, 0, st>>>(rows, cols, seed, r, c, vals, signs, pattern); break;
        case TOMOS_F16: csr_sketch_pattern_kernel<I, TOMOS_F16><<<g, 256, 0, st>>>(rows, cols, seed, r, c, vals, signs, pattern); break;
        default: csr_sketch_pattern_kernel<I, TOMOS_BF16><<<g, 256, 0, st>>>(rows, cols, seed, r, c, vals, signs, pattern); break;
    }
    TOMOS_LAUNCH_CHECK("csr_sketch_pattern_kernel");
}

}  // namespace
}  // namespace tomos_hip

using namespace tomos_hip;

extern "C" int tomos_csr_sketch(int kind, int val_type, int idx_type, int64_t rows, int64_t cols, void* vals,
                                void* row_ptrs, void* col_idxs, uint64_t seed, tomos_stream_t st) {
    return guarded([&] {
        require(kind >= 0 && kind <= 3,
                "tomos_csr_sketch: kind must be 0 (+-1), 1 (Gaussian), 2 (pattern only) or 3 (+-1 values only)");
        require(val_type == TOMOS_F64 || val_type == TOMOS_F32 || val_type == TOMOS_F16 || val_type == TOMOS_BF16,
                "tomos_csr_sketch: values must be F64, F32, F16 or BF16");
        require(idx_type == TOMOS_INDEX_INT32 || idx_type == TOMOS_INDEX_INT64, "tomos_csr_sketch: bad index type");
        require(rows >= 0 && cols >= 1, "tomos_csr_sketch: need rows >= 0 and cols >= 1");
        require(idx_type == TOMOS_INDEX_INT64 || (rows <= 0x7FFFFFFF && cols <= 0x7FFFFFFF),
                "tomos_csr_sketch: sizes exceed INT32 indices");
        const bool pattern = kind != 3, signs = kind == 0 || kind == 3;
        require((!pattern || row_ptrs) && (rows == 0 || ((vals || kind == 2) && (col_idxs || kind == 3))),
                "tomos_csr_sketch: null output");
        if (idx_type == TOMOS_INDEX_INT64)
            launch_pattern<int64_t>(val_type, rows, cols, seed, row_ptrs, col_idxs, vals, signs, pattern, st);
        else
            launch_pattern<int32_t>(val_type, rows, cols, seed, row_ptrs, col_idxs, vals, signs, pattern, st);
        if (kind == 1 && rows > 0) {
            switch (val_type) {
                case TOMOS_F64: launch_fill<TOMOS_F64>(rows, 1, vals, rows, seed, st); break;
                case TOMOS_F32: launch_fill<TOMOS_F32>(rows, 1, vals, rows, seed, st); break;
                case TOMOS_F16: launch_fill<TOMOS_F16>(rows, 1, vals, rows, seed, st); break;
                default: launch_fill<TOMOS_BF16>(rows, 1, vals, rows, seed, st); break;
            }
        }
    });
}

extern "C" int tomos_gaussian_fill(int type, int64_t rows, int64_t cols, void* out, int64_t ld,
                                   uint64_t seed, tomos_stream_t st) {
    return guarded([&] {
        require(rows >= 0 && cols >= 0, "tomos_gaussian_fill: negative size");
        require(ld >= (rows > 1 ? rows : 1), "tomos_gaussian_fill: ld < rows");
        if (rows == 0 || cols == 0) return;
        require(out != nullptr, "tomos_gaussian_fill: null output");
        require(ceil_div((rows + 1) >> 1, kGaussThreads) <= 0x7FFFFFFF, "tomos_gaussian_fill: too many rows");
        switch (type) {
            case TOMOS_F64: launch_fill<TOMOS_F64>(rows, cols, out, ld, seed, st); break;
            case TOMOS_F32: launch_fill<TOMOS_F32>(rows, cols, out, ld, seed, st); break;
            case TOMOS_F16: launch_fill<TOMOS_F16>(rows, cols, out, ld, seed, st); break;
            case TOMOS_BF16: launch_fill<TOMOS_BF16>(rows, cols, out, ld, seed, st); break;
            default: throw Error(kErrUnsupported, "tomos_gaussian_fill: type must be F64, F32, F16 or BF16");
        }
    });
}
