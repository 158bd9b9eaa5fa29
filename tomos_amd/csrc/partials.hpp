// Column totals of a problem's partial sums [items][n], for the grouped
// solvers: 64 columns a block, 16 waves that take every sixteenth item with
// eight loads in flight each, their sums added in wave order in LDS.
// A thread that walked its column alone paid one memory latency for every
// few items (100 items of a 200000 x 512 problem: 50 us, with one block a
// problem; 9 us so, on 8 blocks a problem).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tomos_hip {

constexpr int kPartCols = 64;
constexpr int kPartSlices = 16;
constexpr int kPartThreads = kPartCols * kPartSlices;

// Total of column j = col0 + (threadIdx.x & 63), valid in the first wave
// (0 for j >= n); every thread of the block takes part.
template <typename T>
__device__ __forceinline__ double column_total(const T* __restrict__ part, int items, int64_t n, int64_t col0) {
    constexpr int kU = 8;
    __shared__ double sums[kPartSlices][kPartCols];
    const int lane = threadIdx.x & (kPartCols - 1), slice = threadIdx.x / kPartCols;
    const int64_t j = col0 + lane;
    double a = 0.0;
    if (j < n)
        for (int k = slice; k < items; k += kU * kPartSlices) {
            T v[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int i = k + u * kPartSlices;
                v[u] = i < items ? part[static_cast<int64_t>(i) * n + j] : T(0);
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) a += static_cast<double>(v[u]);
        }
    sums[slice][lane] = a;
    __syncthreads();
    if (slice != 0) return 0.0;
    a = 0.0;
    for (int q = 0; q < kPartSlices; ++q) a += sums[q][lane];
    return a;
}

}  // namespace tomos_hip
