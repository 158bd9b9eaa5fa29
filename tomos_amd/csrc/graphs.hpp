// Capturing a launch sequence as a graph that the batched solvers keep.
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <type_traits>

#include "common.hpp"
#include "shared_cache.hpp"

namespace tomos_hip {

using GraphExec = std::remove_pointer_t<hipGraphExec_t>;
using SharedGraph = std::shared_ptr<GraphExec>;

// What `body` enqueues on s, instantiated; destroyed with its last share.
template <class F>
SharedGraph capture_graph(hipStream_t s, F&& body) {
    TOMOS_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
    hipGraph_t graph = nullptr;
    try {
        body();
    } catch (...) {
        (void)hipStreamEndCapture(s, &graph);
        if (graph) (void)hipGraphDestroy(graph);
        throw;
    }
    TOMOS_HIP_CHECK(hipStreamEndCapture(s, &graph));
    hipGraphExec_t exec = nullptr;
    const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    TOMOS_HIP_CHECK(e);
    return SharedGraph(exec, [](hipGraphExec_t x) { (void)hipGraphExecDestroy(x); });
}

// The graph of `key`: kept, or captured from `body` and kept.
template <class Key, class F>
SharedGraph cached_graph(SharedCache<Key, GraphExec>& cache, const Key& key, hipStream_t s, F&& body) {
    SharedGraph g = cache.find(key);
    if (!g) {
        g = capture_graph(s, body);
        cache.insert(key, g);
    }
    return g;
}

}  // namespace tomos_hip
