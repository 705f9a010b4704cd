// jh_graph.h -- kernel launches that can also become the nodes of a graph.
//
// A graph of steps is put together from kernel nodes, not by capturing a
// stream: while any thread of the process captures, the runtime refuses work on
// the legacy stream to all of them (hipMemcpy: "would make the legacy stream
// depend on a capturing blocking stream"), and contexts build graphs that
// nobody asked for.
#pragma once

#include <hip/hip_runtime.h>

#include <tuple>

namespace jh {

// The graph that this thread's launches go to, one node after the other.
struct GraphChain {
  hipGraph_t graph;
  hipGraphNode_t last = nullptr;
  hipError_t err = hipSuccess;  // the first node that could not be added
};
inline thread_local GraphChain *graph_chain = nullptr;

// Launch fn on st, or add it to this thread's graph while one is set.
template <class... P, class... A>
void enqueue(void (*fn)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, A &&...a) {
  if (!graph_chain) {
    hipLaunchKernelGGL(fn, grid, block, lds, st, static_cast<P>(a)...);
    return;
  }
  GraphChain &c = *graph_chain;
  if (c.err != hipSuccess) return;
  std::tuple<P...> v(static_cast<P>(a)...);
  std::apply(
      [&](auto &...x) {
        void *args[] = {const_cast<void *>(static_cast<const void *>(&x))...};
        hipKernelNodeParams k = {};
        k.func = reinterpret_cast<void *>(fn);
        k.gridDim = grid;
        k.blockDim = block;
        k.sharedMemBytes = (unsigned)lds;
        k.kernelParams = args;  // copied with the node
        hipGraphNode_t node = nullptr;
        c.err = hipGraphAddKernelNode(&node, c.graph, c.last ? &c.last : nullptr, c.last ? 1 : 0, &k);
        c.last = node;
      },
      v);
}

}  // namespace jh
