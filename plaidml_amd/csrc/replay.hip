// Replay of a recorded sequence of launches.
//
// hipGraphLaunch takes 16 to 18 us of the host whatever the graph holds, before the device sees the first kernel; a launch of its
// own takes 2.1, which the kernels ahead of it cover.  So a short recording is replayed launch by launch, with the arguments it
// holds (no plan is asked again), and a longer one as a graph: from eight commands on -- a run's launches, its copies up and down by
// kernel and hipStreamSynchronize's own -- retiring them takes the run that waits 13 us more, and a graph is one.  us a call, n dense
// layers of 8 x 64 on arrays in host memory, as a graph -> one by one (medians, roots in turn on one box):
//   n                                    2             3             4             5             6             7             8            10            30           52
//   one behind the other        40.2 -> 30.1  52.4 -> 34.0  47.1 -> 38.2  47.8 -> 41.4  51.0 -> 59.6  59.3 -> 64.3  61.2 -> 66.1  63.6 -> 73.6   130 -> 144    202 -> 227
//   and a wait for the device   45.1 -> 33.3  56.2 -> 37.1  50.8 -> 41.2  51.0 -> 44.4  54.0 -> 61.8  61.3 -> 67.4  64.2 -> 69.1  67.2 -> 76.9   133 -> 147    205 -> 230
//   new arrays, 10 ms later     72.3 -> 48.7  85.2 -> 52.0  73.4 -> 47.8  77.5 -> 61.9  73.2 -> 80.5  79.9 -> 89.4  76.7 -> 96.8  78.3 -> 94.5   147 -> 156    219 -> 237
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <new>

#include "plans.h"

namespace pml {

namespace {

constexpr size_t kFewLaunches = 5;  // one by one up to here

// The kernels of a short recording that is one chain of nothing else, in their order (the arguments stay the recording's own);
// their number, or 0.
size_t kernel_chain(hipGraph_t g, hipKernelNodeParams (&chain)[kFewLaunches]) {
  size_t n = 0, edges = 0;
  if (hipGraphGetNodes(g, nullptr, &n) != hipSuccess || n == 0 || n > kFewLaunches) return 0;
  if (hipGraphGetEdges(g, nullptr, nullptr, &edges) != hipSuccess || edges != n - 1) return 0;
  hipGraphNode_t nodes[kFewLaunches], from[kFewLaunches], to[kFewLaunches], at = nullptr;
  if (hipGraphGetNodes(g, nodes, &n) != hipSuccess) return 0;
  if (edges > 0 && hipGraphGetEdges(g, from, to, &edges) != hipSuccess) return 0;
  for (size_t i = 0; i < n; ++i)
    if (std::count(to, to + edges, nodes[i]) == 0) {
      if (at) return 0;
      at = nodes[i];
    }
  size_t count = 0;
  while (at) {
    hipGraphNodeType type;
    hipKernelNodeParams p = {};
    if (count == n || hipGraphNodeGetType(at, &type) != hipSuccess || type != hipGraphNodeTypeKernel) return 0;
    if (hipGraphKernelNodeGetParams(at, &p) != hipSuccess || !p.func || !p.kernelParams || p.extra) return 0;
    chain[count++] = p;
    if (std::count(from, from + edges, at) > 1) return 0;
    const size_t edge = (size_t)(std::find(from, from + edges, at) - from);
    at = edge == edges ? nullptr : to[edge];
  }
  return count == n ? count : 0;
}

}  // namespace

struct Replay {
  hipGraph_t recorded = nullptr;              // of launches that go out one by one
  hipKernelNodeParams launches[kFewLaunches];  // (their arguments are `recorded`'s)
  size_t n = 0;                               // 0: as a graph
  hipGraphExec_t exec = nullptr;
  ~Replay() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (recorded) (void)hipGraphDestroy(recorded);
  }
};

// (called by entry points of a C library: nothing here throws)
hipError_t replay_create(hipGraph_t recorded, Replay** out) {
  std::unique_ptr<Replay> r(new (std::nothrow) Replay);
  if (!r) {
    (void)hipGraphDestroy(recorded);
    return hipErrorOutOfMemory;
  }
  r->recorded = recorded;
  r->n = kernel_chain(recorded, r->launches);
  if (r->n == 0) {
    (void)hipGetLastError();
    if (hipError_t e = hipGraphInstantiate(&r->exec, recorded, nullptr, nullptr, 0); e != hipSuccess) return e;
    (void)hipGraphDestroy(recorded);
    r->recorded = nullptr;
  }
  *out = r.release();
  return hipSuccess;
}

hipError_t replay_launch(const Replay& r, hipStream_t s) {
  for (size_t i = 0; i < r.n; ++i) {
    const hipKernelNodeParams& p = r.launches[i];
    if (hipError_t e = hipLaunchKernel(p.func, p.gridDim, p.blockDim, p.kernelParams, p.sharedMemBytes, s); e != hipSuccess) return e;
  }
  return r.exec ? hipGraphLaunch(r.exec, s) : hipSuccess;
}

void replay_destroy(Replay* r) { delete r; }

}  // namespace pml
