// Replay of a recorded sequence of launches.
//
// hipGraphLaunch takes 16 to 18 us of the host whatever the graph holds, before the device sees the first kernel; a launch of its
// own takes 2.1, which the kernels ahead of it cover.  So a recording is replayed launch by launch, with the arguments it holds (no
// plan is asked again), and only a long one as a graph.  us a run, host to host, as a graph -> one by one, one box:
//   dense layers of 4 x 64 (3.3 us each on the device)   7 of them 48.9 -> 38.4, 14 66.7 -> 59.0, 80 264 -> 257 (another box 270 -> 276)
//   ResNet-50 on one image, 52 kernels                   389 -> 375
// (The first 4 or 8 one by one and the rest as a graph: as a graph.  Both sides with the results' mark in host memory; waiting for
// the stream takes 13 us more from eight queued commands on.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <vector>

#include "plans.h"

namespace pml {

namespace {

constexpr size_t kFewLaunches = 64;  // one by one up to here

// The kernels of a recording that is one chain of nothing else, in their order (the arguments stay the recording's own).
bool kernel_chain(hipGraph_t g, std::vector<hipKernelNodeParams>* chain) {
  size_t n = 0, edges = 0;
  if (hipGraphGetNodes(g, nullptr, &n) != hipSuccess || n == 0) return false;
  if (hipGraphGetEdges(g, nullptr, nullptr, &edges) != hipSuccess || edges != n - 1) return false;
  std::vector<hipGraphNode_t> nodes(n), from(edges), to(edges);
  if (hipGraphGetNodes(g, nodes.data(), &n) != hipSuccess) return false;
  if (edges > 0 && hipGraphGetEdges(g, from.data(), to.data(), &edges) != hipSuccess) return false;
  hipGraphNode_t at = nullptr;
  for (hipGraphNode_t node : nodes)
    if (std::count(to.begin(), to.end(), node) == 0) {
      if (at) return false;
      at = node;
    }
  while (at) {
    hipGraphNodeType type;
    hipKernelNodeParams p = {};
    if (hipGraphNodeGetType(at, &type) != hipSuccess || type != hipGraphNodeTypeKernel) return false;
    if (hipGraphKernelNodeGetParams(at, &p) != hipSuccess || !p.func || !p.kernelParams || p.extra) return false;
    chain->push_back(p);
    if (chain->size() > n) return false;
    const auto edge = std::find(from.begin(), from.end(), at);
    if (edge != from.end() && std::find(edge + 1, from.end(), at) != from.end()) return false;
    at = edge == from.end() ? nullptr : to[edge - from.begin()];
  }
  return chain->size() == n;
}

}  // namespace

struct Replay {
  hipGraph_t recorded = nullptr;
  std::vector<hipKernelNodeParams> launches;  // one by one (their arguments are `recorded`'s); empty: as a graph
  hipGraphExec_t exec = nullptr;
  ~Replay() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (recorded) (void)hipGraphDestroy(recorded);
  }
};

hipError_t replay_create(hipGraph_t recorded, Replay** out) {
  std::unique_ptr<Replay> r(new Replay);
  r->recorded = recorded;
  if (!kernel_chain(recorded, &r->launches)) {
    (void)hipGetLastError();
    r->launches.clear();
  }
  if (r->launches.size() > kFewLaunches) r->launches.clear();
  if (r->launches.empty())
    if (hipError_t e = hipGraphInstantiate(&r->exec, recorded, nullptr, nullptr, 0); e != hipSuccess) return e;
  *out = r.release();
  return hipSuccess;
}

hipError_t replay_launch(const Replay& r, hipStream_t s) {
  for (const hipKernelNodeParams& p : r.launches)
    if (hipError_t e = hipLaunchKernel(p.func, p.gridDim, p.blockDim, p.kernelParams, p.sharedMemBytes, s); e != hipSuccess) return e;
  return r.exec ? hipGraphLaunch(r.exec, s) : hipSuccess;
}

void replay_destroy(Replay* r) { delete r; }

}  // namespace pml
