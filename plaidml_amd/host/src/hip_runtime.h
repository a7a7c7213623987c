// The `hip` runtime: device "hip.<n>" and its executables.  It fills the seam
// the reference defines with pmlc::rt::Runtime / Device / Executable
// (pmlc/rt/runtime.h:19-26, device.h:14-21, executable.h:13-25) and registers
// under the name "hip" the way `llvm_cpu` does (pmlc/rt/llvm/runtime.cc:12-35).
// An executable owns device buffers for every value of the plan, uploads
// constants and re-lays-out constant weights once when it is built (the
// reference runs its `init` closure once, pmlc/rt/jit_executable.cc:404-418),
// and on every invoke copies inputs in, launches the plan on one stream and
// copies outputs back, long copies on streams of their own beside the launches.
#pragma once

#include <memory>
#include <string>
#include <vector>

#include "hip_plan.h"
#include "tile.h"
#include "util.h"

namespace pmlc::rt {

// A program input or output in host memory; f32: a bf16 tensor held as fp32 values there
struct HostSpan {
  void* data;
  size_t bytes;
  bool f32;
};

class Executable {
 public:
  virtual ~Executable() = default;
  // the same on plain memory (inputs are only read)
  virtual double invokeHost(const std::vector<HostSpan>& inputs, const std::vector<HostSpan>& outputs) = 0;
  // the results of the last run, from the device
  virtual void download(const std::vector<HostSpan>& outputs) = 0;
  // returns the wall time of the run in milliseconds, host-device transfers included
  virtual double invoke(const std::vector<util::BufferPtr>& inputs, const std::vector<util::BufferPtr>& outputs) = 0;
};

class Device {
 public:
  virtual ~Device() = default;
  virtual std::unique_ptr<Executable> compile(const std::shared_ptr<tile::Program>& program) = 0;
};

class Runtime {
 public:
  virtual ~Runtime() = default;
  virtual size_t getDeviceCount() const = 0;
  virtual std::shared_ptr<Device> getDevice(size_t ordinal) = 0;
};

// registry keyed by runtime name; device ids are "<runtime>.<ordinal>" (pmlc/rt/device_id.cc:13-38)
void registerRuntime(const std::string& id, std::shared_ptr<Runtime> runtime);
void initRuntimes();
std::vector<std::string> listDevices();
std::shared_ptr<Device> getDevice(const std::string& deviceID);

// Host memory the GPU can read and write directly (page-locked), for buffers the library allocates itself: a
// copy to or from it runs at the link's rate instead of being staged through the driver's own bounce buffers.
// Zero-initialised (pinnedAllocRaw: not).  nullptr when no GPU is visible (the caller falls back to ordinary memory).
// Freed blocks up to a bound are kept for the next allocation: page-locking costs about as much as copying the block.
void* pinnedAlloc(size_t bytes);
void* pinnedAllocRaw(size_t bytes);  // not zeroed
void pinnedFree(void* p);
// whether [p, p + bytes) lies in one live block of it
bool isPinned(const void* p, size_t bytes);

// statistics of the most recent invoke of any hip executable in this thread (for benchmarks)
struct InvokeStats {
  // The wall time in three parts.  Where the link's share ends is not seen from here (another mark would cost a launch of its
  // own): h2d_ms is the host's time up to the last upload it queues, rounding and staging included; kernel_ms the device's, first
  // launch -> last launch, by the device's clock as the kernels that copy small operands and results read it (by events where
  // steps are timed); d2h_ms the rest -- what of the uploads is still under way then, the downloads, the passes over the results.
  // A run whose copies and launches go on streams of their own: kernel_ms is the sum, by events, over its runs of launches, each
  // from where it could begin (what it needs up, the run before it done) to its end -- the time between two streams is in it, time
  // in which launches wait for the link is not.
  double kernel_ms = 0;
  double h2d_ms = 0;
  double d2h_ms = 0;
  size_t launches = 0;             // steps of the plan; one that runs on parts counts once a part
  double wall_ms = 0;              // the whole run, transfers included (what invoke returns)
  size_t arena_bytes = 0;          // device memory shared by the temporaries
  size_t unshared_temp_bytes = 0;  // what the temporaries would take with memory of their own
  size_t device_bytes = 0;         // arena + inputs + outputs + constants + what the kernel plans hold
  std::vector<double> step_ms;     // per step of the plan, over its parts; only with PLAIDML_PROFILE=1
  bool replayed = false;           // the launches came from a recording
  std::string graph_note;          // why they did not, when recording was tried and failed
};
InvokeStats lastInvokeStats();

}  // namespace pmlc::rt
