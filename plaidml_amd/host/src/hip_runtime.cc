#include "hip_runtime.h"

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <regex>
#include <sstream>

#include "host_copy.h"
#include "pinned_pool.h"
#include "pml_hip.h"

namespace pmlc::rt {

using target::hip::BufferInfo;
using target::hip::Plan;
using target::hip::Step;

namespace {

thread_local InvokeStats g_stats;

constexpr size_t kAlign = 256;  // arena offsets; also the slack behind every value (kernels read whole 16-byte vectors)
size_t padded(size_t bytes) { return (bytes + 16 + kAlign - 1) / kAlign * kAlign; }

bool profileRequested() {
  const char* e = std::getenv("PLAIDML_PROFILE");
  return e && std::string(e) == "1";
}

void hipCheck(int status, const char* what) {
  if (status != 0) throw std::runtime_error(std::string(what) + ": " + pml_hip_last_error());
}

double nowMs() {
  using clock = std::chrono::steady_clock;
  return std::chrono::duration<double, std::milli>(clock::now().time_since_epoch()).count();
}

class HipExecutable final : public Executable {
 public:
  HipExecutable(std::shared_ptr<tile::Program> program, std::shared_ptr<Plan> plan, int ordinal)
      : program_(std::move(program)), plan_(std::move(plan)), ordinal_(ordinal) {
    hipCheck(pml_hip_init(ordinal_), "pml_hip_init");
    device_.assign(plan_->buffers.size(), nullptr);
    owned_.assign(plan_->buffers.size(), false);
    try {
      // Inputs, outputs and constants keep memory of their own for the life of the executable; temporaries
      // share one arena, each placed by the span of steps in which it is live (what the reference's
      // resize-tmps / dealloc placement does for its heap temporaries, pmlc/target/x86/pipeline.cc:289-360).
      const std::vector<size_t> offsets = placeTemporaries();
      if (arena_bytes_) hipCheck(pml_hip_malloc(&arena_, arena_bytes_), "pml_hip_malloc (arena)");
      for (size_t i = 0; i < plan_->buffers.size(); ++i) {
        const BufferInfo& b = plan_->buffers[i];
        if (b.kind == BufferInfo::Temp) {
          device_[i] = static_cast<char*>(arena_) + offsets[i];
          continue;
        }
        hipCheck(pml_hip_malloc(&device_[i], b.bytes + 16), "pml_hip_malloc");
        owned_[i] = true;
        fixed_bytes_ += padded(b.bytes);
        if (b.kind == BufferInfo::Constant)
          hipCheck(pml_hip_memcpy_h2d(device_[i], b.constant->data(), b.constant->size(), nullptr), "upload constant");
      }
      handles_.resize(plan_->steps.size());
      for (size_t i = 0; i < plan_->steps.size(); ++i) dispatch(i < plan_->sliced.size() ? plan_->sliced[i] : plan_->steps[i], &handles_[i]);
      if (plan_->uneven) {
        last_handles_.resize(plan_->sliced.size());
        for (size_t i = 0; i < plan_->sliced.size(); ++i) dispatch(plan_->sliced_last[i], &last_handles_[i]);
      }
      // Where a run begins and ends on the device is read off its clock by the kernels that copy, or by one of their kind
      // (two events around the launches cost a run 8 us); with events where that cannot be had, and under PLAIDML_PROFILE.
      clock_khz_ = pml_hip_clock_khz();
      void* stamps = nullptr;
      if (clock_khz_ > 0 && pml_hip_host_alloc(&stamps, 2 * sizeof(uint64_t)) == 0) stamps_ = static_cast<uint64_t*>(stamps);
      hipCheck(pml_hip_event_create(&ev0_), "event");
      hipCheck(pml_hip_event_create(&ev1_), "event");
      hipCheck(pml_hip_stream_create(&stream_), "stream");
      hipCheck(pml_hip_stream_sync(nullptr), "sync");
      // Recording is for runs of plain kernel launches and device-to-device copies: the sort, scatter, gather, index and random-number steps keep
      // state or sizes on the host side of their entry points and stay with one-by-one launches.
      graphable_ = plan_->graph && (plan_->steps.size() > 1 || plan_->slices > 1);
      for (const Step& s : plan_->steps)
        if (s.kind != Step::Gemm && s.kind != Step::Conv2d && s.kind != Step::Dwconv2d && s.kind != Step::Pool2d &&
            s.kind != Step::Eltwise && s.kind != Step::Contract && s.kind != Step::Select && s.kind != Step::Copy &&
            s.kind != Step::Softmax && s.kind != Step::Product && s.kind != Step::ConvGrad && s.kind != Step::Rows &&
            s.kind != Step::Argmax && s.kind != Step::TopK)
          graphable_ = false;
      findSegments();
      if (segments_.size() > 1) {
        for (pml_hip_stream* q : {&up_stream_, &down_stream_}) hipCheck(pml_hip_stream_create(q), "stream");
        for (Segment& seg : segments_)
          for (pml_hip_event* e : {&seg.up, &seg.done, &seg.down}) hipCheck(pml_hip_event_create(e), "event");
      }
    } catch (...) {
      release();
      throw;
    }
  }

  ~HipExecutable() override { release(); }

  double invoke(const std::vector<util::BufferPtr>& inputs, const std::vector<util::BufferPtr>& outputs) override {
    std::vector<HostSpan> in, out;
    for (const auto& b : inputs) in.push_back({b->data(), b->size(), false});
    for (const auto& b : outputs) out.push_back({b->data(), b->size(), false});
    return invokeHost(in, out);
  }

  // One run.  Everything is queued on the executable's stream -- uploads, launches, downloads -- and waited for once, or, where
  // long copies can go beside launches, on three (overlapped).
  //   inputs   in page-locked memory already: straight from there.  Elsewhere (or fp32 values of a bf16 tensor): through
  //            the executable's page-locked staging, a few megabytes at a time, so that the link carries one piece
  //            while the host passes over the next.
  //   outputs  the mirror image: pieces are passed on as they arrive, the last ones after the wait.
  // Short transfers are made by one kernel each way (pml_hip_copy_spans), long ones by the copy engines.
  double invokeHost(const std::vector<HostSpan>& inputs, const std::vector<HostSpan>& outputs) override {
    hipCheck(pml_hip_init(ordinal_), "pml_hip_init");
    if (inputs.size() != plan_->input_buffers.size() || outputs.size() != plan_->output_buffers.size())
      throw std::runtime_error("executable invoked with the wrong number of buffers");
    InvokeStats st;
    const double start = nowMs();
    const bool profile = profileRequested();
    for (size_t i = 0; i < outputs.size(); ++i)
      if (outputs[i].bytes < spanBytes(plan_->output_buffers[i], outputs[i])) throw std::runtime_error("output buffer #" + std::to_string(i) + " is too small");
    for (size_t i = 0; i < inputs.size(); ++i)
      if (inputs[i].bytes < spanBytes(plan_->input_buffers[i], inputs[i])) throw std::runtime_error("input buffer #" + std::to_string(i) + " is too small");
    if (segments_.size() > 1 && !profile && !shared(inputs, outputs) && overlapped(inputs, outputs, start, &st)) {
      g_stats = st;
      return st.wall_ms;
    }
    Spans up, down;
    std::vector<Piece> arriving;  // what waits in the staging to be passed on, in the order it is sent
    std::vector<size_t> unstaged;  // outputs that go without it
    Staging stage;
    try {
      std::vector<size_t> staged;
      auto needs = [&](const std::vector<int>& buffers, const std::vector<HostSpan>& spans) {
        for (size_t i = 0; i < spans.size(); ++i)
          if (!direct(buffers[i], spans[i])) staged.push_back(plan_->buffers[buffers[i]].bytes);
      };
      needs(plan_->input_buffers, inputs);
      needs(plan_->output_buffers, outputs);
      stage = staging(staged);
      for (size_t i = 0; i < inputs.size(); ++i) {
        const int buf = plan_->input_buffers[i];
        const size_t bytes = plan_->buffers[buf].bytes;
        if (direct(buf, inputs[i])) {
          upload(device_[buf], inputs[i].data, bytes, &up);
        } else if (stage.base) {
          stageIn(&stage, inputs[i], bytes, static_cast<char*>(device_[buf]), &up);
        } else {
          // (no page-locked memory to be had)
          std::vector<uint16_t> tmp;
          const void* from = inputs[i].data;
          if (inputs[i].f32) {
            tmp.resize(bytes / 2);
            hostToBf16(tmp.data(), static_cast<const float*>(from), tmp.size());
            from = tmp.data();
          }
          hipCheck(pml_hip_memcpy_h2d(device_[buf], from, bytes, stream_), "h2d");
        }
      }
      const bool stamped = stamps_ && !profile;
      up.issue(stream_, stamped ? &stamps_[0] : nullptr, true);
      st.h2d_ms = nowMs() - start;
      launchAll(profile, &st);
      // (ahead of what the copy engines fetch; otherwise by the kernel that fetches the results)
      uint64_t* end = stamped ? &stamps_[1] : nullptr;
      for (int buf : plan_->output_buffers)
        if (end && plan_->buffers[buf].bytes > kKernelCopy) {
          Spans().issue(stream_, end, false);
          end = nullptr;
        }
      for (size_t i = 0; i < outputs.size(); ++i) {
        const int buf = plan_->output_buffers[i];
        const size_t bytes = plan_->buffers[buf].bytes;
        if (direct(buf, outputs[i]))
          download(outputs[i].data, device_[buf], bytes, &down);
        else if (stage.base)
          stageOut(&stage, outputs[i], bytes, static_cast<const char*>(device_[buf]), &arriving, &down);
        else
          unstaged.push_back(i);
      }
      down.issue(stream_, end, false);
      collect(&stage, arriving);
    } catch (...) {
      (void)pml_hip_stream_sync(stream_);  // queued copies may still use the caller's memory
      throw;
    }
    for (size_t i : unstaged) {
      const int buf = plan_->output_buffers[i];
      const size_t bytes = plan_->buffers[buf].bytes;
      if (!outputs[i].f32) {
        hipCheck(pml_hip_memcpy_d2h(outputs[i].data, device_[buf], bytes, stream_), "d2h");
        continue;
      }
      std::vector<uint16_t> tmp(bytes / 2);
      hipCheck(pml_hip_memcpy_d2h(tmp.data(), device_[buf], bytes, stream_), "d2h");
      hostFromBf16(static_cast<float*>(outputs[i].data), tmp.data(), tmp.size());
    }
    st.wall_ms = nowMs() - start;
    finish(profile, &st);
    st.d2h_ms = std::max(0.0, st.wall_ms - st.h2d_ms - st.kernel_ms);
    g_stats = st;
    // wall time of the whole run, transfers included, as the reference returns the time around its jitted main
    // (pmlc/rt/jit_executable.cc:484-490); the device time alone is in the statistics
    return st.wall_ms;
  }

  void download(const std::vector<HostSpan>& outputs) override {
    hipCheck(pml_hip_init(ordinal_), "pml_hip_init");
    if (outputs.size() != plan_->output_buffers.size()) throw std::runtime_error("executable asked for the wrong number of results");
    for (size_t i = 0; i < outputs.size(); ++i) {
      const int buf = plan_->output_buffers[i];
      if (outputs[i].f32 || outputs[i].bytes < plan_->buffers[buf].bytes) throw std::runtime_error("output buffer #" + std::to_string(i) + " is too small");
      hipCheck(pml_hip_memcpy_d2h(outputs[i].data, device_[buf], plan_->buffers[buf].bytes, stream_), "d2h");
    }
  }

 private:
  std::shared_ptr<tile::Program> program_;
  std::shared_ptr<Plan> plan_;
  int ordinal_;
  std::vector<void*> device_;
  std::vector<bool> owned_;
  void* arena_ = nullptr;
  size_t arena_bytes_ = 0, fixed_bytes_ = 0, unshared_temp_bytes_ = 0;
  struct Launch {
    size_t step;
    int slice;  // its part of the leading dimension, -1: the whole step
  };
  struct Handles {
    int64_t own = 0, next = 0;  // next: the second product of a step that has one behind its first (Step::chained)
  };
  std::vector<Handles> handles_, last_handles_;  // per step; of the sliced ones' last, shorter part
  pml_hip_event ev0_ = nullptr, ev1_ = nullptr;
  uint64_t* stamps_ = nullptr;  // page-locked: the device's clock ahead of and behind a run's launches
  int clock_khz_ = 0;
  std::vector<pml_hip_event> step_events_;
  pml_hip_stream stream_ = nullptr;  // every copy and launch of this executable
  pml_hip_graph graph_ = nullptr;    // the launches of one run, recorded
  bool graphable_ = false;
  int runs_ = 0;
  std::string graph_note_;
  void* staging_ = nullptr;          // page-locked: what a run passes between the caller's memory and the device
  size_t staging_bytes_ = 0;
  std::vector<pml_hip_event> half_events_;  // the last copies from or into each half of its slots

  // transfers up to this many bytes go by kernel, longer ones by copy engine
  static constexpr size_t kKernelCopy = 512 << 10;
  // bytes the host stages before it hands them to the copy engine; slots for such pieces, filled a half at a time (an event
  // between copies costs the link about 10 us: 134 MB in 2.8 ms with one after every piece, 2.3 with one after every fourth)
  static constexpr size_t kStageRun = 4 << 20;
  static constexpr size_t kStageHalf = 4, kStageSlots = 2 * kStageHalf;

  struct Spans {
    std::vector<void*> dst;
    std::vector<const void*> src;
    std::vector<size_t> bytes;
    void add(void* d, const void* s, size_t n) {
      dst.push_back(d);
      src.push_back(s);
      bytes.push_back(n);
    }
    void issue(pml_hip_stream stream, uint64_t* stamp, bool after) {
      if (!dst.empty() || stamp)
        hipCheck(pml_hip_copy_spans_stamped(static_cast<int>(dst.size()), dst.data(), src.data(), bytes.data(), stamp, after ? 1 : 0, stream), "copy");
    }
  };

  // Whether a result lies in the memory of an operand, or of another result.  On one stream everything is up before anything goes
  // down, and results arrive in their order; between queues of their own a result would reach an operand that is still to go up.
  bool shared(const std::vector<HostSpan>& inputs, const std::vector<HostSpan>& outputs) const {
    auto meet = [](const HostSpan& a, size_t a_bytes, const HostSpan& b, size_t b_bytes) {
      const uintptr_t p = reinterpret_cast<uintptr_t>(a.data), q = reinterpret_cast<uintptr_t>(b.data);
      return p < q + b_bytes && q < p + a_bytes;
    };
    for (size_t o = 0; o < outputs.size(); ++o) {
      const size_t bytes = spanBytes(plan_->output_buffers[o], outputs[o]);
      for (size_t i = 0; i < inputs.size(); ++i)
        if (meet(outputs[o], bytes, inputs[i], spanBytes(plan_->input_buffers[i], inputs[i]))) return true;
      for (size_t q = 0; q < o; ++q)
        if (meet(outputs[o], bytes, outputs[q], spanBytes(plan_->output_buffers[q], outputs[q]))) return true;
    }
    return false;
  }

  // bytes the caller's side of a value takes
  size_t spanBytes(int buf, const HostSpan& h) const { return plan_->buffers[buf].bytes * (h.f32 ? 2 : 1); }
  bool direct(int buf, const HostSpan& h) const { return !h.f32 && isPinned(h.data, plan_->buffers[buf].bytes); }

  // The page-locked staging of one run.  Values that go by kernel have a place each; the others share what is behind them:
  // a place each as well where that takes no more than the slots, else the slots in turn, a piece at a time.  Page-locking
  // memory takes longer than copying through it, and what is locked is kept as long as the executable: a first run with
  // 134 MB of inputs takes 14.4 ms, 21.8 with all of them locked, 22.7 from pageable memory (later runs 4.0, 4.1, 11.1).
  struct Staging {
    char* base = nullptr;
    char* next = nullptr;    // the next place of a value of its own
    char* slots = nullptr;   // the slots, or nullptr: every value has its own place
    size_t turn = 0;         // pieces that have gone through the slots
  };
  struct Piece {
    char* at;                // in the staging; nullptr: in a slot, when its turn comes
    const char* dev;
    char* host;
    size_t bytes;            // on the device
    bool f32;
  };

  Staging staging(const std::vector<size_t>& values) {
    size_t by_kernel = 0, others = 0;
    for (size_t bytes : values) (bytes <= kKernelCopy ? by_kernel : others) += padded(bytes);
    Staging s;
    const bool in_turn = others > kStageSlots * kStageRun;
    const size_t need = by_kernel + (in_turn ? kStageSlots * kStageRun : others);
    if (need == 0) return s;
    if (need > staging_bytes_) {
      if (staging_) pinnedFree(staging_);
      staging_bytes_ = 0;
      staging_ = pinnedAllocRaw(need);
      if (!staging_) return s;  // (none now: the next run asks again)
      staging_bytes_ = need;
    }
    if (in_turn) needHalfEvents();
    s.base = s.next = static_cast<char*>(staging_);
    if (in_turn) s.slots = s.base + by_kernel;
    return s;
  }
  void needHalfEvents() {
    while (half_events_.size() < 2) {
      half_events_.push_back(nullptr);
      hipCheck(pml_hip_event_create(&half_events_.back()), "event");
    }
  }
  // the place of a value that has its own
  static char* place(Staging* s, size_t bytes) {
    char* p = s->next;
    s->next += padded(bytes);
    return p;
  }

  void upload(void* dst, const void* src, size_t bytes, Spans* spans) {
    if (bytes <= kKernelCopy)
      spans->add(dst, src, bytes);
    else
      hipCheck(pml_hip_memcpy_h2d_async(dst, src, bytes, stream_), "h2d");
  }
  void download(void* dst, const void* src, size_t bytes, Spans* spans) {
    if (bytes <= kKernelCopy)
      spans->add(dst, src, bytes);
    else
      hipCheck(pml_hip_memcpy_d2h_async(dst, src, bytes, stream_), "d2h");
  }
  void stageIn(Staging* stage, const HostSpan& in, size_t bytes, char* dev, Spans* spans) {
    const bool by_kernel = bytes <= kKernelCopy, in_turn = !by_kernel && stage->slots;
    char* const own = in_turn ? nullptr : place(stage, bytes);
    for (size_t at = 0; at < bytes; at += kStageRun) {
      const size_t n = std::min(kStageRun, bytes - at), turn = stage->turn, half = turn / kStageHalf % 2;
      char* to = own + at;
      if (in_turn) {
        to = stage->slots + turn % kStageSlots * kStageRun;
        if (turn >= kStageSlots && turn % kStageHalf == 0) hipCheck(pml_hip_event_sync(half_events_[half]), "event sync");
        ++stage->turn;
      }
      if (in.f32)
        hostToBf16(reinterpret_cast<uint16_t*>(to), static_cast<const float*>(in.data) + at / 2, n / 2);
      else
        hostCopy(to, static_cast<const char*>(in.data) + at, n);
      if (by_kernel)
        spans->add(dev + at, to, n);
      else
        hipCheck(pml_hip_memcpy_h2d_async(dev + at, to, n, stream_), "h2d");
      if (in_turn && turn % kStageHalf == kStageHalf - 1) hipCheck(pml_hip_event_record(half_events_[half], stream_), "event record");
    }
  }

  // An output that comes back through the staging: queues what has a place of its own, leaves the rest to collect().
  void stageOut(Staging* stage, const HostSpan& out, size_t bytes, const char* dev, std::vector<Piece>* pieces, Spans* spans) {
    char* const host = static_cast<char*>(out.data);
    if (bytes > kKernelCopy && stage->slots) {
      for (size_t at = 0; at < bytes; at += kStageRun)
        pieces->push_back({nullptr, dev + at, host + at * (out.f32 ? 2 : 1), std::min(kStageRun, bytes - at), out.f32});
      return;
    }
    char* const own = place(stage, bytes);
    download(own, dev, bytes, spans);
    pieces->push_back({own, dev, host, bytes, out.f32});
  }

  // Waits for everything queued and passes on what comes back through the staging: pieces that go through the slots while
  // the ones behind them are on the link, the others at the end.  (A piece may go into its slot right away: the uploads
  // from there are before it on the stream.)
  void collect(Staging* stage, const std::vector<Piece>& pieces) {
    std::vector<const Piece*> in_turn;
    for (const Piece& p : pieces)
      if (!p.at) in_turn.push_back(&p);
    const size_t halves = (in_turn.size() + kStageHalf - 1) / kStageHalf;
    auto each = [&](size_t h, auto&& fn) {  // fn(piece, its slot) for the pieces of one half
      for (size_t k = h * kStageHalf; k < std::min(in_turn.size(), (h + 1) * kStageHalf); ++k) fn(*in_turn[k], stage->slots + k % kStageSlots * kStageRun);
    };
    auto send = [&](size_t h) {
      each(h, [&](const Piece& p, char* slot) { hipCheck(pml_hip_memcpy_d2h_async(slot, p.dev, p.bytes, stream_), "d2h"); });
      hipCheck(pml_hip_event_record(half_events_[h % 2], stream_), "event record");
    };
    auto pass = [](const char* from, const Piece& p) {
      if (p.f32)
        hostFromBf16(reinterpret_cast<float*>(p.host), reinterpret_cast<const uint16_t*>(from), p.bytes / 2);
      else
        hostCopy(p.host, from, p.bytes);
    };
    for (size_t h = 0; h < halves && h < 2; ++h) send(h);
    for (size_t h = 0; h < halves; ++h) {
      hipCheck(pml_hip_event_sync(half_events_[h % 2]), "event sync");
      each(h, [&](const Piece& p, char* slot) { pass(slot, p); });
      if (h + 2 < halves) send(h + 2);
    }
    hipCheck(pml_hip_stream_sync(stream_), "stream sync");
    for (const Piece& p : pieces)
      if (p.at) pass(p.at, p);
  }

  void launchAll(bool profile, InvokeStats* st) {
    const std::vector<Launch>& launches = order_;
    if (profile && step_events_.size() != launches.size() + 1) {
      step_events_.assign(launches.size() + 1, nullptr);
      for (auto& e : step_events_) hipCheck(pml_hip_event_create(&e), "event");
    }
    // The launches of a run never change (same plans, same device buffers), so from the third run on they are
    // replayed from a recording made during that run; the first two run one by one (first runs of a kernel plan may
    // allocate, which cannot be recorded).  A recording that fails leaves the executable with one-by-one launches.
    if (graphable_ && !profile && !graph_ && runs_ >= 2) graph_ = record(launches);
    ++runs_;
    const bool events = profile || !stamps_;
    if (events) hipCheck(pml_hip_event_record(ev0_, stream_), "event record");
    if (graph_ && !profile) {
      hipCheck(pml_hip_graph_launch(graph_, stream_), "graph launch");
      st->replayed = true;
    } else {
      for (size_t k = 0; k < launches.size(); ++k) {
        if (profile) hipCheck(pml_hip_event_record(step_events_[k], stream_), "event record");
        launch(launches[k].step, launches[k].slice);
      }
    }
    if (profile) hipCheck(pml_hip_event_record(step_events_.back(), stream_), "event record");
    if (events) hipCheck(pml_hip_event_record(ev1_, stream_), "event record");
  }

  // statistics of a run that has been waited for
  void finish(bool profile, InvokeStats* st) {
    if (stamps_ && !profile) {
      st->kernel_ms = static_cast<double>(stamps_[1] - stamps_[0]) / clock_khz_;
    } else {
      float ms = 0;
      hipCheck(pml_hip_event_elapsed_ms(ev0_, ev1_, &ms), "event elapsed");
      st->kernel_ms = ms;
    }
    describe(st);
    if (!profile) return;
    report(st);
  }

  // what does not depend on the run
  void describe(InvokeStats* st) const {
    st->launches = order_.size();
    st->graph_note = graph_note_;
    st->arena_bytes = arena_bytes_;
    st->unshared_temp_bytes = unshared_temp_bytes_;
    st->device_bytes = arena_bytes_ + fixed_bytes_;
    for (const auto* handles : {&handles_, &last_handles_})
      for (const Handles& h : *handles)
        for (int64_t plan : {h.own, h.next})
          if (plan) st->device_bytes += pml_hip_plan_bytes(plan);
  }

  void report(InvokeStats* st) {
    // One row per launch, in the reference's format (pmlc/rt/instrument.cc:22-43: id, loc, tag, seconds since
    // the previous point, seconds since the start); loc is the plan's line for the step, tag its kind.
    std::printf("\"id\",\"loc\",\"tag\",\"elapsed\",\"accumulated\"\n");
    double total = 0;
    st->step_ms.assign(plan_->steps.size(), 0);
    const std::vector<Launch>& launches = order_;
    for (size_t k = 0; k < launches.size(); ++k) {
      const size_t i = launches[k].step;
      float step = 0;
      hipCheck(pml_hip_event_elapsed_ms(step_events_[k], step_events_[k + 1], &step), "event elapsed");
      st->step_ms[i] += step;
      total += step;
      std::printf("%03d,\"%s\",%d,%7.6f,%7.6f\n", static_cast<int>(i), plan_->steps[i].text.c_str(), static_cast<int>(plan_->steps[i].kind),
                  step * 1e-3, total * 1e-3);
    }
    std::printf("%03d,%s,%d,%7.6f,%7.6f\n", 9999, "endTime", 9999, 0.0, total * 1e-3);
    std::fflush(stdout);
  }

  // The launches as a recording, or nullptr (and one-by-one launches from then on).
  pml_hip_graph record(const std::vector<Launch>& launches) {
    if (pml_hip_capture_begin(stream_) != 0) {
      graph_note_ = pml_hip_last_error();
      graphable_ = false;
      return nullptr;
    }
    bool ok = true;
    try {
      for (const Launch& l : launches) launch(l.step, l.slice);
    } catch (const std::exception& e) {
      graph_note_ = e.what();
      ok = false;
    }
    pml_hip_graph g = nullptr;
    if (pml_hip_capture_end(stream_, &g) != 0 || !ok) {
      if (ok) graph_note_ = pml_hip_last_error();
      if (g) pml_hip_graph_destroy(g);
      graphable_ = false;
      return nullptr;
    }
    return g;
  }

  // ---- overlapped runs: copies up, launches and copies down in three queues ------------------------------------------

  // A run of launches, what of the inputs has to be up before them, and what of the outputs may go down behind them.
  struct Range {
    size_t index, offset, bytes;
  };
  struct Segment {
    std::vector<Launch> launches;
    std::vector<Range> needs, yields;
    pml_hip_graph graph = nullptr;
    pml_hip_event up = nullptr, done = nullptr, down = nullptr;
    double ms = 0;  // of its launches in the last run
  };
  std::vector<Segment> segments_;
  std::vector<Launch> order_;  // of all the segments
  pml_hip_stream up_stream_ = nullptr, down_stream_ = nullptr;
  int overlapped_runs_ = 0;
  static constexpr double kPassMs = 0.05;  // of the host over kStageRun bytes, at least

  void findSegments() {
    const Plan& p = *plan_;
    std::vector<int> input_of(p.buffers.size(), -1);
    for (size_t i = 0; i < p.input_buffers.size(); ++i) input_of[p.input_buffers[i]] = static_cast<int>(i);
    std::vector<char> up(p.input_buffers.size(), 0);
    std::vector<int> writer(p.buffers.size(), -1);  // the last step that writes a buffer
    for (size_t i = 0; i < p.steps.size(); ++i) {
      for (int b : {p.steps[i].c, p.steps[i].out2})
        if (b >= 0) writer[b] = static_cast<int>(i);
      for (int b : p.steps[i].outs) writer[b] = static_cast<int>(i);
    }
    auto reads = [&](const Step& s) {
      std::vector<size_t> in;
      auto note = [&](int b) {
        if (b >= 0 && input_of[b] >= 0) in.push_back(static_cast<size_t>(input_of[b]));
      };
      for (int b : {s.a, s.b, s.init, s.a2, s.b2, s.init2, s.next_b, s.next_init, s.out2, s.c}) note(b);
      for (int b : s.operands) note(b);
      return in;
    };
    const size_t n = p.sliced.size();
    for (int slice = 0; slice < (n ? p.slices : 0); ++slice) {
      Segment seg;
      for (size_t i = 0; i < n; ++i) {
        seg.launches.push_back({i, slice});
        for (size_t in : reads(p.steps[i])) {
          const int buf = p.input_buffers[in];
          const size_t part = p.part_bytes[buf], bytes = p.buffers[buf].bytes;
          if (part == 0 && !up[in]) seg.needs.push_back({in, 0, bytes});
          if (part > 0 && up[in] <= slice) seg.needs.push_back({in, slice * part, std::min(part, bytes - slice * part)});
          up[in] = static_cast<char>(part > 0 ? slice + 1 : p.slices);
        }
      }
      for (size_t o = 0; o < p.output_buffers.size(); ++o) {
        const int buf = p.output_buffers[o];
        if (writer[buf] < 0 || static_cast<size_t>(writer[buf]) >= n) continue;
        const size_t part = p.part_bytes[buf], bytes = p.buffers[buf].bytes;
        seg.yields.push_back({o, slice * part, std::min(part, bytes - slice * part)});
      }
      segments_.push_back(std::move(seg));
    }
    for (size_t i = n; i < p.steps.size(); ++i) {
      if (segments_.empty() || std::count(p.runs.begin(), p.runs.end(), i)) segments_.emplace_back();
      Segment& seg = segments_.back();
      seg.launches.push_back({i, -1});
      for (size_t in : reads(p.steps[i]))
        if (!up[in]) {
          up[in] = 1;
          seg.needs.push_back({in, 0, p.buffers[p.input_buffers[in]].bytes});
        }
      for (size_t o = 0; o < p.output_buffers.size(); ++o)
        if (writer[p.output_buffers[o]] == static_cast<int>(i)) seg.yields.push_back({o, 0, p.buffers[p.output_buffers[o]].bytes});
    }
    for (const Segment& seg : segments_) order_.insert(order_.end(), seg.launches.begin(), seg.launches.end());
    if (segments_.empty()) return;
    for (size_t in = 0; in < up.size(); ++in)
      if (!up[in]) segments_.front().needs.push_back({in, 0, p.buffers[p.input_buffers[in]].bytes});
    for (size_t o = 0; o < p.output_buffers.size(); ++o)
      if (writer[p.output_buffers[o]] < 0) segments_.back().yields.push_back({o, 0, p.buffers[p.output_buffers[o]].bytes});
  }

  // One run, segment by segment: what a segment needs is staged and sent up, its launches wait for that, and what is final behind
  // it goes down while the link carries the next one's needs up.  Inputs that take more than the slots go through them in turn,
  // and so do outputs behind the last launch.  False (and nothing done) where the staging has no place for the other values, or there is none.  An output's place is that of an input which is up before the output exists, where there is one.
  bool overlapped(const std::vector<HostSpan>& inputs, const std::vector<HostSpan>& outputs, double start, InvokeStats* st) {
    constexpr size_t kNowhere = ~size_t{0}, kInTurn = kNowhere - 1, kAll = kStageSlots * kStageRun;
    std::vector<size_t> in_at, out_at, up_by(inputs.size(), 0), from(outputs.size(), 0);
    size_t need = 0;
    auto bytes_of = [&](int buf) { return plan_->buffers[buf].bytes; };
    for (size_t k = 0; k < segments_.size(); ++k) {
      for (const Range& r : segments_[k].needs) up_by[r.index] = k;
      for (size_t q = segments_[k].yields.size(); q-- > 0;)
        if (segments_[k].yields[q].offset == 0) from[segments_[k].yields[q].index] = k;
    }
    size_t staged = 0;
    for (size_t i = 0; i < inputs.size(); ++i)
      if (!direct(plan_->input_buffers[i], inputs[i])) staged += padded(bytes_of(plan_->input_buffers[i]));
    // a place for every value, or the slots for the long ones: inputs in turn, and outputs that half as much has no place for, at the end
    auto place_all = [&](bool in_turn) {
      in_at.assign(inputs.size(), kNowhere);
      out_at.assign(outputs.size(), kNowhere);
      std::vector<char> lent(inputs.size(), 0);
      need = 0;
      for (size_t i = 0; i < inputs.size(); ++i) {
        const size_t bytes = bytes_of(plan_->input_buffers[i]);
        if (direct(plan_->input_buffers[i], inputs[i])) continue;
        in_at[i] = in_turn && bytes > kKernelCopy ? kInTurn : need;
        if (in_at[i] != kInTurn) need += padded(bytes);
      }
      for (size_t o = 0; o < outputs.size(); ++o) {
        const int buf = plan_->output_buffers[o];
        if (direct(buf, outputs[o])) continue;
        for (size_t i = 0; i < inputs.size() && out_at[o] == kNowhere; ++i) {
          const int in = plan_->input_buffers[i];
          if (in_at[i] >= kInTurn || lent[i] || bytes_of(in) < bytes_of(buf)) continue;
          const bool parts = plan_->slices > 1 && plan_->part_bytes[in] > 0 && plan_->part_bytes[buf] > 0;
          if (parts ? plan_->part_bytes[in] >= plan_->part_bytes[buf] : up_by[i] <= from[o]) {
            out_at[o] = in_at[i];
            lent[i] = 1;
          }
        }
        if (out_at[o] != kNowhere) continue;
        const size_t bytes = padded(bytes_of(buf));
        out_at[o] = in_turn && bytes > kKernelCopy && need + bytes > kAll / 2 ? kInTurn : need;
        if (out_at[o] != kInTurn) need += bytes;
      }
      return need <= (in_turn ? kAll / 2 : kAll);
    };
    bool in_turn = staged > kAll;
    if (!place_all(in_turn) && (in_turn || !place_all(in_turn = true))) return false;
    const size_t slots = need;
    if (in_turn) need += kAll;
    if (need > staging_bytes_) {
      if (staging_) pinnedFree(staging_);
      staging_bytes_ = 0;
      staging_ = pinnedAllocRaw(need);
      if (!staging_) return false;
      staging_bytes_ = need;
    }
    if (in_turn) needHalfEvents();
    char* const base = static_cast<char*>(staging_);
    // (an output lies in its lender's place part behind part, as far apart as the lender's are)
    auto out_place = [&](const Range& r) {
      const size_t part = plan_->slices > 1 ? plan_->part_bytes[plan_->output_buffers[r.index]] : 0;
      size_t at = out_at[r.index] + r.offset;
      if (part > 0)
        for (size_t i = 0; i < inputs.size(); ++i)
          if (in_at[i] == out_at[r.index] && plan_->part_bytes[plan_->input_buffers[i]] > 0)
            at = out_at[r.index] + r.offset / part * plan_->part_bytes[plan_->input_buffers[i]];
      return base + at;
    };
    auto sync = [&] {
      for (pml_hip_stream s : {up_stream_, stream_, down_stream_}) (void)pml_hip_stream_sync(s);
    };
    try {
      const bool record_now = graphable_ && overlapped_runs_++ >= 2;
      size_t turn = 0, sent = 0, last_up = 0;  // last_up: of the segments, whose operands go up by copy engine
      for (size_t k = 0; k < segments_.size(); ++k)
        for (const Range& r : segments_[k].needs)
          if (r.bytes > kKernelCopy) last_up = k;
      // What goes down last so far is marked when the next copies down, or no more launches, are to be queued: a mark waits for the
      // copies, and where the streams share one of the device's queues, which a process's many streams do, launches behind it on
      // another stream wait with it.  (A product of 1024 x 1024 and two small launches behind it 186 us on one stream; marked
      // ahead of the small ones 165 to 230 by what shares a queue, now 163.)
      Segment* marked = nullptr;
      auto mark = [&] {
        if (marked) hipCheck(pml_hip_event_record(marked->down, down_stream_), "event record");
      };
      auto send = [&](Segment& seg) {
        if (seg.yields.empty()) return;
        mark();
        marked = &seg;
        Spans down;
        hipCheck(pml_hip_stream_wait_event(down_stream_, seg.done), "wait");
        for (const Range& r : seg.yields) {
          const HostSpan& out = outputs[r.index];
          const char* const dev = static_cast<const char*>(device_[plan_->output_buffers[r.index]]) + r.offset;
          if (out_at[r.index] == kInTurn) continue;
          char* const to = out_at[r.index] == kNowhere ? static_cast<char*>(out.data) + r.offset : out_place(r);
          if (r.bytes <= kKernelCopy)
            down.add(to, dev, r.bytes);
          else
            hipCheck(pml_hip_memcpy_d2h_async(to, dev, r.bytes, down_stream_), "d2h");
        }
        down.issue(down_stream_, nullptr, false);
      };
      // Whether segment k is done before the next copy up is queued: it is a part, its launches took less in the last run than a
      // pass over a piece does, and the next part's operand takes several.  (Its results go down at once then: 4096 x 1000 fp32
      // normalised 660 us a call, 700 with a look between pieces.  Otherwise a look is better: batched products with 2.4 MB a part
      // 520 us at once, 495, gradients whose second operand is 5.9 MB 463 and 410.)
      auto quick = [&](size_t k) {
        if (k + 1 >= static_cast<size_t>(plan_->slices) || segments_[k].ms <= 0 || segments_[k].ms >= kPassMs) return false;
        for (const Range& r : segments_[k + 1].needs)
          if (r.bytes > kKernelCopy) return in_at[r.index] != kNowhere && r.bytes > kStageRun;
        return false;
      };
      // Sends down what the first `launched` segments yield: of those that are done, or (all) of all of them.  A copy down that waits
      // for its launches holds up whatever is queued behind it on its copy engine, and which engine a copy up gets depends on the
      // process's other streams: a copy down is queued once its launches are done, or behind the last copy up that goes by
      // engine.  (Both gradients of 10 x 49 x 49 x 117 (*) 5 x 5 x 26 with torch's streams in the process: 855 us with the second operand up behind the first
      // result, 836 on one stream, 589 now; on engines of their own 612 and 586.)
      auto send_down = [&](size_t launched, bool all) {
        for (; sent < launched && (all || pml_hip_event_done(segments_[sent].done)); ++sent) send(segments_[sent]);
      };
      for (size_t k = 0; k < segments_.size(); ++k) {
        Segment& seg = segments_[k];
        Spans up;
        for (const Range& r : seg.needs) {
          const int buf = plan_->input_buffers[r.index];
          const HostSpan& in = inputs[r.index];
          char* const dev = static_cast<char*>(device_[buf]) + r.offset;
          const bool slotted = in_at[r.index] == kInTurn, by_kernel = r.bytes <= kKernelCopy && !slotted;
          for (size_t at = 0; at < r.bytes;) {
            const size_t n = in_at[r.index] == kNowhere ? r.bytes : std::min(kStageRun, r.bytes - at);
            const char* src = static_cast<const char*>(in.data) + (r.offset + at) * (in.f32 ? 2 : 1);
            if (in_at[r.index] != kNowhere) {
              char* const to = base + (slotted ? slots + turn % kStageSlots * kStageRun : in_at[r.index] + r.offset + at);
              if (slotted && turn >= kStageSlots && turn % kStageHalf == 0) hipCheck(pml_hip_event_sync(half_events_[turn / kStageHalf % 2]), "event sync");
              if (in.f32)
                hostToBf16(reinterpret_cast<uint16_t*>(to), reinterpret_cast<const float*>(src), n / 2);
              else
                hostCopy(to, src, n);
              src = to;
            }
            if (by_kernel)
              up.add(dev + at, src, n);
            else
              hipCheck(pml_hip_memcpy_h2d_async(dev + at, src, n, up_stream_), "h2d");
            if (slotted && ++turn % kStageHalf == 0) hipCheck(pml_hip_event_record(half_events_[(turn / kStageHalf - 1) % 2], up_stream_), "event record");
            at += n;
            send_down(k, false);
          }
        }
        send_down(k, k >= last_up);
        up.issue(up_stream_, nullptr, false);
        if (!seg.needs.empty()) {
          hipCheck(pml_hip_event_record(seg.up, up_stream_), "event record");
          hipCheck(pml_hip_stream_wait_event(stream_, seg.up), "wait");
          st->h2d_ms = nowMs() - start;
        } else if (k == 0) {
          hipCheck(pml_hip_event_record(seg.up, stream_), "event record");  // (where it could begin)
        }
        if (record_now && !seg.graph && graphable_ && seg.launches.size() > 1) seg.graph = record(seg.launches);
        if (seg.graph) {
          hipCheck(pml_hip_graph_launch(seg.graph, stream_), "graph launch");
          st->replayed = true;
        } else {
          for (const Launch& l : seg.launches) launch(l.step, l.slice);
        }
        hipCheck(pml_hip_event_record(seg.done, stream_), "event record");
        send_down(k + 1, k >= last_up || quick(k));
      }
      mark();
      for (Segment& seg : segments_) {
        bool waited = false;
        for (const Range& r : seg.yields) {
          if (out_at[r.index] >= kInTurn) continue;
          if (!waited) hipCheck(pml_hip_event_sync(seg.down), "event sync");
          waited = true;
          const HostSpan& out = outputs[r.index];
          char* const to = static_cast<char*>(out.data) + r.offset * (out.f32 ? 2 : 1);
          if (out.f32)
            hostFromBf16(reinterpret_cast<float*>(to), reinterpret_cast<const uint16_t*>(out_place(r)), r.bytes / 2);
          else
            hostCopy(to, out_place(r), r.bytes);
        }
      }
      // (behind the launches, and so behind every copy out of the slots)
      Staging late;
      late.slots = base + slots;
      std::vector<Piece> arriving;
      Spans none;
      for (size_t o = 0; o < outputs.size(); ++o)
        if (out_at[o] == kInTurn) stageOut(&late, outputs[o], bytes_of(plan_->output_buffers[o]), static_cast<const char*>(device_[plan_->output_buffers[o]]), &arriving, &none);
      if (!arriving.empty()) collect(&late, arriving);
      for (pml_hip_stream s : {up_stream_, stream_, down_stream_}) hipCheck(pml_hip_stream_sync(s), "stream sync");
    } catch (...) {
      sync();  // queued copies may still use the caller's memory
      throw;
    }
    st->wall_ms = nowMs() - start;
    // A segment's time is from where it could begin -- its needs up, the one before it done -- to its end.
    for (size_t k = 0; k < segments_.size(); ++k) {
      float ms = 0, behind = 0;
      Segment& seg = segments_[k];
      if (k == 0 || !seg.needs.empty()) hipCheck(pml_hip_event_elapsed_ms(seg.up, seg.done, &ms), "event elapsed");
      if (k > 0) hipCheck(pml_hip_event_elapsed_ms(segments_[k - 1].done, seg.done, &behind), "event elapsed");
      seg.ms = k == 0 ? ms : seg.needs.empty() ? behind : std::min(ms, behind);
      st->kernel_ms += seg.ms;
    }
    describe(st);
    st->kernel_ms = std::min(st->kernel_ms, st->wall_ms);
    st->h2d_ms = std::min(st->h2d_ms, st->wall_ms - st->kernel_ms);
    st->d2h_ms = st->wall_ms - st->h2d_ms - st->kernel_ms;
    return true;
  }

  // Offsets of the temporaries in the arena.  A temporary is live from the first to the last step that names
  // it; steps run in order on one stream, so two temporaries whose spans do not overlap may share bytes.  A
  // value freed by step i is not handed to a value that step i itself defines (kernels read while they write).
  std::vector<size_t> placeTemporaries() {
    const size_t nb = plan_->buffers.size(), ns = plan_->steps.size();
    std::vector<int> first(nb, -1), last(nb, -1);
    auto touch = [&](int buf, size_t step) {
      if (buf < 0 || static_cast<size_t>(buf) >= nb) return;
      if (first[buf] < 0) first[buf] = static_cast<int>(step);
      last[buf] = static_cast<int>(step);
    };
    for (size_t i = 0; i < ns; ++i) {
      const Step& s = plan_->steps[i];
      for (int b : {s.a, s.b, s.c, s.init, s.out2, s.a2, s.b2, s.init2}) touch(b, i);
      for (int b : s.operands) touch(b, i);
      for (int b : s.outs) touch(b, i);
    }
    // (what outlives the sliced steps is written from their first part on)
    if (plan_->slices > 1)
      for (size_t b = 0; b < nb; ++b)
        if (plan_->part_bytes[b] > 0 && first[b] >= 0) first[b] = 0;
    std::vector<size_t> offsets(nb, 0);
    struct Block { size_t off, size; };
    std::vector<Block> free_blocks;
    std::vector<std::vector<int>> starts(ns + 1), ends(ns + 1);
    for (size_t b = 0; b < nb; ++b) {
      if (plan_->buffers[b].kind != BufferInfo::Temp) continue;
      if (first[b] < 0) continue;  // a value no launch touches (its producer was fused away) takes no memory
      unshared_temp_bytes_ += padded(plan_->buffers[b].bytes);
      const size_t f = first[b] < 0 ? 0 : static_cast<size_t>(first[b]);
      const size_t l = last[b] < 0 ? 0 : static_cast<size_t>(last[b]);
      starts[f].push_back(static_cast<int>(b));
      ends[l].push_back(static_cast<int>(b));
    }
    auto release_block = [&](size_t off, size_t size) {
      free_blocks.push_back({off, size});
      std::sort(free_blocks.begin(), free_blocks.end(), [](const Block& x, const Block& y) { return x.off < y.off; });
      for (size_t k = 0; k + 1 < free_blocks.size();) {
        if (free_blocks[k].off + free_blocks[k].size == free_blocks[k + 1].off) {
          free_blocks[k].size += free_blocks[k + 1].size;
          free_blocks.erase(free_blocks.begin() + static_cast<long>(k) + 1);
        } else {
          ++k;
        }
      }
    };
    for (size_t i = 0; i <= ns; ++i) {
      // larger values first: they are the hard ones to place
      std::sort(starts[i].begin(), starts[i].end(),
                [&](int x, int y) { return plan_->buffers[x].bytes > plan_->buffers[y].bytes; });
      for (int b : starts[i]) {
        const size_t need = padded(plan_->buffers[b].bytes);
        size_t best = free_blocks.size();
        for (size_t k = 0; k < free_blocks.size(); ++k)
          if (free_blocks[k].size >= need && (best == free_blocks.size() || free_blocks[k].size < free_blocks[best].size)) best = k;
        if (best < free_blocks.size()) {
          offsets[b] = free_blocks[best].off;
          free_blocks[best].off += need;
          free_blocks[best].size -= need;
          if (!free_blocks[best].size) free_blocks.erase(free_blocks.begin() + static_cast<long>(best));
        } else if (!free_blocks.empty() && free_blocks.back().off + free_blocks.back().size == arena_bytes_) {
          // grow the free block at the end of the arena
          offsets[b] = free_blocks.back().off;
          arena_bytes_ = offsets[b] + need;
          free_blocks.pop_back();
        } else {
          offsets[b] = arena_bytes_;
          arena_bytes_ += need;
        }
      }
      for (int b : ends[i]) release_block(offsets[b], padded(plan_->buffers[b].bytes));
    }
    return offsets;
  }

  void release() {
    for (auto* handles : {&handles_, &last_handles_}) {
      for (const Handles& h : *handles)
        for (int64_t plan : {h.own, h.next})
          if (plan) pml_hip_plan_free(plan);
      handles->clear();
    }
    for (Segment& s : segments_) {
      if (s.graph) pml_hip_graph_destroy(s.graph);
      for (pml_hip_event e : {s.up, s.done, s.down})
        if (e) pml_hip_event_destroy(e);
    }
    segments_.clear();
    if (up_stream_) pml_hip_stream_destroy(up_stream_);
    if (down_stream_) pml_hip_stream_destroy(down_stream_);
    up_stream_ = down_stream_ = nullptr;
    for (size_t i = 0; i < device_.size(); ++i)
      if (device_[i] && owned_[i]) pml_hip_free(device_[i]);
    device_.clear();
    if (arena_) pml_hip_free(arena_);
    arena_ = nullptr;
    for (auto& e : step_events_)
      if (e) pml_hip_event_destroy(e);
    step_events_.clear();
    for (auto& e : half_events_)
      if (e) pml_hip_event_destroy(e);
    half_events_.clear();
    if (ev0_) pml_hip_event_destroy(ev0_);
    if (ev1_) pml_hip_event_destroy(ev1_);
    ev0_ = ev1_ = nullptr;
    if (stamps_) pml_hip_host_free(stamps_);
    stamps_ = nullptr;
    if (graph_) pml_hip_graph_destroy(graph_);
    graph_ = nullptr;
    if (stream_) pml_hip_stream_destroy(stream_);
    stream_ = nullptr;
    if (staging_) pinnedFree(staging_);
    staging_ = nullptr;
  }

  char* ptr(int buf, int64_t elem_off = 0, size_t elem_size = 1) const {
    if (buf < 0) return nullptr;
    return static_cast<char*>(device_[buf]) + elem_off * static_cast<int64_t>(elem_size);
  }

  static size_t elemSize(int dt) { return util::byteSize(static_cast<util::DataType>(dt)); }

  void dispatch(const Step& s, Handles* handles) {
    int64_t h = 0;
    switch (s.kind) {
      case Step::Gemm: {
        h = pml_hip_gemm_dispatch(&s.gemm);
        break;
      }
      case Step::Conv2d: h = pml_hip_conv2d_dispatch(&s.conv); break;
      case Step::Dwconv2d: h = pml_hip_dwconv2d_dispatch(&s.dw); break;
      case Step::Pool2d: h = pml_hip_pool2d_dispatch(&s.pool); break;
      case Step::Eltwise: h = pml_hip_eltwise_dispatch(&s.elt); break;
      case Step::Contract: h = pml_hip_contract_dispatch(&s.con); break;
      case Step::Product: h = pml_hip_product_dispatch(&s.prod); break;
      case Step::ConvGrad: h = pml_hip_conv2d_grad_dispatch(&s.conv, s.grad_which); break;
      case Step::Select:
      case Step::Index:
      case Step::Gather:
      case Step::Scatter:
      case Step::ArgSort:
      case Step::Prng:
      case Step::Softmax:
      case Step::Rows:
      case Step::Argmax:
      case Step::TopK:
      case Step::Copy: return;
    }
    if (!h) throw std::runtime_error("hip dispatch failed for '" + s.text + "': " + pml_hip_last_error());
    handles->own = h;
    // constant right-hand sides are re-laid-out once, here
    if (s.kind == Step::Gemm && s.b_constant && !s.b_is_nk)
      hipCheck(pml_hip_gemm_pack_b(h, ptr(s.b, s.b_off, elemSize(s.gemm.in_dtype)), nullptr), "pack_b");
    if (s.kind == Step::Gemm && s.gemm.k2 > 0 && s.b2_constant && !s.b_is_nk)
      hipCheck(pml_hip_gemm_pack_b2(h, ptr(s.b2, s.b2_off, elemSize(s.gemm.in_dtype)), nullptr), "pack_b2");
    if (s.chained) {
      handles->next = pml_hip_gemm_dispatch(&s.next_gemm);
      if (!handles->next) throw std::runtime_error("hip dispatch failed for '" + s.text + "': " + pml_hip_last_error());
      hipCheck(pml_hip_gemm_pack_b(handles->next, ptr(s.next_b, s.next_b_off, elemSize(s.next_gemm.in_dtype)), nullptr), "pack_b");
    }
    if (s.kind == Step::Conv2d && s.b_constant) hipCheck(pml_hip_conv2d_pack_filter(h, ptr(s.b), nullptr), "pack_filter");
    if (s.kind == Step::Dwconv2d && s.b_constant) hipCheck(pml_hip_dwconv2d_pack_filter(h, ptr(s.b), nullptr), "pack_filter");
  }

  // Step i, or its part `slice` of the leading dimension.
  void launch(size_t i, int slice = -1) {
    const bool last = slice >= 0 && slice == plan_->slices - 1;
    const Step& s = slice < 0 ? plan_->steps[i] : last ? plan_->sliced_last[i] : plan_->sliced[i];
    const Handles& h = last && plan_->uneven ? last_handles_[i] : handles_[i];
    auto ptr = [&](int buf, int64_t elem_off = 0, size_t elem_size = 1) -> char* {
      if (buf < 0) return nullptr;
      return static_cast<char*>(device_[buf]) + (slice > 0 ? static_cast<size_t>(slice) * plan_->part_bytes[buf] : 0) + elem_off * static_cast<int64_t>(elem_size);
    };
    const void* operands[PML_HIP_MAX_EPI_OPERANDS] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    void* outs[PML_HIP_MAX_EPI_OPERANDS] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    for (size_t k = 0; k < s.operands.size() && k < PML_HIP_MAX_EPI_OPERANDS; ++k) operands[k] = ptr(s.operands[k]);
    for (size_t k = 0; k < s.outs.size() && k < PML_HIP_MAX_EPI_OPERANDS; ++k) outs[k] = ptr(s.outs[k]);
    switch (s.kind) {
      case Step::Gemm: {
        const size_t es = elemSize(s.gemm.in_dtype);
        if (s.chained) {
          hipCheck(pml_hip_gemm_chain_invoke(h.own, h.next, ptr(s.a), ptr(s.c), ptr(s.init), ptr(s.a2), ptr(s.init2), operands, ptr(s.out2),
                                             ptr(s.next_init), stream_),
                   s.text.c_str());
          break;
        }
        const void* b = ptr(s.b, s.b_off, es);
        if (s.b_constant && !s.b_is_nk) b = nullptr;  // packed when the executable was built
        if (s.gemm.k2 > 0) {
          const void* b2 = ptr(s.b2, s.b2_off, es);
          if (s.b2_constant && !s.b_is_nk) b2 = nullptr;
          hipCheck(pml_hip_gemm_invoke2(h.own, ptr(s.a, s.a_off, es), b, ptr(s.c, s.c_off, elemSize(s.gemm.c_dtype)), ptr(s.init),
                                        ptr(s.a2, s.a2_off, es), b2, ptr(s.init2), operands, outs, stream_),
                   s.text.c_str());
          break;
        }
        hipCheck(pml_hip_gemm_invoke(h.own, ptr(s.a, s.a_off, es), b, ptr(s.c, s.c_off, elemSize(s.gemm.c_dtype)),
                                     ptr(s.init), operands, outs, stream_),
                 s.text.c_str());
        break;
      }
      case Step::Conv2d:
        hipCheck(pml_hip_conv2d_invoke(h.own, ptr(s.a), s.b_constant ? nullptr : ptr(s.b), ptr(s.c), ptr(s.init), operands,
                                       outs, stream_),
                 s.text.c_str());
        break;
      case Step::Dwconv2d:
        hipCheck(pml_hip_dwconv2d_invoke(h.own, ptr(s.a), s.b_constant ? nullptr : ptr(s.b), ptr(s.c), operands, outs, stream_),
                 s.text.c_str());
        break;
      case Step::Pool2d:
        hipCheck(pml_hip_pool2d_invoke(h.own, ptr(s.a), ptr(s.c), ptr(s.out2), stream_), s.text.c_str());
        break;
      case Step::Eltwise:
        hipCheck(pml_hip_eltwise_invoke(h.own, ptr(s.a), ptr(s.c), operands, outs, stream_), s.text.c_str());
        break;
      case Step::Select:
        hipCheck(pml_hip_select(&s.sel, operands[0], operands[1], operands[2], ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::Softmax:
        hipCheck(pml_hip_softmax(&s.sm, ptr(s.a), ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::Rows:
        hipCheck(pml_hip_rows(&s.rows, operands, outs, stream_), s.text.c_str());
        break;
      case Step::Argmax:
        hipCheck(pml_hip_argmax_rows(s.sm.dtype, s.sm.rows, s.sm.cols, ptr(s.a), reinterpret_cast<int32_t*>(ptr(s.c)), stream_), s.text.c_str());
        break;
      case Step::TopK:
        hipCheck(pml_hip_topk_rows(s.sm.dtype, s.topk_descending, s.sm.rows, s.sm.cols, s.topk, ptr(s.a), ptr(s.c),
                                   reinterpret_cast<int32_t*>(ptr(s.out2)), stream_),
                 s.text.c_str());
        break;
      case Step::Index:
        hipCheck(pml_hip_index(ptr(s.c), static_cast<int32_t>(s.index_sizes.size()), s.index_sizes.data(), s.index_axis, stream_),
                 s.text.c_str());
        break;
      case Step::Contract:
        hipCheck(pml_hip_contract_invoke(h.own, operands, ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::Product:
        hipCheck(pml_hip_product_invoke(h.own, ptr(s.a, s.a_off, elemSize(s.prod.in_dtype)), ptr(s.b, s.b_off, elemSize(s.prod.in_dtype)),
                                        ptr(s.c), ptr(s.init), operands, stream_),
                 s.text.c_str());
        break;
      case Step::ConvGrad:
        hipCheck(pml_hip_conv2d_grad_invoke(h.own, ptr(s.a), ptr(s.b), ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::Copy:
        hipCheck(pml_hip_memcpy_d2d(ptr(s.c), ptr(s.a), s.copy_bytes, stream_), s.text.c_str());
        break;
      case Step::Gather:
        hipCheck(pml_hip_gather(&s.gat, operands[0], operands[1], ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::Scatter:
        hipCheck(pml_hip_scatter(&s.sca, operands[0], operands[1], operands[2], ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::ArgSort:
        hipCheck(pml_hip_argsort(&s.srt, operands[0], ptr(s.c), stream_), s.text.c_str());
        break;
      case Step::Prng:
        hipCheck(pml_hip_prng(operands[0], s.prng_count, s.prng_state ? nullptr : ptr(s.c), s.prng_state ? ptr(s.c) : nullptr, stream_),
                 s.text.c_str());
        break;
    }
  }
};

class HipDevice final : public Device {
 public:
  explicit HipDevice(int ordinal) : ordinal_(ordinal) {}
  std::unique_ptr<Executable> compile(const std::shared_ptr<tile::Program>& program) final {
    if (!program->compiled || program->target != "hip")
      throw std::runtime_error("the program was not compiled for target 'hip'");
    auto plan = std::static_pointer_cast<Plan>(program->compiled);
    return std::make_unique<HipExecutable>(program, plan, ordinal_);
  }

 private:
  int ordinal_;
};

class HipRuntime final : public Runtime {
 public:
  HipRuntime() {
    count_ = static_cast<size_t>(pml_hip_device_count());
    if (count_ == 0) throw std::runtime_error("no HIP device is visible");
  }
  size_t getDeviceCount() const final { return count_; }
  std::shared_ptr<Device> getDevice(size_t ordinal) final {
    if (ordinal >= count_) throw std::out_of_range("hip device ordinal out of range");
    return std::make_shared<HipDevice>(static_cast<int>(ordinal));
  }

 private:
  size_t count_ = 0;
};

std::map<std::string, std::shared_ptr<Runtime>>& registry() {
  static std::map<std::string, std::shared_ptr<Runtime>> r;
  return r;
}

}  // namespace

InvokeStats lastInvokeStats() { return g_stats; }

void registerRuntime(const std::string& id, std::shared_ptr<Runtime> runtime) {
  if (registry().count(id)) throw std::runtime_error("Multiple runtime registrations for id: " + id);
  registry()[id] = std::move(runtime);
}

// Page-locked host memory for buffers the library allocates itself.  Asking for it initialises the GPU runtime as a
// side effect, so a process that must not touch the GPU (one that only builds programs, or that will exec another
// program) sets PLAIDML_PINNED=0; the total of all blocks, those kept for the next allocation among them, is capped
// (PLAIDML_PINNED_MAX_MB, default 4096) because page-locked memory is taken from what the host can page.  Beyond the
// cap, and on any failure, the caller falls back to ordinary memory (nullptr here).
namespace {
PinnedPool& pinnedPool() {  // (never destroyed: buffers may be freed while the process ends)
  static PinnedPool* pool = new PinnedPool(
      [](size_t bytes) -> void* {
        initRuntimes();
        if (listDevices().empty()) return nullptr;
        void* p = nullptr;
        return pml_hip_host_alloc(&p, bytes) == 0 ? p : nullptr;
      },
      [](void* p) { (void)pml_hip_host_free(p); }, size_t{256} << 20);
  return *pool;
}
}  // namespace

void* pinnedAlloc(size_t bytes) {
  void* p = pinnedAllocRaw(bytes);
  if (p) std::memset(p, 0, bytes);
  return p;
}

void* pinnedAllocRaw(size_t bytes) {
  const std::string enabled = util::Settings::Instance()->get("PLAIDML_PINNED");
  if (enabled == "0" || enabled == "false" || enabled == "off") return nullptr;
  const std::string cap_text = util::Settings::Instance()->get("PLAIDML_PINNED_MAX_MB");
  const size_t cap = (cap_text.empty() ? size_t{4096} : static_cast<size_t>(std::strtoull(cap_text.c_str(), nullptr, 10))) << 20;
  return pinnedPool().take(bytes, cap);
}

void pinnedFree(void* p) {
  if (p) pinnedPool().put(p);
}

bool isPinned(const void* p, size_t bytes) { return pinnedPool().holds(p, bytes); }

void initRuntimes() {
  static bool done = false;
  if (done) return;
  done = true;
  // a runtime whose construction fails (no GPU) is skipped, as the reference skips a throwing factory
  // (pmlc/rt/runtime_registry.cc:48-59)
  try {
    registerRuntime("hip", std::make_shared<HipRuntime>());
  } catch (const std::exception&) {
  }
}

std::vector<std::string> listDevices() {
  std::vector<std::string> out;
  for (const auto& kv : registry())
    for (size_t i = 0; i < kv.second->getDeviceCount(); ++i) out.push_back(kv.first + "." + std::to_string(i));
  return out;
}

std::shared_ptr<Device> getDevice(const std::string& deviceID) {
  static const std::regex re("([[:alpha:]][_[:alnum:]]*(?:-[[:alpha:]][_[:alnum:]]*)*)\\.([[:digit:]]+)");
  std::smatch m;
  if (!std::regex_match(deviceID, m, re)) throw std::runtime_error("Invalid device name: " + deviceID);
  auto it = registry().find(m[1].str());
  if (it == registry().end()) throw std::runtime_error("Unable to find " + m[1].str() + " runtime");
  return it->second->getDevice(std::stoul(m[2].str()));
}

}  // namespace pmlc::rt
