#include "host_copy.h"

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>

namespace pmlc::rt {

namespace {

// One core moves 20-30 GB/s between memory and memory, the link to the GPU 57: a long pass is cut into pieces that up to
// eight threads take in order.  The threads are started by the first long pass and wait on a condition variable in
// between; a pass that finds them at work for another thread runs alone.  They are never joined (a process may end
// while they wait).
class Helpers {
 public:
  static Helpers& instance() {
    static Helpers* h = new Helpers();
    return *h;
  }

  // fn(i) for every i < n, on this thread and the helpers; returns when all are done
  void run(size_t n, const std::function<void(size_t)>& fn) {
    std::unique_lock<std::mutex> busy(busy_, std::try_to_lock);
    if (!busy.owns_lock() || n < 2 || !start()) {
      for (size_t i = 0; i < n; ++i) fn(i);
      return;
    }
    {
      std::lock_guard<std::mutex> lock(mutex_);
      fn_ = &fn;
      total_ = n;
      next_.store(0, std::memory_order_relaxed);
      ++generation_;
    }
    wake_.notify_all();
    work(fn, n);
    // the last pieces may still be with helpers; none may hold `fn` when this returns
    std::unique_lock<std::mutex> lock(mutex_);
    fn_ = nullptr;
    while (active_ != 0) idle_.wait(lock);
  }

 private:
  std::mutex busy_, mutex_;
  std::condition_variable wake_, idle_;
  const std::function<void(size_t)>* fn_ = nullptr;
  size_t total_ = 0, generation_ = 0;
  std::atomic<size_t> next_{0};
  int active_ = 0, threads_ = -1;

  bool start() {
    if (threads_ >= 0) return threads_ > 0;
    cpu_set_t set;
    int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    threads_ = 0;
    for (int t = 1; t < std::min(cpus, 8); ++t) {
      try {
        std::thread([this] { loop(); }).detach();
        ++threads_;
      } catch (const std::exception&) {
        break;
      }
    }
    return threads_ > 0;
  }

  void work(const std::function<void(size_t)>& fn, size_t n) {
    for (size_t i; (i = next_.fetch_add(1, std::memory_order_relaxed)) < n;) fn(i);
  }

  void loop() {
    size_t seen = 0;
    std::unique_lock<std::mutex> lock(mutex_);
    for (;;) {
      while (seen == generation_ || fn_ == nullptr) {
        seen = generation_;
        wake_.wait(lock);
      }
      seen = generation_;
      const std::function<void(size_t)>* fn = fn_;
      const size_t n = total_;
      ++active_;
      lock.unlock();
      work(*fn, n);
      lock.lock();
      if (--active_ == 0) idle_.notify_all();
    }
  }
};

constexpr size_t kPiece = 256 << 10;  // bytes of the wider side per piece

__attribute__((target_clones("avx512f", "avx2", "default"))) void narrow(uint16_t* dst, const float* src, size_t n) {
  const uint32_t* bits = reinterpret_cast<const uint32_t*>(src);
  for (size_t i = 0; i < n; ++i) {
    const uint32_t u = bits[i];
    const uint32_t r = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
    dst[i] = static_cast<uint16_t>((u & 0x7fffffffu) > 0x7f800000u ? 0x7fc0u : r);
  }
}

__attribute__((target_clones("avx512f", "avx2", "default"))) void widen(float* dst, const uint16_t* src, size_t n) {
  uint32_t* bits = reinterpret_cast<uint32_t*>(dst);
  for (size_t i = 0; i < n; ++i) bits[i] = static_cast<uint32_t>(src[i]) << 16;
}

template <typename F>
void pieces(size_t n, size_t per, F&& f) {
  // (two pieces are not worth waking anybody)
  if (n <= 2 * per) {
    f(size_t{0}, n);
    return;
  }
  Helpers::instance().run((n + per - 1) / per, [&](size_t i) { f(i * per, std::min(n - i * per, per)); });
}

}  // namespace

void hostCopy(void* dst, const void* src, size_t bytes) {
  pieces(bytes, kPiece, [&](size_t at, size_t n) { std::memcpy(static_cast<char*>(dst) + at, static_cast<const char*>(src) + at, n); });
}
void hostToBf16(uint16_t* dst, const float* src, size_t n) {
  pieces(n, kPiece / 4, [&](size_t at, size_t m) { narrow(dst + at, src + at, m); });
}
void hostFromBf16(float* dst, const uint16_t* src, size_t n) {
  pieces(n, kPiece / 4, [&](size_t at, size_t m) { widen(dst + at, src + at, m); });
}

}  // namespace pmlc::rt
