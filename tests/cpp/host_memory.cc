// The parts of the host runtime that make no GPU calls, for tests/test_host_memory.py: the passes over arrays
// (host_copy.cc) and the pool of page-locked blocks (pinned_pool.cc) on memory of this file's own.
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "host_copy.h"
#include "pinned_pool.h"

namespace {
size_t g_limit = ~size_t{0}, g_made = 0, g_most = 0;  // bytes the system has, has given, has ever given
void* make(size_t bytes) {
  if (g_made + bytes > g_limit) return nullptr;
  g_made += bytes;
  if (g_made > g_most) g_most = g_made;
  size_t* p = static_cast<size_t*>(std::malloc(bytes + 64));
  *p = bytes;
  return p + 8;
}
void giveBack(void* p) {
  size_t* b = static_cast<size_t*>(p) - 8;
  g_made -= *b;
  std::free(b);
}
}  // namespace

extern "C" {
void to_bf16(uint16_t* dst, const float* src, size_t n) { pmlc::rt::hostToBf16(dst, src, n); }
void from_bf16(float* dst, const uint16_t* src, size_t n) { pmlc::rt::hostFromBf16(dst, src, n); }
void copy(void* dst, const void* src, size_t n) { pmlc::rt::hostCopy(dst, src, n); }

void* pool_new(size_t keep, size_t limit) {
  g_limit = limit;
  g_made = g_most = 0;
  return new pmlc::rt::PinnedPool(make, giveBack, keep);
}
void* pool_take(void* pool, size_t bytes, size_t cap) { return static_cast<pmlc::rt::PinnedPool*>(pool)->take(bytes, cap); }
void pool_put(void* pool, void* p) { static_cast<pmlc::rt::PinnedPool*>(pool)->put(p); }
int pool_holds(void* pool, void* p, size_t bytes) { return static_cast<pmlc::rt::PinnedPool*>(pool)->holds(p, bytes); }
size_t pool_total(void* pool) { return static_cast<pmlc::rt::PinnedPool*>(pool)->total(); }
size_t system_given() { return g_made; }
size_t system_most() { return g_most; }
}

// Under a sanitizer: long passes from several threads at once, of which all but one find the helper threads at work.
int main() {
  const size_t n = 3 << 20;
  std::vector<std::thread> threads;
  std::vector<int> wrong(4, 0);
  for (int t = 0; t < 4; ++t)
    threads.emplace_back([&, t] {
      std::vector<float> a(n), b(n);
      std::vector<uint16_t> h(n);
      for (size_t i = 0; i < n; ++i) a[i] = static_cast<float>((i + static_cast<size_t>(t)) & 255);
      for (int round = 0; round < 3; ++round) {
        pmlc::rt::hostToBf16(h.data(), a.data(), n);
        pmlc::rt::hostFromBf16(b.data(), h.data(), n);
        wrong[t] += std::memcmp(a.data(), b.data(), n * 4) != 0;
        pmlc::rt::hostCopy(b.data() + 1, a.data(), n * 4 - 4);
        wrong[t] += std::memcmp(a.data(), b.data() + 1, n * 4 - 4) != 0;
      }
    });
  for (auto& t : threads) t.join();
  for (int w : wrong)
    if (w) return 1;
  return 0;
}
