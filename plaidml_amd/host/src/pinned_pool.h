// Blocks of page-locked host memory and what is kept of them for the next allocation.  No GPU calls of its own: the two
// that make and give back a block come with the pool.
#pragma once

#include <cstddef>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace pmlc::rt {

// Page-locking a block costs about as much as copying it, so a freed block is kept for the next allocation of its size as
// long as all kept ones together stay under `keep` bytes; the one kept longest goes back first.  Blocks come in sizes of
// 1/8 steps between powers of two.  All blocks, in use and kept, at their own sizes, stay within the cap that an allocation
// names: kept ones are given back for it, and when the system has no more to give.
class PinnedPool {
 public:
  PinnedPool(void* (*make)(size_t), void (*give_back)(void*), size_t keep) : make_(make), give_back_(give_back), keep_(keep) {}
  void* take(size_t bytes, size_t cap);              // nullptr: beyond the cap, or the system has none
  void put(void* p);                                 // (what is no block in use is left alone)
  bool holds(const void* p, size_t bytes) const;     // whether [p, p + bytes) lies in one block in use
  size_t total() const;                              // bytes of all blocks, in use and kept

 private:
  void* (*make_)(size_t);
  void (*give_back_)(void*);
  const size_t keep_;
  mutable std::mutex mutex_;
  std::map<const char*, size_t> live_;               // block -> its size
  std::vector<std::pair<char*, size_t>> kept_;       // free blocks, the one freed first in front
  size_t live_total_ = 0, kept_total_ = 0;
};

}  // namespace pmlc::rt
