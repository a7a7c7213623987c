#include "pinned_pool.h"

#include <algorithm>

namespace pmlc::rt {

void* PinnedPool::take(size_t bytes, size_t cap) {
  if (bytes > cap) return nullptr;
  size_t step = 4096;
  while (step * 16 <= bytes) step *= 2;
  size_t size = (std::max<size_t>(bytes, 1) + step - 1) / step * step;
  if (size > cap) size = bytes;  // (up to the cap itself is to be had)
  char* p = nullptr;
  std::vector<char*> back;
  {
    std::lock_guard<std::mutex> lock(mutex_);
    for (size_t i = kept_.size(); i-- > 0;) {
      if (kept_[i].second != size || live_total_ + kept_total_ > cap) continue;
      p = kept_[i].first;
      kept_.erase(kept_.begin() + static_cast<long>(i));
      kept_total_ -= size;
      live_[p] = size;
      live_total_ += size;
      return p;
    }
    if (live_total_ + size > cap) return nullptr;
    while (live_total_ + kept_total_ + size > cap) {
      back.push_back(kept_.front().first);
      kept_total_ -= kept_.front().second;
      kept_.erase(kept_.begin());
    }
    live_total_ += size;  // (taken before the lock goes, so that two threads cannot both have the last of it)
  }
  for (char* b : back) give_back_(b);
  p = static_cast<char*>(make_(size));
  if (!p) {
    std::vector<std::pair<char*, size_t>> all;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      all.swap(kept_);
      kept_total_ = 0;
    }
    for (const auto& b : all) give_back_(b.first);
    if (!all.empty()) p = static_cast<char*>(make_(size));
  }
  std::lock_guard<std::mutex> lock(mutex_);
  if (p)
    live_[p] = size;
  else
    live_total_ -= size;
  return p;
}

void PinnedPool::put(void* p) {
  std::vector<char*> back;
  {
    std::lock_guard<std::mutex> lock(mutex_);
    const auto it = live_.find(static_cast<const char*>(p));
    if (it == live_.end()) return;
    const size_t size = it->second;
    live_.erase(it);
    live_total_ -= size;
    if (size > keep_) {
      back.push_back(static_cast<char*>(p));
    } else {
      kept_.emplace_back(static_cast<char*>(p), size);
      kept_total_ += size;
      while (kept_total_ > keep_) {
        back.push_back(kept_.front().first);
        kept_total_ -= kept_.front().second;
        kept_.erase(kept_.begin());
      }
    }
  }
  for (char* b : back) give_back_(b);
}

bool PinnedPool::holds(const void* p, size_t bytes) const {
  std::lock_guard<std::mutex> lock(mutex_);
  auto it = live_.upper_bound(static_cast<const char*>(p));
  if (it == live_.begin()) return false;
  --it;
  return static_cast<const char*>(p) + bytes <= it->first + it->second;
}

size_t PinnedPool::total() const {
  std::lock_guard<std::mutex> lock(mutex_);
  return live_total_ + kept_total_;
}

}  // namespace pmlc::rt
