// Blocks of scratch memory that calls borrow. Host code only: the memory comes from the two functions a
// pool is made with, so a host build checks it with malloc.
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <vector>

namespace dyng_hip {

struct scratch_block {
  void* p = nullptr;
  size_t bytes = 0;
};

/// A call takes a block, its work on the block ends, and it gives the block back; calls of several threads
/// hold a block each. At most kKept blocks stay with the pool between calls (the largest), and none when
/// its last user has left.
class scratch_pool {
 public:
  using get_fn = void* (*)(size_t);  ///< null when there is no memory left
  using put_fn = void (*)(void*);
  static constexpr int kKept = 2;

  scratch_pool(get_fn get, put_fn put) : get_(get), put_(put) {}
  scratch_pool(const scratch_pool&) = delete;
  scratch_pool& operator=(const scratch_pool&) = delete;
  ~scratch_pool() { clear(); }

  void join() {
    std::lock_guard<std::mutex> hold(lock_);
    ++users_;
  }
  void leave() {
    bool last = false;
    {
      std::lock_guard<std::mutex> hold(lock_);
      last = --users_ == 0;
    }
    if (last) clear();
  }

  /// The smallest kept block of at least `bytes`, or a new one, which takes the place of the largest kept
  /// one that is too small. New ones are rounded up by at most an eighth, so that a stream of slowly
  /// growing calls does not allocate in each. A null block when there is no memory left.
  scratch_block take(size_t bytes) {
    scratch_block small;
    {
      std::lock_guard<std::mutex> hold(lock_);
      auto it = std::lower_bound(kept_.begin(), kept_.end(), bytes,
                                 [](const scratch_block& b, size_t want) { return b.bytes < want; });
      if (it != kept_.end()) {
        const scratch_block b = *it;
        kept_.erase(it);
        return b;
      }
      if (!kept_.empty()) {
        small = kept_.back();
        kept_.pop_back();
      }
    }
    if (small.p != nullptr) put_(small.p);
    size_t step = 4096;
    while (step * 16 < bytes) step *= 2;
    scratch_block b;
    b.bytes = (bytes + step - 1) / step * step;
    b.p = get_(b.bytes);
    if (b.p == nullptr) {  // with what the pool keeps given up, and no more than was asked for
      clear();
      b.bytes = bytes;
      b.p = get_(bytes);
    }
    return b.p != nullptr ? b : scratch_block{};
  }

  /// All work on the block has ended.
  void give(scratch_block b) {
    if (b.p == nullptr) return;
    {
      std::lock_guard<std::mutex> hold(lock_);
      if (users_ > 0) {
        kept_.insert(std::lower_bound(kept_.begin(), kept_.end(), b.bytes,
                                      [](const scratch_block& k, size_t want) { return k.bytes < want; }),
                     b);
        b = scratch_block{};
        if (static_cast<int>(kept_.size()) > kKept) {
          b = kept_.front();
          kept_.erase(kept_.begin());
        }
      }
    }
    if (b.p != nullptr) put_(b.p);
  }

 private:
  void clear() {
    std::vector<scratch_block> all;
    {
      std::lock_guard<std::mutex> hold(lock_);
      all.swap(kept_);
    }
    for (const scratch_block& b : all) put_(b.p);
  }

  std::mutex lock_;
  std::vector<scratch_block> kept_;  ///< by size
  int users_ = 0;
  get_fn get_;
  put_fn put_;
};

}  // namespace dyng_hip
