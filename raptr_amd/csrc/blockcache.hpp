// blockcache.hpp -- bounded cache of freed device blocks: its rules, over a
// driver D that makes the device calls (HIP in runtime.hip, a model in
// tests/cpp/test_block_cache.cpp).
//
// A reconstruction of 30M entries allocates and frees 2.2 GB in 60 blocks: 8 ms
// of a 19 ms call in the driver, and 85 ms once the device's cleared memory is
// used up, since the driver clears a freed block before it hands it out again.
// Freed blocks of kLeast to kBlock bytes are kept, up to kBytes per device, the
// oldest given back first, all of them when an allocation finds no memory or on
// request (raptr_release_cached: other allocators cannot ask for them).  A
// kept block is cleared when it is freed, so a caller sees what it saw before:
// idle, cleared memory.  Sizes are rounded to eighths of a power of two, so that
// lists of similar length find each other's blocks.
//
// Blocks of less than 2 MiB the driver hands out of its own store: 0.7 us an
// allocation and 0.6 a free, 0.8 and 11.8 through the cache (which waits and
// clears).  From there on 22 and 161 us (60 blocks of 1 to 8 MB at a time), 28
// and 218 (40 of 8 to 64 MB), 32 and 227 (12 of 64 to 300 MB); through the cache
// 0.9 and 12.7, 1.1 and 16.5, 5.4 and 35.
#pragma once

#include <cstddef>
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>

namespace raptr {

// D: Error with kOk, kNoMemory and kInvalid; device(int*) (the current one),
// alloc(void**, bytes), release(p), extent(p) (bytes of the driver's block that
// starts at p, 0 if none), wait() (all work of the current device has ended),
// clear(p, bytes, dev) (queued), wait_clear(dev) (all of them have ended) and
// forget_error().
template <class D>
class BlockCache {
 public:
  using Error = typename D::Error;
  static constexpr size_t kLeast = size_t(2) << 20;
  static constexpr size_t kBlock = size_t(1) << 30;
  static constexpr size_t kBytes = size_t(4) << 30;

  static size_t rounded(size_t bytes) {
    size_t step = kLeast / 16;
    while (step * 16 < bytes) step *= 2;  // bytes in (8, 16] steps
    return (bytes + step - 1) / step * step;
  }

  // No exception leaves these (they serve C entry points): without host memory
  // for the cache's own lists, kNoMemory.
  Error malloc(void** p, size_t bytes) noexcept {
    *p = nullptr;
    try {
      return take_or_alloc(p, bytes);
    } catch (...) {
      if (*p) (void)d_.release(*p);
      *p = nullptr;
      return D::kNoMemory;
    }
  }

  // idle: the caller has waited for the device
  Error free(void* p, bool idle) noexcept {
    try {
      return keep_or_release(p, idle);
    } catch (...) {
      return D::kNoMemory;
    }
  }

  // Kept blocks of a device given back to the driver, the oldest first, down to
  // most bytes; the bytes given back.
  size_t give_back(int dev, size_t most) noexcept {
    try {
      return release_kept(dev, most);
    } catch (...) {
      return 0;
    }
  }

  // of the current device
  size_t kept_bytes() {
    int dev = 0;
    if (d_.device(&dev) != D::kOk) return 0;
    std::lock_guard<std::mutex> lock(mu_);
    const auto it = kept_bytes_.find(dev);
    return it == kept_bytes_.end() ? 0 : it->second;
  }

  D& driver() { return d_; }

 private:
  struct Block {
    size_t bytes;
    int dev;
    bool kept;  // freed by its owner, in kept_
  };

  Error take_or_alloc(void** p, size_t bytes) {
    const bool ours = bytes >= kLeast && bytes <= kBlock;
    if (!ours) {
      Error e = d_.alloc(p, bytes);
      if (e != D::kNoMemory) return e;
    }
    int dev = 0;
    Error e = d_.device(&dev);
    if (e != D::kOk) return e;
    const size_t need = ours ? rounded(bytes) : bytes;
    if (ours) {
      std::lock_guard<std::mutex> lock(mu_);
      while (take(dev, need, p)) {
        Block& b = blocks_[*p];
        const bool there = d_.extent(*p) >= b.bytes;
        // (its clearing, asked for when it was freed, has mostly long ended)
        if (there && d_.wait_clear(dev) == D::kOk) return D::kOk;
        d_.forget_error();
        if (there) {
          keep(*p, b, true);
          *p = nullptr;
          break;
        }
        blocks_.erase(*p);  // released behind the cache's back
        *p = nullptr;
      }
    }
    size_t got = need;
    e = ours ? d_.alloc(p, need) : D::kNoMemory;
    if (e == D::kNoMemory && release_kept(dev, 0)) {
      d_.forget_error();
      e = d_.alloc(p, need);
    }
    if (e == D::kNoMemory && need > bytes) {  // without the rounding
      d_.forget_error();
      e = d_.alloc(p, got = bytes);
    }
    if (e == D::kOk && ours) {
      std::lock_guard<std::mutex> lock(mu_);
      blocks_[*p] = Block{got, dev, false};
    }
    return e;
  }

  Error keep_or_release(void* p, bool idle) {
    if (!p) return D::kOk;
    Block b{0, 0, false};
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = blocks_.find(p);
      if (it != blocks_.end()) {
        if (it->second.kept && d_.extent(p) >= it->second.bytes) return D::kInvalid;  // freed twice
        b = it->second;
        if (b.kept) {  // the driver's no more; p is another block, not the cache's
          kept_.remove(p);
          kept_bytes_[b.dev] -= b.bytes;
          b.bytes = 0;
        }
        blocks_.erase(it);
      }
    }
    int dev = 0;
    // not the cache's, another device's, released and allocated again elsewhere
    // with fewer bytes, or a device that cannot be waited for (a capture): the
    // driver's own free
    if (!b.bytes || d_.device(&dev) != D::kOk || dev != b.dev || d_.extent(p) < b.bytes ||
        (!idle && d_.wait() != D::kOk)) {
      d_.forget_error();
      const Error e = d_.release(p);
      if (e != D::kOk && b.bytes) {  // still the caller's
        std::lock_guard<std::mutex> lock(mu_);
        blocks_[p] = b;
      }
      return e;
    }
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (d_.clear(p, b.bytes, dev) != D::kOk) {
        d_.forget_error();
        return d_.release(p);
      }
      keep(p, b, false);
    }
    (void)release_kept(dev, kBytes);
    return D::kOk;
  }

  // (A release can wait for the device: the lock is not held meanwhile.)
  size_t release_kept(int dev, size_t most) {
    std::list<std::pair<void*, Block>> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      for (auto it = kept_.begin(); kept_bytes_[dev] > most && it != kept_.end();) {
        const Block b = blocks_[*it];
        if (b.dev != dev) {
          ++it;
          continue;
        }
        out.emplace_back(*it, b);
        kept_bytes_[dev] -= b.bytes;
        blocks_.erase(*it);
        it = kept_.erase(it);
      }
    }
    size_t bytes = 0;
    for (auto& [p, b] : out) {
      if (d_.release(p) == D::kOk) {
        bytes += b.bytes;
        continue;
      }
      d_.forget_error();
      if (d_.extent(p) < b.bytes) continue;  // the driver's no more
      std::lock_guard<std::mutex> lock(mu_);
      keep(p, b, true);
    }
    return bytes;
  }

  void keep(void* p, Block b, bool front) {
    b.kept = true;
    blocks_[p] = b;
    kept_bytes_[b.dev] += b.bytes;
    front ? kept_.push_front(p) : kept_.push_back(p);
  }

  // the smallest kept block of the device with need bytes and at most a quarter
  // more, out of kept_
  bool take(int dev, size_t need, void** p) {
    auto best = kept_.end();
    size_t least = need + need / 4 + 1;
    for (auto it = kept_.begin(); it != kept_.end(); ++it) {
      const Block& b = blocks_[*it];
      if (b.dev == dev && b.bytes >= need && b.bytes < least) {
        best = it;
        least = b.bytes;
      }
    }
    if (best == kept_.end()) return false;
    *p = *best;
    blocks_[*p].kept = false;
    kept_bytes_[dev] -= least;
    kept_.erase(best);
    return true;
  }

  D d_;
  std::mutex mu_;
  std::unordered_map<void*, Block> blocks_;  // handed out or kept
  std::list<void*> kept_;                    // oldest first
  std::map<int, size_t> kept_bytes_;
};

}  // namespace raptr
