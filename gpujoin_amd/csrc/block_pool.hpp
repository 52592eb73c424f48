// block_pool.hpp - device blocks that dropped indexes and build temporaries leave for the
// next build.  Host-only and free of HIP: Mem allocates and frees.
#pragma once

#include <cstddef>
#include <mutex>
#include <vector>

namespace gj {

// Mem::alloc(void** p, size_t bytes): false when the device is out of memory (other errors
// throw); Mem::release(void* p) noexcept.  Kept: blocks of up to kBlock bytes, at most kBytes
// and kBlocks of them in all; the oldest go back first, and all of them do before an
// allocation through alloc() or take() fails, or when trim(0, 0) asks for it.
template <class Mem>
class BlockPool {
 public:
  static constexpr size_t kBytes = 512ull << 20;
  static constexpr size_t kBlock = kBytes / 2;
  static constexpr size_t kBlocks = 64;

  // Sizes in steps of an eighth of their power of two (4 KiB at least), so that builds over
  // columns of about the same size share blocks; larger ones than the pool keeps as they are.
  static size_t size_of(size_t bytes) {
    if (bytes > kBlock) return bytes;
    size_t step = 4096;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
  }

  // `bytes` of device memory from outside the pool; null: there are none, with the pool empty.
  void* alloc(size_t bytes) {
    void* p = nullptr;
    if (Mem::alloc(&p, bytes)) return p;
    trim(0, 0);
    return Mem::alloc(&p, bytes) ? p : nullptr;
  }

  // A block of at least `bytes`, its true size in `cap`, kept or new; null as for alloc().
  void* take(size_t bytes, size_t& cap, int dev) {
    cap = size_of(bytes);
    if (void* p = find(cap, dev)) return p;
    void* p = alloc(cap);
    if (!p && cap != bytes) p = alloc(cap = bytes);  // what the caller needs may fit
    return p;
  }

  // Keeps a block that nothing on the device uses any more; false: the caller frees it.
  bool keep(void* p, size_t cap, int dev) noexcept {
    if (cap > kBlock || cap != size_of(cap)) return false;
    try {
      std::lock_guard<std::mutex> g(mu_);
      blocks_.push_back({p, cap, dev});
      held_ += cap;
    } catch (...) {
      return false;
    }
    trim(kBytes, kBlocks);
    return true;
  }

  // Frees the oldest blocks until the pool holds no more than this.
  void trim(size_t max_bytes, size_t max_blocks) noexcept {
    for (;;) {
      void* p = nullptr;
      {
        std::lock_guard<std::mutex> g(mu_);
        if (held_ <= max_bytes && blocks_.size() <= max_blocks) return;
        p = blocks_.front().p;
        held_ -= blocks_.front().cap;
        blocks_.erase(blocks_.begin());
      }
      Mem::release(p);
    }
  }

 private:
  struct Block {
    void* p;
    size_t cap;
    int dev;
  };

  void* find(size_t cap, int dev) {
    std::lock_guard<std::mutex> g(mu_);
    for (size_t i = blocks_.size(); i-- > 0;) {
      if (blocks_[i].cap != cap || blocks_[i].dev != dev) continue;
      void* p = blocks_[i].p;
      blocks_.erase(blocks_.begin() + static_cast<std::ptrdiff_t>(i));
      held_ -= cap;
      return p;
    }
    return nullptr;
  }

  std::mutex mu_;
  std::vector<Block> blocks_;  // oldest first
  size_t held_ = 0;
};

}  // namespace gj
