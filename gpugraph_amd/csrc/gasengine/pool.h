// Device memory kept between uses, for programs that load a graph, query it
// and drop it again: hipMalloc and hipFree (which waits for the whole device)
// were more than half of such a pass (a 300k-vertex, 4.8M-edge directed graph
// loaded, four BFS trees, unloaded: 28 pairs, 3.7 of 6.6 ms; 3.0 ms with
// the blocks kept).
//
// A block may be given back only when nothing on the device can still use it:
// the caller has synchronised the stream (or the device) that did.  Blocks are
// kept per device, at most kPoolBlocks of them and kPoolBytes in all (larger
// ones than kPoolBlock go back to the runtime at once).  Every allocation of
// the engine and its programs goes through take() or device_alloc(): one that
// fails for want of memory returns all kept blocks to the runtime and tries
// again.  Any thread may call.  Contents are whatever the last user left.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

namespace GASengine {

constexpr size_t kPoolBytes = (size_t)256 << 20;
constexpr size_t kPoolBlock = (size_t)64 << 20;
constexpr size_t kPoolBlocks = 128;

class BlockPool {
 public:
  static BlockPool &get() {
    static BlockPool *pool = new BlockPool();  // never destroyed: the runtime may be gone by then
    return *pool;
  }

  // At least `want` bytes (> 0) on the current device; *bytes gets the size.
  hipError_t take(size_t want, void **p, size_t *bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      size_t best = blocks_.size();
      for (size_t i = 0; i < blocks_.size(); i++) {
        const Block &b = blocks_[i];
        if (b.device == dev && b.bytes >= want && b.bytes <= 2 * want &&
            (best == blocks_.size() || b.bytes < blocks_[best].bytes))
          best = i;
      }
      if (best < blocks_.size()) {
        *p = blocks_[best].p;
        *bytes = blocks_[best].bytes;
        held_ -= *bytes;
        blocks_[best] = blocks_.back();
        blocks_.pop_back();
        return hipSuccess;
      }
    }
    e = hipMalloc(p, want);
    if (e == hipErrorOutOfMemory && drain()) {
      (void)hipGetLastError();
      e = hipMalloc(p, want);
    }
    *bytes = e == hipSuccess ? want : 0;
    if (e != hipSuccess) {
      *p = nullptr;
      (void)hipGetLastError();  // reported by the return value alone
    }
    return e;
  }

  // Keeps a block of the current device, or frees it.
  void give(void *p, size_t bytes) {
    if (!p) return;
    int dev = 0;
    if (bytes <= kPoolBlock && hipGetDevice(&dev) == hipSuccess) {
      std::lock_guard<std::mutex> lock(mutex_);
      if (held_ + bytes <= kPoolBytes && blocks_.size() < kPoolBlocks) {
        blocks_.push_back({p, bytes, dev});
        held_ += bytes;
        return;
      }
    }
    (void)hipFree(p);
  }

  // Frees every kept block; whether there was one.
  bool drain() {
    std::vector<Block> old;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      old.swap(blocks_);
      held_ = 0;
    }
    for (const Block &b : old) (void)hipFree(b.p);
    return !old.empty();
  }

 private:
  struct Block {
    void *p;
    size_t bytes;
    int device;
  };
  std::mutex mutex_;
  std::vector<Block> blocks_;
  size_t held_ = 0;
};

// hipMalloc for memory that is freed with hipFree: kept blocks are returned to
// the runtime before it fails.  *p is null on failure.
template <class T>
inline hipError_t device_alloc(T **p, size_t bytes) {
  void *q = nullptr;
  hipError_t e = hipMalloc(&q, bytes);
  if (e == hipErrorOutOfMemory && BlockPool::get().drain()) {
    (void)hipGetLastError();
    e = hipMalloc(&q, bytes);
  }
  if (e != hipSuccess) (void)hipGetLastError();  // reported by the return value alone
  *p = e == hipSuccess ? static_cast<T *>(q) : nullptr;
  return e;
}

// Scratch of one function that ends with its stream synchronised: released()
// says so, after which the blocks are kept; otherwise they are freed (which
// waits for the device).
class PoolScratch {
 public:
  ~PoolScratch() {
    for (const auto &b : blocks_) {
      if (idle_)
        BlockPool::get().give(b.p, b.bytes);
      else
        (void)hipFree(b.p);
    }
  }
  template <class T>
  hipError_t alloc(T **p, size_t bytes) {
    Block b{nullptr, 0};
    const hipError_t e = BlockPool::get().take(bytes ? bytes : 4, &b.p, &b.bytes);
    *p = static_cast<T *>(b.p);
    if (e == hipSuccess) blocks_.push_back(b);
    return e;
  }
  void released() { idle_ = true; }

 private:
  struct Block {
    void *p;
    size_t bytes;
  };
  std::vector<Block> blocks_;
  bool idle_ = false;
};

}  // namespace GASengine
