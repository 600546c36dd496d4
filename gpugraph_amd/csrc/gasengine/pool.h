// Device memory kept between uses, for programs that load a graph, query it
// and drop it again: hipMalloc and hipFree (which waits for the whole device)
// were more than half of such a pass (a 300k-vertex, 4.8M-edge directed graph
// loaded, four BFS trees, unloaded: 28 pairs, 3.7 of 6.7 ms; 4.5 ms with
// the blocks kept).
//
// A block may be given back only when nothing on the device can still use it:
// the caller has synchronised the stream (or the device) that did.  Blocks are
// kept per device, at most kPoolBlocks of them and kPoolBytes in all (larger
// ones than kPoolBlock go back to the runtime at once, the oldest ones when
// there is no room).  Every allocation of the engine and its programs goes
// through take() or device_alloc(): one that fails for want of memory returns
// all kept blocks to the runtime and tries again.  drain() returns them on
// request (a program that resets the device does so first: the blocks do not
// outlive it).  Nothing here allocates host memory or throws.  Any thread may
// call.  Contents are whatever the last user left.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <new>

namespace GASengine {

constexpr size_t kPoolBytes = (size_t)256 << 20;
constexpr size_t kPoolBlock = (size_t)64 << 20;
constexpr int kPoolBlocks = 128;

class BlockPool {
 public:
  static BlockPool &get() {
    // Never destroyed (the runtime may be gone by then), no allocation of its own.
    alignas(BlockPool) static unsigned char storage[sizeof(BlockPool)];
    static BlockPool *pool = ::new (storage) BlockPool();
    return *pool;
  }

  // At least `want` bytes (> 0) on the current device; *bytes gets the size.
  hipError_t take(size_t want, void **p, size_t *bytes) {
    *p = nullptr;
    *bytes = 0;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      int best = -1;
      for (int i = 0; i < count_; i++) {
        const Block &b = blocks_[i];
        if (b.device == dev && b.bytes >= want && b.bytes <= 2 * want &&
            (best < 0 || b.bytes < blocks_[best].bytes))
          best = i;
      }
      if (best >= 0) {
        *p = blocks_[best].p;
        *bytes = blocks_[best].bytes;
        remove(best);
        return hipSuccess;
      }
    }
    e = hipMalloc(p, want);
    if (e == hipErrorOutOfMemory && drain() > 0) {
      (void)hipGetLastError();
      e = hipMalloc(p, want);
    }
    if (e == hipSuccess) {
      *bytes = want;
    } else {
      *p = nullptr;
      (void)hipGetLastError();  // reported by the return value alone
    }
    return e;
  }

  // Keeps a block of the current device, or frees it.
  void give(void *p, size_t bytes) {
    if (!p) return;
    int dev = 0;
    if (bytes > kPoolBlock || hipGetDevice(&dev) != hipSuccess) {
      (void)hipFree(p);
      return;
    }
    void *old[kPoolBlocks];
    int olds = 0;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      while (count_ == kPoolBlocks || held_ + bytes > kPoolBytes) {
        old[olds++] = blocks_[0].p;
        remove(0);
      }
      blocks_[count_++] = {p, bytes, dev};
      held_ += bytes;
    }
    for (int i = 0; i < olds; i++) (void)hipFree(old[i]);
  }

  // Frees every kept block; the bytes they held.
  size_t drain() {
    void *old[kPoolBlocks];
    int olds = 0;
    size_t bytes = 0;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      while (olds < count_) {
        old[olds] = blocks_[olds].p;
        olds++;
      }
      bytes = held_;
      count_ = 0;
      held_ = 0;
    }
    for (int i = 0; i < olds; i++) (void)hipFree(old[i]);
    return bytes;
  }

 private:
  struct Block {
    void *p;
    size_t bytes;
    int device;
  };
  void remove(int at) {  // the order of age is kept
    held_ -= blocks_[at].bytes;
    count_--;
    for (int i = at; i < count_; i++) blocks_[i] = blocks_[i + 1];
  }
  std::mutex mutex_;
  Block blocks_[kPoolBlocks];  // oldest first
  int count_ = 0;
  size_t held_ = 0;
};

// hipMalloc for memory that is freed with hipFree: kept blocks are returned to
// the runtime before it fails.  *p is null on failure.
template <class T>
inline hipError_t device_alloc(T **p, size_t bytes) {
  void *q = nullptr;
  hipError_t e = hipMalloc(&q, bytes);
  if (e == hipErrorOutOfMemory && BlockPool::get().drain() > 0) {
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
  PoolScratch() = default;
  PoolScratch(const PoolScratch &) = delete;
  PoolScratch &operator=(const PoolScratch &) = delete;
  ~PoolScratch() {
    for (int i = 0; i < count_; i++) {
      if (idle_)
        BlockPool::get().give(blocks_[i].p, blocks_[i].bytes);
      else
        (void)hipFree(blocks_[i].p);
    }
  }
  // At most kMax blocks.
  template <class T>
  hipError_t alloc(T **p, size_t bytes) {
    *p = nullptr;
    if (count_ == kMax) return hipErrorInvalidValue;
    Block b{nullptr, 0};
    const hipError_t e = BlockPool::get().take(bytes ? bytes : 4, &b.p, &b.bytes);
    if (e != hipSuccess) return e;
    *p = static_cast<T *>(b.p);
    blocks_[count_++] = b;
    return hipSuccess;
  }
  void released() { idle_ = true; }

 private:
  static constexpr int kMax = 8;
  struct Block {
    void *p;
    size_t bytes;
  };
  Block blocks_[kMax];
  int count_ = 0;
  bool idle_ = false;
};

}  // namespace GASengine
