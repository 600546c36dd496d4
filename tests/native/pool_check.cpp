// The block pool on a host-side device of limited memory.  Prints "ok".
#include "gasengine/pool.h"

#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace {
std::mutex mu;
std::map<void *, size_t> live;
std::vector<void *> freed;
size_t used = 0, limit = (size_t)1 << 40, mallocs = 0;
thread_local int device = 0;
thread_local hipError_t last = hipSuccess;
int bad = 0;
}  // namespace

hipError_t hipMalloc(void **p, size_t bytes) {
  std::lock_guard<std::mutex> lock(mu);
  mallocs++;
  if (used + bytes > limit) return last = hipErrorOutOfMemory;
  static uintptr_t next = 4096;
  *p = (void *)next;  // an address only
  next += (bytes + 4095) / 4096 * 4096;
  live[*p] = bytes;
  used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lock(mu);
  if (!live.count(p)) {
    std::printf("freed twice\n");
    bad++;
    return hipErrorInvalidValue;
  }
  used -= live[p];
  live.erase(p);
  freed.push_back(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}

#define CHECK(cond)                                         \
  do {                                                      \
    if (!(cond)) {                                          \
      std::printf("%s:%d %s\n", __FILE__, __LINE__, #cond); \
      bad++;                                                \
    }                                                       \
  } while (0)

using GASengine::BlockPool;
using GASengine::kPoolBlock;
using GASengine::kPoolBlocks;
using GASengine::kPoolBytes;

static void *take(size_t want, size_t *got) {
  void *p = nullptr;
  CHECK(BlockPool::get().take(want, &p, got) == hipSuccess && p && *got >= want);
  return p;
}

int main() {
  BlockPool &pool = BlockPool::get();
  size_t a = 0, b = 0;
  // Reuse: the smallest block that is no more than twice what is wanted, of the same device.
  void *p = take(1000, &a), *q = take(1500, &b);
  pool.give(p, a);
  pool.give(q, b);
  CHECK(take(900, &a) == p && a == 1000);
  CHECK(take(800, &b) == q && b == 1500);
  pool.give(p, a);
  pool.give(q, b);
  size_t c = 0;
  void *r = take(100, &c);
  CHECK(r != p && r != q && c == 100);
  device = 1;
  void *r1 = take(1000, &c);
  CHECK(r1 != p && r1 != q);
  pool.give(r1, c);
  device = 0;
  (void)hipFree(r);
  CHECK(pool.drain() == 3500 && live.empty());
  CHECK(pool.drain() == 0);

  // More blocks than are kept: the oldest make room, first one first.
  std::vector<void *> ps;
  for (int i = 0; i < kPoolBlocks + 3; i++) ps.push_back(take(4096 + i, &a));
  freed.clear();
  for (int i = 0; i < kPoolBlocks + 3; i++) pool.give(ps[i], 4096 + i);
  CHECK(freed.size() == 3 && freed[0] == ps[0] && freed[1] == ps[1] && freed[2] == ps[2]);
  CHECK((int)live.size() == kPoolBlocks);
  // A program that goes on to graphs of another size finds its own blocks again.
  void *big[3];
  for (auto &x : big) x = take(kPoolBlock, &a);
  for (auto &x : big) pool.give(x, kPoolBlock);
  const size_t before = mallocs;
  for (auto &x : big) x = take(kPoolBlock, &a);
  CHECK(mallocs == before);
  for (auto &x : big) pool.give(x, kPoolBlock);
  CHECK(used <= kPoolBytes);
  for (int i = 0; i < 2; i++) pool.give(take(kPoolBlock / 2 + 1, &a), a);
  // Too large to keep.
  p = take(kPoolBlock + 1, &a);
  freed.clear();
  pool.give(p, a);
  CHECK(freed.size() == 1 && freed[0] == p);
  CHECK(used <= kPoolBytes);
  (void)pool.drain();
  CHECK(live.empty() && used == 0);

  // Short of memory: kept blocks go back before an allocation fails, which
  // leaves no error behind for the next call to find.
  limit = 10000;
  pool.give(take(6000, &a), 6000);
  CHECK(take(9000, &a) && used == 9000);
  int *x = nullptr;
  CHECK(GASengine::device_alloc(&x, 2000) == hipErrorOutOfMemory && !x && last == hipSuccess);
  void *y = nullptr;
  CHECK(pool.take(2000, &y, &b) == hipErrorOutOfMemory && !y && b == 0 && last == hipSuccess);
  (void)hipFree(live.begin()->first);
  pool.give(take(6000, &a), 6000);
  CHECK(GASengine::device_alloc(&x, 5000) == hipSuccess && x && used == 5000 && last == hipSuccess);
  (void)hipFree(x);
  limit = (size_t)1 << 40;

  // Scratch: kept when its stream was waited for, freed otherwise.
  for (int released = 0; released < 2; released++) {
    GASengine::PoolScratch s;
    int *z = nullptr;
    for (int i = 0; i < 8; i++) CHECK(s.alloc(&z, (size_t)i << 12) == hipSuccess && z);
    CHECK(s.alloc(&z, 4) == hipErrorInvalidValue && !z);
    if (released) s.released();
  }
  CHECK(live.size() == 8);
  (void)pool.drain();

  // Threads.
  std::vector<std::thread> ts;
  for (int t = 0; t < 4; t++)
    ts.emplace_back([t] {
      for (int i = 0; i < 3000; i++) {
        size_t n = 0, want = (size_t)((i * 7919 + t) % 97 + 1) << 14;
        void *w = take(want, &n);
        if (i % 5 == 4)
          (void)hipFree(w);
        else
          BlockPool::get().give(w, n);
        if (i % 500 == 0) (void)BlockPool::get().drain();
      }
    });
  for (auto &t : ts) t.join();
  CHECK(used <= kPoolBytes && (int)live.size() <= kPoolBlocks);
  (void)pool.drain();
  CHECK(live.empty() && used == 0);
  std::printf(bad ? "failed\n" : "ok\n");
  return bad != 0;
}
