// Allocation failures of the generic engine and the vertex programs, without a
// device: hipMalloc is replaced by one that fails on request, launches and
// copies are counted instead of made.  Prints "ok" when every failure comes
// back as hipErrorOutOfMemory with nothing launched by the program, and when a
// failure that the kept blocks can cure is cured by returning them.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <map>

namespace fake {
int fail_at = 0;      // the fail_at-th allocation from here on fails (0: none), and
bool short_of = false;  // every one fails while blocks are kept
int calls = 0, launches = 0, frees = 0;
std::map<void *, size_t> live;
template <class T>
hipError_t alloc(T **p, size_t bytes) {
  calls++;
  if ((fail_at && calls >= fail_at) || (short_of && !live.empty() && frees == 0)) {
    *p = reinterpret_cast<T *>(16);  // what a caller that ignores the status might use
    return hipErrorOutOfMemory;
  }
  *p = static_cast<T *>(std::malloc(bytes ? bytes : 1));
  live[*p] = bytes;
  return hipSuccess;
}
inline hipError_t release(void *p) {
  frees++;
  if (live.erase(p)) std::free(p);
  return hipSuccess;
}
inline hipError_t device(int *d) {
  *d = 0;
  return hipSuccess;
}
template <class... A>
hipError_t launched(A...) {
  launches++;
  return hipSuccess;
}
template <class... A>
hipError_t done(A...) {
  return hipSuccess;
}
template <class... A>
hipError_t refused(A...) {
  return hipErrorNotSupported;
}
}  // namespace fake

#define hipMalloc fake::alloc
#define hipHostMalloc(p, n) (*(void **)(p) = std::malloc(n), hipSuccess)
#define hipHostFree(p) (std::free(p), hipSuccess)
#define hipFree fake::release
#define hipGetDevice fake::device
#define hipMemcpyAsync fake::launched
#define hipMemcpy fake::launched
#define hipStreamSynchronize fake::done
#define hipGetLastError fake::done
#define hipStreamCreateWithFlags fake::refused  // ends a run whose allocations all succeeded
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) ((void)fake::launches++)

#include "gasengine/enactor_vertex_centric.h"
#include "programs/bfs.h"
#include "programs/cc.h"
#include "programs/pagerank.h"
#include "programs/sssp.h"
#include "programs/variants.h"

static int bad = 0;
#define CHECK(cond)                                                  \
  do {                                                               \
    if (!(cond)) {                                                   \
      std::printf("%s:%d %s\n", __FILE__, __LINE__, #cond);          \
      bad++;                                                         \
    }                                                                \
  } while (0)

static GASengine::DeviceGraph graph() {
  static int32_t ro[9] = {0, 1, 2, 3, 4, 5, 6, 7, 8}, col[8] = {1, 2, 3, 4, 5, 6, 7, 0};
  GASengine::DeviceGraph g;
  g.nodes = 8;
  g.edges = 8;
  g.directed = 1;
  g.row_offsets = g.column_offsets = ro;
  g.column_indices = g.row_indices = col;
  g.edge_values = col;
  return g;
}

// A program's Initialize with its k-th allocation failing launches nothing.
template <class P>
static void initialize_only(const char *name) {
  for (int k = 1;; k++) {
    typename P::VertexType v;
    typename P::EdgeType e;
    int32_t queue[3][8];
    int *keys[3] = {queue[0], queue[1], queue[2]};
    typename P::MiscType *vals[3] = {};
    int src = 1;
    const GASengine::DeviceGraph g = graph();
    fake::calls = fake::launches = 0;
    fake::fail_at = k;
    GASengine::program_error() = hipSuccess;
    P::Initialize(1, 8, 8, 1, &src, (int *)g.row_offsets, (int *)g.column_indices, (int *)g.column_offsets,
                  (int *)g.row_indices, (typename P::DataType *)g.edge_values, v, e, keys, vals);
    fake::fail_at = 0;
    const bool reached = fake::calls >= k;
    if (reached) {
      CHECK(GASengine::program_error() == hipErrorOutOfMemory);
      CHECK(fake::launches == 0);
    } else {
      CHECK(GASengine::program_error() == hipSuccess);
      CHECK(k > 1);
    }
    P::Release(v, e);
    if (bad) std::printf("  in %s, allocation %d\n", name, k);
    if (!reached) break;
  }
}

// A whole run with its k-th allocation failing reports it.
template <class P, bool PREDS>
static void whole_run(const char *name) {
  using Problem = GASengine::CsrProblem<P, int, int, typename P::DataType, PREDS>;
  for (int k = 1; k < 100; k++) {
    Problem prob;
    GASengine::EnactorVertexCentric<Problem, P> enactor;
    int src = 1;
    fake::calls = 0;
    fake::fail_at = k;
    hipError_t e = prob.Attach(graph(), nullptr);
    if (e == hipSuccess) e = enactor.EnactIterativeSearch(prob, nullptr, 1, 1, &src);
    fake::fail_at = 0;
    const bool reached = fake::calls >= k;
    CHECK(e == (reached ? hipErrorOutOfMemory : hipErrorNotSupported));
    P::Release(prob.vertex_list, prob.edge_list);
    if (bad) std::printf("  in a run of %s, allocation %d\n", name, k);
    if (!reached) {
      CHECK(k > 15);
      break;
    }
  }
}

template <class P>
static void program(const char *name) {
  initialize_only<P>(name);
  whole_run<P, false>(name);
  whole_run<P, true>(name);
}

int main() {
  program<bfs>("bfs");
  program<sssp>("sssp");
  program<cc>("cc");
  program<pagerank>("pagerank");
  program<bfs_reverse>("bfs_reverse");
  program<cc_weak>("cc_weak");
  program<pagerank_all>("pagerank_all");
  program<pagerank_share>("pagerank_share");
  program<pagerank_all_share>("pagerank_all_share");
  // A block kept by the pool is what is missing: it is returned, and the
  // allocation succeeds.
  void *p = nullptr;
  size_t got = 0;
  CHECK(GASengine::BlockPool::get().take(4096, &p, &got) == hipSuccess);
  GASengine::BlockPool::get().give(p, got);
  fake::frees = 0;
  fake::short_of = true;
  int *q = nullptr;
  CHECK(GASengine::device_alloc(&q, 100) == hipSuccess && q);
  CHECK(fake::frees == 1);
  fake::short_of = false;
  (void)fake::release(q);
  std::printf(bad ? "failed\n" : "ok\n");
  return bad != 0;
}
