// Connected components by sampled hooking + pointer jumping (GG_CC_HOOK, and
// gg_cc on graphs of 2^17 vertices and more).
//
// Gives the same labels as the reference's label propagation (Algorithms/CC/
// cc.h, checked against CPUCC cc.cu:127-169): the minimum vertex id of each
// component.  parent[] is a union-find forest with parent[x] <= x; a hook
// links the larger of two roots under the smaller one with an atomicCAS, so
// the root of each final tree is the component's minimum id.
//
// Most edges join vertices that a few edges per vertex have already joined,
// so not every edge is hooked (the sampling of Sutton, Ben-Nun and Barak,
// "Optimizing Parallel Graph Connectivity Computation via Subgraph Sampling",
// 2018):
//   1 init     parent[v] = v's first neighbour where that is smaller: a forest
//              without any atomic
//   2 link     every vertex hooks with its second neighbour, then flatten
//   3 giant    the most frequent root among kSamples vertices
//   4 rest     only the vertices outside that tree hook along their rows; an
//              edge between it and them is seen from their side, which holds
//              it as well where the handle's check found the mirror of every
//              entry (rows that are not sorted are not checked: there every
//              vertex hooks); rows of kLongRow edges and more in chunks that
//              the whole grid shares
//   5 labels   parent[v] = root
// The link pass is bound by its chains of dependent loads and by atomics on
// the roots that most trees join (a wave sends one hook per pair of roots, and
// a root is read again before its CAS: 2.4 -> 0.09 ms on an R-MAT), the others
// by latency and launches: each moves 8-16 n bytes, against 8 m for hooking
// every edge.  Per call, against label propagation / hooking every edge:
// 2048 x 2048 lattice (4.2M vertices, 10M edges) 12.4 / 0.66 -> 0.42 ms; R-MAT
// of 1.5M vertices and 35M edges 0.92 -> 0.16-0.20 ms; of 4.2M vertices and 128M
// edges 3.86 / 3.89 -> 0.27 ms, renumbered by degree 2.02 / 6.36 -> 0.32 ms;
// path, band, star and pair graphs of 2M vertices 0.08-0.30 ms.
//
// Loads of parent[] are plain (cached) loads: a value another workgroup has
// replaced since is still an ancestor from an earlier moment, in the same
// tree and smaller than the child, so a walk along stale values ends at a
// vertex of the same tree; a hook decides by the CAS, whose returned value is
// current, and path halving only ever replaces the parent of a vertex that
// is not a root by a smaller vertex of the same tree.  (System-scope loads,
// which bypass the L2, made each walk step a trip past it.)  Halving stores are
// agent-scope: with plain ones, where workgroups of several XCDs halve the same
// path and store different values to one word in a kernel, runs ended with
// labels that were not roots, and with agent-scope ones none did; why was not
// established.  Words with one writer per kernel, or writers that all store the
// same value, take plain stores.
// Symmetric (undirected) graphs only.
//
// Byte model: 44 n (init 12: offsets, first neighbour, parent; two flattens of
// 8: parent and its parent; link 16: offsets, second neighbour, two parents),
// the rest 12 n (flatten, parent) and 8 per edge (neighbour, its parent), the
// labels 8 n.
#include <hip/hip_runtime.h>

#include <cstring>

#include "internal.h"

namespace gg {
namespace {

using namespace GASengine;

constexpr int kSamples = 256;
constexpr int kLinkRounds = 4;  // pairs of trees a wave combines its hooks for
constexpr int kWalk = 4;        // find_root: pairs of steps before it halves the path
constexpr int kJumps = 64;      // k_cc_flatten: jumps per vertex and launch
constexpr int kLaneRow = 8;     // rest: rows up to here are one lane's work, longer ones a wave's
constexpr int kLongRow = 1024;  // rest: a longer row is cut into chunks of this many edges

struct CcCtl {
  int32_t giant;   // root most samples have
  int32_t chunks;  // entries of the chunk list
  int32_t pad[2];
};

__device__ __forceinline__ int32_t load_parent(const int32_t *parent, int32_t x) {
  return __hip_atomic_load(&parent[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Root of x as far as this thread sees.  A path longer than 2 kWalk is halved
// from there on: trees are flattened before a hooking pass and rarely grow
// that deep in it, and every halving store goes past the L2.
__device__ __forceinline__ int32_t find_root(int32_t *parent, int32_t x) {
  for (int hops = 0;; hops++) {
    const int32_t p = load_parent(parent, x);
    if (p == x) return x;
    const int32_t gp = load_parent(parent, p);
    if (gp == p) return p;
    if (hops >= kWalk) __hip_atomic_store(&parent[x], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    x = gp;
  }
}

// Hook the trees of the roots ru and rv (as this thread sees them).  A root is
// read again past this CU's cache before the CAS, since same-address atomics
// queue up: where most trees join the same few roots, most threads find it
// hooked already.  Every retry starts from the value read, which is smaller
// than the vertex it was read from, so the loop ends.
__device__ __forceinline__ void hook_roots(int32_t *parent, int32_t ru, int32_t rv) {
  while (ru != rv) {
    if (ru > rv) {
      const int32_t t = ru;
      ru = rv;
      rv = t;
    }
    int32_t old = __hip_atomic_load(&parent[rv], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (old == rv) old = atomicCAS(&parent[rv], rv, ru);
    if (old == rv) break;
    rv = find_root(parent, old);
    ru = find_root(parent, ru);
  }
}
__device__ __forceinline__ void hook(int32_t *parent, int32_t u, int32_t v) {
  hook_roots(parent, find_root(parent, u), find_root(parent, v));
}

__global__ void __launch_bounds__(256)
k_cc_init(int32_t *__restrict__ parent, const int32_t *__restrict__ ro, const int32_t *__restrict__ col, int32_t n) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const int32_t b = ro[v], e = ro[v + 1];
    int32_t p = (int32_t)v;
    if (b < e) p = min(p, col[b]);
    parent[v] = p;
  }
}

__global__ void __launch_bounds__(256)
k_cc_link(int32_t *parent, const int32_t *__restrict__ ro, const int32_t *__restrict__ col, int32_t n) {
  const int lane = lane_id();
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t v0 = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~(kWave - 1)); v0 < n; v0 += stride) {
    const int64_t v = v0 + lane;
    int32_t ru = 0, rv = 0;
    if (v < n) {
      const int32_t b = ro[v] + 1;
      if (b < ro[v + 1]) {
        ru = find_root(parent, (int32_t)v);
        rv = find_root(parent, col[b]);
      }
    }
    // One lane of those that join the same two trees (kLinkRounds pairs): on
    // skewed graphs most of a wave's lanes want the same hook.
    const int32_t hi = max(ru, rv), lo = min(ru, rv);
    uint64_t todo = ballot(hi != lo);
    bool drop = hi == lo;
    for (int r = 0; r < kLinkRounds && todo; r++) {
      const int l = __builtin_ctzll(todo);
      const bool peer = hi == __builtin_amdgcn_readlane(hi, l) && lo == __builtin_amdgcn_readlane(lo, l);
      if (peer && lane != l) drop = true;
      todo &= ~ballot(peer);
    }
    if (!drop) hook_roots(parent, lo, hi);
  }
}

// Pointer jumping: v's thread, the only writer of parent[v] here, moves it up
// until it is a root, at most kJumps times: paths get at least kJumps times
// shorter however stale the values it reads are (a second launch then leaves
// an n / kJumps^2 part of the longest possible path to find_root).
__global__ void __launch_bounds__(256) k_cc_flatten(int32_t *parent, int32_t n) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    int32_t p = load_parent(parent, (int32_t)v);
    for (int j = 0; j < kJumps; j++) {
      const int32_t gp = load_parent(parent, p);
      if (gp == p) break;
      __hip_atomic_store(&parent[v], gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      p = gp;
    }
  }
}

// Root without path halving: follows parents only.
__device__ __forceinline__ int32_t walk_to_root(const int32_t *parent, int32_t x) {
  for (;;) {
    const int32_t p = load_parent(parent, x);
    if (p == x) return x;
    x = p;
  }
}

// The most frequent root of kSamples vertices spread over the ids (one
// workgroup; every thread counts its own sample's root in LDS).
// mirrored = false: no tree is left out, whatever its size.
__global__ void __launch_bounds__(kSamples)
k_cc_giant(const int32_t *parent, int32_t n, bool mirrored, CcCtl *ctl) {
  __shared__ __align__(16) int32_t s_root[kSamples];
  __shared__ unsigned long long s_best;
  const int t = threadIdx.x;
  if (t == 0) s_best = 0ull;
  const int32_t v = (int32_t)(((uint64_t)((uint32_t)t * 2654435761u) * (uint64_t)n) >> 32);
  const int32_t r = walk_to_root(parent, v);
  s_root[t] = r;
  __syncthreads();
  int32_t same = 0;
#pragma unroll 8
  for (int k = 0; k < kSamples / 4; k++) {
    const int4 q = reinterpret_cast<const int4 *>(s_root)[k];
    same += (q.x == r) + (q.y == r) + (q.z == r) + (q.w == r);
  }
  atomicMax(&s_best, ((unsigned long long)same << 32) | (uint32_t)r);
  __syncthreads();
  if (t == 0) {
    ctl->giant = mirrored ? (int32_t)(uint32_t)s_best : -1;
    ctl->chunks = 0;
  }
}

// Every edge of a vertex outside the giant tree (no such tree: -1) is hooked
// from its side: a vertex that joined the giant tree before its turn leaves its row out, and
// the far end of such an edge has either joined as well or hooks it itself.
// linked: k_cc_init and k_cc_link have run, so a vertex has been joined with
// its second neighbour, and with its first one where that is smaller.
__global__ void __launch_bounds__(256)
k_cc_rest(int32_t *parent, const int32_t *__restrict__ ro, const int32_t *__restrict__ col, int32_t n, CcCtl *ctl,
          int2 *__restrict__ chunks, unsigned long long *edge_counter, bool linked) {
  const int32_t giant = ctl->giant;
  const int lane = lane_id();
  unsigned long long edges = 0;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t v0 = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~(kWave - 1)); v0 < n; v0 += stride) {
    const int64_t v = v0 + lane;
    const bool out = v < n && load_parent(parent, (int32_t)v) != giant;
    if (!ballot(out)) continue;
    int32_t b = 0, e = 0;
    if (out) {
      b = ro[v];
      e = ro[v + 1];
      edges += (unsigned long long)(e - b);
    }
    const int32_t deg = e - b;
    if (deg > 0 && deg <= kLaneRow) {
      const int32_t u0 = col[b];
      if (!linked || u0 > (int32_t)v) hook(parent, (int32_t)v, u0);
      for (int32_t k = b + (linked ? 2 : 1); k < e; k++) hook(parent, (int32_t)v, col[k]);
    }
    uint64_t mask = ballot(deg > kLaneRow);
    while (mask) {
      const int l = __builtin_ctzll(mask);
      mask &= mask - 1;
      const int32_t wb = __shfl(b, l), we = __shfl(e, l), wv = (int32_t)v0 + l;
      if (we - wb < kLongRow) {
        for (int32_t k = wb + lane; k < we; k += kWave) hook(parent, wv, col[k]);
      } else {  // left to k_cc_rest_chunks
        const int32_t count = (we - wb + kLongRow - 1) / kLongRow;
        int32_t at = 0;
        if (lane == 0) at = atomicAdd(&ctl->chunks, count);
        at = __shfl(at, 0);
        for (int32_t c = lane; c < count; c += kWave) chunks[at + c] = make_int2(wv, wb + c * kLongRow);
      }
    }
  }
  block_counter_add<256>(edge_counter, edges);
}

// The long rows outside the giant tree, a wave per chunk.
__global__ void __launch_bounds__(256)
k_cc_rest_chunks(int32_t *parent, const int32_t *__restrict__ ro, const int32_t *__restrict__ col, const CcCtl *ctl,
                 const int2 *__restrict__ chunks) {
  const int32_t count = ctl->chunks;
  const int64_t waves = (int64_t)gridDim.x * (256 / kWave);
  for (int64_t c = (int64_t)blockIdx.x * (256 / kWave) + threadIdx.x / kWave; c < count; c += waves) {
    const int2 ch = chunks[c];
    const int32_t end = min(ch.y + kLongRow, ro[ch.x + 1]);
    for (int32_t k = ch.y + lane_id(); k < end; k += kWave) hook(parent, ch.x, col[k]);
  }
}

// Final labels: parent[v] = root of v.  Each parent[v] is written by v's
// thread only, with the root, and read by other threads' walks, which accept
// an old ancestor or the root alike.  (With path halving here, a walk that
// read parent[v] before v's thread stored the root could store an older
// ancestor after it, leaving a non-root label.)
__global__ void __launch_bounds__(256) k_cc_labels(int32_t *parent, int32_t n) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const int32_t p = load_parent(parent, (int32_t)v), r = walk_to_root(parent, p);
    if (r != p) __hip_atomic_store(&parent[v], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
}

}  // namespace

// Hooks what parent[] (a forest within the components, parent[x] <= x) leaves
// apart and writes the labels; the edges of the rest pass go to counter 32.
int cc_hook_finish(gg_graph *g, int32_t *parent, bool linked) {
  const int32_t n = g->n;
  hipStream_t s = g->stream;
  const int32_t *ro = g->dg.row_offsets, *col = g->dg.column_indices;
  // A row of d >= kLongRow edges makes at most d / kLongRow + 1 <= 2 d / kLongRow chunks.
  GG_TRY(g->batch[6].ensure(sizeof(CcCtl) + sizeof(int2) * (size_t)(2 * g->m / kLongRow + 1)));
  CcCtl *ctl = g->batch[6].as<CcCtl>();
  int2 *chunks = reinterpret_cast<int2 *>(ctl + 1);
  GG_TRY(g->counters.ensure(kCounterWords * sizeof(unsigned long long)));
  auto *ctr = g->counters.as<unsigned long long>();
  const dim3 block(256), grid(grid_for(n, 256, 8192));
  {
    TimedRegion t(g->prof, "cc.rest");
    GG_HIP(slot_resets_async(ctr, {{32, 0ull}}, s));
    hipLaunchKernelGGL(k_cc_flatten, grid, block, 0, s, parent, n);
    hipLaunchKernelGGL(k_cc_giant, dim3(1), dim3(kSamples), 0, s, parent, n, g->mirror_ok, ctl);
    hipLaunchKernelGGL(k_cc_rest, grid, block, 0, s, parent, ro, col, n, ctl, chunks, ctr + 32, linked);
    hipLaunchKernelGGL(k_cc_rest_chunks, dim3(512), block, 0, s, parent, ro, col, ctl, chunks);
    GG_HIP(hipGetLastError());
  }
  {
    TimedRegion t(g->prof, "cc.labels");
    hipLaunchKernelGGL(k_cc_labels, grid, block, 0, s, parent, n);
    GG_HIP(hipGetLastError());
  }
  g->prof.add_bytes("cc.rest", 12.0 * n);  // the caller adds its edges, read back after
  g->prof.add_bytes("cc.labels", 8.0 * n);
  return GG_OK;
}

int cc_hooking(gg_graph *g, int32_t *label_out, uint32_t flags, gg_stats *stats) {
  GG_TRY(activate(g));
  if (g->directed) return set_error(GG_ERR_UNSUPPORTED, "CC needs a symmetric (undirected) graph");
  const int32_t n = g->n;
  hipStream_t s = g->stream;
  int32_t *parent;
  if (flags & GG_OUT_DEVICE) {
    GG_CHECK_ARG(label_out, "label is NULL");
    parent = label_out;
  } else {
    GG_TRY(g->vtx[1].ensure(4 * (size_t)n));
    parent = g->vtx[1].as<int32_t>();
  }
  g->prof.enabled = (flags & GG_INSTRUMENT) != 0;
  hipEvent_t e0, e1;
  GG_HIP(g->cc_ev.get(&e0, &e1));
  GG_HIP(hipEventRecord(e0, s));
  {
    TimedRegion t(g->prof, "cc.link");
    const dim3 block(256), grid(grid_for(n, 256, 8192));
    hipLaunchKernelGGL(k_cc_init, grid, block, 0, s, parent, g->dg.row_offsets, g->dg.column_indices, n);
    hipLaunchKernelGGL(k_cc_flatten, grid, block, 0, s, parent, n);
    hipLaunchKernelGGL(k_cc_flatten, grid, block, 0, s, parent, n);
    hipLaunchKernelGGL(k_cc_link, grid, block, 0, s, parent, g->dg.row_offsets, g->dg.column_indices, n);
    GG_HIP(hipGetLastError());
  }
  GG_TRY(cc_hook_finish(g, parent, true));
  GG_HIP(hipEventRecord(e1, s));
  GG_TRY(read_counters(g, 33));
  const int64_t rest = g->h64()[32];
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  g->prof.add_bytes("cc.link", 44.0 * n);
  g->prof.add_bytes("cc.rest", 8.0 * (double)rest);
  finish_profile(g);
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    stats->iterations = 3;
    stats->edges_inspected = std::min<int64_t>(2 * (int64_t)n, g->m) + rest;
    stats->alg_bytes = 44.0 * n + cc_finish_bytes(n, rest);
    stats->gpu_ms = ms;
    stats->reached_vertices = n;  // every vertex has a component
    stats->reached_edges = g->m;
  }
  if (flags & GG_OUT_DEVICE) return GG_OK;
  return copy_out(g, label_out, parent, 4 * (size_t)n, flags);
}

}  // namespace gg
