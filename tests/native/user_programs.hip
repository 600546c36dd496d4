// Vertex programs as a user of the headers writes them, for tests/
// test_gpu_user_programs.py: a BFS whose contract takes the 8-argument form
// (with and without a look at the bitmap it is handed), and programs that
// derive from pagerank and set ranks or degrees themselves.
#include "gasengine/enactor_vertex_centric.h"
#include "programs/bfs.h"
#include "programs/pagerank.h"

#include <vector>

namespace {

// bfs.h:252 of the reference's fork: (rank_id, iteration, bitmap, vertex, ...).
struct bfs8 : bfs {
  struct contract {
    __device__ void operator()(int, const int iteration, unsigned char *, int &vertex_id, VertexType &vertex_list,
                               EdgeType &edge_list, GatherType *tmp, int &misc) {
      bfs::contract()(iteration, vertex_id, vertex_list, edge_list, tmp, misc);
    }
  };
};

// Drops a vertex that the next frontier's bitmap already has.
struct bfs8_bitmap : bfs {
  struct contract {
    __device__ void operator()(int, const int iteration, unsigned char *bitmap, int &vertex_id,
                               VertexType &vertex_list, EdgeType &edge_list, GatherType *tmp, int &misc) {
      if (bitmap[vertex_id >> 3] & (1 << (vertex_id & 7)))
        vertex_id = -1;
      else
        bfs::contract()(iteration, vertex_id, vertex_list, edge_list, tmp, misc);
    }
  };
};

// Half the damping, a tight stop; sets the rank without the base's apply.
struct own_apply : pagerank {
  struct apply {
    __device__ void operator()(const int vertex_id, const int, GatherType gathervalue, VertexType &vertex_list,
                               EdgeType &, char &changed) {
      const DataType old = vertex_list.d_dists[vertex_id];
      const DataType now = 0.15f + 0.425f * gathervalue;
      changed = fabsf(old - now) < 1e-6f ? 0 : 1;
      vertex_list.d_dists[vertex_id] = now;
    }
  };
};

__global__ void k_double(int *x, int n) {
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) x[v] *= 2;
}

// Every degree counted twice, which halves the damping as well.
struct own_degrees : pagerank {
  static void Initialize(const int directed, const int nodes, const int edges, int num_srcs, int *srcs,
                         int *d_row_offsets, int *d_column_indices, int *d_column_offsets, int *d_row_indices,
                         DataType *d_edge_values, VertexType &vertex_list, EdgeType &edge_list,
                         int *d_frontier_keys[3], MiscType *d_frontier_values[3]) {
    pagerank::Initialize(directed, nodes, edges, num_srcs, srcs, d_row_offsets, d_column_indices, d_column_offsets,
                         d_row_indices, d_edge_values, vertex_list, edge_list, d_frontier_keys, d_frontier_values);
    hipLaunchKernelGGL(k_double, dim3(GASengine::grid_for(nodes, 256)), dim3(256), 0, GASengine::engine_stream(),
                       vertex_list.d_num_out_edge, nodes);
  }
  struct apply {
    __device__ void operator()(const int vertex_id, const int, GatherType gathervalue, VertexType &vertex_list,
                               EdgeType &, char &changed) {
      const DataType old = vertex_list.d_dists[vertex_id];
      const DataType now = 0.15f + 0.85f * gathervalue;
      changed = fabsf(old - now) < 1e-6f ? 0 : 1;
      vertex_list.d_dists[vertex_id] = now;
    }
  };
};

// One run on a directed host CSR; 0 on success.
template <class P, bool PREDS>
int run(int n, int m, int *ro, int *col, int src, int threshold, typename P::DataType *out, int *preds) {
  using Problem = GASengine::CsrProblem<P, int, int, typename P::DataType, PREDS>;
  Problem prob;
  int rc = (int)prob.FromHostProblem(false, n, m, col, ro, nullptr, nullptr, nullptr, 1, 1);
  if (rc == 0) {
    GASengine::EnactorVertexCentric<Problem, P> enactor;
    rc = (int)enactor.EnactIterativeSearch(prob, nullptr, 1, 1, &src, 2147483647, threshold);
  }
  if (rc == 0) rc = (int)prob.ExtractResults(out);
  if (rc == 0 && PREDS) rc = (int)prob.ExtractPreds(preds);
  P::Release(prob.vertex_list, prob.edge_list);
  return rc;
}

}  // namespace

extern "C" {
int up_bfs8(int n, int m, int *ro, int *col, int src, int threshold, int look, int *out, int *preds) {
  if (preds)
    return look ? run<bfs8_bitmap, true>(n, m, ro, col, src, threshold, out, preds)
                : run<bfs8, true>(n, m, ro, col, src, threshold, out, preds);
  return look ? run<bfs8_bitmap, false>(n, m, ro, col, src, threshold, out, nullptr)
              : run<bfs8, false>(n, m, ro, col, src, threshold, out, nullptr);
}
int up_own_apply(int n, int m, int *ro, int *col, int threshold, float *out) {
  return run<own_apply, false>(n, m, ro, col, 0, threshold, out, nullptr);
}
int up_own_degrees(int n, int m, int *ro, int *col, int threshold, float *out) {
  return run<own_degrees, false>(n, m, ro, col, 0, threshold, out, nullptr);
}
}
