// dense.hip -- dense distance matrices of whole graphs (K = 1 jobs).
//
// For a standalone graph the reference pipeline with K = 1 has no boundary
// vertices: stage 1 is empty and stage 2 closes the matrix built by
// MysubMatBuild_path (fap/utils/util_Myalgorithm.h:30-73) from all arcs --
// INF, then every arc in CSR order (the last duplicate wins, :50), then a
// zero diagonal (:67-72).  These kernels build that matrix for one graph or
// for a batch of graphs in one launch.
#include <algorithm>
#include <vector>

#include "batch_desc.h"
#include "common.h"

namespace fapk {

// A wave builds a row, 1,024 columns at a time in its own LDS buffer: INF,
// the row's arcs one after another (the last duplicate wins), the diagonal,
// then out with 16-byte stores, each step behind wave_order.  Bound:
// writing the matrices once.  512 graphs (1.19 GB): 0.31 ms; 1.62 ms as a
// fill kernel that searched its job and divided once per cell, followed by a
// kernel with a thread per row of arcs.
constexpr int DR_COLS = 1024, DR_WAVES = 4;

// What lanes of a wave have written to LDS comes before what any of them
// writes or reads after this.  (No instruction: a wave's LDS accesses are in
// order; it keeps the compiler to theirs.)
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(64 * DR_WAVES) void dense_rows_kernel(const DenseJob *__restrict__ jobs,
                                                                   int count, int32_t rows) {
  typedef int vec4 __attribute__((ext_vector_type(4), aligned(4)));
  __shared__ __attribute__((aligned(16))) int32_t buf[DR_WAVES * DR_COLS];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  int32_t *w = buf + wave * DR_COLS;
  for (int x = blockIdx.x * DR_WAVES + wave; x < rows; x += gridDim.x * DR_WAVES) {
    int lo = 0, hi = count - 1;  // the job whose rows hold x
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (jobs[mid].row_base <= x) lo = mid;
      else hi = mid - 1;
    }
    const DenseJob &jb = jobs[lo];
    const int u = x - jb.row_base, n = jb.n;
    int32_t *row = jb.mat + (int64_t)u * jb.ld;
    const int e0 = jb.row_offset[u], e1 = jb.row_offset[u + 1];
    const int2 *__restrict__ edges = jb.edges;
    for (int c0 = 0; c0 < n; c0 += DR_COLS) {
#pragma unroll
      for (int i = 0; i < DR_COLS; i += 256)
        *reinterpret_cast<int4 *>(w + i + 4 * lane) =
            make_int4(0x3FFFFFFF, 0x3FFFFFFF, 0x3FFFFFFF, 0x3FFFFFFF);
      wave_order();
      for (int e = e0; e < e1; e += 64) {
        const int2 ed = e + lane < e1 ? edges[e + lane] : make_int2(-1, 0);
        const unsigned at = (unsigned)(ed.x - c0);
        const int m = e1 - e < 64 ? e1 - e : 64;
        for (int k = 0; k < m; k++) {  // one after another: duplicates
          if (lane == k && at < (unsigned)DR_COLS) w[at] = ed.y;
          wave_order();
        }
      }
      if (lane == 0 && (unsigned)(u - c0) < (unsigned)DR_COLS) w[u - c0] = 0;
      wave_order();
      const int m = n - c0 < DR_COLS ? n - c0 : DR_COLS;
#pragma unroll
      for (int i = 0; i < DR_COLS; i += 256) {
        const int j = i + 4 * lane;
        const vec4 v = *reinterpret_cast<const vec4 *>(w + j);
        if (j + 4 <= m) {
          *reinterpret_cast<vec4 *>(row + c0 + j) = v;
        } else {
#pragma unroll
          for (int q = 0; q < 3; q++)
            if (j + q < m) row[c0 + j + q] = v[q];
        }
      }
      wave_order();
    }
  }
}

}  // namespace fapk

namespace fapi {

int launch_dense_jobs(fap_ctx *ctx, const fapk::DenseJob *d_jobs, int32_t njobs, int64_t rows,
                      hipStream_t s) {
  if (njobs <= 0 || rows <= 0) return FAP_OK;
  if (rows > INT32_MAX) return fail(FAP_E_ARG, "dense build: too many rows");
  const int64_t blocks = std::min<int64_t>((rows + fapk::DR_WAVES - 1) / fapk::DR_WAVES,
                                           (int64_t)ctx->num_cus * 32);
  hipLaunchKernelGGL(fapk::dense_rows_kernel, dim3((unsigned)blocks), dim3(64 * fapk::DR_WAVES), 0,
                     s, d_jobs, njobs, (int32_t)rows);
  FAP_CHECK_LAUNCH();
  return FAP_OK;
}

int run_dense_from_graphs(fap_ctx *ctx, int32_t count, const fap_graph_dev *const *graphs,
                          int32_t *const *mats, const int64_t *ld, hipStream_t s) {
  std::vector<fapk::DenseJob> jobs;
  jobs.reserve(count);
  int64_t rows = 0;
  for (int32_t j = 0; j < count; j++) {
    const fap_graph_dev *g = graphs[j];
    if (g->V == 0) continue;
    jobs.push_back(fapk::DenseJob{g->row_offset, g->edges, mats[j], ld[j], (int32_t)rows, g->V});
    rows += g->V;
  }
  if (jobs.empty()) return FAP_OK;
  if (rows > INT32_MAX) return fail(FAP_E_ARG, "dense build: too many rows");
  const size_t bytes = sizeof(fapk::DenseJob) * jobs.size();
  FAP_TRY(ensure_ws(ctx, ctx->ws_dense, bytes));
  FAP_HIP(hipMemcpyAsync(ctx->ws_dense.ptr, jobs.data(), bytes, hipMemcpyHostToDevice, s));
  FAP_TRY(launch_dense_jobs(ctx, (const fapk::DenseJob *)ctx->ws_dense.ptr, (int32_t)jobs.size(),
                            rows, s));
  // the descriptor copy reads `jobs` asynchronously
  FAP_HIP(hipStreamSynchronize(s));
  return FAP_OK;
}

}  // namespace fapi

using namespace fapi;

extern "C" int fap_dense_from_graphs(fap_ctx *ctx, int32_t count,
                                     const fap_graph_dev *const *graphs, int32_t *const *d_mats,
                                     const int64_t *ld, void *stream) {
  if (!ctx) return fail(FAP_E_ARG, "ctx is null");
  if (count < 0 || (count > 0 && (!graphs || !d_mats || !ld)))
    return fail(FAP_E_ARG, "dense build: bad arguments");
  for (int32_t j = 0; j < count; j++) {
    if (!graphs[j]) return fail(FAP_E_ARG, "dense build: null graph");
    if (graphs[j]->V > 0 && (!d_mats[j] || ld[j] < graphs[j]->V))
      return fail(FAP_E_ARG, "dense build: bad matrix/stride for job " + std::to_string(j));
  }
  return run_dense_from_graphs(ctx, count, graphs, d_mats, ld, pick_stream(ctx, stream));
}
