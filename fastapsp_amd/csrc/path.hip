// path.hip -- predecessor rows from exact distance rows (is_path_needed).
//
// The reference carries a path matrix beside every distance matrix: the
// Dijkstra parent (fap/kernel/batch_sssp.h:82-83,110), the FW update
// path[i][j] = path[k][j] (fap/kernel/floyd.h:44), the min-plus update
// path = B_path[k][j] (fap/kernel/minplus.h:60), the part matrix's arcs and
// diagonal (fap/utils/util_Myalgorithm.h:50-51,71).  In every case
// path[i][j] is the vertex before j on a shortest path from row i's vertex
// to j, the row's own vertex for j itself, and -1 when j is unreachable.
//
// Here the distances are computed first (exact, unique) and the predecessor
// is read off them afterwards: u is a valid predecessor of j on row i iff an
// arc u -> j of weight w has d[i][u] + w == d[i][j].  One pass picks, per
// cell, the smallest such u with w > 0 (so d[i][u] < d[i][j]; following
// predecessors strictly decreases the distance and ends at the row's vertex).
// Cells whose only tight arcs have weight 0 (a plateau of equal distance) are
// marked and resolved in further passes: a marked cell takes the smallest
// tight zero-weight in-neighbour resolved in an earlier pass, so walks
// through a plateau end at a vertex resolved earlier, and the rows are a
// function of the distances alone (the same on every run).  Which valid predecessor is
// chosen when several exist is not fixed by the reference (its CPU, CUDA and
// HIP paths differ); validity is.
//
// In-arcs come from the transposed CSR, built once per graph on first use.
#include <algorithm>
#include <vector>

#include "common.h"

namespace fapk {

constexpr int32_t kUnresolved = -2;

// A workgroup takes kPredBlock vertices, two a thread, and walks rows with
// their in-arcs in registers.  Where all in-neighbours lie within kPredSpan
// vertices, that stretch of each row is staged in LDS by wide loads (the next
// two rows' in flight meanwhile) and the neighbours are read from there;
// otherwise they are gathered from memory.  What bounds it: a gather of 64
// lanes holds the vector cache 16 cycles and more, wherever its lanes point,
// and a cell has one per arc (1024 rows of a 256 x 256 grid, 537 MB read and
// written: 560 us with the arcs read again for every row too, 240 with gathers
// alone, 125 from LDS).  Workgroups of neighbouring vertices go to one XCD,
// whose L2 then holds the lines that they share.
constexpr int kPredThreads = 512, kPredBlock = 2 * kPredThreads;
constexpr int kPredArcs = 8;     // more: the arcs are read from memory for every row
constexpr int kPredSpan = 3072;  // words of a row in LDS (two rows, two buffers: 48 KB)

// A vertex's in-arcs of positive weight, padded by arcs that are never tight
// (from the vertex itself, weight -1).  The sources ascend.
template <int K>
struct PredArcs {
  int u[K], w[K];
  __device__ __forceinline__ PredArcs(int j, const int2 *arcs, int deg, int lo) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      u[k] = j - lo;
      w[k] = -1;
      if (k < deg) {
        const int2 a = arcs[k];  // {source vertex, weight}
        if (a.y > 0) {
          u[k] = a.x - lo;
          w[k] = a.y;
        }
      }
    }
  }
  // The predecessor, from the row's words at d (vertex lo at 0): the first
  // tight arc's source is the smallest.  With none, a plateau cell, resolved
  // by the passes below (which report rows that no arc makes tight).
  __device__ __forceinline__ int pick(const int (&du)[K], int dj, int j, int own, int lo) const {
    int p = kUnresolved;
#pragma unroll
    for (int k = K - 1; k >= 0; k--) p = du[k] + w[k] == dj ? u[k] + lo : p;
    if (dj >= 0x3FFFFFFF) p = -1;
    return own == j ? j : p;
  }
};

struct PredRows {
  const int32_t *dist, *own;
  int32_t *pred;
  int64_t ld, ldp;
  int i0, i1;  // rows
};

// One cell with its arcs read from memory; returns 1 for a plateau cell.
__device__ __forceinline__ unsigned int pred_scan(const PredRows &x, int i, int j,
                                                  const int2 *arcs, int deg) {
  const int32_t *d = x.dist + (int64_t)i * x.ld;
  const int dj = d[j];
  int p = kUnresolved;
  if (x.own[i] == j) {
    p = j;
  } else if (dj >= 0x3FFFFFFF) {
    p = -1;
  } else {
    // four arcs at a time: a load does not wait to see whether the arc before
    // was tight (300 rows of 65,536 vertices, 12 random in-arcs: 743 us, 1,226
    // one by one; 20 in-arcs nearby: 504, 1,445, and 1,321 with all of them read)
    for (int e = 0; e < deg && p == kUnresolved; e += 4) {
      int2 a[4];
      int du[4];
#pragma unroll
      for (int k = 0; k < 4; k++) a[k] = arcs[min(e + k, deg - 1)];
#pragma unroll
      for (int k = 0; k < 4; k++) du[k] = d[a[k].x];
#pragma unroll
      for (int k = 3; k >= 0; k--)  // the first tight one is the smallest
        if (a[k].y > 0 && du[k] + a[k].y == dj) p = a[k].x;
    }
  }
  x.pred[(int64_t)i * x.ldp + j] = p;
  return p == kUnresolved;
}

template <int K>
__device__ __forceinline__ unsigned int pred_gather(const PredRows &x, int j, bool valid,
                                                    const int2 *arcs, int deg) {
  constexpr int R = 4;  // rows in flight
  const PredArcs<K> in(j, arcs, deg, 0);
  unsigned int marked = 0;
  for (int i = x.i0; i < x.i1; i += R) {
    int dj[R], du[R][K];
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int32_t *d = x.dist + (int64_t)min(i + r, x.i1 - 1) * x.ld;
      dj[r] = d[j];
#pragma unroll
      for (int k = 0; k < K; k++) du[r][k] = d[in.u[k]];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (i + r >= x.i1) break;
      const int p = in.pick(du[r], dj[r], j, x.own[i + r], 0);
      marked += p == kUnresolved;
      if (valid) x.pred[(int64_t)(i + r) * x.ldp + j] = p;
    }
  }
  return valid ? marked : 0u;
}

// chunks: 4-word pieces of a row from vertex lo (all inside the row).
template <int K>
__device__ __forceinline__ unsigned int pred_staged(const PredRows &x, const int (&j)[2],
                                                    const bool (&valid)[2],
                                                    const int2 *const (&arcs)[2],
                                                    const int (&deg)[2], int lo, int chunks,
                                                    int32_t *lds) {
  typedef int vec __attribute__((ext_vector_type(4), aligned(4)));
  typedef int lvec __attribute__((ext_vector_type(4)));
  const PredArcs<K> a0(j[0], arcs[0], deg[0], lo), a1(j[1], arcs[1], deg[1], lo);
  const int t = threadIdx.x;
  constexpr int PER = kPredSpan / 4 / kPredThreads + (kPredSpan / 4 % kPredThreads != 0);
  vec v[2][PER];
  auto load = [&](int i) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const int32_t *d = x.dist + (int64_t)min(i + r, x.i1 - 1) * x.ld + lo;
#pragma unroll
      for (int c = 0; c < PER; c++)
        if (t + c * kPredThreads < chunks)
          v[r][c] = *reinterpret_cast<const vec *>(d + 4 * (t + c * kPredThreads));
    }
  };
  unsigned int marked = 0;
  if (x.i0 < x.i1) load(x.i0);
  for (int i = x.i0, b = 0; i < x.i1; i += 2, b ^= 1) {
    int32_t *row = lds + b * (2 * kPredSpan);
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
      for (int c = 0; c < PER; c++)
        if (t + c * kPredThreads < chunks)
          *reinterpret_cast<lvec *>(row + r * kPredSpan + 4 * (t + c * kPredThreads)) = v[r][c];
    __syncthreads();  // the buffer of two rows before has been read before the last one
    if (i + 2 < x.i1) load(i + 2);
#pragma unroll
    for (int r = 0; r < 2; r++) {
      if (i + r >= x.i1) break;
      const int32_t *d = row + r * kPredSpan;
      const int own = x.own[i + r];
      int d0[K], d1[K];
#pragma unroll
      for (int k = 0; k < K; k++) {
        d0[k] = d[a0.u[k]];
        d1[k] = d[a1.u[k]];
      }
      int32_t *out = x.pred + (int64_t)(i + r) * x.ldp;
      const int p0 = a0.pick(d0, d[j[0] - lo], j[0], own, lo);
      const int p1 = a1.pick(d1, d[j[1] - lo], j[1], own, lo);
      if (valid[0]) {
        marked += p0 == kUnresolved;
        out[j[0]] = p0;
      }
      if (valid[1]) {
        marked += p1 == kUnresolved;
        out[j[1]] = p1;
      }
    }
  }
  return marked;
}

__global__ __launch_bounds__(kPredThreads) void pred_kernel(
    const int32_t *__restrict__ dist, int64_t ld, const int32_t *__restrict__ own, int32_t nrows,
    int32_t V, const int32_t *__restrict__ in_off, const int2 *__restrict__ in_arcs,
    int32_t *__restrict__ pred, int64_t ldp, unsigned int *__restrict__ unresolved) {
  __shared__ __attribute__((aligned(16))) int32_t lds[4 * kPredSpan];
  __shared__ int s_lo, s_hi, s_most;
  const int t = threadIdx.x;
  // from 64 on, gridDim.x is 8 q: XCD x takes vertex blocks [x q, x q + q)
  const int q = gridDim.x >> 3;
  const int64_t blk = gridDim.x < 64 ? blockIdx.x
                                     : (int64_t)(blockIdx.x & 7) * q + (blockIdx.x >> 3);
  const int64_t j0 = blk * kPredBlock;
  if (j0 >= V) return;
  if (t == 0) {
    s_lo = V;
    s_hi = s_most = 0;
  }
  __syncthreads();
  int j[2], deg[2];
  bool valid[2];
  const int2 *arcs[2];
  int lo = V, hi = 0;
#pragma unroll
  for (int m = 0; m < 2; m++) {
    valid[m] = j0 + m * kPredThreads + t < V;
    j[m] = valid[m] ? (int)j0 + m * kPredThreads + t : V - 1;
    const int e = in_off[j[m]];
    deg[m] = in_off[j[m] + 1] - e;
    arcs[m] = in_arcs + e;
    lo = min(lo, j[m]);
    hi = max(hi, j[m]);
    if (deg[m] > 0) {  // the sources ascend
      lo = min(lo, arcs[m][0].x);
      hi = max(hi, arcs[m][deg[m] - 1].x);
    }
  }
  int most = max(deg[0], deg[1]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
    most = max(most, __shfl_xor(most, o));
  }
  if ((t & 63) == 0) {
    atomicMin(&s_lo, lo);
    atomicMax(&s_hi, hi);
    atomicMax(&s_most, most);
  }
  __syncthreads();
  const int per = (nrows + gridDim.y - 1) / gridDim.y;
  const PredRows x{dist, own, pred, ld, ldp, (int)blockIdx.y * per,
                   min((int)(blockIdx.y + 1) * per, nrows)};
  const int chunks = (s_hi - s_lo) / 4 + 1;
  const int base = min(s_lo, V - 4 * chunks);
  unsigned int marked = 0;
  if (s_most <= kPredArcs && 4 * chunks <= kPredSpan && base >= 0) {
    const int b = __builtin_amdgcn_readfirstlane(base);
    if (s_most <= 4) marked = pred_staged<4>(x, j, valid, arcs, deg, b, chunks, lds);
    else if (s_most <= 6) marked = pred_staged<6>(x, j, valid, arcs, deg, b, chunks, lds);
    else marked = pred_staged<kPredArcs>(x, j, valid, arcs, deg, b, chunks, lds);
  } else {
    const int wave_most = __builtin_amdgcn_readfirstlane(most);
#pragma unroll 1
    for (int m = 0; m < 2; m++) {
      const int v = m ? j[1] : j[0], dg = m ? deg[1] : deg[0];
      const bool ok = m ? valid[1] : valid[0];
      const int2 *ar = m ? arcs[1] : arcs[0];
      if (wave_most <= 4) {
        marked += pred_gather<4>(x, v, ok, ar, dg);
      } else if (wave_most <= kPredArcs) {
        marked += pred_gather<kPredArcs>(x, v, ok, ar, dg);
      } else if (ok) {
        for (int i = x.i0; i < x.i1; i++) marked += pred_scan(x, i, v, ar, dg);
      }
    }
  }
  if (marked) atomicAdd(unresolved, marked);
}

// Few cells (kPredFew): a thread each, the shortest chain (64 rows of 4,096
// vertices 27 us a call, 31 through pred_kernel; 2^20 cells the same, 2^21 37
// and 35).  And graphs without locality: all vertices of a few rows at a time,
// which the L2 then holds (1024 rows of 65,536 vertices at random, six arcs
// each, one after another: 1.89 ms; pred_kernel's gathers walk many rows at
// once, 1.7 times that; arcs in registers, up to 16 a vertex: 2.15).
constexpr int64_t kPredFew = 1 << 20;

__global__ __launch_bounds__(256) void pred_few_kernel(
    const int32_t *__restrict__ dist, int64_t ld, const int32_t *__restrict__ own, int32_t nrows,
    int32_t V, const int32_t *__restrict__ in_off, const int2 *__restrict__ in_arcs,
    int32_t *__restrict__ pred, int64_t ldp, unsigned int *__restrict__ unresolved) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= V) return;
  const int e = in_off[j];
  const PredRows x{dist, own, pred, ld, ldp, 0, nrows};
  unsigned int marked = 0;
  for (int i = blockIdx.y; i < nrows; i += gridDim.y)
    marked += pred_scan(x, i, (int)j, in_arcs + e, in_off[j + 1] - e);
  if (marked) atomicAdd(unresolved, marked);
}

// One resolution pass over plateau cells: take the smallest tight
// zero-weight in-neighbour resolved BEFORE this pass.  A cell resolved here
// is written as -(u + 3) (readers of the same pass skip it) and made
// positive by pred_settle_kernel after the pass, so the choice does not
// depend on the order in which workgroups run.  Counts the cells resolved.
__global__ void pred_plateau_kernel(const int32_t *__restrict__ dist, int64_t ld, int32_t nrows,
                                    int32_t V, const int32_t *__restrict__ in_off,
                                    const int2 *__restrict__ in_arcs, int32_t *pred, int64_t ldp,
                                    unsigned int *__restrict__ resolved) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= V) return;
  const int e0 = in_off[j], e1 = in_off[j + 1];
  unsigned int n = 0;
  for (int i = blockIdx.y; i < nrows; i += gridDim.y) {
    int32_t *pr = pred + (int64_t)i * ldp;
    if (pr[j] != kUnresolved) continue;
    const int32_t *d = dist + (int64_t)i * ld;
    const int dj = d[j];
    int p = 0x7FFFFFFF;
    for (int e = e0; e < e1; e++) {
      const int2 a = in_arcs[e];
      if (a.y == 0 && d[a.x] == dj &&
          __hip_atomic_load(pr + a.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= -1)
        p = min(p, a.x);
    }
    if (p != 0x7FFFFFFF) {
      __hip_atomic_store(pr + j, -(p + 3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      n++;
    }
  }
  if (n) atomicAdd(resolved, n);
}

// After a plateau pass: cells resolved in it (-(u + 3)) become u.
__global__ void pred_settle_kernel(int32_t *pred, int64_t ldp, int32_t nrows, int32_t V) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= V) return;
  for (int i = blockIdx.y; i < nrows; i += gridDim.y) {
    int32_t *c = pred + (int64_t)i * ldp + j;
    const int32_t v = *c;
    if (v <= -3) *c = -v - 3;
  }
}

}  // namespace fapk

namespace fapi {

// Transposed CSR of g (in-arcs of every vertex as {source, weight}, sources
// ascending, arcs of one source in CSR order), built on the host from the
// device copy.
static int ensure_in_csr(fap_ctx *ctx, fap_graph_dev *g, hipStream_t s) {
  if (g->in_offset) return FAP_OK;
  const int32_t V = g->V;
  const int64_t E = g->E;
  std::vector<int32_t> ro(V + 1);
  std::vector<int2> ed((size_t)E);
  FAP_HIP(hipMemcpyAsync(ro.data(), g->row_offset, sizeof(int32_t) * (V + 1),
                         hipMemcpyDeviceToHost, s));
  if (E) FAP_HIP(hipMemcpyAsync(ed.data(), g->edges, sizeof(int2) * E, hipMemcpyDeviceToHost, s));
  FAP_HIP(hipStreamSynchronize(s));
  std::vector<int32_t> off(V + 1, 0);
  for (int64_t e = 0; e < E; e++) off[ed[e].x + 1]++;
  for (int32_t v = 0; v < V; v++) off[v + 1] += off[v];
  std::vector<int32_t> fill(off.begin(), off.end() - 1);
  std::vector<int2> in((size_t)E);
  for (int32_t u = 0; u < V; u++)
    for (int32_t e = ro[u]; e < ro[u + 1]; e++) in[fill[ed[e].x]++] = make_int2(u, ed[e].y);
  int32_t *d_off = nullptr;
  int2 *d_in = nullptr;
  hipError_t e1 = hipMalloc(&d_off, sizeof(int32_t) * (V + 1));
  hipError_t e2 = hipMalloc(&d_in, sizeof(int2) * std::max<int64_t>(E, 1));
  if (e1 != hipSuccess || e2 != hipSuccess) {
    if (d_off) (void)hipFree(d_off);
    if (d_in) (void)hipFree(d_in);
    (void)hipGetLastError();
    return fail(FAP_E_NOMEM, "transposed CSR allocation failed");
  }
  hipError_t e = hipMemcpyAsync(d_off, off.data(), sizeof(int32_t) * (V + 1),
                                hipMemcpyHostToDevice, s);
  if (e == hipSuccess && E)
    e = hipMemcpyAsync(d_in, in.data(), sizeof(int2) * E, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    (void)hipFree(d_off);
    (void)hipFree(d_in);
    return hip_fail(e, "transposed CSR copy", __FILE__, __LINE__);
  }
  // is the graph laid out so that pred_kernel's blocks stage their rows?
  int64_t staged = 0, blocks = 0;
  for (int64_t j0 = 0; j0 < V; j0 += fapk::kPredBlock, blocks++) {
    const int64_t j1 = std::min<int64_t>(j0 + fapk::kPredBlock, V);
    int64_t lo = j0, hi = j1 - 1, most = 0;
    for (int64_t j = j0; j < j1; j++) {
      most = std::max<int64_t>(most, off[j + 1] - off[j]);
      if (off[j + 1] > off[j]) {
        lo = std::min<int64_t>(lo, in[off[j]].x);
        hi = std::max<int64_t>(hi, in[off[j + 1] - 1].x);
      }
    }
    staged += most <= fapk::kPredArcs && hi - lo < fapk::kPredSpan;
  }
  g->pred_local = 2 * staged >= blocks;
  g->in_offset = d_off;
  g->in_arcs = d_in;
  (void)ctx;
  return FAP_OK;
}

int run_pred_rows(fap_ctx *ctx, fap_graph_dev *g, const int32_t *d_dist, int64_t ld,
                  const int32_t *d_own, int32_t nrows, int32_t *d_pred, int64_t ldp,
                  hipStream_t s) {
  if (nrows <= 0 || g->V <= 0) return FAP_OK;
  FAP_TRY(ensure_in_csr(ctx, g, s));
  FAP_TRY(ensure_ws(ctx, ctx->ws_misc, 64));
  unsigned int *cnt = (unsigned int *)ctx->ws_misc.ptr;
  const int V = g->V;
  dim3 blk(256), grd((V + 255) / 256, std::min(nrows, 256));
  FAP_TRY(launch_fill_u32(cnt, 1, 0u, s));
  if ((int64_t)nrows * V < fapk::kPredFew || !g->pred_local) {
    hipLaunchKernelGGL(fapk::pred_few_kernel, grd, blk, 0, s, d_dist, ld, d_own, nrows, V,
                       g->in_offset, g->in_arcs, d_pred, ldp, cnt);
  } else {
    // about 4 workgroups per CU (3 fit at a time), rows in runs of 4 or more
    int xb = (V + fapk::kPredBlock - 1) / fapk::kPredBlock;
    if (xb >= 64) xb = (xb + 7) & ~7;
    const int64_t yb = std::min<int64_t>(std::max<int64_t>(1, (int64_t)ctx->num_cus * 4 / xb),
                                         std::min((nrows + 3) / 4, 65535));
    hipLaunchKernelGGL(fapk::pred_kernel, dim3(xb, (unsigned)yb), dim3(fapk::kPredThreads), 0, s,
                       d_dist, ld, d_own, nrows, V, g->in_offset, g->in_arcs, d_pred, ldp, cnt);
  }
  FAP_CHECK_LAUNCH();
  unsigned int h = 0;
  FAP_HIP(hipMemcpyAsync(&h, cnt, sizeof(h), hipMemcpyDeviceToHost, s));
  FAP_HIP(hipStreamSynchronize(s));
  int64_t left = h;
  // each pass resolves at least one plateau cell per row that has any
  // (some unresolved cell of a plateau always has a resolved tight
  // in-neighbour), so V passes bound the loop
  for (int pass = 0; left > 0; pass++) {
    if (pass >= V) return fail(FAP_E_STATE, "predecessor plateaus did not resolve");
    FAP_TRY(launch_fill_u32(cnt, 1, 0u, s));
    hipLaunchKernelGGL(fapk::pred_plateau_kernel, grd, blk, 0, s, d_dist, ld, nrows, V,
                       g->in_offset, g->in_arcs, d_pred, ldp, cnt);
    FAP_CHECK_LAUNCH();
    hipLaunchKernelGGL(fapk::pred_settle_kernel, grd, blk, 0, s, d_pred, ldp, nrows, V);
    FAP_CHECK_LAUNCH();
    FAP_HIP(hipMemcpyAsync(&h, cnt, sizeof(h), hipMemcpyDeviceToHost, s));
    FAP_HIP(hipStreamSynchronize(s));
    if (h == 0) return fail(FAP_E_STATE, "predecessor plateaus made no progress");
    left -= h;
  }
  return FAP_OK;
}

}  // namespace fapi

using namespace fapi;

extern "C" int fap_pred_rows(fap_ctx *ctx, fap_graph_dev *g, const int32_t *d_dist, int64_t ld,
                             const int32_t *d_row_vertex, int32_t nrows, int32_t *d_pred,
                             int64_t ld_pred, void *stream) {
  if (!ctx || !g) return fail(FAP_E_ARG, "null ctx/graph");
  if (nrows < 0) return fail(FAP_E_ARG, "pred: negative row count");
  if (nrows == 0) return FAP_OK;
  if (!d_dist || !d_row_vertex || !d_pred || ld < g->V || ld_pred < g->V)
    return fail(FAP_E_ARG, "pred: bad pointers or strides");
  return run_pred_rows(ctx, g, d_dist, ld, d_row_vertex, nrows, d_pred, ld_pred,
                       pick_stream(ctx, stream));
}

extern "C" int fap_subgraph_pred(fap_ctx *ctx, fap_graph_dev *g, int32_t start, int32_t n_sub,
                                 const int32_t *rowblock, int64_t ld_rb, int32_t *predblock,
                                 int64_t ld_pred, void *stream) {
  if (!ctx || !g) return fail(FAP_E_ARG, "null ctx/graph");
  if (!g->st2ed) return fail(FAP_E_STATE, "graph has no partition (fap_graph_set_partition)");
  if (start < 0 || n_sub < 0 || (int64_t)start + n_sub > g->V)
    return fail(FAP_E_ARG, "part range outside the vertex permutation");
  if (n_sub == 0) return FAP_OK;
  if (!rowblock || !predblock || ld_rb < g->V || ld_pred < g->V)
    return fail(FAP_E_ARG, "pred: bad pointers or strides");
  return run_pred_rows(ctx, g, rowblock, ld_rb, g->st2ed + start, n_sub, predblock, ld_pred,
                       pick_stream(ctx, stream));
}
