// hindex.hip -- coarse level of the boundary index: regions of parts.
//
// The boundary index (bindex.hip) finds the distances from a part's boundary
// vertices to all others (stage 1, fap/kernel/batch_sssp.h:254-277) by block
// iterations over the parts.  On a graph of many parts a block settles late:
// the 512 x 512 grid's 256 parts took 243 iterations and 25 updates per block,
// each a pass over X's rows in memory (29 ms for 32 parts).  Here the same
// theorem is used once more, one level up, and without iterations.  The
// boundary graph H (all boundary vertices; arcs: the cut arcs, and inside each
// part the closed local distances) is itself cut into regions of whole parts.
// Made once: per region D, the closure of H inside it; and C2, the closure of
// the graph of region-boundary vertices (those with a cut arc to another
// region; arcs: these cut arcs, and inside each region D).  For sources s of
// region S:
//  1. X2[s][c], c region-boundary: min over region-boundary c' of S of
//     D_S[s][c'] + C2[c'][c], one product;
//  2. X[s][h], h any boundary vertex, of region R: min over region-boundary c
//     of R of X2[s][c] + D_R[c][h], one product, and D_S[s][h] inside S;
//  3. the rows, from X, by the index's own expansion.
// A path from s leaves S for the first time at some c' (or never), enters h's
// region for the last time at some c, and between them is a path of the
// region-boundary graph, so the distances are exact, and integers: the same
// rows as without.
#include <math.h>

#include <algorithm>
#include <new>
#include <vector>

#include "common.h"
#include "host.h"
#include "mfma_tile.h"

// Region-local entries: entry e of region r's columns is the H id colid[e];
// ent[e] = {its part, its H position}.
struct HidxRegion {
  int64_t off;  // of D_r (row stride ldd)
  int32_t start, n, ldd;
  int32_t hoff, b;  // its region-boundary ids: hoff .. hoff + b - 1, local positions 0 .. b - 1
  int32_t pad;
};

struct fap_hidx {
  fap_bidx *c = nullptr;              // expansions inside regions (owns D)
  int32_t nbp2 = 0;                   // region-boundary ids, padding included
  int32_t max_b = 0;                  // most region-boundary vertices of a region (padded)
  std::vector<int32_t> region, lpos;  // of every H id
  HidxRegion *regs = nullptr;         // device
  const int32_t *D = nullptr;         // device (owned by c)
  int32_t *C2 = nullptr;              // device: nbp2 x nbp2
  size_t bytes = 0;
};

// Rows of one step-1 tile: X2 rows row0 .. row0 + rows - 1, all of region reg.
struct HidxTile {
  int32_t row0, rows, reg, pad;
};

namespace fapk {

// D_r before its closure: inside a part the closed local distances, else INF
// (the cut arcs follow).  One row per workgroup row.
__global__ void hidx_fill_kernel(HidxRegion R, const int2 *__restrict__ ent,
                                 const int64_t *__restrict__ lbb_off,
                                 const int32_t *__restrict__ ldb, const int32_t *__restrict__ lbb,
                                 int32_t *__restrict__ D) {
  const int i = blockIdx.y;
  const int2 a = ent[R.start + i];
  const int32_t *row = lbb + lbb_off[a.x] + (int64_t)a.y * ldb[a.x];
  int32_t *out = D + R.off + (int64_t)i * R.ldd;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < R.ldd; j += gridDim.x * blockDim.x) {
    int v = kInf;
    if (j < R.n) {
      const int2 b = ent[R.start + j];
      if (b.x == a.x) v = row[b.y];
      if (i == j) v = 0;
    }
    out[j] = v;
  }
}

// C2 before its closure: inside a region D, else INF (the cut arcs between
// regions follow); padding ids are isolated.  One workgroup row per id.
__global__ void hidx_top_kernel(const HidxRegion *__restrict__ regs, int32_t nreg, int32_t nbp2,
                                const int32_t *__restrict__ D, int32_t *__restrict__ C2) {
  const int i = blockIdx.y;
  int lo = 0, hi = nreg - 1;  // the region of id i (or of the ids before its padding)
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (regs[mid].hoff <= i) lo = mid;
    else hi = mid - 1;
  }
  const HidxRegion R = regs[lo];
  const int32_t *own = D + R.off + (int64_t)(i - R.hoff) * R.ldd;
  const bool real = i - R.hoff < R.b;
  int32_t *out = C2 + (int64_t)i * nbp2;
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < nbp2; j += gridDim.x * blockDim.x) {
    int v = kInf;
    if (real && j >= R.hoff && j < R.hoff + R.b) v = own[j - R.hoff];
    if (i == j) v = 0;
    out[j] = v;
  }
}

// Cut arcs: {word of the matrix, weight} (no two alike: duplicate arcs
// leave a graph without an index).
__global__ void hidx_arcs_kernel(const int64_t *__restrict__ at, const int32_t *__restrict__ w,
                                 int64_t count, int32_t *__restrict__ D) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) D[at[i]] = w[i];
}

// X[s][h] = min(X[s][h], D_S[s][h]) for every h of the source's own region.
__global__ void hidx_own_kernel(int32_t *__restrict__ X, int64_t ldx, const int2 *__restrict__ rowq,
                                const HidxRegion *__restrict__ regs,
                                const int32_t *__restrict__ colid,
                                const int32_t *__restrict__ D) {
  const int2 qi = rowq[blockIdx.x];
  const HidxRegion R = regs[qi.x];
  const int32_t *own = D + R.off + (int64_t)qi.y * R.ldd;
  int32_t *x = X + (int64_t)blockIdx.x * ldx;
  for (int j = blockIdx.y * blockDim.x + threadIdx.x; j < R.n; j += gridDim.y * blockDim.x) {
    const int h = colid[R.start + j];
    const int v = own[j];
    if (v < x[h]) x[h] = v;
  }
}

// What step 1 and 2 read of the sources: S2[s][k] = D_S[s][k] for the
// region-boundary k of the source's region, and the rows of X.
__global__ void hidx_sources_kernel(const int2 *__restrict__ rowq,
                                    const HidxRegion *__restrict__ regs,
                                    const int32_t *__restrict__ D, int32_t *__restrict__ S2,
                                    int32_t lds2, int32_t *X, int64_t ldx, int32_t **rowptr) {
  const int2 qi = rowq[blockIdx.x];
  const HidxRegion R = regs[qi.x];
  const int32_t *own = D + R.off + (int64_t)qi.y * R.ldd;
  int32_t *out = S2 + (int64_t)blockIdx.x * lds2;
  for (int k = threadIdx.x; k < R.b; k += blockDim.x) out[k] = own[k];
  if (threadIdx.x == 0) rowptr[blockIdx.x] = X + (int64_t)blockIdx.x * ldx;
}

// Step 1: 128 x 128 tiles of X2 = S2 (x) C2[region-boundary of S, .], K = b of
// the rows' region (0 where the region has no boundary: INF).
__global__ __launch_bounds__(MP_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4))) void hidx_cross_kernel(
    const HidxTile *__restrict__ tiles, const HidxRegion *__restrict__ regs,
    const int32_t *__restrict__ S2, int32_t lds2, const int32_t *__restrict__ C2, int32_t nbp2,
    int32_t *__restrict__ X2) {
  __shared__ __attribute__((aligned(16))) int32_t lds[MxBig::LDS_WORDS];
  const HidxTile T = tiles[blockIdx.y];
  const HidxRegion R = regs[T.reg];
  const int c0 = blockIdx.x * 128;
  MxBig::run(S2 + (int64_t)T.row0 * lds2, lds2, C2 + (int64_t)R.hoff * nbp2 + c0, nbp2,
             X2 + (int64_t)T.row0 * nbp2 + c0, nbp2, T.rows, imin(128, nbp2 - c0), R.b, false,
             MP_VEC_A | MP_VEC_B | MP_VEC_C, lds);
}

}  // namespace fapk

namespace fapi {

namespace {

// Memory for D and the smallest graph that gets a coarse level.
constexpr int64_t kMaxWords = (int64_t)1 << 28;  // 1 GiB of int32
constexpr int32_t kMaxTop = 12288;               // C2: 604 MB, closed in ~50 ms
constexpr int32_t kMinParts = 32;
constexpr size_t kFreeShare = 16;  // of the free memory

struct Regions {
  std::vector<BidxPartDesc> parts;  // of the coarse index
  std::vector<HidxRegion> regs;
  std::vector<int32_t> colid, region, lpos, part_region;
  std::vector<int2> ent;
  std::vector<int64_t> arc_at, top_at;  // cut arcs: words of D, of C2
  std::vector<int32_t> arc_w, top_w;
  int64_t words = 0;
  int32_t nbp2 = 0, nb2 = 0;
};

// Region-boundary vertices of a grouping of the parts.
int32_t boundary_of(const BidxDesc &d, const std::vector<int32_t> &part_region) {
  std::vector<uint8_t> on(d.nbp, 0);
  for (const BidxCut &c : *d.cuts)
    if (part_region[c.pu] != part_region[c.pv]) on[c.u] = on[c.v] = 1;
  return (int32_t)std::count(on.begin(), on.end(), (uint8_t)1);
}

// R regions of whole parts: runs of part ids (neighbours where the partitioner
// numbers its parts recursively, as the built-in one does) or the built-in
// bisection of the graph of parts, whichever leaves the smaller region
// boundary (512 x 512 grid, 16 regions: 6,250 and 9,445 vertices).
void group_parts(const BidxDesc &d, int32_t R, std::vector<int32_t> *part_region) {
  HostCSR pg;
  pg.V = d.K;
  std::vector<std::pair<int32_t, int32_t>> edges;
  for (const BidxCut &c : *d.cuts) {
    edges.push_back({c.pu, c.pv});
    edges.push_back({c.pv, c.pu});
  }
  std::sort(edges.begin(), edges.end());
  edges.erase(std::unique(edges.begin(), edges.end()), edges.end());
  pg.row_offset.assign(d.K + 1, 0);
  for (auto &e : edges) {
    pg.row_offset[e.first + 1]++;
    pg.col.push_back(e.second);
    pg.w.push_back(1);
  }
  for (int32_t q = 0; q < d.K; q++) pg.row_offset[q + 1] += pg.row_offset[q];
  pg.E = (int64_t)pg.col.size();
  bisection_partition(pg, R, part_region);
  for (int32_t &r : *part_region) r--;
  std::vector<int32_t> runs(d.K);
  for (int32_t q = 0; q < d.K; q++) runs[q] = (int32_t)((int64_t)q * R / d.K);
  if (boundary_of(d, runs) <= boundary_of(d, *part_region)) part_region->swap(runs);
}

// The regions' local matrices laid out; region-boundary vertices come first in
// a region, grouped by the region of their first cut arc.
void make_regions(const BidxDesc &d, int32_t R, Regions *o) {
  group_parts(d, R, &o->part_region);
  o->region.assign(d.nbp, -1);
  o->lpos.assign(d.nbp, -1);
  std::vector<int2> entry(d.nbp, make_int2(-1, -1));  // {part, H position} of an H id
  std::vector<std::vector<int32_t>> ids(R);
  for (int32_t q = 0; q < d.K; q++)
    for (int32_t i = 0; i < d.parts[q].b; i++) {
      const int32_t h = d.parts[q].hoff + i;
      o->region[h] = o->part_region[q];
      entry[h] = make_int2(q, i);
      ids[o->part_region[q]].push_back(h);
    }
  std::vector<int32_t> first(d.nbp, INT32_MAX);  // region of the first cut arc out of the region
  for (const BidxCut &c : *d.cuts) {
    const int32_t a = o->region[c.u], b = o->region[c.v];
    if (a == b) continue;
    first[c.u] = std::min(first[c.u], b);
    first[c.v] = std::min(first[c.v], a);
  }
  int32_t start = 0;
  for (int32_t r = 0; r < R; r++) {
    std::stable_sort(ids[r].begin(), ids[r].end(),
                     [&](int32_t a, int32_t b) { return first[a] < first[b]; });
    int32_t b2 = 0;
    for (size_t i = 0; i < ids[r].size(); i++) {
      o->lpos[ids[r][i]] = (int32_t)i;
      b2 += first[ids[r][i]] != INT32_MAX;
      o->colid.push_back(ids[r][i]);
      o->ent.push_back(entry[ids[r][i]]);
    }
    const int32_t n = (int32_t)ids[r].size(), ldd = (n + 3) & ~3;
    o->parts.push_back(BidxPartDesc{start, n, b2, o->nbp2, o->words, ldd});
    o->regs.push_back(HidxRegion{o->words, start, n, ldd, o->nbp2, b2, 0});
    o->nbp2 += (b2 + 3) & ~3;
    o->nb2 += b2;
    o->words += (int64_t)ldd * n;
    start += n;
  }
  for (const BidxCut &c : *d.cuts) {
    const int32_t a = o->region[c.u], b = o->region[c.v];
    if (a == b) {
      o->arc_at.push_back(o->regs[a].off + (int64_t)o->lpos[c.u] * o->regs[a].ldd + o->lpos[c.v]);
      o->arc_w.push_back(c.w);
    } else {
      o->top_at.push_back((int64_t)(o->regs[a].hoff + o->lpos[c.u]) * o->nbp2 + o->regs[b].hoff +
                          o->lpos[c.v]);
      o->top_w.push_back(c.w);
    }
  }
}

template <typename T>
hipError_t to_device(const std::vector<T> &h, T **d, hipStream_t s) {
  hipError_t e = hipMalloc((void **)d, std::max<size_t>(h.size(), 1) * sizeof(T));
  if (e == hipSuccess && !h.empty())
    e = hipMemcpyAsync(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s);
  return e;
}

int write_arcs(const std::vector<int64_t> &at, const std::vector<int32_t> &w, int32_t *D,
               hipStream_t s, void **keep) {
  if (at.empty()) return FAP_OK;
  int64_t *dat = nullptr;
  int32_t *dw = nullptr;
  hipError_t e = to_device(at, &dat, s);
  keep[0] = dat;
  if (e == hipSuccess) e = to_device(w, &dw, s);
  keep[1] = dw;
  if (e != hipSuccess) return hip_fail(e, "coarse index", __FILE__, __LINE__);
  hipLaunchKernelGGL(fapk::hidx_arcs_kernel, dim3((unsigned)((at.size() + 255) / 256)), dim3(256),
                     0, s, dat, dw, (int64_t)at.size(), D);
  FAP_CHECK_LAUNCH();
  return FAP_OK;
}

// D of every region and C2: filled, arcs written, closed.
int close_levels(fap_ctx *ctx, const BidxDesc &d, const Regions &o, const HidxRegion *d_regs,
                 int32_t *D, int32_t *C2, hipStream_t s) {
  std::vector<int64_t> off;
  std::vector<int32_t> ldb;
  for (const BidxPartDesc &p : d.parts) {
    off.push_back(p.lbb_off);
    ldb.push_back(p.ldb);
  }
  void *keep[7] = {};
  int2 *ent = nullptr;
  int64_t *doff = nullptr;
  int32_t *dldb = nullptr;
  hipError_t e = to_device(o.ent, &ent, s);
  if (e == hipSuccess) e = to_device(off, &doff, s);
  if (e == hipSuccess) e = to_device(ldb, &dldb, s);
  keep[0] = ent;
  keep[1] = doff;
  keep[2] = dldb;
  std::vector<int32_t *> mats;
  std::vector<int32_t> ns;
  std::vector<int64_t> lds;
  for (size_t r = 0; r < o.regs.size() && e == hipSuccess; r++) {
    const HidxRegion &R = o.regs[r];
    if (R.n == 0) continue;
    hipLaunchKernelGGL(fapk::hidx_fill_kernel, dim3((R.ldd + 255) / 256, R.n), dim3(256), 0, s, R,
                       ent, doff, dldb, d.lbb, D);
    e = hipGetLastError();
    mats.push_back(D + R.off);
    ns.push_back(R.n);
    lds.push_back(R.ldd);
  }
  int rc = e == hipSuccess ? FAP_OK : hip_fail(e, "coarse index", __FILE__, __LINE__);
  if (rc == FAP_OK) rc = write_arcs(o.arc_at, o.arc_w, D, s, keep + 3);
  if (rc == FAP_OK)
    rc = fap_fw_batched(ctx, (int32_t)mats.size(), mats.data(), ns.data(), lds.data(), s);
  if (rc == FAP_OK) {
    hipLaunchKernelGGL(fapk::hidx_top_kernel, dim3((o.nbp2 + 255) / 256, o.nbp2), dim3(256), 0, s,
                       d_regs, (int32_t)o.regs.size(), o.nbp2, D, C2);
    e = hipGetLastError();
    if (e != hipSuccess) rc = hip_fail(e, "coarse index", __FILE__, __LINE__);
  }
  if (rc == FAP_OK) rc = write_arcs(o.top_at, o.top_w, C2, s, keep + 5);
  if (rc == FAP_OK) rc = fap_fw_blocked(ctx, C2, o.nbp2, o.nbp2, s);
  e = hipStreamSynchronize(s);  // before the descriptors go
  if (rc == FAP_OK && e != hipSuccess) rc = hip_fail(e, "coarse index", __FILE__, __LINE__);
  for (void *b : keep)
    if (b) (void)hipFree(b);
  return rc;
}

}  // namespace

static void free_hidx(fap_hidx *h) {
  if (!h) return;
  if (h->c) bidx_free(h->c);  // D with it
  if (h->regs) (void)hipFree(h->regs);
  if (h->C2) (void)hipFree(h->C2);
  delete h;
}

void hidx_release(fap_graph_dev *g) {
  free_hidx(g->hidx.exchange(nullptr));
  g->hidx_tried = false;
  g->batch_parts = 0;
}

// About sqrt(K) regions (a power of two: bisection cuts them evenly), more
// when their matrices would pass kMaxWords; kept when they leave at most half
// of the boundary vertices as region boundary (a graph without locality has no
// use for it) and take a small share of the memory that is free.
static bool choose_regions(const BidxDesc &d, Regions *o) {
  if (d.K < kMinParts) return false;
  for (int32_t R = 1 << (int)lround(log2((double)d.K) / 2); 2 * R <= d.K; R *= 2) {
    *o = Regions();
    make_regions(d, R, o);
    if (o->words > kMaxWords) continue;
    if (2 * (int64_t)o->nb2 > d.nb || o->nb2 == 0 || o->nbp2 > kMaxTop) return false;
    const size_t bytes = sizeof(int32_t) * ((size_t)o->words + (size_t)o->nbp2 * o->nbp2);
    size_t left = 0, total = 0;
    if (hipMemGetInfo(&left, &total) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return bytes <= left / kFreeShare;
  }
  return false;
}

static int make_level(fap_ctx *ctx, const BidxDesc &d, hipStream_t s, fap_hidx *h, int32_t **D) {
  Regions o;
  if (!choose_regions(d, &o)) return FAP_E_STATE;
  const size_t d_bytes = sizeof(int32_t) * (size_t)o.words;
  const size_t c_bytes = sizeof(int32_t) * (size_t)o.nbp2 * o.nbp2;
  FAP_HIP(hipMalloc((void **)D, d_bytes));
  FAP_HIP(hipMalloc((void **)&h->C2, c_bytes));
  FAP_HIP(to_device(o.regs, &h->regs, s));
  FAP_TRY(close_levels(ctx, d, o, h->regs, *D, h->C2, s));
  FAP_TRY(bidx_coarse(o.parts, o.colid, *D, o.nbp2, s, &h->c));
  BidxDesc cd;
  bidx_describe(h->c, &cd);
  h->D = *D;
  h->nbp2 = o.nbp2;
  for (const HidxRegion &r : o.regs) h->max_b = std::max(h->max_b, (r.b + 3) & ~3);
  h->bytes = cd.bytes + d_bytes + c_bytes + sizeof(HidxRegion) * o.regs.size();
  h->region = std::move(o.region);
  h->lpos = std::move(o.lpos);
  return FAP_OK;
}

// Tried once; a level that does not pay or cannot be made (memory) leaves the
// graph with the index alone.  The caller holds g->index_mu; the stream has
// drained on return, so the level may be used on any other.
int hidx_build(fap_ctx *ctx, fap_graph_dev *g, hipStream_t s) {
  if (g->hidx_tried || !g->bidx) return FAP_OK;
  g->hidx_tried = true;
  BidxDesc d;
  bidx_describe(g->bidx, &d);
  fap_hidx *h = new (std::nothrow) fap_hidx();
  if (!h) return FAP_OK;
  int32_t *D = nullptr;
  int rc = FAP_E_NOMEM;
  try {
    rc = make_level(ctx, d, s, h, &D);
  } catch (const std::bad_alloc &) {
  }
  if (rc == FAP_OK) {
    g->hidx.store(h, std::memory_order_release);
    return FAP_OK;
  }
  (void)hipStreamSynchronize(s);
  if (D && !h->c) (void)hipFree(D);
  free_hidx(h);
  (void)hipGetLastError();
  clear_error();
  return FAP_OK;
}

// Arguments as bidx_rows; everything is enqueued on s.  Uses ctx->ws_bidx
// (nsrc x nbp words, as there) and ctx->ws_hidx; without room for the latter,
// or with more tiles than a grid has rows, the block iterations do the work.
int hidx_rows(fap_ctx *ctx, const fap_graph_dev *g, int32_t count, const int32_t *qidx,
              const int32_t *rowoff, int32_t nsrc, int32_t *const *d_rowptr, hipStream_t s) {
  const fap_hidx *h = g->hidx.load(std::memory_order_acquire);
  if (!h) return bidx_rows(ctx, g, count, qidx, rowoff, nsrc, d_rowptr, s);
  if (nsrc <= 0) return FAP_OK;
  if ((nsrc + 63) / 64 > 65535)
    return fail(FAP_E_ARG, "boundary rows: too many sources in one call");
  BidxDesc d;
  bidx_describe(g->bidx, &d);
  // every source's region and place in it; runs of rows of one region in tiles
  std::vector<int2> rowq(nsrc);
  for (int32_t p = 0; p < count; p++) {
    const int32_t q = qidx[p];
    for (int32_t i = 0; i < d.parts[q].b; i++) {
      const int32_t id = d.parts[q].hoff + (*d.hpos)[(*d.boff)[q] + i];
      rowq[rowoff[p] + i] = make_int2(h->region[id], h->lpos[id]);
    }
  }
  std::vector<HidxTile> tiles;
  for (int32_t r = 0; r < nsrc;) {
    int32_t e = r + 1;
    while (e < nsrc && e < r + 128 && rowq[e].x == rowq[r].x) e++;
    tiles.push_back(HidxTile{r, e - r, rowq[r].x, 0});
    r = e;
  }
  if (tiles.size() > 65535) return bidx_rows(ctx, g, count, qidx, rowoff, nsrc, d_rowptr, s);
  const int64_t ldx = d.nbp, ldx2 = h->nbp2;
  const int32_t lds2 = h->max_b;
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  const size_t o_x2 = up(sizeof(int32_t) * (size_t)nsrc * lds2);
  const size_t o_rp = o_x2 + up(sizeof(int32_t) * (size_t)nsrc * ldx2);
  const size_t o_rq = o_rp + up(sizeof(int32_t *) * (size_t)nsrc);
  const size_t o_tl = up(sizeof(int2) * (size_t)nsrc);  // from o_rq: uploaded together
  const size_t staged = o_tl + sizeof(HidxTile) * tiles.size();
  FAP_TRY(ensure_ws(ctx, ctx->ws_bidx, sizeof(int32_t) * (size_t)nsrc * ldx));
  if (ensure_ws(ctx, ctx->ws_hidx, o_rq + staged) != FAP_OK) {
    (void)hipGetLastError();
    clear_error();
    return bidx_rows(ctx, g, count, qidx, rowoff, nsrc, d_rowptr, s);
  }
  char *w = (char *)ctx->ws_hidx.ptr;
  int32_t *X = (int32_t *)ctx->ws_bidx.ptr, *S2 = (int32_t *)w, *X2 = (int32_t *)(w + o_x2);
  int32_t **d_rp = (int32_t **)(w + o_rp);
  const int2 *d_rq = (const int2 *)(w + o_rq);
  void *stage = nullptr;
  FAP_TRY(acquire_host_stage(ctx, staged, &stage));
  std::copy(rowq.begin(), rowq.end(), (int2 *)stage);
  std::copy(tiles.begin(), tiles.end(), (HidxTile *)((char *)stage + o_tl));
  FAP_HIP(hipMemcpyAsync(w + o_rq, stage, staged, hipMemcpyHostToDevice, s));
  FAP_TRY(release_host_stage(ctx, s));
  hipLaunchKernelGGL(fapk::hidx_sources_kernel, dim3(nsrc), dim3(128), 0, s, d_rq, h->regs, h->D,
                     S2, lds2, X, ldx, d_rp);
  FAP_CHECK_LAUNCH();
  hipLaunchKernelGGL(fapk::hidx_cross_kernel,
                     dim3((unsigned)((ldx2 + 127) / 128), (unsigned)tiles.size()),
                     dim3(fapk::MP_THREADS), 0, s, (const HidxTile *)(w + o_rq + o_tl), h->regs, S2,
                     lds2, h->C2, h->nbp2, X2);
  FAP_CHECK_LAUNCH();
  FAP_TRY(bidx_expand(h->c, X2, ldx2, nsrc, d_rp, s));
  hipLaunchKernelGGL(fapk::hidx_own_kernel, dim3(nsrc, 4), dim3(256), 0, s, X, ldx, d_rq, h->regs,
                     bidx_columns(h->c), h->D);
  FAP_CHECK_LAUNCH();
  return bidx_expand(g->bidx, X, ldx, nsrc, d_rowptr, s);
}

}  // namespace fapi

using namespace fapi;

extern "C" int fap_graph_build_index(fap_ctx *ctx, fap_graph_dev *g, int32_t *built) {
  if (!ctx || !g) return fail(FAP_E_ARG, "null ctx/graph");
  FAP_HIP(hipSetDevice(ctx->device));
  std::lock_guard<std::mutex> lock(g->index_mu);
  FAP_TRY(bidx_build(ctx, g));
  FAP_TRY(hidx_build(ctx, g, ctx->stream));
  if (built) *built = g->bidx ? 1 : 0;
  return FAP_OK;
}

extern "C" int fap_graph_index_info(const fap_graph_dev *g, int32_t *boundary, int64_t *bytes) {
  if (!g) return fail(FAP_E_ARG, "null graph");
  BidxDesc d;
  if (g->bidx) bidx_describe(g->bidx, &d);
  if (boundary) *boundary = d.nb;
  const fap_hidx *h = g->hidx.load(std::memory_order_acquire);
  if (bytes) *bytes = (int64_t)(d.bytes + (h ? h->bytes : 0));
  return FAP_OK;
}
