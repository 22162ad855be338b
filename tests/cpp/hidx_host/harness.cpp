// Host check of the boundary index's coarse level
// (fastapsp_amd/csrc/hindex.hip): regions, layouts, uploads, workspaces and
// fallbacks, compiled as they are against the host-only stand-in of the HIP
// runtime (tests/cpp/bidx_host/mock) and CPU emulations of the kernels, under
// AddressSanitizer / UBSan.  Builds the index and its coarse level for a
// partitioned graph, solves boundary rows in calls of several sizes, with and
// without room for the coarse workspace, and compares rows with Dijkstra.
// Usage: hidx_host <graph.bin> <coarse level expected: 0 or 1>
// Prints "checked N rows, 0 bad" and exits 0 when everything matches.
#include <math.h>
#include <stdio.h>

#include <numeric>
#include <queue>
#include <string>
#include <vector>

#include "common.h"
#include "host.h"

static size_t g_ws_limit = SIZE_MAX;
inline hipError_t hipMemGetInfo(size_t *left, size_t *total) {
  *left = *total = (size_t)1 << 36;
  return hipSuccess;
}
namespace fapi {
void set_error(const std::string &m) { fprintf(stderr, "error: %s\n", m.c_str()); }
void clear_error() {}
int fail(int code, const std::string &m) { set_error(m); return code; }
int hip_fail(hipError_t, const char *w, const char *f, int l) {
  fprintf(stderr, "hip %s %s:%d\n", w, f, l);
  return FAP_E_HIP;
}
int ensure_ws(fap_ctx *ctx, Workspace &ws, size_t bytes) {
  if (&ws == &ctx->ws_hidx && bytes > g_ws_limit) return FAP_E_NOMEM;
  if (ws.bytes >= bytes) return FAP_OK;
  free(ws.ptr);
  ws.ptr = malloc(bytes);
  ws.bytes = bytes;
  return FAP_OK;
}
static std::vector<char> g_stage;
int acquire_host_stage(fap_ctx *, size_t bytes, void **out) {
  g_stage.assign(bytes, 0);
  *out = g_stage.data();
  return FAP_OK;
}
int release_host_stage(fap_ctx *, hipStream_t) { return FAP_OK; }
int launch_fill_i32(int32_t *d, int64_t n, int32_t v, hipStream_t) {
  std::fill(d, d + n, v);
  return FAP_OK;
}
int launch_gather(const fap_graph_dev *g, int32_t start, int32_t n, int32_t n_bdy, const int32_t *,
                  int64_t, int32_t *sub, int64_t ld, hipStream_t) {
  if (n_bdy != 0) abort();
  for (int i = 0; i < n; i++) {
    for (int j = 0; j < n; j++) sub[(int64_t)i * ld + j] = i == j ? 0 : kInf;
    const int u = g->st2ed[start + i];
    for (int e = g->row_offset[u]; e < g->row_offset[u + 1]; e++) {
      const int j = g->ed2st[g->edges[e].x] - start;
      if (j >= 0 && j < n && j != i) sub[(int64_t)i * ld + j] = g->edges[e].y;
    }
  }
  return FAP_OK;
}
}  // namespace fapi
extern "C" int fap_fw_batched(fap_ctx *, int32_t count, int32_t *const *m, const int32_t *ns,
                              const int64_t *lds, void *);
extern "C" int fap_fw_blocked(fap_ctx *ctx, int32_t *m, int32_t n, int64_t ld, void *s) {
  return fap_fw_batched(ctx, 1, &m, &n, &ld, s);
}
#include "bindex_host.inc"
#include "hindex_host.inc"

static std::vector<int32_t> dijkstra(const std::vector<int32_t> &ro, const std::vector<int2> &ed, int s) {
  std::vector<int32_t> d(ro.size() - 1, fapi::kInf);
  std::priority_queue<std::pair<int, int>, std::vector<std::pair<int, int>>, std::greater<>> pq;
  d[s] = 0;
  pq.push({0, s});
  while (!pq.empty()) {
    auto [du, u] = pq.top();
    pq.pop();
    if (du != d[u]) continue;
    for (int e = ro[u]; e < ro[u + 1]; e++)
      if (du + ed[e].y < d[ed[e].x]) {
        d[ed[e].x] = du + ed[e].y;
        pq.push({d[ed[e].x], ed[e].x});
      }
  }
  return d;
}

int main(int, char **argv) {
  FILE *f = fopen(argv[1], "rb");
  const bool expect = atoi(argv[2]) != 0;
  int64_t hdr[3];
  if (!f || fread(hdr, 8, 3, f) != 3) return 1;
  const int V = hdr[0], E = hdr[1], K = hdr[2];
  auto rd = [&](size_t n) {
    std::vector<int32_t> v(n);
    if (fread(v.data(), 4, n, f) != n) abort();
    return v;
  };
  auto ro = rd(V + 1), col = rd(E), wt = rd(E), gid = rd(V), st2ed = rd(V), ed2st = rd(V);
  auto vn = rd(K + 1), vo = rd(K + 1), bn = rd(K + 1);
  fclose(f);
  std::vector<int2> ed(E);
  for (int e = 0; e < E; e++) ed[e] = int2{col[e], wt[e]};
  fap_graph_dev g;
  g.V = V;
  g.E = E;
  g.row_offset = ro.data();
  g.edges = ed.data();
  g.graph_id = gid.data();
  g.st2ed = st2ed.data();
  g.ed2st = ed2st.data();
  g.h_st2ed = st2ed;
  g.h_graph_id = gid;
  fap_ctx *ctx = new fap_ctx();
  ctx->num_cus = 256;
  int32_t built = 0;
  if (fap_graph_build_index(ctx, &g, &built) || !built) return 1;
  const bool coarse = g.hidx.load() != nullptr;
  printf("index of %d parts, coarse level %s\n", K, coarse ? "built" : "not built");
  if (coarse != expect) return 1;
  long checked = 0, bad = 0;
  for (const size_t limit : {SIZE_MAX, (size_t)64})  // the second: the block iterations do the work
    for (const int group : {3, K}) {
      g_ws_limit = limit;
      for (int p0 = 1; p0 <= K; p0 += std::max(group, K / 3)) {
        const int cnt = std::min(group, K + 1 - p0);
        std::vector<int32_t> qidx(cnt), rowoff(cnt);
        int nsrc = 0;
        for (int i = 0; i < cnt; i++) {
          const int p = p0 + i;
          qidx[i] = fapi::bidx_part(&g, vo[p], vn[p], bn[p]);
          if (qidx[i] < 0) return 1;
          rowoff[i] = nsrc;
          nsrc += bn[p];
        }
        std::vector<int32_t> out((size_t)nsrc * V, -7);
        std::vector<int32_t *> rp(nsrc);
        for (int r = 0; r < nsrc; r++) rp[r] = out.data() + (size_t)r * V;
        if (fapi::hidx_rows(ctx, &g, cnt, qidx.data(), rowoff.data(), nsrc, rp.data(), nullptr))
          return 1;
        for (int i = 0, r = 0; i < cnt; i++)
          for (int j = 0; j < bn[p0 + i]; j++, r++) {
            if (r % 23 && r != nsrc - 1) continue;
            const auto want = dijkstra(ro, ed, st2ed[vo[p0 + i] + j]);
            checked++;
            bad += memcmp(want.data(), rp[r], 4 * (size_t)V) != 0;
          }
      }
    }
  fapi::hidx_release(&g);
  fapi::bidx_release(&g);
  printf("checked %ld rows, %ld bad\n", checked, bad);
  return bad != 0;
}
