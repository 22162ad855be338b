// CPU emulations of hindex.hip's kernels for the host check: each follows its
// kernel's indexing, so that AddressSanitizer sees every access the device
// code would make.
#pragma once
namespace fapk {

inline void hidx_fill_kernel(dim3 g, dim3 b, HidxRegion R, const int2 *ent, const int64_t *lbb_off,
                             const int32_t *ldb, const int32_t *lbb, int32_t *D) {
  assert((int)g.y == R.n && (int)(g.x * b.x) >= R.ldd);
  for (int i = 0; i < R.n; i++) {
    const int2 a = ent[R.start + i];
    for (int j = 0; j < R.ldd; j++) {
      int v = kInf;
      if (j < R.n) {
        const int2 c = ent[R.start + j];
        if (c.x == a.x) v = lbb[lbb_off[a.x] + (int64_t)a.y * ldb[a.x] + c.y];
        if (i == j) v = 0;
      }
      D[R.off + (int64_t)i * R.ldd + j] = v;
    }
  }
}

inline void hidx_top_kernel(dim3 g, dim3, const HidxRegion *regs, int32_t nreg, int32_t nbp2,
                            const int32_t *D, int32_t *C2) {
  assert((int)g.y == nbp2);
  for (int i = 0; i < nbp2; i++) {
    int lo = 0, hi = nreg - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (regs[mid].hoff <= i) lo = mid;
      else hi = mid - 1;
    }
    const HidxRegion R = regs[lo];
    const bool real = i - R.hoff < R.b;
    for (int j = 0; j < nbp2; j++) {
      int v = kInf;
      if (real && j >= R.hoff && j < R.hoff + R.b)
        v = D[R.off + (int64_t)(i - R.hoff) * R.ldd + j - R.hoff];
      C2[(int64_t)i * nbp2 + j] = i == j ? 0 : v;
    }
  }
}

inline void hidx_arcs_kernel(dim3 g, dim3 b, const int64_t *at, const int32_t *w, int64_t count,
                             int32_t *D) {
  assert((int64_t)g.x * b.x >= count);
  for (int64_t i = 0; i < count; i++) D[at[i]] = w[i];
}

inline void hidx_own_kernel(dim3 g, dim3, int32_t *X, int64_t ldx, const int2 *rowq,
                            const HidxRegion *regs, const int32_t *colid, const int32_t *D) {
  for (unsigned r = 0; r < g.x; r++) {
    const HidxRegion R = regs[rowq[r].x];
    for (int j = 0; j < R.n; j++) {
      int32_t &x = X[r * ldx + colid[R.start + j]];
      x = std::min(x, D[R.off + (int64_t)rowq[r].y * R.ldd + j]);
    }
  }
}

inline void hidx_sources_kernel(dim3 g, dim3, const int2 *rowq, const HidxRegion *regs,
                                const int32_t *D, int32_t *S2, int32_t lds2, int32_t *X, int64_t ldx,
                                int32_t **rowptr) {
  for (unsigned r = 0; r < g.x; r++) {
    const HidxRegion R = regs[rowq[r].x];
    for (int k = 0; k < R.b; k++)
      S2[(int64_t)r * lds2 + k] = D[R.off + (int64_t)rowq[r].y * R.ldd + k];
    rowptr[r] = X + r * ldx;
  }
}

inline void hidx_cross_kernel(dim3 g, dim3, const HidxTile *tiles, const HidxRegion *regs,
                              const int32_t *S2, int32_t lds2, const int32_t *C2, int32_t nbp2,
                              int32_t *X2) {
  for (unsigned t = 0; t < g.y; t++) {
    const HidxTile T = tiles[t];
    const HidxRegion R = regs[T.reg];
    assert(T.rows > 0 && T.rows <= 128 && R.b <= lds2);
    for (int i = T.row0; i < T.row0 + T.rows; i++)
      for (int c = 0; c < std::min<int>(g.x * 128, nbp2); c++) {
        int v = kInf;
        for (int k = 0; k < R.b; k++)
          v = std::min(v, S2[(int64_t)i * lds2 + k] + C2[(int64_t)(R.hoff + k) * nbp2 + c]);
        X2[(int64_t)i * nbp2 + c] = v;
      }
  }
}

}  // namespace fapk
