// floyd.hip -- blocked Floyd-Warshall closure, in place.
//
// Replaces the reference's stage-2 operator floyd_path (fap/kernel/floyd.h:
// 150-158; CPU semantics floyd_CPU_path :38-49: k-i-j order, strict relax).
// The closure of a non-negative matrix is unique, so the blocked order gives
// the same distances as the k-i-j loop.  With block size T (64 or 128) and
// nb = ceil(n / T) blocks, round r (pivot block r) runs:
//   1. diagonal tile (r, r): closed in one workgroup, in registers;
//   2. row panel (r, J) = min(C, D_rr (x) C) and column panel
//      (I, r) = min(C, C (x) D_rr) for all I, J != r: one launch;
//   3. every other tile (I, J) = min(C, D_Ir (x) D_rJ): one launch.
// Phases 2 and 3 run T x T tiles with their additions on the matrix cores
// (mfma_tile.h; the panels of T = 128 in 64 x 64 quarters on the VALU).
// T = 128 halves the number of rounds and the passes over the matrix, which
// bound phase 3 (T = 64, n = 3800: 116 MB in 38 us, 19 us of arithmetic);
// T = 64 has a cheaper chain of diagonal and panels.  128 is the default for
// large n, 64 below (launch_fw).
#include <type_traits>

#include "common.h"
#include "mfma_tile.h"

namespace fapk {

// Closure of a 128 x 128 diagonal block (kb <= 128 valid rows/columns) by
// one workgroup of 1024 / NC threads: the blocked algorithm itself one level
// down, its 64-blocks closed in registers and multiplied from LDS (Blk64).
// The four blocks stay in registers throughout, so memory is read and
// written once.  `lds` holds CLOSE128_WORDS.
constexpr int CLOSE128_WORDS = 2 * T64_WORDS + CLOSE64_WORDS;

template <int NC>
__device__ __forceinline__ void close_block128(int32_t *blk, int64_t ld, int kb, int32_t *lds) {
  using B = Blk64<NC>;
  int32_t *X = lds, *Y = lds + T64_WORDS, *buf = lds + 2 * T64_WORDS;
  const int n0 = imin(64, kb), n1 = kb - 64;
  int d00[4][NC], d01[4][NC], d10[4][NC], d11[4][NC];
  int32_t *p01 = blk + 64, *p10 = blk + 64 * ld, *p11 = blk + 64 * ld + 64;
  if (n1 <= 0) {
    close_block64<NC>(blk, ld, n0, buf);
    return;
  }
  B::load(blk, ld, n0, n0, d00);
  B::load(p01, ld, n0, n1, d01);
  B::load(p10, ld, n1, n0, d10);
  B::load(p11, ld, n1, n1, d11);
  B::close(d00, n0, buf);
  B::to_lds(X, d00);
  B::to_lds(Y, d01);
  __syncthreads();
  B::product(X, Y, d01);  // D01 (+)= D00 D01
  __syncthreads();
  B::to_lds(Y, d10);
  __syncthreads();
  B::product(Y, X, d10);  // D10 (+)= D10 D00
  __syncthreads();
  B::to_lds(X, d10);
  B::to_lds(Y, d01);
  __syncthreads();
  B::product(X, Y, d11);  // D11 (+)= D10 D01
  B::close(d11, n1, buf);
  B::to_lds(X, d11);  // X's readers have passed a barrier of the closure
  __syncthreads();
  B::product(Y, X, d01);  // D01 (+)= D01 D11
  __syncthreads();
  B::to_lds(Y, d10);
  __syncthreads();
  B::product(X, Y, d10);  // D10 (+)= D11 D10
  __syncthreads();
  B::to_lds(X, d01);
  B::to_lds(Y, d10);
  __syncthreads();
  B::product(X, Y, d00);  // D00 (+)= D01 D10
  B::store(blk, ld, n0, n0, d00);
  B::store(p01, ld, n0, n1, d01);
  B::store(p10, ld, n1, n0, d10);
  B::store(p11, ld, n1, n1, d11);
}

// As a function of its own, for the phase-3 kernel (as close_block64_call).
__device__ __attribute__((noinline)) void close_block128_call(mp_out_ptr blk, int64_t ld, int kb,
                                                              mp_lds_ptr lds) {
  close_block128<4>((int32_t *)blk, ld, kb, (int32_t *)lds);
}

constexpr int FW_DIAG_THREADS = 512;  // workgroups alone on their CU: Blk64<2>

// Phase 1: the diagonal tile (r, r) alone, one workgroup.
template <int T>
__global__ __launch_bounds__(FW_DIAG_THREADS) void fw_diag_kernel(int32_t *d, int n, int64_t ld,
                                                                  int r) {
  __shared__ __attribute__((aligned(16))) int32_t lds[T == 64 ? CLOSE64_WORDS : CLOSE128_WORDS];
  const int base = r * T;
  const int kb = imin(T, n - base);
  int32_t *blk = d + (int64_t)base * ld + base;
  if (T == 64) close_block64<2>(blk, ld, kb, lds);
  else close_block128<2>(blk, ld, kb, lds);
}

// One whole round of T = 64 in a launch, for matrices whose rounds are
// latency and not work: the workgroup of tile (I, J) closes the pivot block
// itself, forms the row panel tile it needs, B' = min(B, D* (x) B), and
// updates C = min(C, A (x) B').  Sibling workgroups may already be writing
// the closed pivot block and panels over the tiles read here; every value in
// between is the length of a path through block r, no shorter than the
// closed one, and min-plus with the closed block makes the same result of
// both (D* D* = D*), so the bits do not depend on what was seen.
__global__ __launch_bounds__(FW_DIAG_THREADS) void fw_round_kernel(int32_t *d, int n, int64_t ld,
                                                                   int r, int nb) {
  using Blk = Blk64<2>;
  __shared__ __attribute__((aligned(16))) int32_t lds[3 * T64_WORDS + CLOSE64_WORDS];
  int32_t *X = lds, *Y = lds + T64_WORDS, *Z = lds + 2 * T64_WORDS;
  const int I = blockIdx.x / nb, J = blockIdx.x - I * nb;
  const int base = r * 64;
  const int kb = imin(64, n - base), rows = imin(64, n - I * 64), cols = imin(64, n - J * 64);
  int32_t *tile = d + (int64_t)I * 64 * ld + (int64_t)J * 64;
  int dd[4][2], a[4][2], b[4][2], c[4][2];
  Blk::load(d + (int64_t)base * ld + base, ld, kb, kb, dd);
  Blk::load(tile, ld, rows, cols, c);
  if (I != r && J != r) {
    Blk::load(d + (int64_t)base * ld + (int64_t)J * 64, ld, kb, cols, b);
    Blk::load(d + (int64_t)I * 64 * ld + base, ld, rows, kb, a);
  }
  Blk::close(dd, kb, lds + 3 * T64_WORDS);
  if (I == r && J == r) {
    Blk::store(tile, ld, rows, cols, dd);
    return;
  }
  Blk::to_lds(X, dd);
  const bool rest = I != r && J != r;
  if (rest) {
    Blk::to_lds(Y, b);
    Blk::to_lds(Z, a);
    __syncthreads();
    Blk::product(X, Y, b);
    __syncthreads();
    Blk::to_lds(Y, b);
  } else {
    Blk::to_lds(Y, c);
  }
  __syncthreads();
  Blk::product(rest ? Z : I == r ? X : Y, J == r ? X : Y, c);
  Blk::store(tile, ld, rows, cols, c);
}

// Phase 2: workgroups [0, nb-1) take row-panel tiles (r, J), the next nb-1
// take column-panel tiles (I, r).  Each tile is owned by one workgroup and
// aliases one operand; the tile reads all operands before writing C.  On the
// matrix-core tile, as phase 3, for any alignment (n = 2999 at an odd row
// stride 2.95 -> 2.01 ms with both; the 4 x 4 integer tile before).
__global__ __launch_bounds__(MP_THREADS) __attribute__((amdgpu_waves_per_eu(6, 6))) void fw_panel_kernel(
    int32_t *d, int n, int64_t ld, int r, int nb, int flags) {
  using Tile = MxSmall;
  constexpr int T = Tile::BM;
  __shared__ __attribute__((aligned(16))) int32_t lds[Tile::LDS_WORDS];
  const int base = r * T;
  const int kb = imin(T, n - base);
  const int32_t *diag = d + (int64_t)base * ld + base;
  int bid = blockIdx.x;
  if (bid < nb - 1) {
    const int J = bid < r ? bid : bid + 1;
    int32_t *c = d + (int64_t)base * ld + (int64_t)J * T;
    Tile::run(diag, ld, c, ld, c, ld, kb, imin(T, n - J * T), kb, true, flags, lds);
  } else {
    bid -= nb - 1;
    const int I = bid < r ? bid : bid + 1;
    int32_t *c = d + (int64_t)I * T * ld + base;
    Tile::run(c, ld, diag, ld, c, ld, imin(T, n - I * T), kb, kb, true, flags, lds);
  }
}

// Phase 2 for T = 128 in 64 x 64 pieces: each panel tile (r, J) or (I, r)
// is split into four 64 x 64 output quarters, one workgroup each (K = 128,
// 4 x 4 cells per lane), so the phase runs 4 (2 nb - 2) short workgroups
// instead of 2 nb - 2 long ones (n = 8192: 19 us per round against 40).
// A quarter reads the other row (column) half of its own panel tile while a
// sibling writes it; every value it can see there is the length of a path
// through pivot block r no shorter than the finished one, so the minimum it
// forms is the same either way.  (Staging the whole 128-deep operands in
// LDS at once, 67 KB per workgroup, measured 21 us.)
__global__ __launch_bounds__(MP_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void fw_panel128_kernel(
    int32_t *d, int n, int64_t ld, int r, int nb, int flags) {
  __shared__ __attribute__((aligned(16))) int32_t lds[MpSmall::LDS_WORDS];
  const int base = r * 128;
  const int kb = imin(128, n - base);
  const int32_t *diag = d + (int64_t)base * ld + base;
  const int q = blockIdx.x & 3, hr = q >> 1, hc = q & 1;
  int bid = blockIdx.x >> 2;
  if (bid < nb - 1) {
    const int J = bid < r ? bid : bid + 1;
    const int rows = kb - 64 * hr, cols = imin(128, n - J * 128) - 64 * hc;
    if (rows <= 0 || cols <= 0) return;
    int32_t *c = d + (int64_t)base * ld + (int64_t)J * 128;
    MpSmall::run(diag + (int64_t)(64 * hr) * ld, ld, c + 64 * hc, ld,
                 c + (int64_t)(64 * hr) * ld + 64 * hc, ld, imin(64, rows), imin(64, cols), kb,
                 true, flags, lds);
  } else {
    bid -= nb - 1;
    const int I = bid < r ? bid : bid + 1;
    const int rows = imin(128, n - I * 128) - 64 * hr, cols = kb - 64 * hc;
    if (rows <= 0 || cols <= 0) return;
    int32_t *c = d + (int64_t)I * 128 * ld + base;
    MpSmall::run(c + (int64_t)(64 * hr) * ld, ld, diag + 64 * hc, ld,
                 c + (int64_t)(64 * hr) * ld + 64 * hc, ld, imin(64, rows), imin(64, cols), kb,
                 true, flags, lds);
  }
}

// Phase 3 over a set of tiles, selected by `mode` (p = r + 1):
//   0: every tile outside row r and column r, (nb-1)^2 of them;
//   1: the look-ahead tiles, row p and column p minus row/column r (2nb-3);
//   2: the rest, outside rows/columns r and p, (nb-2)^2.
// Modes 1 and 2 together equal mode 0; splitting them lets the next round's
// diagonal and panels (which only touch row/column p) start while mode 2
// runs.
//
// With `fuse` (mode 0, r + 1 < nb) workgroup 0 takes tile (r+1, r+1) --
// swapping with the workgroup that had it -- and after its update closes
// it (in LDS for T = 64, by close_block128 for T = 128): the next round's
// diagonal phase, done while the other tiles of this phase run, so that
// round launches only its panels.  T = 64 wants 6 waves per SIMD (78 to 80 VGPRs, no
// call inside): n = 3500 2.58 ms, 2.73 at the 4 that its callees would leave.
template <int TM, bool fuse>
__global__ __launch_bounds__(MP_THREADS) __attribute__((amdgpu_waves_per_eu(TM == 4 ? 6 : 4, TM == 4 ? 6 : 4))) void fw_rest_kernel(
    int32_t *d, int n, int64_t ld, int r, int nb, int flags, int mode) {
  using Tile = typename std::conditional<TM == 8, MxBig, MxSmall>::type;
  constexpr int T = Tile::BM;
  constexpr int CLOSE_WORDS = TM == 4 ? CLOSE64_WORDS : CLOSE128_WORDS;
  constexpr int LDS_WORDS = CLOSE_WORDS > Tile::LDS_WORDS ? CLOSE_WORDS : Tile::LDS_WORDS;
  __shared__ __attribute__((aligned(16))) int32_t lds[LDS_WORDS];
  int I, J;
  if (mode == 0) {
    const int m = nb - 1;
    int t = xcd_remap(blockIdx.x, m * m);
    if (fuse) {
      const int tp = r * m + r;  // tile (r+1, r+1) in the compressed index
      if (blockIdx.x == 0) t = tp;
      else if (t == tp) t = xcd_remap(0, m * m);
    }
    I = t / m;
    J = t - I * m;
    I += (I >= r);
    J += (J >= r);
  } else if (mode == 1) {
    const int p = r + 1;
    const int t = blockIdx.x;
    if (t < nb - 1) {
      I = p;
      J = t + (t >= r);
    } else {
      const int u = t - (nb - 1);
      I = u < r ? u : u + 2;
      J = p;
    }
  } else {
    const int m = nb - 2;
    const int t = xcd_remap(blockIdx.x, m * m);
    I = t / m;
    J = t - I * m;
    I = I < r ? I : I + 2;
    J = J < r ? J : J + 2;
  }
  const int base = r * T;
  const int kb = imin(T, n - base);
  int32_t *c = d + (int64_t)I * T * ld + (int64_t)J * T;
  const int32_t *a = d + (int64_t)I * T * ld + base;
  const int32_t *b = d + (int64_t)base * ld + (int64_t)J * T;
  Tile::run(a, ld, b, ld, c, ld, imin(T, n - I * T), imin(T, n - J * T), kb, true, flags, lds);
  if (fuse && blockIdx.x == 0) {
    __syncthreads();  // the tile's writes above come before the closure reads it
    if constexpr (T == 64) close_block64<4>(c, ld, imin(T, n - I * T), lds);
    else close_block128_call((mp_out_ptr)c, ld, imin(T, n - I * T), (mp_lds_ptr)lds);
  }
}

}  // namespace fapk

namespace fapi {

int vec_flags(const void *A, int64_t lda, const void *B, int64_t ldb, const void *C,
              int64_t ldc);

namespace {

template <int TM>
struct Fw {
  static constexpr int T = 16 * TM;

  static int diag_panel(int32_t *d, int32_t n, int64_t ld, int r, int nb, int flags,
                        hipStream_t s, bool diag = true) {
    if (diag) {
      hipLaunchKernelGGL(fapk::fw_diag_kernel<T>, dim3(1), dim3(fapk::FW_DIAG_THREADS), 0, s, d,
                         n, ld, r);
      FAP_CHECK_LAUNCH();
    }
    if (nb > 1) {
      if constexpr (TM == 8)
        hipLaunchKernelGGL(fapk::fw_panel128_kernel, dim3(8 * (nb - 1)), dim3(fapk::MP_THREADS),
                           0, s, d, n, ld, r, nb, flags);
      else
        hipLaunchKernelGGL(fapk::fw_panel_kernel, dim3(2 * (nb - 1)), dim3(fapk::MP_THREADS), 0, s,
                           d, n, ld, r, nb, flags);
      FAP_CHECK_LAUNCH();
    }
    return FAP_OK;
  }

  static int rest(int32_t *d, int32_t n, int64_t ld, int r, int nb, int flags, int mode,
                  hipStream_t s, int fuse = 0) {
    const int tiles =
        mode == 0 ? (nb - 1) * (nb - 1) : mode == 1 ? 2 * nb - 3 : (nb - 2) * (nb - 2);
    if (tiles <= 0) return FAP_OK;
    if (fuse)
      hipLaunchKernelGGL((fapk::fw_rest_kernel<TM, true>), dim3(tiles), dim3(fapk::MP_THREADS), 0,
                         s, d, n, ld, r, nb, flags, mode);
    else
      hipLaunchKernelGGL((fapk::fw_rest_kernel<TM, false>), dim3(tiles), dim3(fapk::MP_THREADS), 0,
                         s, d, n, ld, r, nb, flags, mode);
    FAP_CHECK_LAUNCH();
    return FAP_OK;
  }

  // With look-ahead, round r's phase 3 is split: the tiles of row/column
  // r+1 first (mode 1), then, on the auxiliary stream, round r+1's diagonal
  // and panels run while the main stream finishes round r's other tiles
  // (mode 2).  All work is ordered before later work on `s` on return.
  static int run(fap_ctx *ctx, int32_t *d, int32_t n, int64_t ld, bool lookahead,
                 hipStream_t s) {
    const int nb = (n + T - 1) / T;
    const int flags = vec_flags(d, ld, d, ld, d, ld);
    FAP_TRY(diag_panel(d, n, ld, 0, nb, flags, s));
    const bool overlap = lookahead && ctx && ctx->aux_stream && nb >= 3;
    // phase 3 also closes the next diagonal block, beside its other tiles,
    // from one tile per CU on: no launch for it, and it starts a phase early
    // (T = 64: n = 1250 0.73 -> 0.62 ms, 2048 1.13 -> 0.94, 2560 -> 1.22;
    // T = 128: 4096 3.89 -> 3.67)
    const int64_t cus = ctx ? ctx->num_cus : 256;
    const bool fuse_ok = (int64_t)(nb - 1) * (nb - 1) >= cus;
    for (int r = 0; r < nb; r++) {
      if (r + 1 < nb && overlap) {
        FAP_TRY(rest(d, n, ld, r, nb, flags, 1, s));
        FAP_HIP(hipEventRecord(ctx->ev_fw_la, s));
        FAP_HIP(hipStreamWaitEvent(ctx->aux_stream, ctx->ev_fw_la, 0));
        FAP_TRY(diag_panel(d, n, ld, r + 1, nb, flags, ctx->aux_stream));
        FAP_HIP(hipEventRecord(ctx->ev_fw_panel, ctx->aux_stream));
        FAP_TRY(rest(d, n, ld, r, nb, flags, 2, s));
        FAP_HIP(hipStreamWaitEvent(s, ctx->ev_fw_panel, 0));
      } else {
        const int fuse = (fuse_ok && r + 1 < nb) ? 1 : 0;
        FAP_TRY(rest(d, n, ld, r, nb, flags, 0, s, fuse));
        if (r + 1 < nb) FAP_TRY(diag_panel(d, n, ld, r + 1, nb, flags, s, !fuse));
      }
    }
    return FAP_OK;
  }
};

}  // namespace

// Rounds of T = 64 as single launches (fw_round_kernel).
static int run_rounds(int32_t *d, int32_t n, int64_t ld, hipStream_t s) {
  const int nb = (n + 63) / 64;
  for (int r = 0; r < nb; r++) {
    hipLaunchKernelGGL(fapk::fw_round_kernel, dim3(nb * nb), dim3(fapk::FW_DIAG_THREADS), 0, s,
                       d, n, ld, r, nb);
    FAP_CHECK_LAUNCH();
  }
  return FAP_OK;
}

// Block size and look-ahead: the context options if set, else the tune
// cache, else 128 for large n and 64 below, without look-ahead (fw_settings,
// with both sides measured).  T = 128 halves the passes over the matrix, but
// its chain of diagonal and panels is longer.
int launch_fw(fap_ctx *ctx, int32_t *d, int32_t n, int64_t ld, hipStream_t s) {
  if (n <= 0) return FAP_OK;
  int tile;
  bool lookahead;
  fw_settings(ctx, n, &tile, &lookahead);
  if (tile == 128) return Fw<8>::run(ctx, d, n, ld, lookahead, s);
  // Up to a workgroup per CU a round in one launch wins although every
  // workgroup closes the pivot block and makes its own panel tile (us, a
  // launch a round / phases: n = 97 44 / 66, 512 160 / 243, 900 346 / 483,
  // 1024 325 / 470; past it 1088 484 / 465, 1216 546 / 527).
  const int64_t nb = (n + 63) / 64;
  if (!lookahead && nb * nb <= (int64_t)(ctx ? ctx->num_cus : 256))
    return run_rounds(d, n, ld, s);
  return Fw<4>::run(ctx, d, n, ld, lookahead, s);
}

}  // namespace fapi

using namespace fapi;

extern "C" int fap_fw_blocked(fap_ctx *ctx, int32_t *d_mat, int32_t n, int64_t ld,
                              void *stream) {
  if (!ctx) return fail(FAP_E_ARG, "ctx is null");
  if (n < 0) return fail(FAP_E_ARG, "fw: negative n");
  if (n == 0) return FAP_OK;
  if (!d_mat) return fail(FAP_E_ARG, "fw: null matrix");
  if (ld < n) return fail(FAP_E_ARG, "fw: ld < n");
  if ((int64_t)(n + 63) / 64 > 46340) return fail(FAP_E_ARG, "fw: n too large");
  return launch_fw(ctx, d_mat, n, ld, pick_stream(ctx, stream));
}
