// mfma_tile.h -- min-plus tile whose additions run on the matrix cores.
//
// A min-plus update is an addition and a minimum.  On the VALU alone the pair
// costs 1.5 instructions (v_add_u32 and half a v_min3_i32), and the tile of
// minplus_tile.h runs at that limit.  Here the additions are an outer sum on
// the matrix cores: with operands split in two f16 digits,
//   (a.lo, a.hi, w0, w1) . (w0, w1, b.lo, b.hi) = w0 (a.lo + b.lo) + w1 (a.hi + b.hi),
// one v_mfma_f32_32x32x4_2b_f16 (K = 4, two blocks: k and k + 1) makes
// 2 x 32 x 32 sums a + b, and the VALU only folds them: one v_min3_i32 per
// two updates.
//
// Exactness.  A digit is an 11-bit integer x stored as the f16 with bits x,
// which is x 2^-24 exactly (subnormal below 1024, the first binade above; the
// matrix cores of this target keep f16 subnormals).  With w0 = 1, w1 = 2048
// the result is (a + b) 2^-24 for values below 2^22: every product and sum is
// an integer below 2^24 times 2^-24, exact in float; sums are not negative, so
// the minimum is taken on the floats' bits, as integers.  Operands are stored
// plus one, so that INF = 2^30 - 1 becomes the single bit 30, which lands in
// the exponent of the high digit: it reads as 2.0, the sum as at least 4096,
// above every finite one.  A value that is neither below 2^22 - 1 nor INF or
// above (bits 22..29 or the sign after the increment) raises a flag while it
// is staged; the workgroup takes the k from that chunk on with integer
// additions (MpTile), on top of what it has: results are the same for all
// inputs.  Distances past 4.19 million are ordinary in road networks; all
// values there, integer kernels alone -> here: 8192^3 17.4 -> 17.4 ms,
// 909 x 262144 x 115 1.01 -> 1.03, closures of n = 1024..3456 585 us -> 341 to
// 2.57 -> 2.56 ms, 4096 3.43 -> 3.63, 8192 19.9 -> 20.5; large values in the
// last chunk alone cost nothing (8192^3 16.4 -> 10.8).  Left: what the first
// look costs products of few k (4096 x 65536 x 16 241 -> 272 us).
//
// What bounds it: the VALU port, 16 v_min3_i32 and one MFMA issue for 2048
// sums.  Measured in registers and LDS alone (4 waves per SIMD): 104 TOP/s at
// 2 ops per update against 70.3 of add, add, min3 (MFMA alone 149, v_min3
// alone 137; the clock falls to 2.1 GHz with both units busy).  Kernels on the
// 128 x 128 tile, integer tile before: the 8192^3 product 16.4 -> 10.8 ms
// (102 TOP/s), 909 x 262144 x 115 0.936 -> 0.66 ms, the n = 8192 closure
// 18.9 -> 15.1 ms.  It takes every 128-row tile of a product of 16 k and more
// (row tails are in minplus.hip).
#ifndef FAP_MFMA_TILE_H_
#define FAP_MFMA_TILE_H_

#include "minplus_tile.h"

namespace fapk {

typedef _Float16 mx_half4 __attribute__((ext_vector_type(4)));
typedef float mx_f32x32 __attribute__((ext_vector_type(32)));
typedef int mx_int2 __attribute__((ext_vector_type(2)));

constexpr int MX_BK = 8;                            // k per staged chunk
constexpr uint32_t MX_WEIGHTS = 0x68003C00u;        // f16 {1.0, 2048.0}
constexpr uint32_t MX_BAD = 0xBFC00000u;            // bits of v + 1 that leave the digits
// v + 1 as two 11-bit f16 digits (high digit in the high half); bit 30, set
// for INF alone among valid values, stays in place.
__device__ __forceinline__ uint32_t mx_digits(uint32_t w) {
  return __umul24((w >> 11) & 0x7FFu, 65536u - 2048u) + w;
}

// The tile: (64 NI) x (64 NJ) outputs by 256 threads, a wave (32 NI) x (32 NJ)
// as NI x NJ MFMA blocks.  Element (k, row) of A and (k, column) of B are
// 8 bytes in LDS, {digits, weights} and {weights, digits}; a fragment is one
// ds_read_b64, lanes 0..31 at k and 32..63 at k + 1.  Lane l holds column
// (l & 31) of a block and rows 8 (r / 4) + 4 (l / 32) + r % 4, r < 16.
// k is staged in chunks of 8 in two LDS buffers (one barrier per chunk); the
// next chunk's global loads are in flight while the current one is computed.
// 128 VGPRs for 2 x 2 blocks: 64 accumulators, 32 sums, 8 staged words.
template <int NI, int NJ>
struct MxTile {
  static constexpr int BM = 64 * NI, BN = 64 * NJ;
  static constexpr int LDA = BM + 1, LDB = BN + 1;  // elements per k row
  static constexpr int EA = 2 * NI, EB = 2 * NJ;    // staged words per thread
  static constexpr int A_TPR = MX_BK / EA;          // threads per A row when staging
  static constexpr int B_OFF = 2 * MX_BK * LDA;     // words from A to B of a buffer
  static constexpr int BUF = 2 * MX_BK * (LDA + LDB);
  static constexpr int FLAG = 2 * BUF;
  static constexpr int LDS_WORDS = FLAG + 4;

  template <int E>
  __device__ static __forceinline__ void load_vec(const int32_t *base, uint32_t off, int v[E]) {
    typedef int vec __attribute__((ext_vector_type(E), aligned(4)));
    const vec x = *reinterpret_cast<const vec *>(reinterpret_cast<const char *>(base) + off);
#pragma unroll
    for (int i = 0; i < E; i++) v[i] = x[i];
  }

  using Int = MpTile<4 * NI, 4 * NJ>;  // the same tile with integer additions
  // The small tile begins with two chunks at once, loaded as the integer
  // tile's first one of 16 k.
  static constexpr bool PAIR = NI * NJ == 1;

  // What the staging below asks of an operand: full first chunks and vectors
  // of columns, and byte offsets inside a chunk that fit 32 bits.  (The large
  // tile asks for 8 k though products of fewer than 16 go elsewhere: told of 16,
  // the compiler makes its k loop slower, 128 x 128 x 8192 1.55 -> 1.65 ms.)
  __device__ static __forceinline__ bool fits(int64_t lda, int64_t ldb, int n_valid, int K) {
    return K >= (PAIR ? MP_BK : MX_BK) && n_valid >= 4 * NJ / (PAIR ? 1 : 2) &&
           lda < (1 << 22) && ldb < (1 << 26);
  }

  // Where this thread's words of a chunk are: A row t / A_TPR, k
  // (t % A_TPR) * EA ..; B k row t / 32, columns (t % 32) * EB ...  Rows past
  // m_valid repeat the last one, columns past n_valid the last EB valid ones
  // (at their own place): neither reaches a stored output.
  struct Stage {
    uint32_t a_off, b_off;  // bytes from the chunk's corner
    int a_lds, b_lds;       // words from the buffer's start
    __device__ __forceinline__ Stage(int64_t lda, int64_t ldb, int m_valid, int n_valid) {
      const int t = threadIdx.x;
      const int col = imin((t & 31) * EB, n_valid - EB);
      a_off = 4u * ((uint32_t)imin(t / A_TPR, m_valid - 1) * (uint32_t)lda +
                    (uint32_t)((t % A_TPR) * EA));
      b_off = 4u * ((uint32_t)(t >> 5) * (uint32_t)ldb + (uint32_t)col);
      a_lds = 2 * ((t % A_TPR) * EA * LDA + t / A_TPR);
      b_lds = B_OFF + 2 * ((t >> 5) * LDB + col) + 1;
    }
  };

  // Writes the digits of a loaded chunk to buffer `par`, and sets its flag if
  // a value did not fit them.
  __device__ static __forceinline__ void store_chunk(int32_t *lds, int par, const Stage &st,
                                                     const int ra[EA], const int rb[EB]) {
    uint32_t seen = 0;
    int32_t *buf = lds + par * BUF, *pa = buf + st.a_lds;
#pragma unroll
    for (int i = 0; i < EA; i++) {
      const uint32_t w = (uint32_t)ra[i] + 1u;
      seen |= w;
      pa[2 * i * LDA] = (int32_t)mx_digits(w);
    }
    int32_t *pb = buf + st.b_lds;
#pragma unroll
    for (int i = 0; i < EB; i++) {
      const uint32_t w = (uint32_t)rb[i] + 1u;
      seen |= w;
      pb[2 * i] = (int32_t)mx_digits(w);
    }
    if (seen & MX_BAD) lds[FLAG + par] = 1;
  }

  // The first two chunks: A row t / 4, k (t % 4) * 4 ..; B k row t / 16,
  // columns (t % 16) * 4 .. (those at the edges as in Stage).
  __device__ static __forceinline__ int pair_col(int n_valid) {
    return imin(((int)threadIdx.x & 15) * 4, n_valid - 4);
  }
  __device__ static __forceinline__ void load_pair(const int32_t *A, int64_t lda, const int32_t *B,
                                                   int64_t ldb, int m_valid, int n_valid,
                                                   int (&ha)[4 * NI], int (&hb)[4 * NJ]) {
    const int t = threadIdx.x;
    load_vec<4>(A, 4u * ((uint32_t)imin(t >> 2, m_valid - 1) * (uint32_t)lda + (t & 3) * 4u), ha);
    load_vec<4>(B, 4u * ((uint32_t)(t >> 4) * (uint32_t)ldb + (uint32_t)pair_col(n_valid)), hb);
  }
  __device__ static __forceinline__ void store_pair(int32_t *lds, int n_valid,
                                                    const int (&ha)[4 * NI],
                                                    const int (&hb)[4 * NJ]) {
    const int t = threadIdx.x, ca = (t & 3) >> 1, cb = t >> 7;  // the words' chunks
    int32_t *pa = lds + ca * BUF + 2 * ((t & 1) * 4 * LDA + (t >> 2));
    int32_t *pb = lds + cb * BUF + B_OFF + 2 * (((t >> 4) & 7) * LDB + pair_col(n_valid)) + 1;
    uint32_t sa = 0, sb = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      sa |= (uint32_t)ha[i] + 1u;
      sb |= (uint32_t)hb[i] + 1u;
    }
    // no digits where the first chunk will not be used (n = 4096, all values
    // past them: 3.79 -> 3.72 ms)
    if (__any((((ca ? 0u : sa) | (cb ? 0u : sb)) & MX_BAD) != 0)) {
      lds[FLAG] = 1;
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t a = (uint32_t)ha[i] + 1u, b = (uint32_t)hb[i] + 1u;
      pa[2 * i * LDA] = (int32_t)mx_digits(a);
      pb[2 * i] = (int32_t)mx_digits(b);
    }
    if (sa & MX_BAD) lds[FLAG + ca] = 1;
    if (sb & MX_BAD) lds[FLAG + cb] = 1;
  }

  // The flag, after the barrier that follows: the same for every thread (a
  // faster one may be writing the other buffer's).
  __device__ static __forceinline__ int unfit(const int32_t *lds, int par) {
    return __builtin_amdgcn_readfirstlane(lds[FLAG + par]);
  }

  // The constant halves of both buffers' elements, and the flags: once.
  __device__ static __forceinline__ void init_lds(int32_t *lds) {
#pragma unroll
    for (int b = 0; b < 2; b++) {
      for (int i = threadIdx.x; i < MX_BK * LDA; i += MP_THREADS)
        lds[b * BUF + 2 * i + 1] = (int32_t)MX_WEIGHTS;
      for (int i = threadIdx.x; i < MX_BK * LDB; i += MP_THREADS)
        lds[b * BUF + B_OFF + 2 * i] = (int32_t)MX_WEIGHTS;
    }
    if (threadIdx.x < 2) lds[FLAG + threadIdx.x] = 0;
  }

  // acc = min(acc, A (x) B) over the staged chunk's k from kbeg (even) on, as
  // float bits.  A block of 16 minima follows each MFMA; the other waves of
  // the SIMD issue while its result is in flight.
  __device__ static __forceinline__ void compute(const int32_t *buf, int kbeg,
                                                 int acc[NI][NJ][16]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const mx_int2 *pa = reinterpret_cast<const mx_int2 *>(buf) + (kbeg + (lane >> 5)) * LDA +
                        (wave >> 1) * (32 * NI) + (lane & 31);
    const mx_int2 *pb = reinterpret_cast<const mx_int2 *>(buf + B_OFF) + (kbeg + (lane >> 5)) * LDB +
                        (wave & 1) * (32 * NJ) + (lane & 31);
    mx_f32x32 zero;
#pragma unroll
    for (int r = 0; r < 32; r++) zero[r] = 0.0f;
#pragma unroll 1
    for (int kk = kbeg; kk < MX_BK; kk += 2) {
      mx_half4 a[NI], b[NJ];
#pragma unroll
      for (int i = 0; i < NI; i++) a[i] = __builtin_bit_cast(mx_half4, pa[32 * i]);
#pragma unroll
      for (int j = 0; j < NJ; j++) b[j] = __builtin_bit_cast(mx_half4, pb[32 * j]);
      pa += 2 * LDA;
      pb += 2 * LDB;
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          const mx_f32x32 d = __builtin_amdgcn_mfma_f32_32x32x4f16(a[i], b[j], zero, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 16; r++)
            acc[i][j][r] = imin(acc[i][j][r], imin(__float_as_int(d[r]), __float_as_int(d[16 + r])));
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  }

  // The value of an accumulator: the sum less both operands' + 1.  The
  // instruction saturates (a C++ cast need not), so every sum with an INF in
  // it comes out as INF.
  __device__ static __forceinline__ int value(int bits) {
    int v;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(v) : "v"(fmaf(__int_as_float(bits), 16777216.0f, -2.0f)));
    return imin(v, kInf);
  }

  // Row of a block held in accumulator r by lanes 0..31 (4 more above).
  __device__ static constexpr int acc_row(int r) { return 8 * (r >> 2) + (r & 3); }

  // The k loop: staging pipelined with compute.  The last chunk ends at K
  // and skips (pairwise) the k that the one before it has taken.  Returns how
  // many k are in acc, the same for every thread: K, or a multiple of 8 when
  // a value of the chunk that follows did not fit its digits.
  __device__ static __forceinline__ int product(const int32_t *A, int64_t lda, const int32_t *B,
                                                int64_t ldb, int m_valid, int n_valid, int K,
                                                int32_t *lds, int acc[NI][NJ][16],
                                                int (&ha)[4 * NI], int (&hb)[4 * NJ]) {
    int ra[EA], rb[EB];
    const Stage st(lda, ldb, m_valid, n_valid);
    int par = 0, kbeg = 0, k0 = MX_BK;  // k0: start of the next chunk
    int bad = 0;
    if constexpr (PAIR) {
      load_pair(A, lda, B, ldb, m_valid, n_valid, ha, hb);
      init_lds(lds);
      __syncthreads();  // the flags are cleared
      store_pair(lds, n_valid, ha, hb);
      __syncthreads();
      if (unfit(lds, 0)) return 0;
      compute(lds, 0, acc);
      __syncthreads();  // the loop's first turn stores over what this has read
      par = 1;
      k0 = 2 * MX_BK;
    } else {
      load_vec<EA>(A, st.a_off, ra);
      load_vec<EB>(B, st.b_off, rb);
      init_lds(lds);
      __syncthreads();  // the flags are cleared
      store_chunk(lds, 0, st, ra, rb);
      __syncthreads();
    }
    while (k0 < K) {
      const int kc = imin(k0, K - MX_BK);
      load_vec<EA>(A + kc, st.a_off, ra);
      load_vec<EB>(B + (int64_t)kc * ldb, st.b_off, rb);
      asm volatile("" ::: "memory");  // the loads stay ahead of the look
      bad = unfit(lds, par);
      if (bad) break;
      compute(lds + par * BUF, 0, acc);
      par ^= 1;
      kbeg = (k0 - kc) & ~1;
      store_chunk(lds, par, st, ra, rb);
      __syncthreads();
      k0 += MX_BK;
    }
    if (!bad) {
      bad = unfit(lds, par);
      if (!bad) {
        compute(lds + par * BUF, kbeg, acc);
        return K;
      }
    }
    return k0 - MX_BK;
  }

  // The accumulators as values, in the integer tile's layout: a wave holds the
  // same (32 NI) x (32 NJ) cells in both, so they change lanes through a part
  // of LDS that is its own, 32 rows at a time.
  __device__ static __forceinline__ void hand_over(const int (&acc)[NI][NJ][16], int32_t *lds,
                                                   int (&out)[4 * NI][4 * NJ]) {
    constexpr int W = 32 * NJ;  // cells of a row
    const int lane = threadIdx.x & 63;
    int32_t *own = lds + (threadIdx.x >> 6) * (32 * W);
    int32_t *to = own + (lane >> 5) * (4 * W) + (lane & 31);
    const int32_t *from = own + (lane >> 3) * W + (lane & 7) * 4;
#pragma unroll
    for (int i = 0; i < NI; i++) {
#pragma unroll
      for (int r = 0; r < 16; r++)
#pragma unroll
        for (int j = 0; j < NJ; j++) to[acc_row(r) * W + 32 * j] = value(acc[i][j][r]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int h = 0; h < NJ; h++) {
          const int4 v = *reinterpret_cast<const int4 *>(from + 8 * r * W + 32 * h);
          int *o = out[4 * i + r] + 4 * h;
          o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }

  // The k from `done` on with integer additions, on top of the accumulators.
  __device__ static __forceinline__ void finish(const int32_t *A, int64_t lda, const int32_t *B,
                                                int64_t ldb, int m_valid, int n_valid, int K,
                                                int flags, int32_t *lds, int done, bool have,
                                                int (&ha)[4 * NI], int (&hb)[4 * NJ],
                                                const int (&acc)[NI][NJ][16],
                                                int (&out)[4 * NI][4 * NJ]) {
    // a slower wave may still read a flag, which neither of these reaches
    static_assert(4 * 32 * 32 * NJ <= FLAG && Int::LDS_WORDS <= FLAG);
    if (done > 0) {
      hand_over(acc, lds, out);
      __syncthreads();  // the integer tile stages over it
    } else {
#pragma unroll
      for (int r = 0; r < 4 * NI; r++)
#pragma unroll
        for (int c = 0; c < 4 * NJ; c++) out[r][c] = kInf;
    }
    Int::fold(A + done, lda, B + (int64_t)done * ldb, ldb, m_valid, n_valid, K - done, flags, lds,
              PAIR && have && done == 0, ha, hb, out);
  }

  // Compute the tile, arguments as MpTile::run (m_valid, n_valid >= 1).  C
  // may alias A or B: every operand is read before the epilogue writes (the
  // last chunk's loads end before its barrier).
  // Integer additions, where needed, come after the matrix cores' epilogue and
  // from arguments that the compiler cannot relate to those used before (their
  // address space kept: flat loads cost the n = 4096 closure 3%), and the way
  // there is an int and not a bool: in any other form the accumulators, or the
  // registers that a function of its own would keep for its caller, went
  // through scratch memory, 85 KB a tile (n = 8192, all values past the digits,
  // 24.9 ms; 4096 x 65536 x 16 533 us).
  __device__ static __forceinline__ void run(const int32_t *A, int64_t lda, const int32_t *B,
                                             int64_t ldb, int32_t *C, int64_t ldc, int m_valid,
                                             int n_valid, int K, bool accumulate, int flags,
                                             int32_t *lds) {
    int acc[NI][NJ][16];
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][j][r] = 0x7F800000;  // above every sum: INF
    int done = 0, have = 0, ha[4 * NI], hb[4 * NJ];
    if (fits(lda, ldb, n_valid, K)) {
      have = n_valid == BN;
      done = product(A, lda, B, ldb, m_valid, n_valid, K, lds, acc, ha, hb);
    }
    if (done == K) store(C, ldc, m_valid, n_valid, accumulate, acc);
    mp_in_ptr a = (mp_in_ptr)A, b = (mp_in_ptr)B;
    mp_out_ptr c = (mp_out_ptr)C;
    asm volatile("" : "+s"(a), "+s"(lda), "+s"(b), "+s"(ldb), "+s"(c), "+s"(ldc));
    asm volatile("" : "+s"(m_valid), "+s"(n_valid), "+s"(K), "+s"(flags), "+s"(done));
    if (done < K) {
      int out[4 * NI][4 * NJ];
      finish((const int32_t *)a, lda, (const int32_t *)b, ldb, m_valid, n_valid, K, flags, lds, done,
             have != 0, ha, hb, acc, out);
      Int::store((int32_t *)c, ldc, m_valid, n_valid, accumulate, flags, out);
    }
  }

  // C = the accumulators' values, or the minimum with them.
  __device__ static __forceinline__ void store(int32_t *C, int64_t ldc, int m_valid, int n_valid,
                                               bool accumulate, const int (&acc)[NI][NJ][16]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = (wave >> 1) * (32 * NI) + (lane >> 5) * 4;
    const int col0 = (wave & 1) * (32 * NJ) + (lane & 31);
    const bool full = m_valid == BM && n_valid == BN;
#pragma unroll
    for (int i = 0; i < NI; i++) {
      int32_t *c = C + (int64_t)(row0 + 32 * i) * ldc + col0;
      if (full) {
        // the C words of a row of blocks are all loaded before any is
        // stored: the compiler must assume that a store changes later loads
        int o[NJ][16];
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
          for (int j = 0; j < NJ; j++) o[j][r] = kInf;  // no value is above it
        if (accumulate) {
#pragma unroll
          for (int r = 0; r < 16; r++)
#pragma unroll
            for (int j = 0; j < NJ; j++) o[j][r] = c[(int64_t)acc_row(r) * ldc + 32 * j];
        }
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
          for (int j = 0; j < NJ; j++)
            c[(int64_t)acc_row(r) * ldc + 32 * j] = imin(value(acc[i][j][r]), o[j][r]);
      } else {
        // as above, G rows of every block at a time, from addresses clamped to
        // the valid cells: a load, a store and the next load each waited for
        // the one before (the n = 2999 closure 1.88 -> 1.66 ms).  More at once
        // would take the larger tile's registers from its k loop (8192^3 10.9
        // -> 12.2 ms)
        constexpr int G = NI * NJ == 1 ? 16 : 4;
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += G) {
          int o[NJ][G];
          if (accumulate) {
#pragma unroll
            for (int r = 0; r < G; r++) {
              const int row = imin(row0 + 32 * i + acc_row(r0 + r), m_valid - 1);
#pragma unroll
              for (int j = 0; j < NJ; j++)
                o[j][r] = C[(int64_t)row * ldc + imin(col0 + 32 * j, n_valid - 1)];
            }
          }
#pragma unroll
          for (int r = 0; r < G; r++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
              if (row0 + 32 * i + acc_row(r0 + r) < m_valid && col0 + 32 * j < n_valid) {
                const int v = value(acc[i][j][r0 + r]);
                c[(int64_t)acc_row(r0 + r) * ldc + 32 * j] = accumulate ? imin(v, o[j][r]) : v;
              }
        }
      }
    }
  }
};

using MxBig = MxTile<2, 2>;    // 128 x 128
using MxSmall = MxTile<1, 1>;  // 64 x 64

}  // namespace fapk

#endif  // FAP_MFMA_TILE_H_
