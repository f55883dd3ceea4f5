/*
 * k_batched.hip -- thousands of small, uneven-size problems in ONE
 * persistent launch (no ATLAS counterpart: ATLAS has no batched interface;
 * each instance here follows the same algorithms as its single-problem
 * routines, src/lapack/ATL_potrfL.c:104-262, ATL_getrfC.c:46-361,
 * ATL_potrs.c:13-86, ATL_getrs.c:8-89, and GEMM's C = alpha op(A) op(B) +
 * beta C of interfaces/blas/C/src/cblas_dgemm.c:16-134).
 *
 * A persistent grid of workgroups takes work items from one atomic counter
 * in the order the host planned (largest first), so uneven sizes balance
 * themselves.  A factor+solve instance is one workgroup's work:
 *
 *   posv (lower Cholesky): left-looking, 32-column panels; the panel's
 *     32-row tiles, the right-hand sides among them, are accumulated from
 *     the finished columns on the matrix cores and multiplied by the diagonal
 *     block's inverse.
 *   gesv (LU, partial pivoting), orders up to 256: 32-column panels one row
 *     per thread in registers, the columns right of them and the right-hand
 *     sides in 16-column strips, each one wavefront's.  Larger orders: the
 *     (n-k) x NB panel lives in LDS while it is factored (workgroup arg-max
 *     per column, ties to the lower row, NaN never wins, like cblas_idamax),
 *     its interchanges are applied to the other columns, U12 is solved column
 *     by column and the trailing matrix is updated in 64 x 64 tiles.
 *
 * The GEMM work item is one 64 x 64 tile of one instance.
 */
#include <hip/hip_runtime.h>
#include <float.h>
#include <math.h>
#include <type_traits>
#include "kernels.h"
#include "lu_panel.h"
#include "chol_block.h"

namespace {

using namespace atlmx;

constexpr int NT = ATLMX_BATCH_ROWS;
constexpr int TS = 64;                 /* trailing-update / GEMM tile */
constexpr int MAXR = ATLMX_BATCH_MAXRHS;

/* ---------------------------------------------------------------------- */
/* Trailing updates on the matrix cores, one 64 x 64 tile per wavefront    */
/* ---------------------------------------------------------------------- */
/* C(tile) -= X Y^T for a 64 x 64 tile by one wavefront, K <= KMAX: X(r, k)
 * = X[r + k ldx], Y(c, k) = Y[c*ycs + k*yks] (NT:
 * ycs = 1, yks = ld; NN with Y = U^T: ycs = ld, yks = 1).  Operands go from
 * memory straight into the MFMA lanes (lane l: row or column l&15 of a
 * 16-block, k = 4s + (l>>4)), no LDS and no barrier, so the wavefronts of a
 * workgroup work on different tiles at once. */
template <typename T, int KMAX>
__device__ void wave_tile_update(T *C, long ldc, const T *X, long ldx, const T *Y, long ycs,
                                 long yks, int K, int mr, int mc) {
  typedef TMfma<T> MF;
  typedef typename MF::acc_t acc_t;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  acc_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < KMAX / 4; ++s) {
    const int k = 4 * s + lk;
    if (4 * s >= K) break;                        /* uniform */
    T a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * i + li;
      a[i] = (r < mr && k < K) ? X[(size_t)r + (size_t)k * ldx] : T(0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 16 * j + li;
      b[j] = (c < mc && k < K) ? Y[(size_t)c * ycs + (size_t)k * yks] : T(0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = MF::mma(a[i], b[j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rr = 16 * i + MF::drow(lane, r), cc = 16 * j + li;
        if (rr < mr && cc < mc) C[(size_t)cc * ldc + rr] -= acc[i][j][r];
      }
}

/* ---------------------------------------------------------------------- */
/* Triangular solve of one instance's right-hand side by one workgroup     */
/* ---------------------------------------------------------------------- */
/* op(A) X = X for the nrhs (<= MAXR) vectors of X in LDS (column r at
 * X + r n), A's triangle in global memory (lower: the stored triangle is
 * the lower one; trans: op(A) = A^T; unit: the diagonal is taken as 1).
 * Left-looking over blocks of SB rows in solve order (top first when
 * lower != trans), RCH right-hand sides at a time: the block's entries less
 * the solved entries' contributions (all four wavefronts, one pass over A
 * for the RCH vectors, then one barrier), then the SB x SB diagonal
 * triangle -- staged in LDS -- by wavefront 0 alone, one row per lane,
 * each solved value broadcast from its lane: no barrier per row.  s_blk
 * holds SB x (SB + 1), s_part 4 RCH SB elements. */
constexpr int SB = 32;
constexpr int RCH = 4;                             /* right-hand sides per pass */
constexpr int RCT = 2;                             /* the transposed GEMV's accumulator set */
constexpr int SOLVE_LDS = SB * (SB + 1) + 4 * RCH * SB;   /* s_blk and s_part */
template <typename T>
__device__ void wg_trsv(int n, int nrhs, const T *A, long lda, bool lower, bool trans, bool unit,
                        T *X, T *s_blk, T *s_part) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool fwd = lower != trans;
  const int nb = (n + SB - 1) / SB;
  for (int bs = 0; bs < nb; ++bs) {
    const int b = fwd ? bs : nb - 1 - bs;
    const int R0 = b * SB, rb = min(SB, n - R0);
    /* solved range: [0, R0) forward, [R0 + rb, n) backward */
    const int k0 = fwd ? 0 : R0 + rb, k1 = fwd ? R0 : n;
    __syncthreads();
    /* the diagonal block of op(A), [row][col] */
    for (int e = tid; e < SB * SB; e += NT) {
      const int i = e % SB, j = e / SB;
      T v = T(0);
      if (i < rb && j < rb && (fwd ? i >= j : i <= j))
        v = trans ? A[(size_t)(R0 + i) * lda + R0 + j] : A[(size_t)(R0 + j) * lda + R0 + i];
      s_blk[i * (SB + 1) + j] = v;
    }
    for (int rc = 0; rc < nrhs; rc += RCH) {
      if (rc > 0) __syncthreads();               /* wavefront 0 is done with s_part */
      if (!trans) {
        /* op(A)(i, k) = A[k lda + i]: thread (row l, chunk q) sums k = k0 + q, k0 + q + 8, ...;
         * the two chunks of a wavefront are added by a lane exchange */
        constexpr int ST = NT / SB, U = 8;       /* stride, loads in flight */
        const int l = tid & (SB - 1), q = tid / SB;
        T part[RCH];
#pragma unroll
        for (int r = 0; r < RCH; ++r) part[r] = T(0);
        if (l < rb) {
          int k = k0 + q;
          for (; k + (U - 1) * ST < k1; k += U * ST) {
            T a[U];
#pragma unroll
            for (int u = 0; u < U; ++u) a[u] = A[(size_t)(k + u * ST) * lda + R0 + l];
#pragma unroll
            for (int r = 0; r < RCH; ++r)
              if (rc + r < nrhs)
#pragma unroll
                for (int u = 0; u < U; ++u) part[r] += a[u] * X[(size_t)(rc + r) * n + k + u * ST];
          }
          for (; k < k1; k += ST) {
            const T a = A[(size_t)k * lda + R0 + l];
#pragma unroll
            for (int r = 0; r < RCH; ++r)
              if (rc + r < nrhs) part[r] += a * X[(size_t)(rc + r) * n + k];
          }
        }
#pragma unroll
        for (int r = 0; r < RCH; ++r) {
          const T v = part[r] + __shfl_xor(part[r], 32);
          if (lane < 32) s_part[(r * 4 + wave) * SB + l] = v;
        }
      } else {
        /* op(A)(i, k) = A[i lda + k]: wavefront w takes rows w, w + 4, ...,
         * lanes run along k, all loads of a step issued together */
        constexpr int RW = SB / (NT / 64);
        for (int rt = 0; rt < RCH && rc + rt < nrhs; rt += RCT) {
          T part[RW][RCT];
#pragma unroll
          for (int m = 0; m < RW; ++m)
#pragma unroll
            for (int r = 0; r < RCT; ++r) part[m][r] = T(0);
          for (int k = k0 + lane; k < k1; k += 64) {
            T a[RW];
#pragma unroll
            for (int m = 0; m < RW; ++m) {
              const int l = wave + m * (NT / 64);
              a[m] = l < rb ? A[(size_t)(R0 + l) * lda + k] : T(0);
            }
#pragma unroll
            for (int r = 0; r < RCT; ++r)
              if (rc + rt + r < nrhs) {
                const T xk = X[(size_t)(rc + rt + r) * n + k];
#pragma unroll
                for (int m = 0; m < RW; ++m) part[m][r] += a[m] * xk;
              }
          }
#pragma unroll
          for (int m = 0; m < RW; ++m)
#pragma unroll
            for (int r = 0; r < RCT; ++r) {
              T v = part[m][r];
              for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
              if (lane == 0) s_part[((rt + r) * 4) * SB + wave + m * (NT / 64)] = v;
            }
        }
      }
      __syncthreads();
      if (wave == 0) {
        T c[RCH];
#pragma unroll
        for (int r = 0; r < RCH; ++r) {
          c[r] = T(0);
          if (rc + r < nrhs && lane < rb) {
            T sum = s_part[(r * 4) * SB + lane];
            if (!trans)
              for (int w = 1; w < NT / 64; ++w) sum += s_part[(r * 4 + w) * SB + lane];
            c[r] = X[(size_t)(rc + r) * n + R0 + lane] - sum;
          }
        }
        for (int s = 0; s < SB; ++s) {
          const int j = fwd ? s : SB - 1 - s;
          if (j < rb) {
            const T dj = unit ? T(1) : s_blk[j * (SB + 1) + j];
            const T lj = (lane < rb && (fwd ? (lane > j) : (lane < j)))
                             ? s_blk[lane * (SB + 1) + j] : T(0);
#pragma unroll
            for (int r = 0; r < RCH; ++r) {
              if (rc + r < nrhs) {
                if (lane == j) c[r] /= dj;
                const T xj = __shfl(c[r], j);
                c[r] -= lj * xj;
              }
            }
          }
        }
        if (lane < rb)
#pragma unroll
          for (int r = 0; r < RCH; ++r)
            if (rc + r < nrhs) X[(size_t)(rc + r) * n + R0 + lane] = c[r];
      }
    }
  }
  __syncthreads();
}

/* g / d from rd = 1 / d, d and rd both normal numbers: the product and one
 * correction round like the division (the product alone: 3% on a small
 * solve's error), in a chain half as long */
template <typename T>
__device__ __forceinline__ T quotient(T g, T d, T rd) {
  const T q = g * rd, c = fma(fma(-q, d, g), rd, q);
  return __builtin_isfinite(c) ? c : q;
}

/* ---------------------------------------------------------------------- */
/* Cholesky factor + solve of one instance by one workgroup                */
/* ---------------------------------------------------------------------- */
/* Left-looking in panels of PB = 32 columns.  Panel k's 32 x 32 row tiles
 * are each one wavefront's: A's tile less L(rows, 0:k) L(k.., 0:k)^T on the
 * matrix cores from the finished columns, then times the diagonal block's
 * inverse (tile_times_inv: refined where the block is not well conditioned),
 * and written once -- no tile of the trailing matrix is read and written again
 * for every panel, as the right-looking form did.  The right-hand sides are
 * one more row tile, [A; B^T], so the forward substitution costs no pass of
 * its own.  Products are formed transposed (D[column][row]): a lane's 16
 * neighbours run down a column of A, and an accumulator is itself the operand
 * of the product with the inverse (its element e on lane group g is the k
 * index drow(e) there).
 *
 * What bounds an instance is the chain of panels: the diagonal tile (its
 * sum split over the four wavefronts), its factor and inverse by wavefront 0
 * alone, then the tiles below; the other wavefronts accumulate their first
 * tile meanwhile, and two workgroups share a compute unit (three in FP32).
 * Panels of 64 columns, which read the finished columns half as often, were
 * no faster (4000 of order 8..512: 3.02 against 2.85 ms).  FP64, 4000
 * instances of order 8..512, one right-hand side, with the inputs' copies:
 * 15.8 -> 3.95 ms; 512 of order 256 with 8: 2.17 -> 0.31 ms.
 *
 * Rounding: 16 products at a time (8 in the diagonal tile) are summed apart
 * and subtracted from A's entry; subtracted one by one, every product would
 * round at the entry's size, and in one sum over all columns at the size it
 * had before any.  FP32 factors of order 512: 1.1e-7 off, 6.1e-8 off, and
 * 4.9e-8 so (updates 16 or 32 columns at a time with substitutions: 7.1e-8);
 * eigenvalues from 1 to 1e-3, order 256: a residual of 1.92 u in one sum,
 * 1.07 u so, 1.41 u with the updates. */
/* s_blk: 4 blocks of PB x PLD elements, or 2 where LDS is short (split =
 * false: then wavefront 0 sums the diagonal tile alone); s_x: n x nrhs;
 * s_ctl: 4 */
template <typename T>
__device__ void wg_posv(int n, T *A, const long lda0, int nrhs, T *B, long ldb, int *info,
                        T *s_blk, bool split, T *s_x, int *s_ctl) {
  typedef TMfma<T> MF;
  typedef typename MF::acc_t acc_t;
  constexpr int BLK = PB * PLD, UT = 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15;
  T *s_d = s_blk, *s_inv = s_blk + BLK;
  if (tid == 0) s_ctl[0] = s_ctl[2] = 0;
  for (int e = tid; e < n * nrhs; e += NT) s_x[e] = B[(size_t)(e / n) * ldb + e % n];
  __syncthreads();

  for (int k = 0; k < n; k += PB) {
    const int kb = min(PB, n - k), epoch = k / PB + 1;
    const long lda = fresh(lda0);
    const T *yp[2] = {A + min(k + li, n - 1), A + min(k + 16 + li, n - 1)};
    /* ---- the diagonal tile's sum, split over the wavefronts ---- */
    if (split || wave == 0) {
      acc_t acc[2][2];
      zero_tile(acc);
      const int w = split ? k / 4 : k;             /* a multiple of 8 */
      panel_acc<T, 2, 2, 2, ADD>(acc, yp, lda, yp, lda, wave * w, wave * w + w);
      T *sp = s_blk + wave * BLK;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sp[(16 * c + MF::drow(lane, e)) * PLD + 16 * r + li] = acc[c][r][e];
    }
    __syncthreads();
    for (int e = tid; e < PB * PB; e += NT) {
      const int c = e / PB, r = e % PB;
      T *o = s_blk + c * PLD + r;
      T v = r == c ? T(1) : T(0);                  /* beyond the matrix: the identity */
      if (r < kb && c < kb && r >= c) {
        T sum = *o;
        if (split) sum = (sum + o[BLK]) + (o[2 * BLK] + o[3 * BLK]);
        v = A[(size_t)(k + c) * lda + k + r] - sum;
      }
      *o = v;
    }
    if (tid == 0) s_ctl[1] = 1;                    /* the next row tile to take */
    __syncthreads();

    if (wave == 0) {
      T v[PB];
      bool refine;
      const int fail = block_factor(v, s_d, kb, refine);
      const long lda = fresh(lda0);
      const int ln = fresh_lane();
      if (!fail && ln < kb) {
#pragma unroll
        for (int c = 0; c < PB; ++c)
          if (c <= ln) A[(size_t)(k + c) * lda + k + ln] = v[c];
      }
      /* the rows' lanes L over the block, the columns' the inverse */
      T *dst = ln < PB ? s_d + ln : s_inv + (ln - PB) * PLD;
      const int step = ln < PB ? PLD : 1;
#pragma unroll
      for (int c = 0; c < PB; ++c) dst[c * step] = ln < c ? T(0) : v[c];
      if (ln == 0) {
        if (fail) s_ctl[2] = k + fail;
        s_ctl[3] = refine;
        __hip_atomic_store(&s_ctl[0], epoch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    /* ---- the row tiles below, and last the right-hand sides' tile; a
     * wavefront waits for the inverse (wavefront 0 always gets there) only
     * with its sum complete ---- */
    const int nt = (n - k + PB - 1) / PB, ntile = nt + (nrhs > 0 ? 1 : 0);
    for (;;) {
      int t = 0;
      if (lane == 0) t = atomicAdd(&s_ctl[1], 1);
      t = __builtin_amdgcn_readfirstlane(t);
      if (t >= ntile) break;
      const long lda = fresh(lda0);
      if (t < nt) {
        const int r0 = k + t * PB;                 /* then kb == PB */
        const int ra = r0 + li, rb = ra + 16;
        const T *xp[2] = {A + min(ra, n - 1), A + min(rb, n - 1)};
        acc_t w[2][2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[c][r][e] = xp[r][(size_t)(k + 16 * c + MF::drow(lane, e)) * lda];
        panel_acc<T, 2, 2, UT, SUBTRACT>(w, yp, lda, xp, lda, 0, k);
        while (__hip_atomic_load(&s_ctl[0], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < epoch)
          __builtin_amdgcn_s_sleep(1);
        if (s_ctl[2]) continue;
        tile_times_inv<T, 2>(w, s_inv, s_d, s_ctl[3]);
        const long ldc = fresh(lda0);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            T *col = A + (size_t)(k + 16 * c + MF::drow(lane, e)) * ldc;
            if (ra < n) col[ra] = w[c][0][e];
            if (rb < n) col[rb] = w[c][1][e];
          }
      } else {
        const T *xp[1] = {s_x + (size_t)min(li, nrhs - 1) * n};
        acc_t w[2][1];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = 16 * c + MF::drow(lane, e);
            w[c][0][e] = j < kb ? xp[0][k + j] : T(0);
          }
        panel_acc<T, 2, 1, UT, SUBTRACT>(w, yp, lda, xp, 1, 0, k);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e)              /* beyond the matrix: its last row again */
            if (16 * c + MF::drow(lane, e) >= kb) w[c][0][e] = T(0);
        while (__hip_atomic_load(&s_ctl[0], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < epoch)
          __builtin_amdgcn_s_sleep(1);
        if (s_ctl[2]) continue;
        tile_times_inv<T, 1>(w, s_inv, s_d, s_ctl[3]);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = 16 * c + MF::drow(lane, e);
            if (j < kb && li < nrhs) s_x[(size_t)li * n + k + j] = w[c][0][e];
          }
      }
    }
    __syncthreads();
    if (s_ctl[2]) {
      if (tid == 0) *info = s_ctl[2];
      return;                               /* ATL_potrfL.c:238-240: stop */
    }
  }
  if (tid == 0) *info = 0;
  if (nrhs <= 0) return;

  /* ---- L^T x = y, blocks from the last: the rows below block k
   * contribute L(r, c) x(r), split over the wavefronts by 16 rows (lane
   * group lk takes rows 4 lk + s at step s: four neighbours in memory); then
   * the 32 x 32 triangle, one unknown per lane, wavefront w solving
   * right-hand side w in lanes 0..31 and w + 4 in lanes 32..63 ---- */
  for (int k = (n - 1) / PB * PB; k >= 0; k -= PB) {
    const long lda = fresh(lda0);
    const int kb = min(PB, n - k), lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
    const int ln = lane & (PB - 1), rhs = wave + 4 * (lane / PB);
    T lc[PB], d = T(1);                            /* a square root: 1 / d is normal */
    if (wave < nrhs) {
#pragma unroll
      for (int j = 0; j < PB; ++j)
        lc[j] = (ln < j && j < kb) ? A[(size_t)(k + ln) * lda + k + j] : T(0);
      if (ln < kb) d = A[(size_t)(k + ln) * lda + k + ln];
    }
    const T rd = T(1) / d;
    acc_t acc[2] = {acc_t{0, 0, 0, 0}, acc_t{0, 0, 0, 0}};
    const T *xr = s_x + (size_t)min(li, nrhs - 1) * n;
    for (int r0 = k + PB + 16 * wave; r0 < n; r0 += 16 * (NT / 64)) {
      T a[2][4], b[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int r = r0 + 4 * lk + s, rr = min(r, n - 1);
        a[0][s] = A[(size_t)(k + li) * lda + rr];
        a[1][s] = A[(size_t)(k + 16 + li) * lda + rr];
        b[s] = r < n ? xr[r] : T(0);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        acc[0] = MF::mma(a[0][s], b[s], acc[0]);
        acc[1] = MF::mma(a[1][s], b[s], acc[1]);
      }
    }
    if (li < nrhs) {
      T *sp = s_blk + wave * MAXR * PB;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) sp[li * PB + 16 * c + MF::drow(lane, e)] = acc[c][e];
    }
    __syncthreads();
    if (wave < nrhs) {
      T g = T(0);
      if (rhs < nrhs && ln < kb) {
        const T *sp = s_blk + rhs * PB + ln;
        g = s_x[(size_t)rhs * n + k + ln] -
            ((sp[0] + sp[MAXR * PB]) + (sp[2 * MAXR * PB] + sp[3 * MAXR * PB]));
      }
#pragma unroll
      for (int j = PB - 1; j >= 0; --j) {          /* steps past kb change nothing */
        const T x = quotient(g, d, rd);            /* lane j's is x_j */
        T xj = bcast(x, j);
        if (nrhs > 4) xj = lane < PB ? xj : bcast(x, PB + j);
        g = ln == j ? x : fma(-lc[j], xj, g);
      }
      if (rhs < nrhs && ln < kb) s_x[(size_t)rhs * n + k + ln] = g;
    }
    __syncthreads();
  }
  for (int e = tid; e < n * nrhs; e += NT) B[(size_t)(e / n) * ldb + e % n] = s_x[e];
}

/* ---------------------------------------------------------------------- */
/* LU (partial pivoting) factor + solve of one instance by one workgroup   */
/* ---------------------------------------------------------------------- */
template <typename T, int NB>
__device__ void wg_gesv(int n, T *A, long lda, int *ipiv, int nrhs, T *B, long ldb, int *info,
                        T *s_p, T *s_t, T *s_x, T *s_v, int *s_i, bool trans) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int first0 = 0;                          /* first exactly-zero pivot, 1-based */
  for (int k = 0; k < n; k += NB) {
    const int kb = min(NB, n - k), mp = n - k;
    /* ---- panel rows k..n-1, columns k..k+kb-1 into LDS (s_p[c*mp + r]) ---- */
    __syncthreads();
    for (int e = tid; e < mp * kb; e += NT) {
      const int r = e % mp, c = e / mp;
      s_p[c * mp + r] = A[(size_t)(k + c) * lda + k + r];
    }
    __syncthreads();
    for (int j = 0; j < kb; ++j) {
      /* arg-max |p(r, j)|, r >= j: first maximum, NaN never wins */
      T bv = T(-1);
      int bi = 0x7fffffff;
      for (int r = j + tid; r < mp; r += NT) {
        const T v = fabs(s_p[j * mp + r]);
        if (v > bv) { bv = v; bi = r; }
      }
      for (int off = 32; off > 0; off >>= 1) {
        const T ov = __shfl_xor(bv, off);
        const int oi = __shfl_xor(bi, off);
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
      }
      if (lane == 0) { s_v[wave] = bv; s_i[wave] = bi; }
      __syncthreads();
      if (tid == 0) {
        T v = s_v[0];
        int p = s_i[0];
        for (int q = 1; q < NT / 64; ++q)
          if (s_v[q] > v || (s_v[q] == v && s_i[q] < p)) { v = s_v[q]; p = s_i[q]; }
        if (!(v > T(0))) p = j;            /* all zero/NaN: cblas_i?amax answers the first */
        s_i[4] = p;
      }
      __syncthreads();
      const int p = s_i[4];
      if (tid == 0) ipiv[k + j] = k + p;
      if (p != j && tid < kb) {
        const T t = s_p[tid * mp + j];
        s_p[tid * mp + j] = s_p[tid * mp + p];
        s_p[tid * mp + p] = t;
      }
      __syncthreads();
      const T piv = s_p[j * mp + j];
      if (piv == T(0)) {
        if (!first0) first0 = k + j + 1;          /* every thread: uniform control flow */
      } else {
        for (int r = j + 1 + tid; r < mp; r += NT) {
          const T l = s_p[j * mp + r] / piv;
          s_p[j * mp + r] = l;
          for (int c = j + 1; c < kb; ++c) s_p[c * mp + r] -= l * s_p[c * mp + j];
        }
      }
      __syncthreads();
    }
    for (int e = tid; e < mp * kb; e += NT) {
      const int r = e % mp, c = e / mp;
      A[(size_t)(k + c) * lda + k + r] = s_p[c * mp + r];
    }
    /* ---- the panel's interchanges on the other columns ---- */
    for (int c = tid; c < n; c += NT) {
      if (c >= k && c < k + kb) continue;
      T *col = A + (size_t)c * lda;
      for (int j = 0; j < kb; ++j) {
        const int p = ipiv[k + j];
        if (p != k + j) { const T t = col[k + j]; col[k + j] = col[p]; col[p] = t; }
      }
    }
    __syncthreads();
    /* ---- U12 = L11^{-1} A12, one column per thread ---- */
    for (int c = k + kb + tid; c < n; c += NT) {
      T x[NB];
#pragma unroll
      for (int r = 0; r < NB; ++r) x[r] = (r < kb) ? A[(size_t)c * lda + k + r] : T(0);
#pragma unroll
      for (int r = 0; r < NB; ++r) {
        if (r < kb) {
          T v = x[r];
#pragma unroll
          for (int l = 0; l < r; ++l) v -= s_p[l * mp + r] * x[l];
          x[r] = v;
        }
      }
#pragma unroll
      for (int r = 0; r < NB; ++r)
        if (r < kb) A[(size_t)c * lda + k + r] = x[r];
    }
    __syncthreads();
    /* ---- A22 -= L21 U12 ---- */
    const int m0 = k + kb, m = n - m0;
    const int nt = (m + TS - 1) / TS;
    for (int t = wave; t < nt * nt; t += NT / 64) {
      const int ti = t % nt, tj = t / nt;         /* wavefront w takes every fourth tile */
      const int r0 = m0 + ti * TS, c0 = m0 + tj * TS;
      wave_tile_update<T, NB>(A + (size_t)c0 * lda + r0, lda, A + (size_t)k * lda + r0, lda,
                              A + (size_t)c0 * lda + k, lda, 1, kb, min(TS, n - r0),
                              min(TS, n - c0));
    }
  }
  if (tid == 0) *info = first0;
  if (nrhs <= 0 || first0) return;
  /* ---- getrs in LDS (ATL_getrs.c:8-89): NoTrans: P b, L y = b (unit),
   * U x = y; Trans (A^T = U^T L^T P): U^T z = b, L^T w = z (unit), x = P^T w.
   * The triangular solves stage through s_t ---- */
  __syncthreads();
  for (int e = tid; e < n * nrhs; e += NT) s_x[e] = B[(size_t)(e / n) * ldb + e % n];
  __syncthreads();
  if (!trans && tid < nrhs) {
    for (int j = 0; j < n; ++j) {
      const int p = ipiv[j];
      if (p != j) { const T t = s_x[tid * n + j]; s_x[tid * n + j] = s_x[tid * n + p]; s_x[tid * n + p] = t; }
    }
  }
  if (!trans) {
    wg_trsv(n, nrhs, A, lda, true, false, true, s_x, s_t, s_t + SB * (SB + 1));
    wg_trsv(n, nrhs, A, lda, false, false, false, s_x, s_t, s_t + SB * (SB + 1));
  } else {
    wg_trsv(n, nrhs, A, lda, false, true, false, s_x, s_t, s_t + SB * (SB + 1));
    wg_trsv(n, nrhs, A, lda, true, true, true, s_x, s_t, s_t + SB * (SB + 1));
  }
  if (trans && tid < nrhs) {                 /* x = P^T w: the swaps in reverse */
    for (int j = n - 1; j >= 0; --j) {
      const int p = ipiv[j];
      if (p != j) { const T t = s_x[tid * n + j]; s_x[tid * n + j] = s_x[tid * n + p]; s_x[tid * n + p] = t; }
    }
  }
  __syncthreads();
  for (int e = tid; e < n * nrhs; e += NT) B[(size_t)(e / n) * ldb + e % n] = s_x[e];
}

/* ---------------------------------------------------------------------- */
/* LU factor + solve of one instance of order <= NT: one panel row a thread */
/* ---------------------------------------------------------------------- */
/* Right-looking, panels of PB = 32 columns held in registers, one row per
 * thread (lu_panel.h), as two halves of 16: after the first the top 16 rows'
 * second half is solved for by one wavefront and every row below takes its
 * products.  The columns right of the panel are taken in strips of 16, each
 * wholly one wavefront's, so a strip's steps need no barrier: gather the 32
 * rows that come to the top, put the displaced top rows where those came
 * from, U12 by substitution in groups of four rows, and the trailing rows -=
 * L21 U12, products on the matrix cores formed transposed (D[column][row]: a
 * lane's 16 neighbours run down a column of A; the U12 accumulators are the
 * operand of the update as they stand).  The right-hand sides are one more
 * strip, in LDS, so the forward substitution costs no pass of its own.  The
 * columns left of a panel get their interchanges once at the end, as one map
 * per panel composed from the later panels' maps.
 *
 * Rounding: multipliers are divisions, the only inverses those of 4 x 4
 * blocks, and products are summed apart, eight to sixteen at a time, before
 * they meet an entry.  FP32, mean residual of the factors of order 32 / 100
 * / 256: 1.32e-7 / 3.08e-7 / 6.5e-7 (LDS panels of 16 or 32 with
 * substitutions, as above order 256: 1.32 / 3.17 / 7.4; reciprocals,
 * panels of 32 and products with inv(L11): 1.41 / 4.30 / 9.2).
 *
 * Bound by the panel's chain (about 1 us a column, two workgroups to a
 * compute unit hiding each other's); the form it replaces at these orders kept
 * the panel in LDS, swapped rows one dependent load at a time in every
 * column, and updated through uncoalesced tiles.  FP64, 4000 of order
 * 8..256, one right-hand side, with the inputs' copies: 9.5 -> 2.9 ms. */
constexpr int MAXPAN = NT / PB;

template <typename T>
struct RowsPanel {
  static constexpr bool DIVIDE = true;
  int w, row0;
  int *ipiv;
  T *s_prow, *s_cand;
  atlmx::u64 *s_key;
  int *s_pos, *s_piv, *s_zero;
  __device__ bool first() const { return true; }
  __device__ void zero_pivot(int C) const { if (*s_zero == 0) *s_zero = row0 + C + 1; }
};

/* The strict part of inv(D) for each 4 x 4 diagonal block D of L11 (unit
 * lower, at s_l[c PLD + r]): row r's four entries at s_n[4 r].  Thread 4 e +
 * c of the first 32 forms column c of block e. */
template <typename T>
__device__ __forceinline__ void unit_lower_inverse4(const T *s_l, T *s_n) {
  const int r0 = (int)threadIdx.x & ~3, k = (int)threadIdx.x & 3;
  T z[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) z[c] = c == k ? T(1) : T(0);
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int c = j + 1; c < 4; ++c) z[c] = fma(-s_l[(r0 + j) * PLD + r0 + c], z[j], z[c]);
#pragma unroll
  for (int c = 0; c < 4; ++c) s_n[4 * (r0 + c) + k] = c > k ? z[c] : T(0);
}

/* An MFMA's 16 rows by the group of four that element e of the accumulators
 * holds: lane group g's element e is row 4 e + g of a tile whose operand
 * row i is row mfma_row(i). */
template <typename T> __device__ __forceinline__ int mfma_row(int i);
template <> __device__ __forceinline__ int mfma_row<double>(int i) { return i; }
template <> __device__ __forceinline__ int mfma_row<float>(int i) { return 4 * (i & 3) + (i >> 2); }

template <typename T>
struct GesvLds {
  T *l11, *inv;            /* PB x PLD; 16 x 16 */
  T *part;                 /* 4 x MAXR x PB */
  T *x;                    /* n x nrhs */
  int *src, *dst;          /* PB each: row now at top j; where top row j went (-1: stays) */
  unsigned char *map;      /* MAXPAN x NT: row -> position, relative to the panel */
  unsigned char *fin;      /* NT */
};

template <typename T>
__device__ void wg_gesv_rows(int n, T *A, const long lda0, int *ipiv, int nrhs, T *B, long ldb,
                             int *info, const GesvLds<T> &S, RowsPanel<T> st, bool trans) {
  typedef TMfma<T> MF;
  typedef typename MF::acc_t acc_t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4, mr = mfma_row<T>(li);
  const int nr_fwd = trans ? 0 : nrhs;             /* right-hand sides carried along */
  if (tid == 0) *st.s_zero = 0;
  for (int e = tid; e < n * nrhs; e += NT) S.x[e] = B[(size_t)(e / n) * ldb + e % n];
  __syncthreads();

  for (int k = 0; k < n; k += PB) {
    const int kb = min(PB, n - k), mp = n - k;
    const long lda = fresh(lda0);
    /* ---- the panel, 16 columns and then 16 ---- */
    T a[16], b[16];
    int pos = tid < mp ? tid : -1;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      a[c] = (c < kb && tid < mp) ? A[(size_t)(k + c) * lda + k + tid] : T(0);
      b[c] = (16 + c < kb && tid < mp) ? A[(size_t)(k + 16 + c) * lda + k + tid] : T(0);
    }
    st.w = min(kb, 16); st.row0 = k; st.ipiv = ipiv + k;
    atlmx::panel_segment<T, NT, 16, 16, false>(st, a, pos);
    if (kb > 16) {
      T *s_u = S.inv;                              /* the first pivot rows' second half */
      if (pos >= 0 && pos < 16)
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          s_u[16 * pos + c] = b[c];
          S.l11[c * PLD + pos] = c < pos ? a[c] : T(0);
        }
      __syncthreads();
      if (wave == 0) {
        /* a column per lane, row j in x[0] at step j; the next step's
         * multipliers are on their way during a step (rows past 15: unused) */
        T x[16], lc[15], ln[15];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = s_u[16 * r + li];
#pragma unroll
        for (int r = 1; r < 16; ++r) ln[r - 1] = S.l11[r];
#pragma unroll 1
        for (int j = 0; j < 16; ++j) {
#pragma unroll
          for (int r = 1; r < 16; ++r) lc[r - 1] = ln[r - 1];
          const T *next = S.l11 + min(j + 1, 14) * (PLD + 1);
#pragma unroll
          for (int r = 1; r < 16; ++r) ln[r - 1] = next[r];
          const T x0 = x[0];
          if (lane < 16) s_u[16 * j + li] = x0;
#pragma unroll
          for (int r = 1; r < 16; ++r) x[r - 1] = fma(-lc[r - 1], x0, x[r]);
        }
      }
      __syncthreads();
      T sum[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) sum[c] = T(0);
#pragma unroll 1
      for (int j = 0; j < 16; j += 4) {            /* a[] comes round once */
        T l[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          T u[16], p = s_u[16 * (j + q) + li];
          asm volatile("" : "+v"(p));              /* one row's entries at a time */
          atlmx::row_spread<T, 0>(u, p);
          l[q] = a[q];
#pragma unroll
          for (int c = 0; c < 16; ++c) sum[c] = fma(l[q], u[c], sum[c]);
        }
#pragma unroll
        for (int c = 0; c < 12; ++c) a[c] = a[c + 4];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[12 + q] = l[q];
      }
#pragma unroll
      for (int c = 0; c < 16; ++c) b[c] = pos >= 16 ? b[c] - sum[c] : b[c];
      if (pos >= 0 && pos < 16)
#pragma unroll
        for (int c = 0; c < 16; ++c) b[c] = s_u[16 * pos + c];
      pos -= 16;                                   /* the top 16 rows, and no row, below zero */
      st.w = kb - 16; st.row0 = k + 16; st.ipiv = ipiv + k + 16;
      atlmx::panel_segment<T, NT, 16, 16, false>(st, b, pos);
      pos += 16;
    }
    if (tid < PB) S.dst[tid] = -1;
    __syncthreads();
    if (pos >= 0) {
      const long ldp = fresh(lda0);
#pragma unroll
      for (int c = 0; c < PB; ++c) {
        const T v = c < 16 ? a[c % 16] : b[c % 16];
        if (c < kb) A[(size_t)(k + c) * ldp + k + pos] = v;
        if (pos < PB) S.l11[c * PLD + pos] = (c < kb && c < pos) ? v : T(0);
      }
      S.map[(k / PB) * NT + tid] = (unsigned char)pos;
      if (pos < kb) S.src[pos] = tid;
      else if (tid < kb) S.dst[tid] = pos;
    } else if (tid < PB) {                         /* beyond the matrix: nothing below the diagonal */
#pragma unroll
      for (int c = 0; c < PB; ++c) S.l11[c * PLD + tid] = T(0);
    }
    if (tid >= kb && tid < PB) S.src[tid] = 0;
    __syncthreads();
    const int ns = (n - k - kb + 15) / 16;         /* strips of A's columns */
    if (ns == 0 && nr_fwd == 0) break;
    if (tid < PB) unit_lower_inverse4(S.l11, S.inv);
    __syncthreads();

    /* ---- strips: columns j0.. of A, then the right-hand sides.  cp(c) is
     * column c's base; clamped columns are read but not written. ---- */
    auto strip = [&](auto cp, int nc) {
      acc_t xv[2], tv[2], u[2], sum[2] = {acc_t{0, 0, 0, 0}, acc_t{0, 0, 0, 0}};
#pragma unroll
      for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 16 * l + 4 * e + lk;
          auto col = cp(min(li, nc - 1));
          xv[l][e] = j < kb ? col[k + S.src[j]] : T(0);
          tv[l][e] = j < kb ? col[k + j] : T(0);
        }
      /* U12: four rows at a time, in element e of each lane group one: the
       * gathered rows less the sum so far, times the block's inverse; then
       * their products join the later rows' sums */
#pragma unroll
      for (int l = 0; l < 2; ++l) {
        const T nv = S.inv[4 * (16 * l + mr) + lk];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const T x = xv[l][e] + sum[l][e];
          const acc_t z = MF::mma((mr >> 2) == e ? nv : T(0), x, acc_t{0, 0, 0, 0});
          u[l][e] = x + z[e];
          const T *Lc = S.l11 + (16 * l + 4 * e + lk) * PLD + mr;
          if (e < 3) sum[l] = MF::mma((mr >> 2) > e ? -Lc[16 * l] : T(0), u[l][e], sum[l]);
          if (l == 0) sum[1] = MF::mma(-Lc[16], u[0][e], sum[1]);
        }
      }
      /* the inverse's zeros times an infinity or a NaN would reach up to
       * three rows above it: then row by row, below it alone */
      bool odd = false;
#pragma unroll
      for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int e = 0; e < 4; ++e) odd |= !__builtin_isfinite(u[l][e]);
      if (__ballot(odd)) {
        const int ln = fresh_lane(), c = ln & 15, g = ln >> 4;
        auto col = cp(min(c, nc - 1));
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = 16 * l + 4 * e + g;
            u[l][e] = j < kb ? col[k + S.src[j]] : T(0);
          }
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll 1
            for (int q = 0; q < 4; ++q) {          /* row j, from lane group q */
              const int j = 16 * l + 4 * e + q;
              const T uj = __shfl(u[l][e], 16 * q + c);
              const T *Lc = S.l11 + j * PLD + g;
#pragma unroll
              for (int r = 4 * l + e; r < 8; ++r) {
                const T v = fma(-Lc[4 * r], uj, u[r / 4][r % 4]);
                u[r / 4][r % 4] = 4 * r + g > j ? v : u[r / 4][r % 4];
              }
            }
      }
      __threadfence_block();                       /* every read above is done */
      if (li < nc) {
        auto col = cp(li);
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int j = 16 * l + 4 * e + lk;
            if (j < kb) {
              const int d = S.dst[j];
              if (d >= 0) col[k + d] = tv[l][e];
              col[k + j] = u[l][e];
            }
          }
      }
      __threadfence_block();                       /* the displaced rows are read below */
      /* the rows below: D'[col][row] = sum over j of U(j, col) L21(row, j) */
      for (int r0 = k + PB; r0 < n; r0 += 32) {    /* then kb == PB */
        const int ra = min(r0 + li, n - 1), rb = min(r0 + 16 + li, n - 1);
        acc_t d0[4], d1[4], c0, c1;                /* sums of eight products each */
        T b0[2][4], b1[2][4];
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const T *Lc = A + (size_t)(k + 16 * l + 4 * e + lk) * lda;
            b0[l][e] = Lc[ra];
            b1[l][e] = Lc[rb];
          }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          auto col = cp(min(MF::drow(lane, e), nc - 1));
          c0[e] = col[ra];
          c1[e] = col[rb];
        }
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int h = 2 * l + e / 2;
            d0[h] = MF::mma(u[l][e], b0[l][e], e & 1 ? d0[h] : acc_t{0, 0, 0, 0});
            d1[h] = MF::mma(u[l][e], b1[l][e], e & 1 ? d1[h] : acc_t{0, 0, 0, 0});
          }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          c0 -= d0[h];
          c1 -= d1[h];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = MF::drow(lane, e);
          if (c < nc) {
            auto col = cp(c);
            if (r0 + li < n) col[ra] = c0[e];
            if (r0 + 16 + li < n) col[rb] = c1[e];
          }
        }
      }
    };
    for (int q = wave; q < ns; q += NT / 64) {
      const int j0 = k + kb + 16 * q;
      T *base = A + (size_t)j0 * lda;
      strip([=](int c) { return base + (size_t)c * lda; }, min(16, n - j0));
    }
    if (nr_fwd > 0 && wave == (ns & 3)) {
      T *xs = S.x;
      strip([=](int c) { return xs + c * n; }, nr_fwd);
    }
    __syncthreads();
  }

  /* ---- the interchanges of the columns left of each panel: fin[i] = where
   * the row at absolute index i ends, composed from the last panel back ---- */
  {
    const int np = (n + PB - 1) / PB;
    if (tid < n) S.fin[tid] = (unsigned char)tid;
    for (int q = np - 2; q >= 0; --q) {
      const int k1 = (q + 1) * PB;                 /* the panel whose map enters now */
      __syncthreads();
      int f = 0;
      if (tid >= k1 && tid < n) f = S.fin[k1 + S.map[(q + 1) * NT + tid - k1]];
      __syncthreads();
      if (tid >= k1 && tid < n) S.fin[tid] = (unsigned char)f;
      const bool moved = tid >= k1 && tid < n && f != tid;
      const long lda = fresh(lda0);
      T v[PB];
      if (moved) {
#pragma unroll
        for (int c = 0; c < PB; ++c) v[c] = A[(size_t)(q * PB + c) * lda + tid];
      }
      __syncthreads();
      if (moved) {
#pragma unroll
        for (int c = 0; c < PB; ++c) A[(size_t)(q * PB + c) * lda + f] = v[c];
      }
    }
  }
  __syncthreads();
  const int first0 = *st.s_zero;
  if (tid == 0) *info = first0;
  if (nrhs <= 0 || first0) return;

  if (trans) {
    /* A^T = U^T L^T P: U^T z = b, L^T w = z (unit), x = P^T w */
    wg_trsv(n, nrhs, A, lda0, false, true, false, S.x, S.l11, S.part);
    wg_trsv(n, nrhs, A, lda0, true, true, true, S.x, S.l11, S.part);
    if (tid < nrhs)
      for (int j = n - 1; j >= 0; --j) {
        const int p = ipiv[j];
        if (p != j) { const T t = S.x[tid * n + j]; S.x[tid * n + j] = S.x[tid * n + p]; S.x[tid * n + p] = t; }
      }
    __syncthreads();
  } else {
    /* ---- U x = y, blocks from the last: the columns right of block k
     * contribute U(r, j) x(j), split over the wavefronts by 16 columns, then
     * the 32 x 32 triangle, one unknown per lane, wavefront w solving
     * right-hand side w in lanes 0..31 and w + 4 in lanes 32..63 ---- */
    for (int k = (n - 1) / PB * PB; k >= 0; k -= PB) {
      const long lda = fresh(lda0);
      const int kb = min(PB, n - k), lane = fresh_lane(), li = lane & 15, lk = lane >> 4;
      const int ln = lane & (PB - 1), rhs = wave + 4 * (lane / PB);
      T uc[PB], d = T(1);
      if (wave < nrhs) {
#pragma unroll
        for (int j = 0; j < PB; ++j)
          uc[j] = (ln < j && j < kb) ? A[(size_t)(k + j) * lda + k + ln] : T(0);
        if (ln < kb) d = A[(size_t)(k + ln) * lda + k + ln];
      }
      /* a pivot can be any nonzero number: where the reciprocal of one in the
       * block would over- or underflow, divide */
      const T rd = T(1) / d, ad = d < T(0) ? -d : d, lo = T(4) * Lim<T>::safmin();
      const bool plain = __ballot(!(ad >= lo && ad <= T(1) / lo)) == 0ull;
      acc_t acc[2][2];                             /* two sums: half the terms in each */
      zero_tile(acc);
      const T *xr = S.x + (size_t)min(li, nrhs - 1) * n;
      for (int j0 = k + PB + 16 * wave; j0 < n; j0 += 16 * (NT / 64)) {
        T ua[2][4], b[4];
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          const int j = j0 + 4 * s4 + lk;
          const T *col = A + (size_t)min(j, n - 1) * lda + k;
          ua[0][s4] = col[li];
          ua[1][s4] = col[16 + li];
          b[s4] = j < n ? xr[j] : T(0);
        }
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          acc[0][s4 / 2] = MF::mma(ua[0][s4], b[s4], acc[0][s4 / 2]);
          acc[1][s4 / 2] = MF::mma(ua[1][s4], b[s4], acc[1][s4 / 2]);
        }
      }
      if (li < nrhs) {
        T *sp = S.part + wave * MAXR * PB;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sp[li * PB + 16 * c + MF::drow(lane, e)] = acc[c][0][e] + acc[c][1][e];
      }
      __syncthreads();
      if (wave < nrhs) {
        T g = T(0);
        if (rhs < nrhs && ln < kb) {
          const T *sp = S.part + rhs * PB + ln;
          g = S.x[(size_t)rhs * n + k + ln] -
              ((sp[0] + sp[MAXR * PB]) + (sp[2 * MAXR * PB] + sp[3 * MAXR * PB]));
        }
        auto solve = [&](auto divide) {
#pragma unroll
          for (int j = PB - 1; j >= 0; --j) {      /* steps past kb change nothing */
            const T x = decltype(divide)::value ? g / d : quotient(g, d, rd);
            T xj = bcast(x, j);                    /* lane j's is x_j */
            if (nrhs > 4) xj = lane < PB ? xj : bcast(x, PB + j);
            g = ln == j ? x : fma(-uc[j], xj, g);
          }
        };
        if (plain) solve(std::false_type());
        else solve(std::true_type());
        if (rhs < nrhs && ln < kb) S.x[(size_t)rhs * n + k + ln] = g;
      }
      __syncthreads();
    }
  }
  for (int e = tid; e < n * nrhs; e += NT) B[(size_t)(e / n) * ldb + e % n] = S.x[e];
}

/* ---------------------------------------------------------------------- */
/* Cholesky adjoint of one instance by one workgroup                       */
/* ---------------------------------------------------------------------- */
/* Given L (lower triangle of A after potrf; its strict upper triangle is
 * overwritten with zeros here), X = A^{-1} B and Bb = A^{-1} Xb (the solve's
 * adjoint), write to G the gradient of <Xb, X> with respect to the lower
 * triangle of A (the entries potrf reads; strict upper part zero).  The
 * Cholesky adjoint (Murray, "Differentiation of the Cholesky decomposition",
 * 2016) of the solve's L-bar is
 *   Lb = -tril(M L),  M = Bb X^T + X Bb^T
 *   P  = Phi(L^T Lb)             (lower triangle, diagonal halved)
 *   S  = L^{-T} P L^{-1}         (two triangular solves)
 *   G  = tril(S + S^T) - diag(S) (off-diagonal entries count twice).
 * With U = L^T X and V = L^T Bb, M L = Bb U^T + X V^T.  An entry i >= j of
 * L^T Lb sums over k >= i >= j, where the tril of Lb masks nothing, so it is
 * -(V U^T + U V^T)(i, j): symmetric of rank 2 nrhs, and P + P^T is all of it.
 * The two solves applied to those factors give back L^{-T} V = Bb and
 * L^{-T} U = X, so
 *   S + S^T = -(Bb X^T + X Bb^T)
 * without forming the n x n intermediates: n^2 nrhs products and one write
 * of G instead of ~2 n^3 flops (FP64, 512 of order 256, 8 right-hand sides:
 * 6.7 -> 0.30 ms, bound by writing G and zeroing L's triangle), and
 * without the solves' rounding. */
constexpr int ADJ_CB = 4;                        /* columns of G at a time */
template <typename T>
__device__ void wg_chol_adjoint(int n, T *L, long lda, int nrhs, const T *Xs, const T *Bb,
                                long ldx, T *G, long ldg) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int j0 = ADJ_CB * wave; j0 < n; j0 += ADJ_CB * (NT / 64)) {
    for (int i = lane; i < n; i += 64) {
      T acc[ADJ_CB];
#pragma unroll
      for (int c = 0; c < ADJ_CB; ++c) acc[c] = T(0);
      if (i >= j0)
        for (int r = 0; r < nrhs; ++r) {
          const T bi = Bb[(size_t)r * ldx + i], xi = Xs[(size_t)r * ldx + i];
#pragma unroll
          for (int c = 0; c < ADJ_CB; ++c) {
            const int j = min(j0 + c, n - 1);
            const T bj = Bb[(size_t)r * ldx + j], xj = Xs[(size_t)r * ldx + j];
            acc[c] += i == j ? bi * xj : bi * xj + xi * bj;
          }
        }
#pragma unroll
      for (int c = 0; c < ADJ_CB; ++c) {
        const int j = j0 + c;
        if (j < n) {
          G[(size_t)j * ldg + i] = i >= j ? -acc[c] : T(0);
          if (i < j) L[(size_t)j * lda + i] = T(0);
        }
      }
    }
  }
}

template <typename T>
struct BatchArgs {
  int count;
  const int *order;              /* instance processing order */
  const int *n;
  T *const *A; const int *lda;
  int *const *ipiv;              /* gesv */
  int nrhs;
  T *const *B; const int *ldb;
  int *info;
  int *counter;                  /* zero on entry; left at count + grid */
};

template <typename T>
__global__ __launch_bounds__(NT, sizeof(T) == 8 ? 2 : 3) void posv_batched_kernel(
    BatchArgs<T> g, int blocks) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T *s_blk = (T *)smem;                                /* blocks x PB x PLD */
  T *s_x = s_blk + blocks * PB * PLD;                  /* n x nrhs */
  __shared__ int s_item, s_ctl[4];
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = atomicAdd(g.counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);   /* scalar: addresses too */
    if (it >= g.count) return;
    const int i = g.order[it];
    wg_posv<T>(g.n[i], g.A[i], g.lda[i], g.nrhs, g.B ? g.B[i] : nullptr, g.ldb ? g.ldb[i] : 1,
               &g.info[i], s_blk, blocks == 4, s_x, s_ctl);
  }
}

template <typename T, int NB>
__global__ __launch_bounds__(NT) void gesv_batched_kernel(BatchArgs<T> g, int maxn, int trans) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T *s_p = (T *)smem;                                  /* maxn x NB */
  T *s_t = s_p + (size_t)maxn * NB;                    /* the solves' staging */
  T *s_x = s_t + SOLVE_LDS;                            /* maxn x nrhs */
  __shared__ T s_v[4];
  __shared__ int s_i[5];
  __shared__ int s_item;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = atomicAdd(g.counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);   /* scalar: addresses too */
    if (it >= g.count) return;
    const int i = g.order[it];
    wg_gesv<T, NB>(g.n[i], g.A[i], g.lda[i], g.ipiv[i], g.nrhs, g.B ? g.B[i] : nullptr,
                   g.ldb ? g.ldb[i] : 1, &g.info[i], s_p, s_t, s_x, s_v, s_i, trans != 0);
  }
}

template <typename T>
__global__ __launch_bounds__(NT, 2) void gesv_rows_batched_kernel(BatchArgs<T> g, int trans) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ __attribute__((aligned(16))) T s_prow[PB];
  __shared__ atlmx::u64 s_key[NT / 64];
  __shared__ int s_pos[NT / 64], s_src[PB], s_dst[PB], s_piv, s_zero, s_item;
  __shared__ unsigned char s_map[MAXPAN * NT], s_fin[NT];
  GesvLds<T> S;
  S.l11 = (T *)smem;
  S.inv = S.l11 + PB * PLD;
  S.part = S.inv + 16 * 16;
  S.x = S.part + 4 * MAXR * PB;                        /* maxn x nrhs */
  S.src = s_src; S.dst = s_dst; S.map = s_map; S.fin = s_fin;
  RowsPanel<T> st;
  st.s_prow = st.s_cand = s_prow; st.s_key = s_key; st.s_pos = s_pos; st.s_piv = &s_piv;
  st.s_zero = &s_zero; st.w = st.row0 = 0; st.ipiv = nullptr;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = atomicAdd(g.counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);
    if (it >= g.count) return;
    const int i = g.order[it];
    wg_gesv_rows<T>(g.n[i], g.A[i], g.lda[i], g.ipiv[i], g.nrhs, g.B ? g.B[i] : nullptr,
                    g.ldb ? g.ldb[i] : 1, &g.info[i], S, st, trans != 0);
  }
}

/* ---------------------------------------------------------------------- */
/* variable-size batched GEMM: one work item = one 64 x 64 tile           */
/* ---------------------------------------------------------------------- */
template <typename T>
struct GemmBatchArgs {
  int count, ta, tb;
  const int *order;              /* instance order of the tile numbering */
  const int *m, *n, *k;
  T alpha, beta;
  const T *const *A; const int *lda;
  const T *const *B; const int *ldb;
  T *const *C; const int *ldc;
  const int *tile_start;         /* prefix sums of tiles per position in order (count + 1) */
  int *counter;
};

template <typename T>
__global__ __launch_bounds__(NT) void gemm_batched_kernel(GemmBatchArgs<T> g) {
  __shared__ T s_a[16 * TS], s_b[16 * TS];
  __shared__ int s_item;
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int total = g.tile_start[g.count];
  for (;;) {
    __syncthreads();
    if (tid == 0) s_item = atomicAdd(g.counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);   /* scalar: addresses too */
    if (it >= total) return;
    /* instance: the last i with tile_start[i] <= it */
    int lo = 0, hi = g.count - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (g.tile_start[mid] <= it) lo = mid; else hi = mid - 1;
    }
    const int i = g.order[lo], t = it - g.tile_start[lo];
    const int M = g.m[i], N = g.n[i], K = g.k[i];
    const int tm = (M + TS - 1) / TS;
    const int r0 = (t % tm) * TS, c0 = (t / tm) * TS;
    const T *A = g.A[i], *B = g.B[i];
    const long lda = g.lda[i], ldb = g.ldb[i], ldc = g.ldc[i];
    T acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = T(0);
    for (int k0 = 0; k0 < K; k0 += 16) {
      __syncthreads();
      for (int e = tid; e < 16 * TS; e += NT) {
        /* op(A)(r0+rr, k0+kk), op(B)(k0+kk, c0+cc) */
        int rr, kk;
        if (g.ta == KX_NOTRANS) { kk = e / TS; rr = e % TS; }
        else                    { rr = e / 16; kk = e % 16; }
        const int gr = r0 + rr, gk = k0 + kk;
        s_a[kk * TS + rr] = (gr < M && gk < K)
            ? (g.ta == KX_NOTRANS ? A[(size_t)gk * lda + gr] : A[(size_t)gr * lda + gk]) : T(0);
        int cc, k2;
        if (g.tb == KX_NOTRANS) { cc = e / 16; k2 = e % 16; }
        else                    { k2 = e / TS; cc = e % TS; }
        const int gc = c0 + cc, gk2 = k0 + k2;
        s_b[k2 * TS + cc] = (gc < N && gk2 < K)
            ? (g.tb == KX_NOTRANS ? B[(size_t)gc * ldb + gk2] : B[(size_t)gk2 * ldb + gc]) : T(0);
      }
      __syncthreads();
#pragma unroll 4
      for (int kk = 0; kk < 16; ++kk) {
        T a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = s_a[kk * TS + ty * 4 + q];
#pragma unroll
        for (int q = 0; q < 4; ++q) b[q] = s_b[kk * TS + tx * 4 + q];
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[p][q] += a[p] * b[q];
      }
    }
    T *C = g.C[i];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int r = r0 + ty * 4 + p, c = c0 + tx * 4 + q;
        if (r < M && c < N) {
          T *pc = C + (size_t)c * ldc + r;
          T v = g.alpha * acc[p][q];
          if (g.beta != T(0)) v += g.beta * *pc;
          *pc = v;
        }
      }
  }
}

template <typename T>
struct AdjArgs {
  int count, nrhs;
  const int *order, *n, *lda, *ldx, *ldg;
  T *const *L; T *const *X; T *const *Bb; T *const *G;
  /* L's strict upper triangle is zeroed */
  int *counter;
};

template <typename T>
__global__ __launch_bounds__(NT) void chol_adjoint_kernel(AdjArgs<T> g) {
  __shared__ int s_item;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_item = atomicAdd(g.counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);
    if (it >= g.count) return;
    const int i = g.order[it];
    wg_chol_adjoint<T>(g.n[i], g.L[i], g.lda[i], g.nrhs, g.X[i], g.Bb[i], g.ldx[i], g.G[i],
                       g.ldg[i]);
  }
}

/* LDS of one workgroup, beside which the kernels keep at most 64 bytes of
 * static words */
constexpr size_t LDS_CAP = 160 * 1024 - 64;
template <typename T>
constexpr size_t posv_lds(size_t maxn, size_t nrhs, size_t blocks) {
  return sizeof(T) * (blocks * PB * PLD + maxn * nrhs);
}
template <typename T>
constexpr size_t gesv_lds(size_t maxn, size_t nb) {
  return sizeof(T) * (maxn * nb + SOLVE_LDS + maxn * MAXR);
}

/* The largest orders of plans (0 Cholesky, 1 LU), with as many right-hand
 * sides as a plan may have */
template <typename T>
constexpr int max_order(int kind) {
  return sizeof(T) == 8 ? (kind == 0 ? 2270 : 768) : (kind == 0 ? 4830 : 1621);
}
static_assert(posv_lds<double>(max_order<double>(0), MAXR, 2) <= LDS_CAP &&
              posv_lds<float>(max_order<float>(0), MAXR, 2) <= LDS_CAP &&
              gesv_lds<double>(max_order<double>(1), 16) <= LDS_CAP &&
              gesv_lds<float>(max_order<float>(1), 16) <= LDS_CAP, "the largest orders fit");

template <typename T>
hipError_t launch_posv(const BatchArgs<T> &g, int maxn, int grid, hipStream_t s) {
  const int blocks = posv_lds<T>(maxn, g.nrhs, 4) <= LDS_CAP ? 4 : 2;
  const size_t lds = posv_lds<T>(maxn, g.nrhs, blocks);
  if (lds > LDS_CAP) return hipErrorInvalidValue;
  hipError_t e = hipFuncSetAttribute((const void *)posv_batched_kernel<T>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((posv_batched_kernel<T>), dim3(grid), dim3(NT), lds, s, g, blocks);
  return hipGetLastError();
}

template <typename T, int NB>
hipError_t launch_gesv(const BatchArgs<T> &g, int maxn, int grid, int trans, hipStream_t s) {
  const size_t lds = gesv_lds<T>(maxn, NB);
  if (lds > LDS_CAP) return hipErrorInvalidValue;
  hipError_t e = hipFuncSetAttribute((const void *)gesv_batched_kernel<T, NB>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((gesv_batched_kernel<T, NB>), dim3(grid), dim3(NT), lds, s, g, maxn, trans);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_gesv_rows(const BatchArgs<T> &g, int maxn, int grid, int trans,
                            hipStream_t s) {
  const size_t lds = sizeof(T) * ((size_t)PB * PLD + 16 * 16 + 4 * MAXR * PB + (size_t)maxn * g.nrhs);
  if (maxn > NT || lds > 64 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL((gesv_rows_batched_kernel<T>), dim3(grid), dim3(NT), lds, s, g, trans);
  return hipGetLastError();
}

template <typename T>
hipError_t batch_factor(int kind, int nb, int count, const int *order, const int *n, T *const *A,
                        const int *lda, int *const *ipiv, int nrhs, T *const *B, const int *ldb,
                        int *info, int *counter, int maxn, int grid, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  if (nrhs < 0 || nrhs > MAXR || maxn <= 0 || grid <= 0) return hipErrorInvalidValue;
  BatchArgs<T> g;
  g.count = count; g.order = order; g.n = n; g.A = A; g.lda = lda; g.ipiv = ipiv;
  g.nrhs = nrhs; g.B = B; g.ldb = ldb; g.info = info; g.counter = counter;
  if (kind == 0) return launch_posv<T>(g, maxn, grid, s);
  if (kind == 1 || kind == 2) {             /* 2: solve with A^T */
    if (maxn <= NT) return launch_gesv_rows<T>(g, maxn, grid, kind == 2, s);
    /* a width timed on another plan of the bucket may not fit this one's order */
    if (nb == 32 && gesv_lds<T>(maxn, 32) <= LDS_CAP)
      return launch_gesv<T, 32>(g, maxn, grid, kind == 2, s);
    if (nb == 16 || nb == 32) return launch_gesv<T, 16>(g, maxn, grid, kind == 2, s);
  }
  return hipErrorInvalidValue;
}

/* The same work items on the matrix cores: a 64 x 64 tile of C per item,
 * NW wavefronts per tile (1: one wavefront holds the whole tile as 4 x 4
 * MFMA blocks of 16 x 16; 4: a 2 x 2 grid of wavefronts, each 32 x 32 =
 * 2 x 2 blocks), K in slices of 16 staged through LDS as [k][row], the next
 * slice's loads issued before the current slice's MFMAs.  FP64:
 * v_mfma_f64_16x16x4f64 (lane l, element r of the accumulator holds
 * D[(l>>4) + 4r][l&15]); FP32: v_mfma_f32_16x16x4f32 (D[4(l>>4) + r][l&15]).
 * In one MFMA lane l supplies op(A)(row l&15, k slot l>>4) and op(B)(k slot
 * l>>4, column l&15); over the four sub-steps s4 the slots l>>4 = 0..3 take
 * k = 4 (l>>4) + s4, so the 16 k of a slice are each used once.  The
 * choice of NW is the autotuner's. */
template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_batched_mfma_kernel(GemmBatchArgs<T> g) {
  typedef TMfma<T> MF;
  typedef typename MF::acc_t acc_t;
  constexpr int NTH = 64 * NW;
  constexpr int KS = 16;                       /* K slice */
  constexpr int LDT = TS + 4;                  /* LDS row: [k][row], padded */
  constexpr int PER = KS * TS / NTH;           /* elements of a slice per thread */
  constexpr int BPW = (NW == 1) ? 4 : 2;       /* 16 x 16 blocks per wavefront side */
  __shared__ T s_a[KS * LDT], s_b[KS * LDT];
  __shared__ int s_item;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (NW == 1) ? 0 : (wave & 1) * 32, wn = (NW == 1) ? 0 : (wave >> 1) * 32;
  const int lr = lane & 15, kq = (lane >> 4) * 4;
  const int total = g.tile_start[g.count];
  for (;;) {
    __syncthreads();
    if (tid == 0) s_item = atomicAdd(g.counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(s_item);   /* scalar: addresses too */
    if (it >= total) return;
    int lo = 0, hi = g.count - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (g.tile_start[mid] <= it) lo = mid; else hi = mid - 1;
    }
    const int i = g.order[lo], t = it - g.tile_start[lo];
    const int M = g.m[i], N = g.n[i], K = g.k[i];
    const int tm = (M + TS - 1) / TS;
    const int r0 = (t % tm) * TS, c0 = (t / tm) * TS;
    const T *A = g.A[i], *B = g.B[i];
    const long lda = g.lda[i], ldb = g.ldb[i], ldc = g.ldc[i];
    /* element e of a slice: op(A)(r0 + ra, k0 + ka) and op(B)(k0 + kb, c0 + cb),
     * numbered so that consecutive threads read consecutive addresses */
    T va[PER], vb[PER];
    auto load = [&](int k0) {
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        const int e = tid + NTH * q;
        int ra, ka, kb, cb;
        if (g.ta == KX_NOTRANS) { ka = e / TS; ra = e % TS; } else { ra = e / KS; ka = e % KS; }
        if (g.tb == KX_NOTRANS) { cb = e / KS; kb = e % KS; } else { kb = e / TS; cb = e % TS; }
        const int gr = r0 + ra, gka = k0 + ka, gc = c0 + cb, gkb = k0 + kb;
        va[q] = (gr < M && gka < K)
                    ? (g.ta == KX_NOTRANS ? A[(size_t)gka * lda + gr] : A[(size_t)gr * lda + gka])
                    : T(0);
        vb[q] = (gc < N && gkb < K)
                    ? (g.tb == KX_NOTRANS ? B[(size_t)gc * ldb + gkb] : B[(size_t)gkb * ldb + gc])
                    : T(0);
      }
    };
    auto store = [&]() {
#pragma unroll
      for (int q = 0; q < PER; ++q) {
        const int e = tid + NTH * q;
        int ra, ka, kb, cb;
        if (g.ta == KX_NOTRANS) { ka = e / TS; ra = e % TS; } else { ra = e / KS; ka = e % KS; }
        if (g.tb == KX_NOTRANS) { cb = e / KS; kb = e % KS; } else { kb = e / TS; cb = e % TS; }
        s_a[ka * LDT + ra] = va[q];
        s_b[kb * LDT + cb] = vb[q];
      }
    };
    acc_t acc[BPW][BPW];
#pragma unroll
    for (int a = 0; a < BPW; ++a)
#pragma unroll
      for (int b = 0; b < BPW; ++b) acc[a][b] = acc_t{0, 0, 0, 0};
    if (K > 0) load(0);
    for (int k0 = 0; k0 < K; k0 += KS) {
      __syncthreads();
      store();
      __syncthreads();
      if (k0 + KS < K) load(k0 + KS);
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        T a[BPW], b[BPW];
#pragma unroll
        for (int x = 0; x < BPW; ++x) {
          a[x] = s_a[(kq + s4) * LDT + wm + 16 * x + lr];
          b[x] = s_b[(kq + s4) * LDT + wn + 16 * x + lr];
        }
#pragma unroll
        for (int x = 0; x < BPW; ++x)
#pragma unroll
          for (int y = 0; y < BPW; ++y) acc[x][y] = MF::mma(a[x], b[y], acc[x][y]);
      }
    }
    T *C = g.C[i];
#pragma unroll
    for (int x = 0; x < BPW; ++x)
#pragma unroll
      for (int y = 0; y < BPW; ++y)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int r = r0 + wm + 16 * x + MF::drow(lane, rr), c = c0 + wn + 16 * y + lr;
          if (r < M && c < N) {
            T *pc = C + (size_t)c * ldc + r;
            T v = g.alpha * acc[x][y][rr];
            if (g.beta != T(0)) v += g.beta * *pc;
            *pc = v;
          }
        }
  }
}

template <typename T>
hipError_t batch_gemm(int count, int ta, int tb, const int *order, const int *m, const int *n,
                      const int *k,
                      T alpha, const T *const *A, const int *lda, const T *const *B,
                      const int *ldb, T beta, T *const *C, const int *ldc,
                      const int *tile_start, int *counter, int variant, int grid,
                      hipStream_t s) {
  if (count <= 0) return hipSuccess;
  if ((ta != KX_NOTRANS && ta != KX_TRANS) || (tb != KX_NOTRANS && tb != KX_TRANS) ||
      grid <= 0 || variant < 0 || variant > 2)
    return hipErrorInvalidValue;
  GemmBatchArgs<T> g;
  g.count = count; g.ta = ta; g.tb = tb; g.order = order; g.m = m; g.n = n; g.k = k;
  g.alpha = alpha;
  g.beta = beta; g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = C; g.ldc = ldc;
  g.tile_start = tile_start; g.counter = counter;
  if (variant == 0)
    hipLaunchKernelGGL(gemm_batched_kernel<T>, dim3(grid), dim3(NT), 0, s, g);
  else if (variant == 1)
    hipLaunchKernelGGL((gemm_batched_mfma_kernel<T, 1>), dim3(grid), dim3(64), 0, s, g);
  else
    hipLaunchKernelGGL((gemm_batched_mfma_kernel<T, 4>), dim3(grid), dim3(256), 0, s, g);
  return hipGetLastError();
}

template <typename T>
hipError_t chol_adjoint(int count, const int *order, const int *n, T *const *L, const int *lda,
                        int nrhs, T *const *Xs, T *const *Bb, const int *ldx, T *const *G,
                        const int *ldg, int *counter, int grid, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  if (nrhs < 0 || grid <= 0) return hipErrorInvalidValue;
  AdjArgs<T> g;
  g.count = count; g.nrhs = nrhs; g.order = order; g.n = n; g.lda = lda; g.ldx = ldx;
  g.ldg = ldg; g.L = L; g.X = Xs; g.Bb = Bb; g.G = G; g.counter = counter;
  hipLaunchKernelGGL(chol_adjoint_kernel<T>, dim3(grid), dim3(NT), 0, s, g);
  return hipGetLastError();
}

}  // namespace

extern "C" hipError_t atlmx_k_dbatch_chol_adjoint(int count, const int *order, const int *n,
                                                  double *const *L, const int *lda, int nrhs,
                                                  double *const *X, double *const *Bb,
                                                  const int *ldx, double *const *G,
                                                  const int *ldg, int *counter, int grid,
                                                  hipStream_t s) {
  return chol_adjoint<double>(count, order, n, L, lda, nrhs, X, Bb, ldx, G, ldg, counter, grid,
                              s);
}
extern "C" hipError_t atlmx_k_sbatch_chol_adjoint(int count, const int *order, const int *n,
                                                  float *const *L, const int *lda, int nrhs,
                                                  float *const *X, float *const *Bb,
                                                  const int *ldx, float *const *G,
                                                  const int *ldg, int *counter, int grid,
                                                  hipStream_t s) {
  return chol_adjoint<float>(count, order, n, L, lda, nrhs, X, Bb, ldx, G, ldg, counter, grid, s);
}

extern "C" hipError_t atlmx_k_dbatch_factor(int kind, int nb, int count, const int *order,
                                            const int *n, double *const *A, const int *lda,
                                            int *const *ipiv, int nrhs, double *const *B,
                                            const int *ldb, int *info, int *counter, int maxn,
                                            int grid, hipStream_t s) {
  return batch_factor<double>(kind, nb, count, order, n, A, lda, ipiv, nrhs, B, ldb, info,
                              counter, maxn, grid, s);
}
extern "C" hipError_t atlmx_k_sbatch_factor(int kind, int nb, int count, const int *order,
                                            const int *n, float *const *A, const int *lda,
                                            int *const *ipiv, int nrhs, float *const *B,
                                            const int *ldb, int *info, int *counter, int maxn,
                                            int grid, hipStream_t s) {
  return batch_factor<float>(kind, nb, count, order, n, A, lda, ipiv, nrhs, B, ldb, info,
                             counter, maxn, grid, s);
}
extern "C" hipError_t atlmx_k_dbatch_gemm(int count, int ta, int tb, const int *order,
                                          const int *m, const int *n,
                                          const int *k, double alpha, const double *const *A,
                                          const int *lda, const double *const *B,
                                          const int *ldb, double beta, double *const *C,
                                          const int *ldc, const int *tile_start, int *counter,
                                          int variant, int grid, hipStream_t s) {
  return batch_gemm<double>(count, ta, tb, order, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                            tile_start, counter, variant, grid, s);
}
extern "C" hipError_t atlmx_k_sbatch_gemm(int count, int ta, int tb, const int *order,
                                          const int *m, const int *n,
                                          const int *k, float alpha, const float *const *A,
                                          const int *lda, const float *const *B, const int *ldb,
                                          float beta, float *const *C, const int *ldc,
                                          const int *tile_start, int *counter, int variant,
                                          int grid, hipStream_t s) {
  return batch_gemm<float>(count, ta, tb, order, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                           tile_start, counter, variant, grid, s);
}

/* kind 0 Cholesky, 1 LU (2, the transposed solve, as 1) */
extern "C" int atlmx_k_batch_max_order(int kind, int dbl) {
  const int k = kind == 0 ? 0 : 1;
  return dbl ? max_order<double>(k) : max_order<float>(k);
}
