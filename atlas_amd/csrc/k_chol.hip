/*
 * k_chol.hip -- Cholesky of one diagonal block (n <= 128) with the inverses
 * of its 64x64 diagonal blocks, and the solve of the panel below (right of)
 * it.
 *
 * Replaces the leaves of ATLAS's recursive Cholesky: the closed-form 4x4,
 * 3x3, 2x2 kernels (src/lapack/ATL_potrfL.c:104-202, ATL_potrfU.c:98-197)
 * and the small-N recursion above them.  A non-positive (or NaN) pivot
 * stops the factorization and records the 1-based global column in *info,
 * as ATL_potrfL.c:238-240 does; later kernels of the same Cholesky see the
 * nonzero info and do nothing.  Only the referenced triangle is read or
 * written.
 */
#include <hip/hip_runtime.h>
#include "kernels.h"
#include "chol_block.h"

namespace {

constexpr int CNB = ATLMX_CHOL_NB;
constexpr int NT = 256;

using namespace atlmx;

/* One workgroup, left-looking in 32-column panels with the pieces of the
 * batched Cholesky (chol_block.h): the diagonal tile's sum split over the
 * four wavefronts, its factor and inverse by wavefront 0, the row tiles
 * below (at most three, one per other wavefront) accumulated meanwhile and
 * then multiplied by the inverse.  Every second panel completes a 64x64
 * diagonal block, whose inverse the panel solve needs, [i11 0; -i22 L21 i11,
 * i22]: formed here from the two 32x32 inverses instead of by a launch of
 * its own.  The ten 32x32 tiles of the triangle stay in LDS from one load to
 * one store, so that no step of the chain waits for memory.  L(i, k) is
 * A[i rs + k cs], so that Upper (A = U^T U, L = U^T) is the same code.  What
 * bounds it: four times the one-wavefront factor of 32 columns.  128
 * columns, FP64: 87 us for one barrier-separated step per column, and 15 for
 * the inverses' launch; 71 for both with the tiles in memory; 49 so: 3 for
 * the load, 6.7 for each panel's factor, 2 to 4 for its products, 4 for the
 * store.  Tiles and column groups beyond the matrix are passed over: one of
 * order 1 takes 6 us (5 in the form with a barrier per step, 13 with the
 * whole block). */
constexpr int TBLK = PB * PLD;
constexpr int NTILE = (CNB / PB) * (CNB / PB + 1) / 2;

template <typename T>
__global__ __launch_bounds__(NT) void potf2_kernel(int lower, int n, T *A, long lda, T *inv,
                                                   int info_base, int *info) {
  typedef TMfma<T> MF;
  typedef typename MF::acc_t acc_t;
  constexpr int IB = 64;
  if (*info != 0) return;
  __shared__ T s_l[NTILE * TBLK], s_blk[4 * TBLK], s_i[2][TBLK];
  __shared__ int s_ready, s_fail, s_refine;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const long rs = lower ? 1 : lda, cs = lower ? lda : 1;
  const int nt = (n + PB - 1) / PB;
  auto tile = [&](int i, int j) { return s_l + (i * (i + 1) / 2 + j) * TBLK; };
  if (tid == 0) s_ready = s_fail = 0;
  /* row and column within a tile: neighbouring threads at neighbouring addresses */
  const int f = tid % PB, g = tid / PB;
  T in[NTILE][PB * PB / NT];                       /* every load before the first use */
#pragma unroll
  for (int i = 0, q = 0; i < CNB / PB; ++i) {
    if (i >= nt) break;
#pragma unroll
    for (int j = 0; j <= i; ++j, ++q)
#pragma unroll
      for (int h = 0; h < PB * PB / NT; ++h) {
        const int r = lower ? f : g + h * (NT / PB), c = lower ? g + h * (NT / PB) : f;
        const int ar = i * PB + r, ac = j * PB + c;
        in[q][h] = ar == ac ? T(1) : T(0);         /* beyond the matrix: the identity */
        if (ar < n && ac <= ar) in[q][h] = A[(long)ar * rs + (long)ac * cs];
      }
  }
#pragma unroll
  for (int i = 0, q = 0; i < CNB / PB; ++i) {
    if (i >= nt) break;                            /* rows of tiles beyond the matrix */
#pragma unroll
    for (int j = 0; j <= i; ++j, ++q)
#pragma unroll
      for (int h = 0; h < PB * PB / NT; ++h) {
        const int r = lower ? f : g + h * (NT / PB), c = lower ? g + h * (NT / PB) : f;
        s_l[q * TBLK + c * PLD + r] = in[q][h];
      }
  }
  __syncthreads();
  for (int p = 0; p < nt; ++p) {
    if (p) {
      acc_t acc[2][2];
      zero_tile(acc);
      for (int t = 0; t < p; ++t) {                /* 8 of each tile's columns */
        const T *y = tile(p, t) + li;
        const T *yp[2] = {y, y + 16};
        panel_acc<T, 2, 2, 2>(acc, yp, PLD, yp, PLD, 8 * wave, 8 * wave + 8);
      }
      T *sp = s_blk + wave * TBLK;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sp[(16 * c + MF::drow(lane, e)) * PLD + 16 * r + li] = acc[c][r][e];
      __syncthreads();
#pragma unroll
      for (int h = 0; h < PB; h += NT / PB) {
        const int r = f, c = g + h;
        T *o = tile(p, p) + c * PLD + r;
        const T *q = s_blk + c * PLD + r;
        if (r >= c && p * PB + r < n) *o -= (q[0] + q[TBLK]) + (q[2 * TBLK] + q[3 * TBLK]);
      }
      __syncthreads();
    }
    if (wave == 0) {
      T v[PB];
      T *d = tile(p, p);
      bool refine;
      const int fail = block_factor(v, d, min(PB, n - p * PB), refine);
      const int ln = fresh_lane();
      if (ln < PB) {
        /* on failure the columns before the failing one; so below */
        const int nc = fail ? fail - 1 : PB;
#pragma unroll
        for (int c = 0; c < PB; ++c)
          if (c <= ln && c < nc) d[c * PLD + ln] = v[c];
      } else {
#pragma unroll
        for (int c = 0; c < PB; ++c) s_i[p & 1][(ln - PB) * PLD + c] = v[c];
      }
      if (ln == 0) {
        if (fail) s_fail = p * PB + fail;
        s_refine = refine;
        __hip_atomic_store(&s_ready, p + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    } else if (p + wave < nt) {                    /* row tile p + wave */
      acc_t acc[2][2], w[2][2];
      T *x = tile(p + wave, p);
      zero_tile(acc);
      for (int t = 0; t < p; ++t) {
        const T *y = tile(p, t) + li, *z = tile(p + wave, t) + li;
        const T *yp[2] = {y, y + 16}, *xp[2] = {z, z + 16};
        panel_acc<T, 2, 2, 2>(acc, yp, PLD, xp, PLD, 0, PB);
      }
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            w[c][r][e] = x[(16 * c + MF::drow(lane, e)) * PLD + 16 * r + li] - acc[c][r][e];
      while (__hip_atomic_load(&s_ready, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < p + 1)
        __builtin_amdgcn_s_sleep(1);
      tile_times_inv<T, 2>(w, s_i[p & 1], tile(p, p), s_refine);
      const int nc = s_fail ? s_fail - 1 - p * PB : PB;
      if (nc == PB) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              x[(16 * c + MF::drow(lane, e)) * PLD + 16 * r + li] = w[c][r][e];
      } else {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int col = 16 * c + MF::drow(lane, e);
            if (col < nc)
#pragma unroll
              for (int r = 0; r < 2; ++r) x[col * PLD + 16 * r + li] = w[c][r][e];
          }
      }
    }
    __syncthreads();
    if (s_fail) break;
    if (!(p & 1) && p + 1 < nt) continue;
    /* ---- inverse of the 64x64 block b: wavefront w forms columns 16 (w & 1)
     * of L21 i11 and from them its 16x16 tile of X21 ---- */
    const int b = p / 2, two = p & 1;
    T *out = inv + (size_t)b * IB * IB;            /* inv(L)(r, c), transposed for Upper */
    auto put = [&](int r, int c, T v) { out[lower ? c * IB + r : r * IB + c] = v; };
#pragma unroll
    for (int h = 0; h < PB; h += NT / PB) {
      const int r = lower ? f : g + h, c = lower ? g + h : f;
      put(r, c, s_i[0][c * PLD + r]);
      put(PB + r, PB + c, two ? s_i[1][c * PLD + r] : (r == c ? T(1) : T(0)));
      put(r, PB + c, T(0));
      if (!two) put(PB + r, c, T(0));
    }
    if (two) {
      const int jb = 16 * (wave & 1), ib = 16 * (wave >> 1);
      const T *l21 = tile(2 * b + 1, 2 * b);
      acc_t t[2], x = acc_t{0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        t[r] = acc_t{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 8; ++s)
          t[r] = MF::mma(l21[(4 * s + lk) * PLD + 16 * r + li], s_i[0][(jb + li) * PLD + 4 * s + lk],
                         t[r]);
      }
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x = MF::mma(s_i[1][(16 * r + MF::drow(lane, e)) * PLD + ib + li], t[r][e], x);
#pragma unroll
      for (int e = 0; e < 4; ++e) put(PB + ib + MF::drow(lane, e), jb + li, -x[e]);
    }
  }
  /* on failure the columns before the failing one are stored, factored in
   * every row of the block; the others stay as they came */
  const int done = s_fail ? s_fail - 1 : n;
  for (int i = 0; i < nt; ++i)
    for (int j = 0; j <= i; ++j)
#pragma unroll
      for (int h = 0; h < PB; h += NT / PB) {
        const int r = lower ? f : g + h, c = lower ? g + h : f;
        const int ar = i * PB + r, ac = j * PB + c;
        if (ar < n && ac <= ar && ac < done) A[(long)ar * rs + (long)ac * cs] = tile(i, j)[c * PLD + r];
      }
  if (s_fail && tid == 0) atomicCAS(info, 0, info_base + s_fail);
}

/* The panel's triangular solve after the diagonal block (jb <= 128 rows)
 * is factored: every panel vector v (a row of A21 for Lower, a column of
 * A12 for Upper) becomes y with L y^T = v^T, L the block's lower factor
 * (Lower: L11; Upper: U11^T).  With L split into 64-row blocks, L = [L00 0;
 * L10 L11'] and the inverted diagonal blocks from potf2_kernel:
 *   y0 = v0 inv(L00)^T,   y1 = (v1 - y0 L10^T) inv(L11')^T
 * -- the two-block TRSM ATLAS's Cholesky makes (ATL_potrfL.c:236-246), as
 * three 64-wide products in one launch.  A workgroup takes 64 vectors,
 * each wavefront 16 of them through all three products on the matrix cores
 * (the MFMA's four k lane groups take k = 16 lk + t in step t); a product's
 * result is turned into the next one's operand layout through the
 * wavefront's own slice of LDS, so no workgroup barrier is needed. */
template <typename T>
__global__ __launch_bounds__(NT) void chol_panel_solve_kernel(int lower, int nr, int jb,
                                                              const T *__restrict__ D, long lda,
                                                              const T *__restrict__ inv, T *P,
                                                              const int *info) {
  typedef TMfma<T> MF;
  typedef typename MF::acc_t acc_t;
  constexpr int B = 64;
  if (*info != 0) return;
  __shared__ T s_w[NT / 64][16][B + 1];           /* per wavefront: 16 vectors x 64 */
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int b0 = min(B, jb), b1 = jb - B;         /* block sizes (b1 <= 0: one block) */
  const int vec = blockIdx.x * 64 + wave * 16 + li;   /* this lane's A-operand vector */
  const bool vok = vec < nr;
  /* v(p, k): Lower P[k lda + p], Upper P[p lda + k] */
  auto vat = [&](int p, int k) -> T * { return lower ? P + (size_t)k * lda + p : P + (size_t)p * lda + k; };
  /* L(i, k) of the factored block: Lower D[k lda + i], Upper D[i lda + k] */
  auto lat = [&](int i, int k) -> T { return lower ? D[(size_t)k * lda + i] : D[(size_t)i * lda + k]; };
  /* inv(L_bb)(i, k): Lower inv_b[k 64 + i], Upper (inv(U_bb)^T) inv_b[i 64 + k] */
  auto iat = [&](int b, int i, int k) -> T {
    const T *ib = inv + (size_t)b * B * B;
    return lower ? ib[(size_t)k * B + i] : ib[(size_t)i * B + k];
  };
  T (*sw)[B + 1] = s_w[wave];

  /* y0 = v0 inv(L00)^T: A operand v0(vec, k), B operand W0(k, i) = inv(L00)(i, k) */
  acc_t acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = acc_t{0, 0, 0, 0};
  /* every operand of a product is requested before its first MFMA */
  T av[16], wv[16][4];
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int k = 16 * lk + t;
    av[t] = (vok && k < b0) ? *vat(vec, k) : T(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = 16 * c + li;
      wv[t][c] = (k < b0 && i < b0) ? iat(0, i, k) : T(0);
    }
  }
#pragma unroll
  for (int t = 0; t < 16; ++t)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = MF::mma(av[t], wv[t][c], acc[c]);
  /* y0 to LDS ([vector][i]) and to P */
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int vr = MF::drow(lane, r), i = 16 * c + li;
      const int p = blockIdx.x * 64 + wave * 16 + vr;
      sw[vr][i] = acc[c][r];
      if (p < nr && i < b0) *vat(p, i) = acc[c][r];
    }
  if (b1 <= 0) return;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  /* v1' = v1 - y0 L10^T: A operand y0(vec, k), B operand L10(i, k) = L(64 + i, k) */
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = acc_t{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int k = 16 * lk + t;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = 16 * c + li;
      wv[t][c] = (i < b1) ? lat(B + i, k) : T(0);
    }
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const T a = sw[li][16 * lk + t];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = MF::mma(a, wv[t][c], acc[c]);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int vr = MF::drow(lane, r), i = 16 * c + li;
      const int p = blockIdx.x * 64 + wave * 16 + vr;
      const T v1 = (p < nr && i < b1) ? *vat(p, B + i) : T(0);
      sw[vr][i] = v1 - acc[c][r];
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  /* y1 = v1' inv(L11')^T */
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = acc_t{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int k = 16 * lk + t;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = 16 * c + li;
      wv[t][c] = (k < b1 && i < b1) ? iat(1, i, k) : T(0);
    }
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const T a = sw[li][16 * lk + t];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = MF::mma(a, wv[t][c], acc[c]);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int vr = MF::drow(lane, r), i = 16 * c + li;
      const int p = blockIdx.x * 64 + wave * 16 + vr;
      if (p < nr && i < b1) *vat(p, B + i) = acc[c][r];
    }
}

template <typename T>
hipError_t launch_chol_panel(int uplo, int nr, int jb, const T *D, long lda, const T *inv, T *P,
                             const int *info, hipStream_t s) {
  if (nr <= 0 || jb <= 0) return hipSuccess;
  if (jb > CNB || lda < jb || !D || !inv || !P || !info) return hipErrorInvalidValue;
  hipLaunchKernelGGL(chol_panel_solve_kernel<T>, dim3((unsigned)((nr + 63) / 64)), dim3(NT), 0,
                     s, uplo == KX_LOWER, nr, jb, D, lda, inv, P, info);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_potf2(int uplo, int n, T *A, long lda, T *inv, int info_base, int *info,
                        hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (n > CNB || lda < n || !A || !inv || !info) return hipErrorInvalidValue;
  hipLaunchKernelGGL(potf2_kernel<T>, dim3(1), dim3(NT), 0, s, uplo == KX_LOWER, n, A, lda,
                     inv, info_base, info);
  return hipGetLastError();
}

}  // namespace

extern "C" hipError_t atlmx_k_dpotf2(int uplo, int n, double *A, long lda, double *inv,
                                     int info_base, int *info, hipStream_t s) {
  return launch_potf2<double>(uplo, n, A, lda, inv, info_base, info, s);
}
extern "C" hipError_t atlmx_k_spotf2(int uplo, int n, float *A, long lda, float *inv,
                                     int info_base, int *info, hipStream_t s) {
  return launch_potf2<float>(uplo, n, A, lda, inv, info_base, info, s);
}
extern "C" hipError_t atlmx_k_dchol_panel(int uplo, int nr, int jb, const double *D, long lda,
                                          const double *inv, double *P, const int *info,
                                          hipStream_t s) {
  return launch_chol_panel<double>(uplo, nr, jb, D, lda, inv, P, info, s);
}
extern "C" hipError_t atlmx_k_schol_panel(int uplo, int nr, int jb, const float *D, long lda,
                                          const float *inv, float *P, const int *info,
                                          hipStream_t s) {
  return launch_chol_panel<float>(uplo, nr, jb, D, lda, inv, P, info, s);
}
