/*
 * chol_block.h -- the 32 x 32 pieces of a Cholesky factorization: sums of
 * row tiles on the matrix cores, a diagonal block's factor and inverse by
 * one wavefront.  Shared by the diagonal block of one large matrix
 * (k_chol.hip) and the batched kernels (k_batched.hip).
 */
#ifndef ATLMX_CHOL_BLOCK_H
#define ATLMX_CHOL_BLOCK_H

#include <hip/hip_runtime.h>
#include <math.h>
#include "mfma16.h"
#include "wave_argmax.h"

namespace atlmx {

/* v from lane `src` (a constant) to every lane of the wavefront */
__device__ inline double bcast(double v, int src) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), src);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline float bcast(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
template <typename T> __device__ inline T dsqrt(T x);
template <> __device__ inline double dsqrt<double>(double x) { return sqrt(x); }
template <> __device__ inline float dsqrt<float>(float x) { return sqrtf(x); }

constexpr int PB = 32;
constexpr int PLD = PB + 1;

template <typename T> struct Rng;
template <> struct Rng<double> {
  __device__ static double rsq(double d) { return __builtin_amdgcn_rsq(d); }
  __device__ static bool plain(double d) { return (d >= 1e-280) & (d <= 1e280); }
};
template <> struct Rng<float> {
  __device__ static float rsq(float d) { return __builtin_amdgcn_rsqf(d); }
  __device__ static bool plain(float d) { return (d >= 1e-30f) & (d <= 1e30f); }
};

/* sd = sqrt(d) and ri = 1 / sd (d > 0), each within an ulp: the hardware
 * reciprocal square root and two coupled Newton steps (one in FP32; the
 * iteration in Markstein, "Software division and square root using
 * Goldschmidt's algorithms", RNC6, 2004), a shorter chain than the library's
 * square root and division; PLAIN: d is in
 * the range where no step can over- or underflow.  Outside it, those. */
template <typename T, bool PLAIN>
__device__ inline void sqrt_inv(T d, T &sd, T &ri) {
  if (PLAIN || Rng<T>::plain(d)) {
    T y = Rng<T>::rsq(d), g = d * y, h = T(0.5) * y;
#pragma unroll
    for (int it = 0; it < (sizeof(T) == 8 ? 2 : 1); ++it) {
      const T r = fma(-h, g, T(0.5));
      g = fma(g, r, g);
      h = fma(h, r, h);
    }
    sd = fma(fma(-g, g, d), h, g);
    ri = T(2) * h;
    ri = fma(fma(-ri, sd, T(1)), ri, ri);
  } else {
    sd = dsqrt(d);
    ri = T(1) / sd;
  }
}

/* acc[ci][rj] += sum over j in [j0, j1) of Y(16 ci + c, j) X(16 rj + r, j):
 * lane (li, lk) reads Y(16 ci + li, j + lk) at y[ci][(j + lk) ys] and X
 * likewise.  j1 - j0 is a multiple of 4 U; the next U steps' operands are
 * loaded before the current steps' MFMAs.  MODE: SUM adds every product to
 * acc; ADD and SUBTRACT sum the 4 U products of a step apart, so that a
 * product rounds at that sum's size and acc once a step. */
enum { SUM, ADD, SUBTRACT };
template <typename T, int NC, int RJ, int U, int MODE = SUM>
__device__ __forceinline__ void panel_acc(typename TMfma<T>::acc_t (&acc)[NC][RJ],
                                          const T *const (&y)[NC], long ys,
                                          const T *const (&x)[RJ], long xs, int j0, int j1) {
  const int lk = (threadIdx.x & 63) >> 4;
  T yc[U][NC], xc[U][RJ];
  auto load = [&](int j) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int c = 0; c < NC; ++c) yc[u][c] = y[c][(size_t)(j + 4 * u + lk) * ys];
#pragma unroll
      for (int r = 0; r < RJ; ++r) xc[u][r] = x[r][(size_t)(j + 4 * u + lk) * xs];
    }
  };
  if (j0 >= j1) return;
  load(j0);
  for (int j = j0; j < j1; j += 4 * U) {
    T ya[U][NC], xa[U][RJ];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int c = 0; c < NC; ++c) ya[u][c] = yc[u][c];
#pragma unroll
      for (int r = 0; r < RJ; ++r) xa[u][r] = xc[u][r];
    }
    if (j + 4 * U < j1) load(j + 4 * U);
    typename TMfma<T>::acc_t t[NC][RJ];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < RJ; ++r) {
          if (u == 0) t[c][r] = acc[c][r];
          if (u == 0 && MODE != SUM) t[c][r] = typename TMfma<T>::acc_t{0, 0, 0, 0};
          t[c][r] = TMfma<T>::mma(ya[u][c], xa[u][r], t[c][r]);
        }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < RJ; ++r) {
        if (MODE == SUM) acc[c][r] = t[c][r];
        else if (MODE == ADD) acc[c][r] += t[c][r];
        else acc[c][r] -= t[c][r];
      }
  }
}

template <typename acc_t, int NC, int RJ>
__device__ __forceinline__ void zero_tile(acc_t (&t)[NC][RJ]) {
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < RJ; ++r) t[c][r] = acc_t{0, 0, 0, 0};
}

/* A scalar, or this lane's number, that the compiler takes for a new value
 * here: without it the products of lda with dozens of column numbers, and
 * one 64-bit mask for every lane compare, are computed ahead of the panel
 * loop and spilled across it (the Cholesky: 252 scalar spills). */
__device__ __forceinline__ long fresh(long v) {
  int lo = __builtin_amdgcn_readfirstlane((int)v);   /* a leading dimension: 31 bits */
  asm volatile("" : "+s"(lo));
  return lo;
}
__device__ __forceinline__ int fresh_lane() {
  int l = threadIdx.x & 63;
  asm volatile("" : "+v"(l));
  return l;
}

/* acc[c][r] += the sum over l <= c, in blocks of 16, of m(c, l) w(l, r), for
 * a lower triangle m(c, l) at s_m[l PLD + c]; NEG: of -m(c, l) w(l, r) */
template <typename T, int RJ, bool NEG>
__device__ __forceinline__ void tri_times_tile(typename TMfma<T>::acc_t (&acc)[2][RJ],
                                               const T *s_m,
                                               const typename TMfma<T>::acc_t (&w)[2][RJ]) {
  const int lane = threadIdx.x & 63, li = lane & 15;
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 16 * l + TMfma<T>::drow(lane, e);
#pragma unroll
      for (int c = l; c < 2; ++c) {                /* zero above the diagonal */
        const T m = s_m[row * PLD + 16 * c + li], a = NEG ? -m : m;
#pragma unroll
        for (int r = 0; r < RJ; ++r) acc[c][r] = TMfma<T>::mma(a, w[l][r][e], acc[c][r]);
      }
    }
}

/* w <- w inv^T for a tile held as accumulators: out[c][r] = the sum over l of
 * inv(c, l) w(l, r), the inverse (lower) at s_inv[l PLD + c] in LDS.
 *
 * The product's error grows with the block's condition, which a
 * substitution's does not (a Gaussian kernel matrix with 1e-10 added to its
 * diagonal, FP64, order 100: a residual of 530 u against 0.9 u; with 1e-13
 * the factorization broke down).  refine: the block L (at s_l) is not well
 * conditioned, and the residual w - out L^T, times inv^T, is added once: as
 * the error of the first product is at most sqrt(u) for a block that has a
 * Cholesky factor, that leaves a substitution's (Higham, Accuracy and
 * Stability, Theorem 12.3).
 *
 * The products run over the inverse's zeros too, so where a sum is not finite
 * all are formed again over l <= c alone: an infinity or a NaN in column l
 * of the tile's row stays in that row, from column l on, as in a
 * substitution. */
template <typename T, int RJ>
__device__ __forceinline__ void tile_times_inv(typename TMfma<T>::acc_t (&w)[2][RJ],
                                               const T *s_inv, const T *s_l, bool refine) {
  typename TMfma<T>::acc_t out[2][RJ];
  zero_tile(out);
  tri_times_tile<T, RJ, false>(out, s_inv, w);
  bool odd = false;
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r = 0; r < RJ; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) odd |= !__builtin_isfinite(out[c][r][e]);
  if (__ballot(odd)) {
    const int ln = fresh_lane();
    zero_tile(out);
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll 1
        for (int g = 0; g < 4; ++g) {              /* lane group g holds w(row, .) */
          const int row = 16 * l + TMfma<T>::drow(16 * g, e);
          T x[RJ];
#pragma unroll
          for (int r = 0; r < RJ; ++r) x[r] = __shfl(w[l][r][e], 16 * g + (ln & 15));
#pragma unroll
          for (int c = l; c < 2; ++c)
#pragma unroll
            for (int f = 0; f < 4; ++f) {
              const int col = 16 * c + TMfma<T>::drow(ln, f);
              const T a = s_inv[row * PLD + col];
#pragma unroll
              for (int r = 0; r < RJ; ++r)
                out[c][r][f] = col >= row ? fma(a, x[r], out[c][r][f]) : out[c][r][f];
            }
        }
  } else if (refine) {
    typename TMfma<T>::acc_t d[2][RJ];
    tri_times_tile<T, RJ, true>(w, s_l, out);
    zero_tile(d);
    tri_times_tile<T, RJ, false>(d, s_inv, w);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int r = 0; r < RJ; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const T v = out[c][r][e] + d[c][r][e];
          out[c][r][e] = __builtin_isfinite(v) ? v : out[c][r][e];
        }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r = 0; r < RJ; ++r) w[c][r] = out[c][r];
}

/* Wavefront 0: the Cholesky factor of the 32 x 32 block at s_d[c PLD + r]
 * (identity beyond the matrix: column nb), lanes 0..31 one row each, and its
 * inverse, lanes 32..63 one column each: both are the same elimination step,
 * v[c] -= v[j] L(c, j), the inverse's columns starting from the identity's.
 * Column j's entries reach all lanes by readlane.  Returns 0 or 1 + the
 * failing column; v holds the row of L or the column of the inverse.
 *
 * The columns are taken in groups (GRP0, then GRP wide).  A group's entries
 * gather the earlier columns' products on their own and are added to the
 * matrix's when the group begins: subtracted from them one by one, every
 * product rounds at the entry's size, 1.4 times the factor's error (FP32,
 * order 32: 1.03e-7; by groups 0.72e-7).  Groups beyond the matrix are left out.
 *
 * The 32 pivots are one serial chain, and a branch at each kept the columns'
 * updates from filling its gaps (FP64: 8.9 us a block).  They are therefore
 * first all taken as plain ones, with no branch between the columns of a
 * group, and only where one was not (too small or large for the short square
 * root, negative, NaN) is the block done again with the tests: the same
 * arithmetic on every column before it.  6.3 us, 6.7 with the groups and the
 * condition estimate. */
constexpr int GRP0 = 4, GRP = 8;
template <typename T, bool PLAIN, int G0, int W>
__device__ __forceinline__ void block_group(T (&v)[PB], T (&in)[GRP], const T *s_d, int nb,
                                            int &fail, bool &plain) {
  if (G0 >= nb || (!PLAIN && fail)) return;        /* uniform */
  const int lane = fresh_lane();
  if (G0 > 0) {
#pragma unroll
    for (int c = 0; c < W; ++c) v[G0 + c] += lane < PB ? in[c] : T(0);
  }
  /* the next group's entries, on their way during this one */
#pragma unroll
  for (int c = 0; c < GRP; ++c)
    if (G0 + W + c < PB) in[c] = s_d[(G0 + W + c) * PLD + (lane & (PB - 1))];
#pragma unroll
  for (int j = G0; j < G0 + W; ++j) {
    if (PLAIN || !fail) {
      const T d = bcast(v[j], j);
      if (!PLAIN && !(d > T(0))) {
        fail = j + 1;                              /* uniform: every lane saw the same d */
      } else {
        if (PLAIN) plain = plain & Rng<T>::plain(d);
        T sd, ri;
        sqrt_inv<T, PLAIN>(d, sd, ri);
        v[j] = lane == j ? sd : v[j] * ri;
#pragma unroll
        for (int c = j + 1; c < PB; ++c) v[c] = fma(-v[j], bcast(v[j], c), v[c]);
      }
    }
  }
}

template <typename T, bool PLAIN>
__device__ __forceinline__ int block_columns(T (&v)[PB], const T *s_d, int nb) {
  const int lane = fresh_lane();
  int fail = 0;
  bool plain = true;
  T in[GRP];
#pragma unroll
  for (int c = 0; c < PB; ++c) {
    v[c] = c == lane - PB ? T(1) : T(0);
    if (c < GRP0 && lane < PB) v[c] = s_d[c * PLD + lane];
  }
  block_group<T, PLAIN, 0, GRP0>(v, in, s_d, nb, fail, plain);
  block_group<T, PLAIN, GRP0, GRP - GRP0>(v, in, s_d, nb, fail, plain);
  block_group<T, PLAIN, GRP, GRP>(v, in, s_d, nb, fail, plain);
  block_group<T, PLAIN, 2 * GRP, GRP>(v, in, s_d, nb, fail, plain);
  block_group<T, PLAIN, 3 * GRP, GRP>(v, in, s_d, nb, fail, plain);
  return PLAIN ? !plain : fail;
}

/* a positive number's upper 32 bits, and the number of those bits alone */
__device__ __forceinline__ unsigned high_bits(double v) {
  return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32);
}
__device__ __forceinline__ unsigned high_bits(float v) { return (unsigned)__float_as_int(v); }
template <typename T> __device__ __forceinline__ T from_high_bits(unsigned b);
template <> __device__ __forceinline__ double from_high_bits<double>(unsigned b) {
  return __longlong_as_double((long long)((unsigned long long)b << 32));
}
template <> __device__ __forceinline__ float from_high_bits<float>(unsigned b) {
  return __int_as_float((int)b);
}

/* refine: the largest column sum of |inv(L)| times the largest row norm of L
 * (the root of A's largest diagonal entry) is above COND, about the condition
 * from which a product with the inverse leaves a larger residual than a
 * substitution (kernel matrices of order 48 to 256). */
constexpr int COND = 16;
template <typename T>
__device__ __forceinline__ int block_factor(T (&v)[PB], const T *s_d, int nb, bool &refine) {
  const int lane = fresh_lane();
  const T dg = s_d[(lane & (PB - 1)) * (PLD + 1)];
  const T dmax = from_high_bits<T>(wave_umax(high_bits(dg > T(0) ? dg : T(0))));
  const int fail = block_columns<T, true>(v, s_d, nb) ? block_columns<T, false>(v, s_d, nb) : 0;
  T sum = T(0);
#pragma unroll
  for (int c = 0; c < PB; ++c) sum += fabs(v[c]);
  refine = __ballot(lane >= PB && !(sum * sum * dmax <= T(COND * COND))) != 0ull;
  return fail;
}

}  // namespace atlmx

#endif
