/*
 * lu_panel.h -- the partial-pivoting elimination of an LU panel whose rows
 * live one per thread in registers: shared by the panel kernel of one large
 * matrix (k_lu.hip) and the batched LU (k_batched.hip).
 */
#ifndef ATLMX_LU_PANEL_H
#define ATLMX_LU_PANEL_H

#include <hip/hip_runtime.h>
#include <float.h>
#include "wave_argmax.h"

namespace atlmx {

typedef unsigned long long u64;

template <typename T> struct Lim;
template <> struct Lim<double> { __device__ static double safmin() { return DBL_MIN; } };
template <> struct Lim<float> { __device__ static float safmin() { return FLT_MIN; } };

/* arg-max over the wavefront of (key, then the lowest position): the key's
 * halves one after the other with 32-bit DPP maxima; the low half and the
 * positions are looked at only where the higher part ties.  key and pos
 * become the winner's, in every lane. */
__device__ __forceinline__ void wave_argmax_key(u64 &key, int &pos) {
  const unsigned hi = (unsigned)(key >> 32), lo = (unsigned)key;
  const unsigned mh = wave_umax(hi);
  u64 tie = __ballot(hi == mh);
  if (tie & (tie - 1)) {
    const unsigned ml = wave_umax(hi == mh ? lo : 0u);
    tie = __ballot(hi == mh && lo == ml);
    if (tie & (tie - 1)) {                         /* equal values: the lowest position */
      const bool in = hi == mh && lo == ml;
      const unsigned mp = wave_umax(in ? ~(unsigned)pos : 0u);
      tie = __ballot(in && ~(unsigned)pos == mp);
    }
  }
  const int w = __ffsll((long long)tie) - 1;
  key = ((u64)mh << 32) | (unsigned)__builtin_amdgcn_readlane((int)lo, w);
  pos = __builtin_amdgcn_readlane(pos, w);
}

/* |v| as an integer that orders like it; NaN never better than zero */
__device__ __forceinline__ u64 abs_key(double v) {
  const u64 b = (u64)__double_as_longlong(v) & 0x7fffffffffffffffull;
  return v == v ? b : 0ull;
}

/* entry n of a row of 16 lanes, to every lane of that row */
template <int N> __device__ __forceinline__ double row_bcast(double v) {
  return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + N, 0xf, 0xf, true);
}
template <int N> __device__ __forceinline__ float row_bcast(float v) {
  return __builtin_amdgcn_update_dpp(0.0f, v, 0x150 + N, 0xf, 0xf, true);
}

/* b[n] = entry n of the 16 that every row of 16 lanes holds in p, to all
 * lanes (all must be enabled: a DPP move from a disabled lane gives 0) */
template <typename T, int N>
__device__ __forceinline__ void row_spread(T (&b)[16], T p) {
  if constexpr (N < 16) {
    b[N] = row_bcast<N>(p);
    row_spread<T, N + 1>(b, p);
  }
}

/* Columns MW - WA .. MW - WA + 15 of an MW-wide panel: a = this thread's row, pos =
 * its position (-1: no row).  The loop is rolled, so that its code stays in
 * the instruction cache (unrolled over the columns it was fetched anew for
 * each, 1.6 us a column at one workgroup): an elimination step writes
 * column k + 1 into register k, so the current column is always a[0], and
 * the finished entry -- the multiplier, or the value a pivot row keeps --
 * goes into the register freed at the end, a[WA - 1].  Step i finds columns
 * C.. in [0, WA - i) and this segment's finished ones in [WA - i, WA), where
 * the pivot row's entries are zero.
 *
 * The pivot row reaches the other lanes by DPP: each lane loads one entry of
 * every 16 from LDS (four loads) and row_newbcast moves hand it on.
 * Broadcast LDS reads return 64 lanes' worth of data for every two entries.
 *
 * Two barriers a column; with several workgroups (MULTI) the wavefront that
 * holds the candidate does the exchange.  State: w, row0, ipiv, s_prow and
 * s_cand (MW entries each), s_key and s_pos (one per wavefront), s_piv,
 * first() (this workgroup records the pivots), zero_pivot(column), DIVIDE
 * (the multipliers by division, not by the pivot's reciprocal as LAPACK
 * scales a column), and with MULTI exchange(). */
template <typename T, int NTH, int MW, int WA, bool MULTI, class State>
__device__ __forceinline__ void panel_segment(const State &st, T (&a)[MW], int &pos) {
  constexpr int NW = NTH / 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = 0; i < 16; ++i) {
    const int C = MW - WA + i;
    const T a0 = a[0];
    if (C >= st.w) {                               /* beyond the panel: only move on */
#pragma unroll
      for (int k = 1; k < WA; ++k) a[k - 1] = a[k];
      a[WA - 1] = a0;
      continue;
    }
    u64 key = pos >= C ? abs_key((double)a0) : 0ull;
    int kp = pos >= C && (key != 0ull || pos == C) ? pos : 0x7fffffff;
    wave_argmax_key(key, kp);
    if (lane == 0) { st.s_key[wave] = key; st.s_pos[wave] = kp; }
    __syncthreads();
    int wsel = 0;
    key = st.s_key[0];
    kp = st.s_pos[0];
#pragma unroll
    for (int q = 1; q < NW; ++q) {
      const u64 k2 = st.s_key[q];
      const int p2 = st.s_pos[q];
      if (k2 > key || (k2 == key && p2 < kp)) { key = k2; kp = p2; wsel = q; }
    }
    kp = __builtin_amdgcn_readfirstlane(kp);
    wsel = __builtin_amdgcn_readfirstlane(wsel);
    if (wave == wsel) {
      /* the candidate's holder lays its row out */
      T *dst = MULTI ? st.s_cand : st.s_prow;
      if (pos == kp) {
#pragma unroll
        for (int k = 0; k < WA; ++k)
          dst[k] = (k < WA - 16 || k < WA - i) ? a[k] : T(0);
      }
      if constexpr (MULTI) kp = st.exchange(C, key, kp, WA);
      if (lane == 0) {
        *st.s_piv = kp;
        if (st.first()) st.ipiv[C] = st.row0 + kp;
      }
    }
    __syncthreads();
    const int p = *st.s_piv;
    if (pos == p) pos = C;
    else if (pos == C) pos = p;
    T pr[WA / 16];
#pragma unroll
    for (int q = 0; q < WA / 16; ++q) pr[q] = st.s_prow[16 * q + (lane & 15)];
    const T pv = st.s_prow[0];
    const bool act = pos > C && pv != T(0);
    const bool recip = !State::DIVIDE && (pv < T(0) ? -pv : pv) >= Lim<T>::safmin(); /* uniform */
    const T l = act ? (recip ? a0 * (T(1) / pv) : a0 / pv) : T(0);
    if (pv == T(0) && st.first() && tid == 0) st.zero_pivot(C);
    bool fin = __builtin_isfinite(l);
#pragma unroll
    for (int q = 0; q < WA / 16; ++q) fin = fin && __builtin_isfinite(pr[q]);
    const bool plain = __ballot(!fin) == 0ull;
#pragma unroll
    for (int q = 0; q < WA / 16; ++q) {
      T b[16];
      row_spread<T, 0>(b, pr[q]);
      if (plain) {                                 /* l = 0 or b = 0 changes nothing */
#pragma unroll
        for (int n = 0; n < 16; ++n)
          if (16 * q + n > 0) a[16 * q + n - 1] = fma(-l, b[n], a[16 * q + n]);
      } else {                                     /* nor may 0 * inf */
#pragma unroll
        for (int n = 0; n < 16; ++n)
          if (16 * q + n > 0) {
            const T v = a[16 * q + n];
            a[16 * q + n - 1] = act && 16 * q + n < WA - i ? fma(-l, b[n], v) : v;
          }
      }
    }
    a[WA - 1] = act ? l : a0;
  }
}

}  // namespace atlmx

#endif
