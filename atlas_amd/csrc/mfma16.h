/*
 * mfma16.h -- the 16 x 16 x 4 matrix instruction of a wavefront: lane l
 * supplies A(l & 15, l >> 4) and B(l >> 4, l & 15), and element r of its
 * accumulator is D(drow(l, r), l & 15).
 */
#ifndef ATLMX_MFMA16_H
#define ATLMX_MFMA16_H

#include <hip/hip_runtime.h>

namespace atlmx {

typedef double td4 __attribute__((ext_vector_type(4)));
typedef float tf4 __attribute__((ext_vector_type(4)));
template <typename T> struct TMfma;
template <> struct TMfma<double> {
  typedef td4 acc_t;
  __device__ static acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int drow(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <> struct TMfma<float> {
  typedef tf4 acc_t;
  __device__ static acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static int drow(int lane, int r) { return 4 * (lane >> 4) + r; }
};

}  // namespace atlmx

#endif
