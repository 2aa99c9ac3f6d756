// mfma.h -- the 16 x 16 x 4 matrix-core product in FP64 and FP32: lane l holds
// A(l % 16, l / 16) and B(l / 16, l % 16) of a step; accumulator register r of
// lane l holds D(row(l / 16, r), l % 16) (measured; the two precisions differ).
#pragma once
#include "la_common.h"

namespace la {

template <class T> struct Mfma;
template <> struct Mfma<double> {
  typedef la_d4 acc_t;
  static __device__ __forceinline__ acc_t op(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};
template <> struct Mfma<float> {
  typedef la_f4 acc_t;
  static __device__ __forceinline__ acc_t op(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

}  // namespace la
