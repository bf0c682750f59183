// los_policy.h — the arithmetic of the fast forms: the type of the products and
// partial sums, and the running sum that a partial sum over some time steps is
// folded into (TwoSum for the FP32-compensated form).
#pragma once

#include <hip/hip_runtime.h>

struct StreamFP64 {
  typedef double real;
  typedef double part_t;
  struct acc_t {
    double s;
  };
  static __device__ __forceinline__ void fold(acc_t &a, double p) { a.s += p; }
  static __device__ __forceinline__ double value(const acc_t &a) { return a.s; }
};

struct StreamFP32C {
  typedef float real;
  typedef float part_t;
  struct acc_t {
    float s, c;  // TwoSum (Knuth) running sum and compensation
  };
  static __device__ __forceinline__ void fold(acc_t &a, float t)
  {
    const float s = a.s + t;
    const float bp = s - a.s;
    const float e = (a.s - (s - bp)) + (t - bp);
    a.s = s;
    a.c += e;
  }
  static __device__ __forceinline__ double value(const acc_t &a) { return (double)a.s + (double)a.c; }
};
