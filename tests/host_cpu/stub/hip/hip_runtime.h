// Lets g++ compile the device headers' arithmetic for the host. The hardware's
// reciprocal and reciprocal square root estimates are stood in for by their
// values rounded to float, whose relative error is the same 2^-24.
#pragma once
#include <cmath>
#include <stdint.h>

#define __device__
#define __host__
#define __forceinline__ inline
#define __shared__ static

using std::fabs;
using std::fma;
using std::fmax;
using std::sqrt;

static struct {
  unsigned x;
} threadIdx, blockDim;
inline void __syncthreads() {}
template <class T>
inline T atomicAdd(T *p, T v) {
  T old = *p;
  *p += v;
  return old;
}

inline double to_float_precision(double x) {
  if (!std::isfinite(x) || x == 0) return x;
  int e;
  const float m = (float)std::frexp(x, &e);
  return std::ldexp((double)m, e);
}
inline double __builtin_amdgcn_rcp(double x) { return to_float_precision(1 / x); }
inline double __builtin_amdgcn_rsq(double x) { return to_float_precision(1 / std::sqrt(x)); }
