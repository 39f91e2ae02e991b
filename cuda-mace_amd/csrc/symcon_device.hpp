// The contraction of one node and channel in the l_max = 3 structure known at build time, shared by symcon.hip and few_nodes.hip:
// both return the same bits.
#pragma once

#include "common.hpp"
#include "symcon_lmax3.inc"

namespace cm {
namespace symcon {

__device__ __forceinline__ float fmad(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fmad(double a, double b, double c) { return fma(a, b, c); }

// value of the cubic form of x, and (GRAD) its gradient
template <typename S, bool GRAD>
__device__ __forceinline__ S contract(const S (&x)[16], const S (&t3)[CM_SYMCON_N3], const S (&t2)[CM_SYMCON_N2], S t1, S (&g)[16]) {
#pragma unroll
  for (int i = 0; i < 16; ++i) g[i] = S(0);
  S acc = t1 * x[0];
  g[0] = t1;
#define CM_TERM3(t, i, j, k)                    \
  {                                             \
    const S w = t3[t];                          \
    const S wjk = w * (x[j] * x[k]);            \
    acc = fmad(wjk, x[i], acc);                 \
    if (GRAD) {                                 \
      g[i] += wjk;                              \
      g[j] = fmad(w * x[i], x[k], g[j]);        \
      g[k] = fmad(w * x[i], x[j], g[k]);        \
    }                                           \
  }
  CM_SYMCON_MONO3(CM_TERM3)
#undef CM_TERM3
#define CM_TERM2(t, i, j)                       \
  {                                             \
    const S w = t2[t];                          \
    acc = fmad(w * x[i], x[j], acc);            \
    if (GRAD) {                                 \
      g[i] = fmad(w, x[j], g[i]);               \
      g[j] = fmad(w, x[i], g[j]);               \
    }                                           \
  }
  CM_SYMCON_MONO2(CM_TERM2)
#undef CM_TERM2
  return acc;
}

}  // namespace symcon
}  // namespace cm
