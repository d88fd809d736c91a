// f16 operands of the MFMA kernels: vector types, and views of 32-bit words as pairs of f16.
#pragma once
#include "common.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

union H8 {  // one MFMA operand
  half8 v;
  uint32_t u[4];
  half2v h[4];
};
__device__ __forceinline__ half2v h2(uint32_t u) {
  union { uint32_t u; half2v h; } c;
  c.u = u;
  return c.h;
}
__device__ __forceinline__ uint32_t u2(half2v h) {
  union { half2v h; uint32_t u; } c;
  c.h = h;
  return c.u;
}
__device__ __forceinline__ uint32_t word(const uint4& q, int s) { return s == 0 ? q.x : s == 1 ? q.y : s == 2 ? q.z : q.w; }
