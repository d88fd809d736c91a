// What a batch needs from a row of x besides its products: one pass.
#pragma once
#include "common.h"
#include "internal.h"

// the chunk's two float4: neighbours, or (layout 2) elements 4w.. and 32 + 4w.. of the 64-block
__device__ __forceinline__ void f16_chunk_src(int layout, int i, int& ia, int& ib) {
  ia = layout == 2 ? (i >> 3) * 16 + (i & 7) : 2 * i;
  ib = layout == 2 ? ia + 8 : ia + 1;
}
__device__ __forceinline__ uint4 f16_chunk(int layout, const float4& u, const float4& v) {
  __half2 a, b, c, e;
  if (layout == 2) {
    a = __floats2half2_rn(u.x, u.z); b = __floats2half2_rn(v.x, v.z);
    c = __floats2half2_rn(u.y, u.w); e = __floats2half2_rn(v.y, v.w);
  } else if (layout == 0) {
    a = __floats2half2_rn(u.x, u.y); b = __floats2half2_rn(u.z, u.w);
    c = __floats2half2_rn(v.x, v.y); e = __floats2half2_rn(v.z, v.w);
  } else {
    a = __floats2half2_rn(u.x, v.x); b = __floats2half2_rn(u.y, v.y);
    c = __floats2half2_rn(u.z, v.z); e = __floats2half2_rn(u.w, v.w);
  }
  uint4 o;
  o.x = *(const uint32_t*)&a; o.y = *(const uint32_t*)&b; o.z = *(const uint32_t*)&c; o.w = *(const uint32_t*)&e;
  return o;
}

// Four (two) values of the gate vector, which may start at any element (moe_set_shared asks for no more; the loads are the same single
// instructions as for aligned ones).
typedef float gate_f32x4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t gate_bf16x4 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t gate_bf16x2 __attribute__((aligned(2)));

// the f16 copy (layout as moe_f32_to_f16's), the mean square, the selection's error bound and the shared expert's gate
// logit (fp64 sum) of row t; each is left out where its pointer is null
// (chunks of 8 columns i0, i0 + step, ...: this thread's part of the row's sums in acc and gate; err: of the squares of what
// rounding to f16 changes)
__device__ __forceinline__ float f16_err2(const float4& u) {
  const float a = u.x - __half2float(__float2half_rn(u.x)), b = u.y - __half2float(__float2half_rn(u.y));
  const float c = u.z - __half2float(__float2half_rn(u.z)), e = u.w - __half2float(__float2half_rn(u.w));
  return (a * a + b * b) + (c * c + e * e);
}
__device__ __forceinline__ void row_extras_part(const float* __restrict__ x, int t, int d, int i0, int step, const moe_row_extras& R,
                                                float& acc, double& gate, float* err = nullptr) {
  const float4* xr = (const float4*)(x + (size_t)t * d);
  uint4* yr = R.x16 ? (uint4*)R.x16 + (size_t)t * (d / 8) : nullptr;
  acc = 0.f;
  gate = 0.0;
#pragma unroll 2
  for (int i = i0; i < d / 8; i += step) {
    int ia, ib;
    f16_chunk_src(R.layout, i, ia, ib);
    const float4 u = xr[ia], v = xr[ib];
    if (yr) {
      yr[i] = f16_chunk(R.layout, u, v);
    }
    acc += ((u.x * u.x + u.y * u.y) + (u.z * u.z + u.w * u.w)) + ((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w));
    if (err) *err += f16_err2(u) + f16_err2(v);
    if (R.wx) {
      float g[8];
      if (R.wx_bf16) {
        const gate_bf16x4 p = ((const gate_bf16x4*)R.wx)[ia], q = ((const gate_bf16x4*)R.wx)[ib];
        g[0] = __uint_as_float(p.x << 16); g[1] = __uint_as_float(p.x & 0xffff0000u);
        g[2] = __uint_as_float(p.y << 16); g[3] = __uint_as_float(p.y & 0xffff0000u);
        g[4] = __uint_as_float(q.x << 16); g[5] = __uint_as_float(q.x & 0xffff0000u);
        g[6] = __uint_as_float(q.y << 16); g[7] = __uint_as_float(q.y & 0xffff0000u);
      } else {
        const gate_f32x4 p = ((const gate_f32x4*)R.wx)[ia], q = ((const gate_f32x4*)R.wx)[ib];
        g[0] = p.x; g[1] = p.y; g[2] = p.z; g[3] = p.w; g[4] = q.x; g[5] = q.y; g[6] = q.z; g[7] = q.w;
      }
      gate = fma((double)g[0], (double)u.x, gate); gate = fma((double)g[1], (double)u.y, gate);
      gate = fma((double)g[2], (double)u.z, gate); gate = fma((double)g[3], (double)u.w, gate);
      gate = fma((double)g[4], (double)v.x, gate); gate = fma((double)g[5], (double)v.y, gate);
      gate = fma((double)g[6], (double)v.z, gate); gate = fma((double)g[7], (double)v.w, gate);
    }
  }
}
// the row's results from its sums (one thread)
__device__ __forceinline__ void row_extras_out(int t, int d, const moe_row_extras& R, float acc, double gate) {
  if (R.xms) R.xms[t] = acc / (float)d;
  if (R.tol) {
    const float tl = R.tol_scale * sqrtf(acc) * 1.01f;
    R.tol[t] = tl >= 0.f ? tl : INFINITY;  // (NaN: nothing is certain)
  }
  if (R.wx) R.out_x[t] = (float)gate;
}
