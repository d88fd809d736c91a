// Selection from a token's logits when some of them are in doubt, shared by the batch routers.
#pragma once
#include "common.h"
#include "internal.h"
#include "topk.h"

// One logit's fp64 sum as the reference's sequential chain (src/ref.cpp:70-77), by one wave: the lanes multiply 256 columns
// at a time into LDS (a single thread's 2 d quarter-rate conversions and its dependent loads took 110 us) -- a product of two
// floats is exact in fp64, so adding products is the chain of FMAs bit for bit --, then every lane adds them up in order.
// buf: 512 doubles of LDS owned by the wave, two halves by turns.  (With both factors in LDS and an FMA each, a read of 16 bytes per column,
// a batch that had such a token spent 34 us in its selecting launch at 48 tokens, 30 at 130; now 26 and 23.)
__device__ __forceinline__ double exact_chain_wave(const moe_rfix& R, int t, int e, double* buf) {
  const int lane = threadIdx.x & 63;
  const float* xr = R.x + (size_t)t * R.d;
  double acc = 0.0;
  float4 w, xv;
  auto load = [&](int c) {
    w = xv = float4{0.f, 0.f, 0.f, 0.f};
    if (c >= R.d) return;
    xv = *(const float4*)(xr + c);
    if (R.bf16) {
      const uint2 u = *(const uint2*)((const uint16_t*)R.W + (size_t)e * R.d + c);
      w = float4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                 __uint_as_float(u.y & 0xffff0000u)};
    } else {
      w = *(const float4*)((const float*)R.W + (size_t)e * R.d + c);
    }
  };
  load(4 * lane);
  for (int c = 0, half = 0; c < R.d; c += 256, half ^= 256) {
    double2* const q = (double2*)(buf + half + 4 * lane);  // this lane's four columns
    q[0] = double2{(double)w.x * (double)xv.x, (double)w.y * (double)xv.y};
    q[1] = double2{(double)w.z * (double)xv.z, (double)w.w * (double)xv.w};
    load(c + 256 + 4 * lane);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's own LDS writes
    __builtin_amdgcn_wave_barrier();
    const int n = R.d - c < 256 ? R.d - c : 256;  // (a multiple of 32)
    for (int i = 0; i < n; i += 32) {
      double2 p[16];
#pragma unroll
      for (int j = 0; j < 16; j++) p[j] = *(const double2*)(buf + half + i + 2 * j);
#pragma unroll
      for (int j = 0; j < 16; j++) {
        acc += p[j].x;
        acc += p[j].y;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  return acc;
}

// A logit whose fp64 sum lies within tol of the reference's sequential one is the reference's float unless a rounding boundary
// lies within tol of the sum.  (true for any finite sum where tol is infinite)  A sum that is not finite is never in doubt: products
// of finite floats and their sums stay finite in fp64, so it has terms that are not, and is then NaN (a NaN among them, or
// infinities of both signs) or the one infinity in every order.  (A row of x with one NaN or infinity has an infinite tol: with
// its 512 logits redone as chains, 2.5 ms of a block, one such row took a batch of 300 tokens from 0.53 to 10.2 ms.)
__device__ __forceinline__ bool logit_doubtful(double sum, float tol) {
  return sum - sum == 0.0 && !((float)(sum - (double)tol) == (float)(sum + (double)tol));
}

// Block of 256 threads: softmax / top-k of token t's logits lg (LDS), of which list[0 .. nlist) are doubtful.  None (two tokens
// in three): the selection is the reference's as it stands.  Otherwise the k + 1 best must be further apart than the doubt
// (topk.h), and where they are not, the doubtful logits alone are redone as the reference's chains -- which leaves none in
// doubt.  (Redoing all 512 logits of such a token, as select_certain does with a true near tie, takes 70 us; one batch of 515
// tokens in ten has one.)  Block-uniform arguments; a barrier stands behind the caller's writes and behind the results.
template <int NPL>
__device__ __forceinline__ void select_listed(float* lg, const int* list, int nlist, float tol, const moe_rfix& RF, int t, int E, int k,
                                              int* sel_ids, float* sel_ws, double (*chain)[512]) {
  float slack = INFINITY;
  if (nlist) slack = topk_block<NPL, false, 256, true>(lg, sel_ids, sel_ws, E, k);
  else (void)topk_block<NPL, false, 256>(lg, sel_ids, sel_ws, E, k);
  if (nlist && !(slack > 2.f * tol)) {
    for (int i = threadIdx.x >> 6; i < nlist; i += 4) {
      const int e = list[i];
      const float v = (float)exact_chain_wave(RF, t, e, chain[threadIdx.x >> 6]) + (RF.bias ? RF.bias[e] : 0.f);
      if ((threadIdx.x & 63) == 0) lg[e] = v;
    }
    __syncthreads();
    (void)topk_block<NPL, false, 256>(lg, sel_ids, sel_ws, E, k);
  }
  __syncthreads();
}
