// Batch router without the dense fp64 pass: bit-exact expert ids at a fraction of the fp64 work.  Three launches, and a
// fourth for the tokens that the selection cannot settle, whose blocks return at once where there are none.
//
// The reference's router (src/ref.cpp:565-594) needs every logit as a sequential fp64 sum, but only the k
// best logits of a token decide its experts and weights; the other ~500 enter through the softmax
// normaliser alone, which cancels in the renormalised weights up to rounding.  So:
//   1. k_router_prep  the router matrix as f16 with its row norms, and one pass over x that leaves everything a batch needs
//                     from it: the f16 copy in the grouped GEMM's order (the router matrix is written in the same order), the
//                     mean square, the error bound of fp64 sums, the shared expert's gate logit;
//   2. k_router_f16   all T x E logits from the two f16 copies on the matrix pipe (f32 accumulation);
//   3. k_router_pick  a wave per token (small batches: four).  A RIGOROUS error bound B_e on each approximate logit (below) gives an interval
//                     [a_e - B_e, a_e + B_e] that holds the exact logit; tau = the k-th largest lower end; every expert whose
//                     upper end reaches tau - 1e-5 is a candidate (the true top k are among them: at least k exact logits are
//                     >= tau, and a true top-k logit is >= the k-th largest exact one).  The candidates' logits (typically
//                     10-12 of 512) are taken as fp64 dot products, in another order than the reference's sequential one:
//                     the reference's float, or in rare cases (a rounding boundary within tol of the sum) its neighbour.  If
//                     every gap between neighbours among the k + 1 best exceeds what can make two probabilities round to one
//                     float, plus two ulps where a logit is in doubt, and all lie within 70 of the maximum, the order by
//                     logit is the reference's order by f32 probability and the ids are final; the weights use these logits
//                     and a normaliser in which the non-candidates' terms are approximate, which moves a renormalised weight
//                     by an ulp or two at most.  Tokens that fail any test (near ties, a logit range where probabilities
//                     underflow, more candidates than slots, non-finite values) are listed; rows of zeros (padding) are
//                     settled by their block, which knows their sums;
//   4. k_router_listed  listed tokens, sixteen at a time, as the reference's chains on the f64 matrix pipe.
// Error bound.  a~ = fl32(sum of x~_c * w~_c) with x~ = f16(x), w~ = f16(w).  |x.w - x~.w~| <= |x - x~||w| + |x~||w - w~| by
// Cauchy-Schwarz; prep, which makes the copies, leaves the norms of what their rounding changed (a bound from the format alone,
// 2^-10 |x||w|, is five times as wide for an f32 router beside activations that came from bf16, thirty times where the router
// is bf16 too and nothing rounds: 13 candidates of 512 instead of 10.8 and 10.1).  The accumulation adds at most (RA_CHUNK *
// 2^-22 + (d / RA_CHUNK + RA_KS) * 2^-23) * 1.001 |x~||w~|: inside a chunk of RA_CHUNK
// columns however the matrix pipe orders and rounds its partial sums (twice the IEEE bound per addition, one addition
// charged per product), plus one IEEE f32 addition per chunk for the running sum and per column share.  Non-finite
// approximations (overflow of the f16 conversions) put the token on the list.
// Measured (512 experts, d = 3072, top-10, nothing beside them; prep + f16 + pick, us): 515 tokens, f32 router 12 + 12 + 20; 2048 16 + 21 + 35,
// bf16 16 + 22 + 30; 4096 bf16 22 + 34 + 55; 16384 f32 62 + 90 + 190.  The f16 launch and the dot products of an f32 router (which two
// XCDs' L2s together could hold, one cannot) run at the L2s' rate, 10.5 TB/s; prep at the memory's.  (With the format's bound, eight lanes
// to a row, sixteen rows a pass whatever their number, x handed round through LDS and v_cvt_f64_f32, pick took 25, 41, 40, 65 and 222.)
#include <type_traits>

#include "common.h"
#include "internal.h"
#include "router_chain.h"
#include "rowx.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int RA_CHUNK = 128;  // columns summed in the matrix pipe's f32 accumulators before they are added to the running sums
constexpr int RA_KS = 4;       // column shares at most
constexpr int RA_NBUF = 4;     // slabs in LDS
constexpr int RC_SLOTS = 32;   // candidates per token at most
constexpr int RL_T = 16;       // listed tokens of a group

// Norm of a row's rounding errors from the sum of their squares; what underflow dropped from that is below the smallest normal
// float a column.
__device__ __forceinline__ float f16_err_norm(float sum2, int d) { return sqrtf(sum2 + (float)d * 1.2e-38f); }

// ---- 1. a wave per row: first the router matrix's, then x's ----
template <bool BF16>
__global__ void __launch_bounds__(256) k_router_prep(const void* __restrict__ W, int E, int d, __half* __restrict__ W16,
                                                     float* __restrict__ wnorm, float* __restrict__ xerr, int* __restrict__ hard,
                                                     const float* __restrict__ x, int P, moe_row_extras R) {
  const int lane = threadIdx.x & 63, nwb = (E + 3) >> 2;
  {  // the list's count and its tickets (first used two launches on)
    const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (i <= (P + RL_T - 1) / RL_T) hard[i] = 0;
  }
  if ((int)blockIdx.x < nwb) {
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= E) return;
    uint4* dst = (uint4*)W16 + (size_t)e * (d / 8);
    float s2 = 0.f, r2 = 0.f;
    for (int i = lane; i < d / 8; i += 64) {
      int ia, ib;
      f16_chunk_src(R.layout, i, ia, ib);
      float4 u, v;
      if (BF16) {
        const uint2* w = (const uint2*)((const uint16_t*)W + (size_t)e * d);
        const uint2 p = w[ia], q = w[ib];
        u = float4{__uint_as_float(p.x << 16), __uint_as_float(p.x & 0xffff0000u), __uint_as_float(p.y << 16), __uint_as_float(p.y & 0xffff0000u)};
        v = float4{__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xffff0000u), __uint_as_float(q.y << 16), __uint_as_float(q.y & 0xffff0000u)};
      } else {
        const float4* w = (const float4*)((const float*)W + (size_t)e * d);
        u = w[ia];
        v = w[ib];
      }
      s2 += ((u.x * u.x + u.y * u.y) + (u.z * u.z + u.w * u.w)) + ((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w));
      r2 += f16_err2(u) + f16_err2(v);
      dst[i] = f16_chunk(R.layout, u, v);
    }
    s2 = wave_sum(s2);
    r2 = wave_sum(r2);
    if (lane == 0) {
      wnorm[e] = sqrtf(s2);
      wnorm[E + e] = f16_err_norm(r2, d);
    }
    return;
  }
  const int t = ((int)blockIdx.x - nwb) * 4 + (threadIdx.x >> 6);
  if (t >= P) return;
  float acc, err = 0.f;
  double gate;
  row_extras_part(x, t, d, lane, 64, R, acc, gate, &err);
  acc = wave_sum(acc);
  err = wave_sum(err);
  if (R.wx) gate = wave_sum(gate);
  if (lane == 0) {
    row_extras_out(t, d, R, acc, gate);
    xerr[t] = f16_err_norm(err, d);
  }
}

// ---- 2. approximate logits: block = 64 MT tokens x 64 MT experts x one column share, 4 waves as 2 x 2 ----
// Both operands go global -> LDS in slabs of KB columns, RA_NBUF - 1 slabs ahead, one barrier per slab; 16-byte chunk c of row
// r lies in slot c ^ (r & 7) of a 128-byte row (64 bytes: c ^ ((r >> 2) & 3)), so that the fragment reads of 8 (16) rows
// cover all banks.  What bounds it is the latency of a slab at few blocks (d / 64 of them in a chain) and the L2's rate at many.
// So small tiles (64 x 64) with the columns split as long as that fills the chip, large ones (128 x 128, half the traffic)
// where there are enough of those.
template <int MT>
__global__ void __launch_bounds__(256, 2) k_router_f16(const __half* __restrict__ W16, const __half* __restrict__ x16, int P, int E,
                                                       int d, float* __restrict__ alog, int ncol, int ntt, int KS) {
  constexpr int BT = 64 * MT, KB = MT == 1 ? 64 : 32, ROW = 2 * KB, HALF = BT * ROW, BUF = 2 * HALF;
  constexpr int LPR = ROW / 16;               // lanes per row of a load
  constexpr int NI = BUF / 1024 / 4;          // loads per wave and slab
  static_assert(NI == 4, "wait counts below");
  __shared__ __attribute__((aligned(16))) uint8_t sm[RA_NBUF * BUF];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5, wm = wv >> 1, wn = wv & 1;
  // the blocks of a token tile share an XCD (and its L2 copy of x)
  const int b = blockIdx.x, xcd = b & 7, q = b >> 3, per = ncol * KS;
  const int sub = q % per, tt = (q / per) * 8 + xcd, col = sub % ncol, ks = sub / ncol;
  if (tt >= ntt) return;
  const int t0 = tt * BT, e0 = col * BT;
  const int nsl = d / KB, s0 = ks * nsl / KS, s1 = (ks + 1) * nsl / KS;
  // waves 0, 1 load activations, 2, 3 weights; rows past the end repeat the last one and are never stored
  const uint8_t* src[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int r = ((wv & 1) * NI + i) * (64 / LPR) + lane / LPR, slot = lane % LPR;
    const int c = KB == 64 ? slot ^ (r & 7) : slot ^ ((r >> 2) & 3);
    const int row = wv < 2 ? (t0 + r < P ? t0 + r : P - 1) : (e0 + r < E ? e0 + r : E - 1);
    src[i] = (const uint8_t*)((wv < 2 ? x16 : W16) + (size_t)row * d) + 16 * c;
  }
  auto issue = [&](int s) {
    uint8_t* dst = sm + (s - s0) % RA_NBUF * BUF + wv * (NI * 1024);
#pragma unroll
    for (int i = 0; i < NI; i++)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (size_t)s * ROW),
                                       (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
  };
  floatx16 acc[MT][MT], run[MT][MT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = run[i][j][r] = 0.f;
  auto slot_of = [](int c, int r) { return KB == 64 ? c ^ (r & 7) : c ^ ((r >> 2) & 3); };
#pragma unroll
  for (int i = 0; i < RA_NBUF - 1; i++)
    if (s0 + i < s1) issue(s0 + i);
  for (int s = s0; s < s1; s++) {
    // slab s has landed when at most the loads of the (up to two) later slabs in flight are outstanding
    const int later = s1 - 1 - s;
    if (later >= 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else if (later == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    moe_lds_barrier();  // everybody's part of slab s has landed; slab s - 1, whose buffer is filled next, has been read
    if (s + RA_NBUF - 1 < s1) issue(s + RA_NBUF - 1);
    const uint8_t* const Xb = sm + (s - s0) % RA_NBUF * BUF;
    const uint8_t* const Wb = Xb + HALF;
#pragma unroll
    for (int kk = 0; kk < KB / 16; kk++) {
      half8 a[MT], w[MT];
#pragma unroll
      for (int i = 0; i < MT; i++) {
        const int r = 32 * (MT * wm + i) + n;
        a[i] = *(const half8*)(Xb + r * ROW + (slot_of(2 * kk + h, r) << 4));
      }
#pragma unroll
      for (int j = 0; j < MT; j++) {
        const int r = 32 * (MT * wn + j) + n;
        w[j] = *(const half8*)(Wb + r * ROW + (slot_of(2 * kk + h, r) << 4));
      }
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < MT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[i], w[j], acc[i][j], 0, 0, 0);
    }
    if ((s - s0 + 1) % (RA_CHUNK / KB) == 0 || s + 1 == s1) {
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < MT; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            run[i][j][r] += acc[i][j][r];
            acc[i][j][r] = 0.f;
          }
    }
  }
  // D[i][j]: j = lane % 32 (expert), i = 8 * (r / 4) + 4 * (lane / 32) + r % 4 (token)
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int t = t0 + 32 * (MT * wm + i) + 8 * (r >> 2) + 4 * h + (r & 3);
      if (t >= P) continue;
#pragma unroll
      for (int j = 0; j < MT; j++) {
        const int e = e0 + 32 * (MT * wn + j) + n;
        if (e < E) alog[((size_t)ks * P + t) * E + e] = run[i][j][r];
      }
    }
}

// fp64 dot products of row x with up to sixteen weight rows (ids: lane i's register holds row i's index, n of them; the lanes
// past n repeat the last), columns c0 .. c1 - 1 of rows of ld (multiples of 64).  The wave keeps a panel of x in registers, four
// columns of every 256 to a lane, widened once, and lets the rows go past it two at a time, the next two requested before
// these are summed: a load covers 1 KB (bf16 512 bytes) of one row, no activation passes through LDS, and no more rows are
// multiplied than there are candidates (one more where their number is odd).  A lane's sums wait in LDS between panels,
// four rows' in a double of each lane: the launch runs beside the shared expert's GEMMs, which want the CUs' LDS (with a double of every
// lane and row, 38 KB a block, it was as fast alone and the layer no faster for it at 4096 tokens).
// What bounds it is widening the weights -- v_cvt_f64_f32 takes four times as long as an FMA -- next to the L2s' rate.  A float's
// exponent and mantissa shifted into a double's places are the value times 2^-896, zeros and subnormals included, so the
// weights are widened with shifts and x carries the 2^896 (|x| < 2^128: no overflow; infinities and NaNs never get here).
// The order of the sums is fixed.
constexpr int DR_ROWS = 16;              // rows of a pass
constexpr int DR_SUMS = DR_ROWS * 16;  // doubles of a wave's sums in LDS
// lanes' a and b -> half as many lanes' sums of each (lanes 0 .. 31 a's, the others b's; by 16: in rows of 16 lanes a, b, a, b)
template <bool BY32>
__device__ __forceinline__ double swap_add(double a, double b) {
  union U { double d; uint32_t i[2]; } x, y, p, q;
  x.d = a;
  y.d = b;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const auto s = BY32 ? __builtin_amdgcn_permlane32_swap(x.i[i], y.i[i], false, false) : __builtin_amdgcn_permlane16_swap(x.i[i], y.i[i], false, false);
    p.i[i] = s[0];
    q.i[i] = s[1];
  }
  return p.d + q.d;
}
__device__ __forceinline__ double widen_m896(uint32_t u) {
  union { double d; uint32_t i[2]; } r;
  r.i[0] = u << 29;
  r.i[1] = (u & 0x80000000u) | ((u >> 3) & 0x0fffffffu);
  return r.d;
}
__device__ __forceinline__ double widen_m896_hi(uint32_t u) {  // (a bf16 in the upper half; the lower half is zero)
  union { double d; uint32_t i[2]; } r;
  r.i[0] = 0u;
  r.i[1] = (u & 0x80000000u) | ((u >> 3) & 0x0fffffffu);
  return r.d;
}
// sums: DR_SUMS doubles of LDS owned by the wave.  Returns row lane % 16's sum.  PP: pieces of 256 columns in a panel.
template <bool BF16, int PP>
__device__ __forceinline__ double dot_rows(__amdgpu_buffer_rsrc_t W, const float* __restrict__ xrow, int ld, int c0, int c1, int ids, int n,
                                           int lane, double* sums) {
  constexpr int ESZ = BF16 ? 2 : 4, WPL = BF16 ? 2 : 4;  // words of four weights
  double* const mine = sums + lane;
  for (int p0 = c0; p0 < c1; p0 += 256 * PP) {
    int off[PP];
    float4 xv[PP];
#pragma unroll
    for (int i = 0; i < PP; i++) {  // (past the end: the first columns again, times zero)
      const int c = p0 + 256 * i + 4 * lane;
      off[i] = (c < c1 ? c : c0) * ESZ;
      xv[i] = *(const float4*)(xrow + (c < c1 ? c : c0));
    }
    uint32_t w[2][2][PP][WPL];  // [pair][row][piece]
    auto load = [&](int r, uint32_t(&q)[2][PP][WPL]) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int at = __builtin_amdgcn_readlane(ids, r + h < DR_ROWS ? r + h : DR_ROWS - 1) * (ld * ESZ);
#pragma unroll
        for (int i = 0; i < PP; i++) {
          if constexpr (BF16) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(W, off[i], at, 0);
            q[h][i][0] = v[0]; q[h][i][1] = v[1];
          } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(W, off[i], at, 0);
            q[h][i][0] = v[0]; q[h][i][1] = v[1]; q[h][i][2] = v[2]; q[h][i][3] = v[3];
          }
        }
      }
    };
    load(0, w[0]);
    double x[PP][4];
#pragma unroll
    for (int i = 0; i < PP; i++) {
      const float f[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
      const double s = p0 + 256 * i + 4 * lane < c1 ? 0x1p896 : 0.0;
#pragma unroll
      for (int k = 0; k < 4; k++) x[i][k] = (double)f[k] * s;
    }
    const bool first = p0 == c0;
    auto sum = [&](const uint32_t(&q)[2][PP][WPL]) {
      double a[2] = {0.0, 0.0};
#pragma unroll
      for (int i = 0; i < PP; i++)
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
          for (int h = 0; h < 2; h++) {
            double wd;
            if constexpr (BF16) wd = widen_m896_hi(k & 1 ? q[h][i][k >> 1] & 0xffff0000u : q[h][i][k >> 1] << 16);
            else wd = widen_m896(q[h][i][k]);
            a[h] = fma(wd, x[i][k], a[h]);
          }
      return swap_add<true>(a[0], a[1]);
    };
    // four rows' sums in the four rows of sixteen lanes: r, r + 2, r + 1, r + 3
#pragma unroll 1
    for (int r = 0; r < n; r += 4) {
      load(r + 2, w[1]);
      __builtin_amdgcn_sched_barrier(0);
      const double lo = sum(w[0]);
      __builtin_amdgcn_sched_barrier(0);
      load(r + 4, w[0]);
      __builtin_amdgcn_sched_barrier(0);
      double hi = 0.0;
      if (r + 2 < n) hi = sum(w[1]);
      __builtin_amdgcn_sched_barrier(0);
      const double v = swap_add<false>(lo, hi);
      mine[16 * r] = first ? v : mine[16 * r] + v;
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's own LDS writes
  __builtin_amdgcn_wave_barrier();
  // lane group g adds four of the sixteen lanes' sums of row lane % 16, two more steps add the groups'
  const int row = lane & 15;
  const double* const q = sums + 64 * (row >> 2) + 16 * (((row & 1) << 1) | (row >> 1 & 1)) + 4 * (lane >> 4);
  double v = 0.0;
  if (c1 > c0) {
#pragma unroll
    for (int i = 0; i < 4; i++) v += q[i];
  }
  v += __shfl_xor(v, 16, 64);
  v += __shfl_xor(v, 32, 64);
  __builtin_amdgcn_wave_barrier();
  return v;
}

// ---- 3. candidates, their exact logits, ids and weights ----
struct PickLds {
  __attribute__((aligned(16))) float lg[512];
  int cid[4][RC_SLOTS], sid[4][RC_SLOTS];
  double sums[4][DR_SUMS], part[4][DR_ROWS];  // [wave]
  float sval[4][RC_SLOTS], sel_ws[64];
  int sel_ids[64], zero[4], nzero;
};

// WPT: waves per token (1, 4).  With four, each wave takes a quarter of the columns of the exact dot products; all else runs
// in every wave alike, so that they agree on every branch.
template <bool BF16, int WPT, int PP>
__device__ __forceinline__ bool pick_token(PickLds& S, const float* __restrict__ alog, int KS, const float* __restrict__ wnorm, int P,
                                           int E, int d, int k, float eps, float bias_max, float xms, float xerr, int t, int lane,
                                           int wv, int* __restrict__ ids, float* __restrict__ ws, const moe_rfix& RF) {
  // |x| of what the matrix pipe has seen at most; a weight row's norm and error norm count (below) with cw and ce
  const float xn = sqrtf(xms * (float)d) + xerr, cw = 1.01f * (xerr + eps * xn), ce = 1.02f * xn;
  // lane l holds experts 8 l .. 8 l + 7
  float a[8], U[8], L[8];
  bool fin = isfinite(xn);
  float maxU = -INFINITY, maxB = 0.f;
  float v8[8], wn8[8], we8[8], bi8[8];
#pragma unroll
  for (int j = 0; j < 8; j++) v8[j] = wn8[j] = we8[j] = bi8[j] = 0.f;
  if (E % 8 == 0) {  // whole lanes, aligned rows
    if (8 * lane < E) {
      auto ld8 = [&](const float* p, float (&o)[8], bool add) {
        const float4 x0 = *(const float4*)p, x1 = *(const float4*)(p + 4);
        const float q[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = add ? o[j] + q[j] : q[j];
      };
      ld8(wnorm + 8 * lane, wn8, false);
      ld8(wnorm + E + 8 * lane, we8, false);
      for (int s = 0; s < KS; s++) ld8(alog + ((size_t)s * P + t) * E + 8 * lane, v8, s > 0);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int e = 8 * lane + j;
      if (e < E) {
        wn8[j] = wnorm[e];
        we8[j] = wnorm[E + e];
        for (int s = 0; s < KS; s++) v8[j] = s ? v8[j] + alog[((size_t)s * P + t) * E + e] : alog[(size_t)t * E + e];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (RF.bias && 8 * lane + j < E) bi8[j] = RF.bias[8 * lane + j];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int e = 8 * lane + j;
    a[j] = U[j] = L[j] = -INFINITY;
    // (an expert whose bias is minus infinity is switched off: its logit is the same minus infinity whatever the sum, its
    //  softmax term zero, and it is no candidate)
    if (e < E && !(bi8[j] == -INFINITY && isfinite(v8[j]))) {
      const float av = v8[j] + bi8[j];
      const float B = cw * wn8[j] + ce * we8[j] + 1e-6f * (1.f + fabsf(av));
      fin = fin && isfinite(av) && isfinite(B);
      a[j] = av;
      maxB = fmaxf(maxB, B);
      U[j] = av + B;
      L[j] = av - B;
    }
    maxU = fmaxf(maxU, U[j]);
  }
  maxU = wave_fmax_dpp(maxU);
  maxB = wave_fmax_dpp(maxB);
  if (!__all(fin)) return false;
  // tau = the k-th largest lower end: each lane's eight sorted, then k rounds of the largest head
#pragma unroll
  for (int pass = 0; pass < 8; pass++)
#pragma unroll
    for (int j = pass & 1; j + 1 < 8; j += 2) {
      const float p = L[j], q = L[j + 1];
      L[j] = fmaxf(p, q);
      L[j + 1] = fminf(p, q);
    }
  float tau = -INFINITY;
  for (int r = 0; r < k; r++) {
    tau = wave_fmax_dpp(L[0]);
    const bool me = lane == (int)__builtin_ctzll(__ballot(L[0] == tau) | (1ull << 63));  // drop one instance
#pragma unroll
    for (int j = 0; j < 7; j++) {
      const float cur = L[j], nxt = L[j + 1];
      L[j] = me ? nxt : cur;
    }
    const float last = L[7];
    L[7] = me ? -INFINITY : last;
  }
  const float thr = tau - 1e-5f;
  // the candidates' rows, by expert index
  int cnt = 0;
  uint64_t mine = 0;
#pragma unroll
  for (int j = 0; j < 8; j++) mine |= (uint64_t)(U[j] >= thr) << j;
  int pos = __popcll(mine), inc = pos;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  cnt = __builtin_amdgcn_readlane(inc, 63);
  if (cnt > RC_SLOTS || cnt < k || !(maxU - thr < 60.f) || !isfinite(tau)) return false;
  pos = inc - pos;
#pragma unroll
  for (int j = 0; j < 8; j++)
    if (mine >> j & 1) S.cid[wv][pos++] = 8 * lane + j;
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_wave_barrier();
  // exact logits, sixteen rows a pass
  const float tol = RF.tol[t];
  const float* xrow = RF.x + (size_t)t * d;
  const __amdgpu_buffer_rsrc_t W = __builtin_amdgcn_make_buffer_rsrc((void*)RF.W, 0, E * d * (BF16 ? 2 : 4), 0x00027000);
  bool doubt = false;
  float cv = -INFINITY;  // lane i < cnt: candidate i's logit
  for (int p0 = 0; p0 < cnt; p0 += DR_ROWS) {
    const int left = cnt - p0 < DR_ROWS ? cnt - p0 : DR_ROWS, s = lane & (DR_ROWS - 1);
    const int c0 = WPT == 1 ? 0 : d / 64 * wv / 4 * 64, c1 = WPT == 1 ? d : d / 64 * (wv + 1) / 4 * 64;  // (WPT 4: may be none)
    const double dot = dot_rows<BF16, PP>(W, xrow, d, c0, c1, S.cid[wv][p0 + (s < left ? s : left - 1)], left, lane, S.sums[wv]);
    if (lane < DR_ROWS) S.part[wv][lane] = dot;
    if (WPT == 1) {
      __builtin_amdgcn_s_waitcnt(0xC07F);
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
    const int i = lane - p0;
    if (i >= 0 && i < DR_ROWS && lane < cnt) {
      const double v = WPT == 1 ? S.part[wv][i] : (S.part[0][i] + S.part[1][i]) + (S.part[2][i] + S.part[3][i]);
      doubt = logit_doubtful(v, tol);
      cv = (float)v + (RF.bias ? RF.bias[S.cid[wv][lane]] : 0.f);
    }
    if (WPT > 1) __syncthreads();  // (S.part has been read)
  }
  doubt = __any(doubt);
  // rank
  const int ci = lane < cnt ? S.cid[wv][lane] : 0;
  int rank = 0;
  for (int i = 0; i < cnt; i++) {  // (equal logits: by expert index, which is the order of the list)
    const float o = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cv), i));
    rank += o > cv || (o == cv && i < lane) ? 1 : 0;
  }
  if (__any(lane < cnt && !isfinite(cv))) return false;
  if (lane < cnt) {
    S.sval[wv][rank] = cv;
    S.sid[wv][rank] = ci;
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_wave_barrier();
  const float la = lane < cnt ? S.sval[wv][lane] : -INFINITY, lb = lane + 1 < cnt ? S.sval[wv][lane + 1] : -INFINITY;
  const float lmax = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(la), 0));
  const int ia = lane < cnt ? S.sid[wv][lane] : 0, ib = lane + 1 < cnt ? S.sid[wv][lane + 1] : 0x7fffffff;
  // softmax terms: the candidates' exact, the others' (which only enter the normaliser) from the approximate logits
  float rest = 0.f;
#pragma unroll
  for (int j = 0; j < 8; j++) rest += (mine >> j & 1) ? 0.f : __expf(a[j] - lmax);
  const float term = lane < cnt ? (float)exp((double)la - (double)lmax) : 0.f;
  const double se = wave_dsum_dpp((double)rest + (double)term);
  // Rank r is certain against rank r + 1 where the logits differ by more than four half ulps of their probabilities
  // fl(fl(exp(l - max)) / s), 2.4e-7 (a doubtful token's logits may be an ulp off each, |dot| <= |logit| + |bias|).  Closer
  // logits that are the reference's own: equal probabilities go by expert index, so nothing is left to decide where the
  // better logit has the lower index; else the terms must be further apart than a probability's ulp (se within 10 %).
  bool good = true;
  if (lane < k) {
    const float need = doubt ? 1e-6f + 0x1p-22f * (fmaxf(fabsf(la), fabsf(lb)) + bias_max) : 3e-7f;
    good = lane + 1 >= cnt || la - lb > need;
    if (!good && !doubt) {
      const float next = (float)exp((double)lb - (double)lmax);
      int pe;
      (void)frexp(1.1 * (double)term / se, &pe);  // term / se < 2^pe: an ulp is at most 2^(pe - 24)
      good = ia < ib || (maxB < 0.09f && 0.9 * (double)(term - next) / se >= ldexp(1.0, pe - 24));
    }
    good = good && lmax - la < 70.f;
  }
  if (!__all(good)) return false;
  const float sc = (float)((double)term / se);
  double wsum = 0.0;
  for (int r = 0; r < k; r++) wsum += (double)__int_as_float(__builtin_amdgcn_readlane(__float_as_int(sc), r));  // selection order, as the reference's loop
  if (lane < k && (WPT == 1 || wv == 0)) {
    ids[lane] = ia;
    ws[lane] = (float)((double)sc / wsum);
  }
  return true;
}

// Batches up to this size give a token to four waves: with one, the chip holds a wave or less per SIMD that walks the 3072
// columns of all candidates by itself.  Four walk a quarter each, but each repeats the selection around it, which counts as
// soon as the SIMDs are full (three blocks per CU: 768 tokens).  The layer with one wave and with four, us, f32 router: 420 tokens 535
// and 530, 600 565 and 558, 700 572 and 567, 800 584.5 and 591, 1020 618 and 629; bf16: 300 553 and 551, 900 639 and 646.
constexpr int PICK_SPLIT_MAX = 768;

// The list of tokens for k_router_listed, ints: [0] their number, [1 + g] the tickets of group g, then the tokens.
__host__ __device__ constexpr int hard_first(int P) { return 1 + (P + RL_T - 1) / RL_T; }

template <bool BF16, int WPT, int PP>
__global__ void __launch_bounds__(256, 3) k_router_pick(const float* __restrict__ alog, int KS, const float* __restrict__ wnorm,
                                                        const float* __restrict__ xms, const float* __restrict__ xerr, int P, int E, int d,
                                                        int k, float eps, float bias_max, int* __restrict__ ids, float* __restrict__ ws, int id_stride,
                                                        int* __restrict__ hard, moe_rfix RF) {
  __shared__ __attribute__((aligned(16))) PickLds S;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t = WPT == 1 ? blockIdx.x * 4 + wv : blockIdx.x;
  if (tid == 0) S.nzero = 0;
  __syncthreads();
  if (t < P) {
    const bool ok = pick_token<BF16, WPT, PP>(S, alog, KS, wnorm, P, E, d, k, eps, bias_max, xms[t], xerr[t], t, lane, wv,
                                     ids + (size_t)t * id_stride, ws + (size_t)t * id_stride, RF);
    if (!ok && lane == 0 && (WPT == 1 || wv == 0)) {
      // an all-zero row (padding): every dot product is zero.  (A mean square that underflows: |dot| < 1e-17, no softmax term
      // moves.)
      if (xms[t] == 0.f) S.zero[atomicAdd(&S.nzero, 1)] = t;
      else hard[hard_first(P) + atomicAdd(hard, 1)] = t;
    }
  }
  __syncthreads();
  const int nzero = S.nzero;
  if (nzero == 0) return;
  // (one selection for all of them: their logits are the biases)
  for (int e = tid; e < E; e += 256) S.lg[e] = RF.bias ? RF.bias[e] : 0.f;
  __syncthreads();
  (void)topk_block<8, false, 256>(S.lg, S.sel_ids, S.sel_ws, E, k);
  __syncthreads();
  for (int i = 0; i < nzero; i++)
    if (tid < k) {
      ids[(size_t)S.zero[i] * id_stride + tid] = S.sel_ids[tid];
      ws[(size_t)S.zero[i] * id_stride + tid] = S.sel_ws[tid];
    }
}

// ---- 4. listed tokens: all E logits as the reference's chains, in groups of sixteen tokens x 64 experts to a block ----
// v_mfma_f64_16x16x4_f64 adds its four k slices one after the other (router.hip), so MFMAs over ascending columns are the
// reference's sums bit for bit and nothing is left in doubt.  A lane's 16-byte load holds four neighbouring columns of a row; the
// 4 x 4 exchange between lane groups and words turns them into the order of the slices: word q of lane group g = column
// 4 q + g of sixteen.  The block that draws a group's last ticket runs its softmax and top-k, a wave per token (hand-over of the
// logits as in k_router_mfma).
// A few tokens wait for one wave's chain of d / 4 dependent MFMAs, so a wave takes one tile (all 512 experts in one block: 280 us
// for one group).  Long lists are bound by the f64 pipe, where an operand's conversion from f32 counts for half an MFMA:
// there a wave takes 2 x 4 tiles, 6 conversions to 8 MFMAs for 2 to 1 (from RL_LONG tokens; all of 8192 tokens: 1050 -> 540 us).
// The router's launches, us (512 experts, d = 3072, f32; in brackets redone by the tokens' own blocks, and by the dense launch that
// was here before): one token of 300 130 (330, 224) where none takes 46 (43, 239); one of 2048 160 (364, 250); 40 of 2048 190
// (358, 264); all of 1024 190 (645, 442), of 2048 345 (1285, 470), of 8192 810 (3830, 1000), of 16384 1580 (-, 1560).  Nothing
// listed: 2.4 us.
constexpr int RL_E = 64, RL_GRID = 512, RL_LONG = 2560;
__device__ __forceinline__ void group_transpose(const float4& f, float (&o)[4]) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(f.x), __float_as_uint(f.z), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(f.y), __float_as_uint(f.w), false, false);
  const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto e = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  o[0] = __uint_as_float(c[0]); o[1] = __uint_as_float(c[1]); o[2] = __uint_as_float(e[0]); o[3] = __uint_as_float(e[1]);
}
// NT x NE: a wave's tiles of sixteen tokens and sixteen experts; RD: 16-column steps in flight.
template <bool BF16, int NT, int NE, int RD>
__device__ __forceinline__ void listed_groups(float (*lg)[512], float (*pbuf)[512], int* s_last, int* __restrict__ hard, int P, int E, int d,
                                              int k, float* logits, int* __restrict__ ids, float* __restrict__ ws, int id_stride,
                                              const moe_rfix& RF) {
  typedef double double4v __attribute__((ext_vector_type(4)));
  constexpr int T = RL_T * NT, EB = 64 * NE;  // tokens and experts of a block
  const int n = hard[0];
  const int* const list = hard + hard_first(P);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, g = lane >> 4, nst = d / 16;
  const int nrb = (E + EB - 1) / EB, nitem = (n + T - 1) / T * nrb;
  for (int item = blockIdx.x; item < nitem; item += gridDim.x) {
    const int grp = item / nrb, i0 = grp * T, e0 = (item % nrb) * EB + 16 * NE * wv + li;
    // rows past the end: the group's first token, the matrix's last row; not stored
    const float* xp[NT];
#pragma unroll
    for (int m = 0; m < NT; m++) xp[m] = RF.x + (size_t)list[i0 + 16 * m + li < n ? i0 + 16 * m + li : i0] * d + 4 * g;
    const uint8_t* wp[NE];
#pragma unroll
    for (int q = 0; q < NE; q++) wp[q] = (const uint8_t*)RF.W + ((size_t)(e0 + 16 * q < E ? e0 + 16 * q : E - 1) * d + 4 * g) * (BF16 ? 2 : 4);
    float4 xr[RD][NT], wr[RD][NE];
    auto fetch = [&](int j, int s) {
      s = s < nst ? s : nst - 1;  // (past the end: a repeat that is never used)
#pragma unroll
      for (int m = 0; m < NT; m++) xr[j][m] = *(const float4*)(xp[m] + (size_t)s * 16);
#pragma unroll
      for (int q = 0; q < NE; q++) {
        if (BF16) {
          const uint2 u = *(const uint2*)(wp[q] + (size_t)s * 32);
          wr[j][q].x = __uint_as_float(u.x); wr[j][q].y = __uint_as_float(u.y);
        } else {
          wr[j][q] = *(const float4*)(wp[q] + (size_t)s * 64);
        }
      }
    };
    double4v acc[NT][NE];
#pragma unroll
    for (int m = 0; m < NT; m++)
#pragma unroll
      for (int q = 0; q < NE; q++) acc[m][q] = double4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < RD; j++) fetch(j, j);
    for (int sb = 0; sb < nst; sb += RD) {
#pragma unroll
      for (int j = 0; j < RD; j++) {
        if (sb + j < nst) {
          float xt[NT][4], wt[NE][4];
#pragma unroll
          for (int m = 0; m < NT; m++) group_transpose(xr[j][m], xt[m]);
#pragma unroll
          for (int q = 0; q < NE; q++) {
            float4 f = wr[j][q];
            if (BF16) {
              const uint32_t u = __float_as_uint(f.x), v = __float_as_uint(f.y);
              f = float4{__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u), __uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)};
            }
            group_transpose(f, wt[q]);
          }
          fetch(j, sb + j + RD);
#pragma unroll
          for (int c = 0; c < 4; c++)
#pragma unroll
            for (int m = 0; m < NT; m++)
#pragma unroll
              for (int q = 0; q < NE; q++)
                acc[m][q] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)xt[m][c], (double)wt[q][c], acc[m][q], 0, 0, 0);
        }
      }
    }
    // D value r of lane l = [token 4r + l/16][expert l%16]
#pragma unroll
    for (int m = 0; m < NT; m++)
#pragma unroll
      for (int q = 0; q < NE; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int i = i0 + 16 * m + 4 * r + g, e = e0 + 16 * q;
          if (i < n && e < E)
            __hip_atomic_store(&logits[(size_t)i * E + e], (float)acc[m][q][r] + (RF.bias ? RF.bias[e] : 0.f), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    if (tid == 0) *s_last = __hip_atomic_fetch_add(&hard[1 + grp], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nrb - 1;
    __syncthreads();
    if (!*s_last) continue;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    for (int h = 0; h < NT; h++) {
      const int ih = i0 + 16 * h, nt = n - ih < RL_T ? n - ih : RL_T;
      for (int j = tid; j < nt * 512; j += 256)
        if ((j & 511) < E)
          lg[j >> 9][j & 511] = __hip_atomic_load(&logits[(size_t)(ih + (j >> 9)) * E + (j & 511)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
#pragma unroll 1
      for (int i = wv; i < nt; i += 4) {
        const size_t row = (size_t)list[ih + i] * id_stride;
        topk_wave<8>(lg[i], ids + row, ws + row, E, k, pbuf[wv]);
      }
      __syncthreads();  // (before the next logits)
    }
  }
}
template <bool BF16>
__global__ void __launch_bounds__(256, 2) k_router_listed(int* __restrict__ hard, int P, int E, int d, int k, float* logits,
                                                       int* __restrict__ ids, float* __restrict__ ws, int id_stride, moe_rfix RF) {
  __shared__ __attribute__((aligned(16))) float lg[RL_T][512];
  __shared__ __attribute__((aligned(16))) float pbuf[4][512];
  __shared__ int s_last;
  const int n = hard[0];
  if (n == 0) return;
  if (n < RL_LONG) listed_groups<BF16, 1, 1, 6>(lg, pbuf, &s_last, hard, P, E, d, k, logits, ids, ws, id_stride, RF);
  else listed_groups<BF16, 2, 4, 3>(lg, pbuf, &s_last, hard, P, E, d, k, logits, ids, ws, id_stride, RF);
}

// Tiles of the f16 launch, and column shares as far as two blocks per CU.  Either tile moves 10.5 TB/s out of the L2s, so the
// large one, with half the traffic, is the faster from the size on at which its shares fill the chip: 15.1 against 16.7 us at
// 2048 x 512 (64 large tiles), 27.4 against 23.6 at 3001 (96), 44.5 against 31 at 5000.
constexpr int RA_SLOTS = 512;
struct F16Shape {
  int mt, ncol, ntt, ks;
};
F16Shape f16_shape(int P, int E, int d) {
  F16Shape s;
  s.mt = (int64_t)((P + 127) / 128) * ((E + 127) / 128) >= 80 ? 2 : 1;
  s.ncol = (E + 64 * s.mt - 1) / (64 * s.mt);
  s.ntt = (P + 64 * s.mt - 1) / (64 * s.mt);
  s.ks = 1;
  while (s.ks < RA_KS && s.ncol * s.ntt * (s.ks + 1) <= RA_SLOTS && d / 64 / (s.ks + 1) >= 8) s.ks++;
  return s;
}

}  // namespace

bool moe_router_cand_supported(const moe_wview* W, int P, int k) {
  const int E = (int)W->rows, d = (int)W->cols;
  if (P < 1 || d % 64 || d < 64 || E > 512 || k + 1 > RC_SLOTS - 1 || k >= E) return false;
  if ((uint64_t)E * (uint64_t)d * 4 >= 1ull << 31) return false;  // (32-bit byte offsets of the candidates' rows)
  return moe_aligned(W->data, 16);
}

static size_t rc_hard_bytes(int tokens) { return ((size_t)(hard_first(tokens) + tokens) * 4 + 255) / 256 * 256; }
static size_t rc_wnorm_bytes(int experts) { return ((size_t)experts * 8 + 255) / 256 * 256; }
static size_t rc_xerr_bytes(int tokens) { return ((size_t)tokens * 4 + 255) / 256 * 256; }
size_t moe_router_cand_scratch_bytes(int max_tokens, int experts, int d) {
  // the rows' norms and error norms (W 2 E, x), the router matrix as f16, the column shares' partial logits (as long as there are shares: at most RA_SLOTS tiles)
  const size_t tiles = (size_t)RA_SLOTS * 128 * 128 * 4, all = (size_t)RA_KS * max_tokens * experts * 4;
  // and the list of hard tokens in front of all
  return rc_hard_bytes(max_tokens) + rc_wnorm_bytes(experts) + rc_xerr_bytes(max_tokens) + (size_t)experts * d * 2 + 256 + (all < tiles ? all : tiles);
}

// Internal: ids / ws of a batch; `logits` [P][E] is scratch.
int moe_router_batch_cand(const moe_wview* W, const float* x, int P, float* logits, int* ids, float* ws, int k, int id_stride,
                          void* scratch, const moe_row_extras& R, const moe_rfix& RF, float bias_max, hipStream_t st,
                          hipEvent_t after_rows) {
  const int E = (int)W->rows, d = (int)W->cols;
  if (!moe_router_cand_supported(W, P, k) || !moe_aligned(x, 16) || !R.x16 || !R.xms || !R.tol) return MOE_E_UNSUPPORTED;
  int* const hard = (int*)scratch;
  float* wnorm = (float*)((uint8_t*)scratch + rc_hard_bytes(P));
  float* xerr = (float*)((uint8_t*)wnorm + rc_wnorm_bytes(E));
  __half* W16 = (__half*)((uint8_t*)xerr + rc_xerr_bytes(P));
  const F16Shape s = f16_shape(P, E, d);
  float* alog = s.ks == 1 ? logits : (float*)((uint8_t*)W16 + ((size_t)E * d * 2 + 255) / 256 * 256);
  // 1.002: second-order terms; 1.01: the f32 norms' own rounding
  const float eps = ((float)RA_CHUNK * 0x1p-22f + (float)(d / RA_CHUNK + 1 + RA_KS) * 0x1p-23f) * 1.002f * 1.01f;
  const bool bf = W->dtype == MOE_DT_BF16;
  const unsigned g1 = (unsigned)((E + 3) / 4 + (P + 3) / 4), g3 = (unsigned)((P + 3) / 4);
  const unsigned g2 = (unsigned)((s.ntt + 7) / 8 * 8 * s.ncol * s.ks);
  if (bf) k_router_prep<true><<<g1, 256, 0, st>>>(W->data, E, d, W16, wnorm, xerr, hard, x, P, R);
  else k_router_prep<false><<<g1, 256, 0, st>>>(W->data, E, d, W16, wnorm, xerr, hard, x, P, R);
  MOE_LAUNCH_CHECK();
  if (after_rows) MOE_HIP(hipEventRecord(after_rows, st));
  if (s.mt == 2) k_router_f16<2><<<g2, 256, 0, st>>>(W16, (const __half*)R.x16, P, E, d, alog, s.ncol, s.ntt, s.ks);
  else k_router_f16<1><<<g2, 256, 0, st>>>(W16, (const __half*)R.x16, P, E, d, alog, s.ncol, s.ntt, s.ks);
  MOE_LAUNCH_CHECK();
  // panels of three, four or five pieces: what leaves the fewest empty pieces (3001 tokens, d = 3072, f32: four 41.5 us, three 42.2)
  const int pieces = ((P <= PICK_SPLIT_MAX ? (d / 64 + 3) / 4 * 64 : d) + 255) / 256;
  int pp = 4;
  for (int i = 3; i <= 5; i += 2)
    if ((pieces + i - 1) / i * i < (pieces + pp - 1) / pp * pp) pp = i;
#define PICK_PP(BF, WPT, PP) k_router_pick<BF, WPT, PP><<<WPT == 1 ? g3 : (unsigned)P, 256, 0, st>>>(alog, s.ks, wnorm, R.xms, xerr, P, E, d, k, eps, bias_max, ids, ws, id_stride, hard, RF)
#define PICK_GO(BF, WPT)                    \
  do {                                      \
    if (pp == 3) PICK_PP(BF, WPT, 3);       \
    else if (pp == 4) PICK_PP(BF, WPT, 4);  \
    else PICK_PP(BF, WPT, 5);               \
  } while (0)
  if (P <= PICK_SPLIT_MAX) {
    if (bf) PICK_GO(true, 4);
    else PICK_GO(false, 4);
  } else {
    if (bf) PICK_GO(true, 1);
    else PICK_GO(false, 1);
  }
#undef PICK_PP
#undef PICK_GO
  MOE_LAUNCH_CHECK();
  const int items = (P + RL_T - 1) / RL_T * ((E + RL_E - 1) / RL_E);
  const unsigned g4 = (unsigned)(items < RL_GRID ? items : RL_GRID);
  if (bf) k_router_listed<true><<<g4, 256, 0, st>>>(hard, P, E, d, k, logits, ids, ws, id_stride, RF);
  else k_router_listed<false><<<g4, 256, 0, st>>>(hard, P, E, d, k, logits, ids, ws, id_stride, RF);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}
