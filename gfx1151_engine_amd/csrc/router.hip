// Router: logits with the CPU path's fp64 accumulation, fp64 softmax, top-k, renormalised weights.
// (reference: src/ref.cpp:68-77,565-594; src/gpu/parts/20_kernels_gemv.inc:1433-1562)
#include "common.h"
#include "hv2.h"
#include "internal.h"
#include "qvec.h"
#include "rowx.h"
#include "topk.h"

namespace {

template <bool BF16>
__device__ __forceinline__ float load_w(const void* W, uint64_t i) {
  if (BF16) return bf16_bits_to_f32(((const uint16_t*)W)[i]);
  return ((const float*)W)[i];
}

// ---- sequential order: bit-identical to `acc += (double)w*x` for c = 0..d-1 ----
// The f32*f32 product is exact in fp64, so a chain of fp64 FMAs over c = 0..d-1 equals the
// reference's multiply-then-add.  v_mfma_f64_16x16x4_f64 is such a chain: it adds its four k
// slices to the accumulator one after the other, each with a single FMA rounding (lane group
// l/16 supplies slice k; checked bit for bit against host fma chains over 3072-long sums with
// heavy cancellation), so successive MFMAs over ascending c reproduce the CPU sum exactly while
// the fp64 work runs on the matrix pipe.
// Block = BT tokens x 128 weight rows, 4 waves as 2 x 2, wave = BT/2 tokens x 64 rows.  Operands
// are staged in LDS as f32 (k permuted so that one 16-byte read feeds four MFMAs) and widened in
// registers; the next K slab is fetched into registers while the current one is consumed.
// D layout: value r of lane l is token 4r + l/16, weight row l%16 of the 16 x 16 tile.
// Block ids are dealt so that the column blocks of one
// token tile run on the same XCD (ids that differ by 8) and share its L2 copy of the activations.
typedef double double4v __attribute__((ext_vector_type(4)));
constexpr int RS_E = 128, RS_K = 32, RS_PITCH = 36;
template <bool BF16, int BT>
__global__ void __launch_bounds__(256, 2) k_router_logits_seq(const void* __restrict__ W,
                                                           const float* __restrict__ bias,
                                                           const float* __restrict__ x, int P, int E,
                                                           int d, float* __restrict__ logits, int ncol, int ntt) {
  constexpr int MT = BT / 32;                 // 16-token MFMA tiles per wave
  constexpr int XL = (BT * RS_K / 4) / 256;   // float4 loads per thread and slab (activations)
  constexpr int WL = (RS_E * RS_K / 4) / 256; // (weights)
  __shared__ __attribute__((aligned(16))) float Xs[BT][RS_PITCH];
  __shared__ __attribute__((aligned(16))) float Ws[RS_E][RS_PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int li = lane & 15, lg = lane >> 4, wm = wv >> 1, wn = wv & 1;
  const int b = blockIdx.x, xcd = b & 7, q = b >> 3;
  const int col = q % ncol, tt = (q / ncol) * 8 + xcd;
  if (tt >= ntt) return;
  const int e0 = col * RS_E, t0 = tt * BT;
  const bool vec = (d % 4 == 0);

  auto fetch_x = [&](int c0, float4* v) {
#pragma unroll
    for (int it = 0; it < XL; it++) {
      const int i = tid + it * 256, r = i >> 3, cc = c0 + (i & 7) * 4;
      const int t = t0 + r;
      float4 f = {0.f, 0.f, 0.f, 0.f};
      if (t < P) {
        const float* src = x + (size_t)t * d + cc;
        if (vec && cc + 3 < d) f = *(const float4*)src;
        else {
          if (cc < d) f.x = src[0];
          if (cc + 1 < d) f.y = src[1];
          if (cc + 2 < d) f.z = src[2];
          if (cc + 3 < d) f.w = src[3];
        }
      }
      v[it] = f;
    }
  };
  auto fetch_w = [&](int c0, float4* v) {
#pragma unroll
    for (int it = 0; it < WL; it++) {
      const int i = tid + it * 256, r = i >> 3, cc = c0 + (i & 7) * 4;
      const int e = e0 + r;
      float4 f = {0.f, 0.f, 0.f, 0.f};
      if (e < E) {
        const uint64_t o = (uint64_t)e * d + cc;
        if (vec && cc + 3 < d) {
          if (BF16) {
            const uint2 u = *(const uint2*)((const uint16_t*)W + o);
            f.x = __uint_as_float(u.x << 16); f.y = __uint_as_float(u.x & 0xffff0000u);
            f.z = __uint_as_float(u.y << 16); f.w = __uint_as_float(u.y & 0xffff0000u);
          } else {
            f = *(const float4*)((const float*)W + o);
          }
        } else {
          if (cc < d) f.x = load_w<BF16>(W, o);
          if (cc + 1 < d) f.y = load_w<BF16>(W, o + 1);
          if (cc + 2 < d) f.z = load_w<BF16>(W, o + 2);
          if (cc + 3 < d) f.w = load_w<BF16>(W, o + 3);
        }
      }
      v[it] = f;
    }
  };
  // slab element k (0..31) of a row sits at [ (k & 3) * 8 + (k >> 2) ]: lane group g reads its
  // slices k = 4*kk + g for kk = 0..7 as two float4
  auto stage = [&](float (*dst)[RS_PITCH], const float4* v, int n) {
#pragma unroll
    for (int it = 0; it < n; it++) {
      const int i = tid + it * 256, r = i >> 3, m = i & 7;
      dst[r][m] = v[it].x; dst[r][8 + m] = v[it].y; dst[r][16 + m] = v[it].z; dst[r][24 + m] = v[it].w;
    }
  };

  double4v acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = double4v{0.0, 0.0, 0.0, 0.0};

  float4 xr[XL], wr[WL];
  fetch_x(0, xr);
  fetch_w(0, wr);
  for (int c0 = 0; c0 < d; c0 += RS_K) {
    moe_lds_barrier();  // everybody is done reading the previous slab (LDS-only barriers: the next slab's loads stay in flight)
    stage(Xs, xr, XL);
    stage(Ws, wr, WL);
    moe_lds_barrier();
    if (c0 + RS_K < d) {
      fetch_x(c0 + RS_K, xr);
      fetch_w(c0 + RS_K, wr);
    }
#pragma unroll
    for (int half = 0; half < 2; half++) {
      float4 xa[MT], wb[4];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) xa[mt] = *(const float4*)&Xs[wm * (BT / 2) + 16 * mt + li][lg * 8 + 4 * half];
#pragma unroll
      for (int nt = 0; nt < 4; nt++) wb[nt] = *(const float4*)&Ws[wn * 64 + 16 * nt + li][lg * 8 + 4 * half];
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        double a[MT], bq[4];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) a[mt] = (double)(kk == 0 ? xa[mt].x : kk == 1 ? xa[mt].y : kk == 2 ? xa[mt].z : xa[mt].w);
#pragma unroll
        for (int nt = 0; nt < 4; nt++) bq[nt] = (double)(kk == 0 ? wb[nt].x : kk == 1 ? wb[nt].y : kk == 2 ? wb[nt].z : wb[nt].w);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int nt = 0; nt < 4; nt++)
            acc[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mt], bq[nt], acc[mt][nt], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = t0 + wm * (BT / 2) + 16 * mt + 4 * r + lg;
      if (t >= P) continue;
#pragma unroll
      for (int nt = 0; nt < 4; nt++) {
        const int e = e0 + wn * 64 + 16 * nt + li;
        if (e >= E) continue;
        float v = (float)acc[mt][nt][r];
        if (bias) v += bias[e];
        logits[(size_t)t * E + e] = v;
      }
    }
  }
}

// The blocks past the rows of the small-batch router launches: the digit planes of x for the integer-dot decode
// kernels (a thread per 32-element group) and, for hgn v2 layers, the planes of rot_in(x, pre) = H(pre . x) / sqrt(128)
// (a thread per 8 elements, 16 lanes per 128-block) -- work that rides along instead of costing a launch.
// q = index among these blocks, bs = block size.
__device__ __forceinline__ void router_plane_blocks(int q, int bs, int tid, const float* __restrict__ x, int P, int d,
                                                    uint32_t* __restrict__ planes, float2* __restrict__ meta,
                                                    bool planes_natural, const moe_rot_planes& R) {
  const int G = d / 32, gb = (G + bs - 1) / bs;
  const int nq = planes ? P * gb : 0;
  if (q < nq) {
    const int t = q / gb, g = (q % gb) * bs + tid;
    if (t < P && g < G) {
      if (planes_natural) qvec_group_from_f32(x, (uint64_t)d, G, t, g, planes, meta);  // GGUF kernels
      else qvec4_group_from_f32(x, (uint64_t)d, G, t, g, planes, meta);                       // q4cp kernels
    }
    return;
  }
  if (!R.planes) return;
  q -= nq;
  const int per_row = d / 8, rb = (per_row + bs - 1) / bs;
  const int t = q / rb, c8 = (q % rb) * bs + tid;
  const bool live = t < P && c8 < per_row;  // (whole groups of 16 lanes: d % 128 == 0)
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = 0.f;
  if (live) {
    const float4* xp = (const float4*)(x + (size_t)t * d + 8 * c8);
    const float4* pp = (const float4*)(R.pre + 8 * c8);
    const float4 a = xp[0], b = xp[1], e = pp[0], f = pp[1];
    v[0] = a.x * e.x; v[1] = a.y * e.y; v[2] = a.z * e.z; v[3] = a.w * e.w;
    v[4] = b.x * f.x; v[5] = b.y * f.y; v[6] = b.z * f.z; v[7] = b.w * f.w;
  }
  moe_fwht128_r8(v, tid);
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] *= MOE_RS128;
  moe_st8_planes(v, tid, R.planes, R.meta, (size_t)t * G + (c8 >> 2), live);
}

// ---- lane-parallel order for 1..4 tokens: one wave per weight row (two rows per block, so that 513 rows cover every CU),
// lanes stride the columns, four independent fp64 chains per lane and token, fixed combination order.  The fp64
// sum differs from the sequential one only in its last bits, so the f32 logit differs with
// probability ~1e-8 per value.  Row E (if Wx given) is the shared-expert gate vector: out_x[t] =
// its logit.  Blocks past the rows (if planes given) turn x into the digit planes of the
// integer-dot decode kernels, so that work rides along instead of costing a launch.
// What bounds it is one trip to memory: a wave's twelve loads of its row (3072 columns) are requested before anything
// is used, with nothing conditional between them.  The weight type and the token count are therefore template
// arguments, and the next token's activations are requested while one token is summed: with the type tested in the loop (the gate vector may differ from the matrix) and tokens tested per
// column step, each step waited for its own loads (512 experts, 3072 columns, bf16 matrix and f32 gate vector: one token 8.4 us,
// three tokens 16.2; now 4.0 and 5.9).  One token on an f32 matrix, where the compiler had untangled the loop: 4.1 before and
// now; with all weights requested ahead of all activations instead of pair by pair 4.5.
// Four tokens take 306 of the 512 registers a wave can have (AGPRs among them).  One body serves rows of any length: with a
// second copy for passes that lie wholly inside the row, without the selects below, three tokens of 3072 columns gain 1 us
// of 120 in two layers, and the compiler keeps 415 registers of the four-token kernel in scratch: 98 -> 130 us (q4cp), 150 ->
// 190 (Q5_K / Q8_0).
// Column steps of 256 requested together: what registers and one trip allow.  Steps past the row's end load its head again.
// Two q4cp layers of 1 / 2 / 3 / 4 tokens, us, against one load in flight per step: 1024 columns 34 / 39 / 48 / 58 (34 / 42 /
// 53 / 60), 2048 37 / 53 / 63 / 78 (42 / 60 / 74 / 93), 2560 38 / 46 / 63 / 80 (45 / 57 / 78 / 94), 4096 86 / 130 / 127 /
// 148 (93 / 148 / 149 / 178), 5120 99 / 134 / 165 / 200 (109 / 158 / 206 / 257).
constexpr int RSM_IT = 12;
template <bool BF>
struct RsmW {
  typedef gate_f32x4 T;
};
template <>
struct RsmW<true> {
  typedef gate_bf16x4 T;
};
template <bool BF, int TT>
__device__ __forceinline__ void router_small_row(const void* __restrict__ Wr, const float* __restrict__ x, int d, int lane,
                                                 bool norms, double (&sum)[TT], float (&n2)[TT]) {
  typedef typename RsmW<BF>::T WT;
  double acc[TT][4];
  float xs[TT];
#pragma unroll
  for (int i = 0; i < TT; i++) {
    xs[i] = 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++) acc[i][q] = 0.0;
  }
  for (int c0 = 0; c0 < d; c0 += 256 * RSM_IT) {
    WT w[RSM_IT];
    float4 xv[2][RSM_IT];  // a token's activations, and the next one's
    auto load_x = [&](int i, int j) {
      const int c = c0 + 256 * j + 4 * lane;
      xv[i & 1][j] = *(const float4*)(x + (size_t)i * d + (c < d ? c : 0));
    };
#pragma unroll
    for (int j = 0; j < RSM_IT; j++) {
      const int c = c0 + 256 * j + 4 * lane;
      w[j] = *(const WT*)((const uint8_t*)Wr + (size_t)(c < d ? c : 0) * (BF ? 2 : 4));  // (past the row: its head, not used)
      load_x(0, j);  // (in the order of use: the sums start when the first pair is there)
    }
#pragma unroll
    for (int i = 0; i < TT; i++) {
#pragma unroll
      for (int j = 0; j < RSM_IT; j++)
        if (i + 1 < TT) load_x(i + 1, j);
      __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, not next to their uses
#pragma unroll
      for (int j = 0; j < RSM_IT; j++) {
        // (columns past the row count as zeros: selects, where a branch would make the step wait for its own loads)
        const bool in = c0 + 256 * j + 4 * lane < d;
        float4 wf, xf = xv[i & 1][j];
        if constexpr (BF) {
          wf.x = __uint_as_float(w[j].x << 16);
          wf.y = __uint_as_float(w[j].x & 0xffff0000u);
          wf.z = __uint_as_float(w[j].y << 16);
          wf.w = __uint_as_float(w[j].y & 0xffff0000u);
        } else {
          wf = float4{w[j].x, w[j].y, w[j].z, w[j].w};
        }
        wf = in ? wf : float4{0.f, 0.f, 0.f, 0.f};
        xf = in ? xf : float4{0.f, 0.f, 0.f, 0.f};
        acc[i][0] = fma((double)wf.x, (double)xf.x, acc[i][0]);
        acc[i][1] = fma((double)wf.y, (double)xf.y, acc[i][1]);
        acc[i][2] = fma((double)wf.z, (double)xf.z, acc[i][2]);
        acc[i][3] = fma((double)wf.w, (double)xf.w, acc[i][3]);
        xs[i] += xf.x * xf.x + xf.y * xf.y + xf.z * xf.z + xf.w * xf.w;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TT; i++) {
    sum[i] = wave_sum((acc[i][0] + acc[i][1]) + (acc[i][2] + acc[i][3]));
    n2[i] = norms ? wave_sum(xs[i]) : 0.f;
  }
}

template <bool BF16, int TT>
__global__ void __launch_bounds__(128) k_router_small(const void* __restrict__ W, const float* __restrict__ bias,
                                                      const void* __restrict__ Wx, bool wx_bf16,
                                                      const float* __restrict__ x, int E, int d,
                                                      float* __restrict__ logits, float* __restrict__ out_x,
                                                      int nrows, uint32_t* __restrict__ planes,
                                                      float2* __restrict__ meta, bool planes_natural, moe_rot_planes rot,
                                                      float* __restrict__ tol_out, float tol_scale) {
  // the wave index as a scalar: row, weight type and base address are then wave-uniform values
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nrb = (nrows + 1) / 2;
  if ((int)blockIdx.x >= nrb) {
    router_plane_blocks((int)blockIdx.x - nrb, (int)blockDim.x, (int)threadIdx.x, x, TT, d, planes, meta, planes_natural, rot);
    return;
  }
  const int row = blockIdx.x * 2 + wv;
  if (row >= nrows) return;
  const bool extra = row == E;
  // the wave of row 0 also takes |x|^2 of every token: the selection that follows needs a bound on how far these
  // sums (lanes, then a tree) can lie from the reference's sequential ones, tol_scale * |x|
  const bool norms = tol_out && row == 0;
  double sum[TT];
  float n2[TT];
  if (extra && wx_bf16 != BF16) router_small_row<!BF16, TT>(Wx, x, d, lane, false, sum, n2);
  else router_small_row<BF16, TT>(extra ? Wx : (const void*)((const uint8_t*)W + (uint64_t)row * d * (BF16 ? 2 : 4)), x, d, lane, norms, sum, n2);
  if (lane != 0) return;
#pragma unroll
  for (int i = 0; i < TT; i++) {
    if (norms) {
      const float tl = tol_scale * sqrtf(n2[i]) * 1.01f;
      tol_out[i] = tl >= 0.f ? tl : INFINITY;  // (NaN: nothing is certain)
    }
    float v = (float)sum[i];
    if (extra) {
      out_x[i] = v;
    } else {
      if (bias) v += bias[row];
      logits[(size_t)i * E + row] = v;
    }
  }
}

// ---- lane-parallel order for 5..32 tokens: four weight rows per block (a wave each); the tokens'
// activations are widened to fp64 ONCE per block and 128-column slab (in LDS) instead of once per
// row, and every weight is read once for all tokens.  Lane l owns columns 2l, 2l+1 of each slab:
// two fp64 chains per token, combined in a fixed order, then the wave sum.  Same accuracy
// statement as k_router_small.  Blocks past the rows build the digit planes of x.
constexpr int RM_C = 128, RM_D = 4;
template <bool BF16, int PMAX>  // PMAX 8 / 16 / 24
__global__ void __launch_bounds__(256) k_router_mid(const void* __restrict__ W, const float* __restrict__ bias,
                                                    const void* __restrict__ Wx, bool wx_bf16,
                                                    const float* __restrict__ x, int P, int E, int d,
                                                    float* __restrict__ logits, float* __restrict__ out_x,
                                                    int nrows, uint32_t* __restrict__ planes,
                                                    float2* __restrict__ meta, bool planes_natural, moe_rot_planes rot) {
  __shared__ __attribute__((aligned(16))) double Xd[2][PMAX][RM_C];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nrb = (nrows + 3) >> 2;
  if ((int)blockIdx.x >= nrb) {
    router_plane_blocks((int)blockIdx.x - nrb, 256, tid, x, P, d, planes, meta, planes_natural, rot);
    return;
  }
  // the wave's row as scalar values: the bf16 / f32 choice is then a scalar branch
  const int row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(wv);
  // (without a gate vector row E is padding like every row past it: it must not take Wx, a null pointer then)
  const bool live = row < nrows, extra = Wx != nullptr && row == E;
  const void* Wr = extra ? Wx : W;
  const uint64_t base = (extra || !live) ? 0 : (uint64_t)row * d;  // rows past the matrix read row 0, never stored
  const bool bf = extra ? wx_bf16 : BF16;
  constexpr int XR = PMAX * RM_C / 256;  // staged activations per thread and slab
  // Register ring of RM_D slabs: slot j holds slab s with s % RM_D == j and is refilled for slab
  // s + RM_D as soon as slab s has gone to LDS, so every load has RM_D slab times to arrive
  // (one slab ahead left the loop waiting a full memory latency per 128 columns).
  // All loads are unconditional (clamped address, value times 0 or 1) and weights stay as raw
  // bits until they are used: a load under a divergent branch, or converted where it is issued,
  // makes the wave wait for every load in flight.  (d is even: c + 1 < d whenever c < d.)
  float xr[RM_D][XR];
  uint2 wr[RM_D];
  auto fetch = [&](int j, int c0) {
#pragma unroll
    for (int i = 0; i < XR; i++) {
      const int e = tid + 256 * i, t = e / RM_C, c = c0 + e % RM_C;
      const bool ok = t < P && c < d;
      xr[j][i] = x[ok ? (size_t)t * d + c : 0] * (ok ? 1.f : 0.f);
    }
    const int c = c0 + 2 * lane;
    const int cc = c < d ? c : 0;
    // two 32-bit loads in either format (bf16: the same word twice), so no branch surrounds them
    const uint8_t* p0 = (const uint8_t*)Wr + (base + cc) * (bf ? 2 : 4);
    wr[j].x = *(const gate_bf16x2*)p0;
    wr[j].y = *(const gate_bf16x2*)(p0 + (bf ? 0 : 4));
  };
  auto weights = [&](int j, int c0, double& w0, double& w1) {
    const float m = c0 + 2 * lane < d ? 1.f : 0.f;
    const float f0 = bf ? __uint_as_float(wr[j].x << 16) : __uint_as_float(wr[j].x);
    const float f1 = bf ? __uint_as_float(wr[j].x & 0xffff0000u) : __uint_as_float(wr[j].y);
    w0 = (double)(f0 * m);
    w1 = (double)(f1 * m);
  };
  double acc[PMAX][2];
#pragma unroll
  for (int t = 0; t < PMAX; t++) acc[t][0] = acc[t][1] = 0.0;
#pragma unroll
  for (int j = 0; j < RM_D; j++) fetch(j, j * RM_C);
  int buf = 0;
  for (int cg = 0; cg < d; cg += RM_D * RM_C) {
#pragma unroll
    for (int j = 0; j < RM_D; j++) {
      const int c0 = cg + j * RM_C;
      if (c0 < d) {  // block-uniform
        // Xd[buf] was last read two slabs ago; every wave has passed the barrier of the slab in
        // between, so it is free
#pragma unroll
        for (int i = 0; i < XR; i++) {
          const int e = tid + 256 * i;
          Xd[buf][e / RM_C][e % RM_C] = (double)xr[j][i];
        }
        double w0, w1;
        weights(j, c0, w0, w1);
        fetch(j, c0 + RM_D * RM_C);  // slabs past d load column 0 and count as zeros
        moe_lds_barrier();  // (LDS only: the ring's loads stay in flight across it)
        // rows past P hold zeros: no predicate, so the LDS reads of a slab go out back to back
#pragma unroll
        for (int t = 0; t < PMAX; t++) {
          const double2 xv = *(const double2*)&Xd[buf][t][2 * lane];
          acc[t][0] = fma(w0, xv.x, acc[t][0]);
          acc[t][1] = fma(w1, xv.y, acc[t][1]);
        }
        buf ^= 1;
      }
    }
  }
#pragma unroll
  for (int t = 0; t < PMAX; t++) {
    if (t < P) {
      const double sum = wave_sum(acc[t][0] + acc[t][1]);
      if (lane == 0 && live) {
        float v = (float)sum;
        if (extra) out_x[t] = v;
        else {
          if (bias) v += bias[row];
          logits[(size_t)t * E + row] = v;
        }
      }
    }
  }
}

// ---- softmax + top-k, one wave per token (E <= 64*NPL): topk_wave in topk.h ----
template <int NPL>
__global__ void __launch_bounds__(256) k_router_topk(const float* __restrict__ logits,
                                                     int* __restrict__ ids, float* __restrict__ ws,
                                                     int P, int E, int k, int id_stride) {
  __shared__ __attribute__((aligned(16))) float pbuf[4][64 * NPL];
  const int wv = threadIdx.x >> 6;
  const int tok = blockIdx.x * 4 + wv;
  if (tok >= P) return;
  topk_wave<NPL>(logits + (size_t)tok * E, ids + (size_t)tok * id_stride, ws + (size_t)tok * id_stride, E, k, pbuf[wv]);
}

template <int NPL>
__global__ void __launch_bounds__(256) k_router_topk_block(const float* __restrict__ logits, int* __restrict__ ids,
                                                           float* __restrict__ ws, int E, int k, int id_stride, moe_rfix RF) {
  __shared__ int sel_ids[64];
  __shared__ float sel_ws[64];
  const int t = blockIdx.x;
  if (!RF.W) {
    topk_block<NPL, false>(logits + (size_t)t * E, ids + (size_t)t * id_stride, ws + (size_t)t * id_stride, E, k);
    return;
  }
  select_certain<NPL, 256>(logits + (size_t)t * E, RF, t, sel_ids, sel_ws, E, k, true);
  __syncthreads();
  if ((int)threadIdx.x < k) {
    ids[(size_t)t * id_stride + threadIdx.x] = sel_ids[threadIdx.x];
    ws[(size_t)t * id_stride + threadIdx.x] = sel_ws[threadIdx.x];
  }
}

// |row|_2 of every row, the maximum as the bits of a non-negative float
__global__ void __launch_bounds__(256) k_row_norm_max(const void* __restrict__ W, int bf16, int E, int d, unsigned* __restrict__ out) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= E) return;
  float a = 0.f;
  for (int c = lane; c < d; c += 64) {
    const float w = bf16 ? bf16_bits_to_f32(((const uint16_t*)W)[(size_t)row * d + c]) : ((const float*)W)[(size_t)row * d + c];
    a += w * w;
  }
  a = wave_sum(a);
  if (lane == 0) atomicMax(out, __float_as_uint(a >= 0.f ? sqrtf(a) : INFINITY));
}

// Launch of the sequential-order kernel: 128-token tiles when there are enough of them to fill the
// chip, 64-token tiles otherwise.
void launch_seq(const void* W, bool bf, const float* bias, const float* x, int P, int E, int d, float* logits, hipStream_t st) {
  const int ncol = (E + RS_E - 1) / RS_E;
  const bool big = (int64_t)((P + 127) / 128) * ncol >= 512;
  const int bt = big ? 128 : 64;
  const int ntt = (P + bt - 1) / bt;
  const unsigned grid = (unsigned)(((ntt + 7) / 8) * 8 * ncol);
#define RS_GO(BF, BT) k_router_logits_seq<BF, BT><<<grid, 256, 0, st>>>(W, bias, x, P, E, d, logits, ncol, ntt)
  if (bf) { if (big) RS_GO(true, 128); else RS_GO(true, 64); }
  else { if (big) RS_GO(false, 128); else RS_GO(false, 64); }
#undef RS_GO
}


// ---- 5..32 tokens on the f64 matrix pipe: a block = 16 weight rows x all tokens x one column split,
// its eight waves each take one eighth of the block's columns and the partial 16 x 16 tiles are added in
// wave order (fixed, so the result does not depend on timing; same accuracy statement as k_router_small).
// v_mfma_f64_16x16x4_f64: lane l supplies A[row l%16][k l/16] and B[k l/16][token l%16]; a 16-byte load
// per lane (4 consecutive columns 4*(l/16)..+3 of its row / token) therefore feeds four MFMAs.
// Every weight is read once, activations come from L2; loads run through a register ring of
// RD 16-column steps.  Needs d % 128 == 0.  Blocks past the rows build the digit planes of x.
// KS > 1 (needs gpart): the columns are split over KS blocks per row group as well, so that
// 16 rows x d columns, one block's work with KS = 1 and the whole time of the launch, become KS blocks on KS
// CUs.  Each block leaves its fp64 partial tile in gpart.  Where the selection is a launch of its own, that one adds the KS shares
// in share order (k_router_split_topk; no tickets).  With tickets (MOE_OPT_GU_TOPK_MAX_TOKENS above 4: the blocks of the gate/up launch
// want logits) each block takes a ticket of its row group, and the block that
// draws the last one adds the KS partial tiles in split order (fixed again) and writes the logits.  Partial
// tiles go out and come back as device-scope accesses, the ticket counters rest at 0 between launches.  That hand-over is a
// store's, a ticket's and a load's trip to memory one behind the other: the launch takes 2 us more, 20 tokens 14.3 for 12.2.
// The shared expert's gate vector has a block per token, which leaves the selection's bound as well: as row 513 of 512 experts it made
// 264 blocks, each a CU's work, for 256 CUs, and 20 tokens took 12.2 us for 7.4, eight 9.4 for 5.8.  Layers, us, with all of
// this, weights from HBM: q4cp 5 tokens (four) 238 -> 216, 8 315 -> 293, 20 (two) 306 -> 292, rotated experts 11 (two) 198 -> 187; and a batch with a near tie, whose logits
// the selecting launch redoes by waves now, 32 tokens 632 -> 243.
template <bool BF16, int NTT, int RD>  // NTT = token tiles of 16 (1 or 2)
__global__ void __launch_bounds__(512, 2) k_router_mfma(const void* __restrict__ W, const float* __restrict__ bias,
                                                        const float* __restrict__ x, int P, int E, int d,
                                                        float* __restrict__ logits, uint32_t* __restrict__ planes,
                                                        float2* __restrict__ meta, bool planes_natural, int KS,
                                                        double* gpart, unsigned* tickets, moe_row_extras R, moe_rot_planes rot) {
  __shared__ double part[8][NTT][4][64];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nrt = (E + 15) >> 4;
  if ((int)blockIdx.x >= nrt * KS) {
    const int nx = R.tol || R.wx ? P : 0, t = (int)blockIdx.x - nrt * KS;
    if (t >= nx) {
      router_plane_blocks(t - nx, 512, tid, x, P, d, planes, meta, planes_natural, rot);
      return;
    }
    // a block per token: |x| as the selection's bound, the shared expert's gate logit
    double* const xp = &part[0][0][0][0];
    float acc;
    double gate;
    row_extras_part(x, t, d, tid, 512, R, acc, gate);
    acc = wave_sum(acc);
    gate = wave_sum(gate);
    if (lane == 0) {
      xp[2 * wv] = (double)acc;
      xp[2 * wv + 1] = gate;
    }
    __syncthreads();
    if (tid == 0) {
      acc = 0.f;
      gate = 0.0;
#pragma unroll
      for (int w = 0; w < 8; w++) {
        acc += (float)xp[2 * w];
        gate += xp[2 * w + 1];
      }
      row_extras_out(t, d, R, acc, gate);
    }
    return;
  }
  const int rg = (int)blockIdx.x % nrt, ks = (int)blockIdx.x / nrt;  // row group, column split
  const int li = lane & 15, lg = lane >> 4;
  const int row = rg * 16 + li;
  // per-lane weight row (rows past the end read row 0 and are never stored); all loads unconditional
  const uint8_t* wrow = (const uint8_t*)W + (row < E ? (uint64_t)row : 0) * d * (BF16 ? 2 : 4);
  const float* xrow[NTT];
  float xm[NTT];
#pragma unroll
  for (int tt = 0; tt < NTT; tt++) {
    const int t = 16 * tt + li;
    xrow[tt] = x + (size_t)(t < P ? t : 0) * d;
    xm[tt] = t < P ? 1.f : 0.f;
  }
  const int nst = d / 16, slot = ks * 8 + wv, s0 = slot * nst / (8 * KS);  // the wave's 16-column steps, one at least
  const int k0 = 16 * s0 + 4 * lg, nit = (slot + 1) * nst / (8 * KS) - s0;  // this lane's first column
  uint4 wr[RD];
  float4 xr[RD][NTT];
  auto fetch = [&](int j, int it) {
    const int c = k0 + 16 * (it < nit ? it : nit - 1);  // past the end: a repeat that is never used
    const uint8_t* p = wrow + (size_t)c * (BF16 ? 2 : 4);
    const gate_bf16x4 lo = *(const gate_bf16x4*)p, hi = *(const gate_bf16x4*)(p + (BF16 ? 0 : 8));
    wr[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
#pragma unroll
    for (int tt = 0; tt < NTT; tt++) xr[j][tt] = *(const float4*)(xrow[tt] + c);
  };
  double4v acc[NTT];
#pragma unroll
  for (int tt = 0; tt < NTT; tt++) acc[tt] = double4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < RD; j++) fetch(j, j);
  for (int ib = 0; ib < nit; ib += RD) {
#pragma unroll
    for (int j = 0; j < RD; j++) {
      if (ib + j < nit) {  // wave-uniform (a wave's steps may be one fewer than another's)
        float w[4];
        if (BF16) {
          w[0] = __uint_as_float(wr[j].x << 16); w[1] = __uint_as_float(wr[j].x & 0xffff0000u);
          w[2] = __uint_as_float(wr[j].y << 16); w[3] = __uint_as_float(wr[j].y & 0xffff0000u);
        } else {
          w[0] = __uint_as_float(wr[j].x); w[1] = __uint_as_float(wr[j].y);
          w[2] = __uint_as_float(wr[j].z); w[3] = __uint_as_float(wr[j].w);
        }
        float4 xv[NTT];
#pragma unroll
        for (int tt = 0; tt < NTT; tt++) xv[tt] = xr[j][tt];
        fetch(j, ib + j + RD);
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const double a = (double)w[q];
#pragma unroll
          for (int tt = 0; tt < NTT; tt++) {
            const float xq = q == 0 ? xv[tt].x : q == 1 ? xv[tt].y : q == 2 ? xv[tt].z : xv[tt].w;
            acc[tt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)(xq * xm[tt]), acc[tt], 0, 0, 0);
          }
        }
      }
    }
  }
#pragma unroll
  for (int tt = 0; tt < NTT; tt++)
#pragma unroll
    for (int r = 0; r < 4; r++) part[wv][tt][r][lane] = acc[tt][r];
  __syncthreads();
  // D value r of lane l = [row 4r + l/16][token l%16]; thread i = (tile, row, token) adds the eight partials
  auto emit = [&](int i, double sum) {
    const int orow = rg * 16 + ((i >> 4) & 15), t = 16 * (i >> 8) + (i & 15);
    if (orow < E && t < P) logits[(size_t)t * E + orow] = (float)sum + (bias ? bias[orow] : 0.f);
  };
  constexpr int NV = NTT * 256;
  for (int i = tid; i < NV; i += 512) {
    const int tt = i >> 8, r = (i >> 6) & 3, l = i & 63;
    double sum = part[0][tt][r][l];
#pragma unroll
    for (int w = 1; w < 8; w++) sum += part[w][tt][r][l];
    if (KS == 1) emit(i, sum);
    else if (!tickets) {  // (the selecting launch adds the column shares)
      const int orow = rg * 16 + ((i >> 4) & 15), t = 16 * tt + (i & 15);
      if (orow < E && t < P) gpart[((size_t)ks * P + t) * E + orow] = sum;
    } else __hip_atomic_store(&gpart[((size_t)ks * nrt + rg) * NV + i], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (KS == 1 || !tickets) return;
  // Hand-over of the partial tiles to the block that draws the row group's last ticket (possibly on another
  // XCD): the tiles are device-scope atomic stores, every storing thread waits until all of its stores have
  // been acknowledged (vmcnt = 0) before the barrier, thread 0 takes the device-scope ticket after the
  // barrier, and the last block reads the tiles back with device-scope atomic loads issued after its own
  // ticket returned.  Both sides go to the device's coherence point; no cache-wide write-back / invalidate.
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __syncthreads();
  if (tid == 0) {
    const unsigned ticket = __hip_atomic_fetch_add(&tickets[rg], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = ticket == (unsigned)KS - 1u;
    if (s_last) __hip_atomic_store(&tickets[rg], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-armed
  }
  __syncthreads();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  for (int i = tid; i < NV; i += 512) {
    double v[8];  // KS <= 8: all partials requested before the first is used
#pragma unroll
    for (int q = 0; q < 8; q++)
      v[q] = __hip_atomic_load(&gpart[((size_t)(q < KS ? q : 0) * nrt + rg) * NV + i], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    double sum = v[0];
#pragma unroll
    for (int q = 1; q < 8; q++)
      if (q < KS) sum += v[q];
    emit(i, sum);
  }
}

}  // namespace

MOE_API int moe_router_logits(const moe_wview* W, const float* bias, const float* x, int P,
                              float* logits, int mode, moe_stream_t st) {
  if (!W || !W->data || !x || !logits) return MOE_E_INVALID;
  if (W->dtype != MOE_DT_F32 && W->dtype != MOE_DT_BF16) return MOE_E_UNSUPPORTED;
  if (P < 0 || W->rows == 0 || W->cols == 0 || W->rows > (1u << 20) || W->cols > (1u << 24))
    return MOE_E_INVALID;
  if (P == 0) return MOE_OK;
  const int E = (int)W->rows, d = (int)W->cols;
  const bool bf = W->dtype == MOE_DT_BF16;
  const bool par = mode == 0 && P <= 32 && d % 4 == 0 && moe_aligned(x, 16) && moe_aligned(W->data, 16);
  if (par) {
    return moe_router_logits_small(W, bias, nullptr, x, P, logits, nullptr, nullptr, nullptr, false, moe_s(st), nullptr,
                                   nullptr);
  } else {
    launch_seq(W->data, bf, bias, x, P, E, d, logits, moe_s(st));
  }
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// Internal: sequential-order logits for any P.
int moe_router_logits_seq(const moe_wview* W, const float* bias, const float* x, int P, float* logits, hipStream_t st) {
  launch_seq(W->data, W->dtype == MOE_DT_BF16, bias, x, P, (int)W->rows, (int)W->cols, logits, st);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

static int column_shares(int P, int E, int d) {
  if (P <= 4 || E + 1 > MOE_ROUTER_KSPLIT_ROWS || d < 256) return 1;
  return d / 128 < 8 ? d / 128 : 8;
}
static bool on_matrix_pipe(int P, int d, int KS) { return P > 4 && (P > 24 || KS > 1) && d % 128 == 0; }
bool moe_router_small_bounds(const moe_wview* W, int P) {
  const int E = (int)W->rows, d = (int)W->cols;
  return P <= 4 || on_matrix_pipe(P, d, column_shares(P, E, d));
}

// Internal: small-P logits plus the shared-expert gate row (and, if planes != nullptr, the digit
// planes of x for the integer-dot decode kernels) in the same launch.
int moe_router_logits_small(const moe_wview* W, const float* bias, const moe_wview* Wx, const float* x,
                            int P, float* logits, float* out_x, uint32_t* planes, float2* meta,
                            bool planes_natural, hipStream_t st, double* kpart, unsigned* ktickets, const moe_rot_planes* rotp,
                            float* tol_out, float tol_scale, int* parts) {
  const int E = (int)W->rows, d = (int)W->cols;
  if (parts) *parts = 0;
  moe_rot_planes rot{nullptr, nullptr, nullptr};
  if (rotp) {  // hgn v2: the planes of rot_in(x, pre) in the same launch
    if (!rotp->pre || !rotp->planes || !rotp->meta || d % 128 || !moe_aligned(rotp->pre, 16) || !moe_aligned(x, 16)) return MOE_E_INVALID;
    rot = *rotp;
  }
  // The f64 matrix pipe kernel (d a multiple of 128).  With the caller's scratch for
  // partial tiles the columns are split over up to eight blocks per 16 rows and it serves 5..32 tokens;
  // without it one block per 16 rows leaves most CUs idle (38 us at 32 tokens), which only beats
  // k_router_mid above 24 tokens.  A shared-expert gate row in the other format (checkpoints: a bf16 matrix, an f32 row)
  // makes no difference to it: that row is read by a block per token, in its own format.
  // (as many shares as leave every wave a step of 16 columns, whether or not they are equal: 2560 columns in eight shares of two and three
  // steps a wave instead of four of five: the launch 13.2 -> 7.5 us at 20 tokens; one layer of 2560 x 640 again and again
  // (up to 12 tokens wholly or mostly out of the last-level cache), q4cp 5 tokens 49.0 -> 46.5, 20 118.2 112.4, table codebook 12 112.4 109.1; 2304 x 512 12
  // 67.5 62.2)
  const int KS = kpart && ktickets ? column_shares(P, E, d) : 1;
  const bool mfma_ok = on_matrix_pipe(P, d, KS);
  if (P > 24 && !mfma_ok) {
    // more than 24 tokens per block cost the kernel its second wave per SIMD (accumulators):
    // two launches of at most 16 tokens read the router matrix twice (L2 / MALL) and are faster
    const int P0 = 16, G = d / 32;
    const size_t pdw = planes_natural ? QV_GROUP_DW : QV4_GROUP_DW;
    int rc = moe_router_logits_small(W, bias, Wx, x, P0, logits, out_x, planes, meta, planes_natural, st, nullptr,
                                     nullptr, rotp);
    if (rc) return rc;
    moe_rot_planes rot2 = rot;
    if (rotp) {
      rot2.planes += (size_t)P0 * G * QV4_GROUP_DW;
      rot2.meta += (size_t)P0 * G;
    }
    return moe_router_logits_small(W, bias, Wx, x + (size_t)P0 * d, P - P0, logits + (size_t)P0 * E,
                                   out_x ? out_x + P0 : nullptr, planes ? planes + (size_t)P0 * G * pdw : nullptr,
                                   meta ? meta + (size_t)P0 * G : nullptr, planes_natural, st, nullptr, nullptr,
                                   rotp ? &rot2 : nullptr);
  }
  const bool bf = W->dtype == MOE_DT_BF16;
  const bool xbf = Wx && Wx->dtype == MOE_DT_BF16;
  const int nrows = E + (Wx ? 1 : 0);
  const int bs = P <= 4 ? 128 : 256, rpb = bs / 64;  // rows per block: one per wave
  const int qblocks = (planes ? P * ((d / 32 + bs - 1) / bs) : 0) + (rot.planes ? P * ((d / 8 + bs - 1) / bs) : 0);
  dim3 g((nrows + rpb - 1) / rpb + qblocks);
  const void* wx = Wx ? Wx->data : nullptr;
  if (P <= 4) {
#define RSM_GO(BF, TT) k_router_small<BF, TT><<<g, bs, 0, st>>>(W->data, bias, wx, xbf, x, E, d, logits, out_x, nrows, planes, meta, planes_natural, rot, tol_out, tol_scale)
#define RSM_T(TT) do { if (bf) RSM_GO(true, TT); else RSM_GO(false, TT); } while (0)
    if (P == 1) RSM_T(1);
    else if (P == 2) RSM_T(2);
    else if (P == 3) RSM_T(3);
    else RSM_T(4);
#undef RSM_T
#undef RSM_GO
  } else {
    if (mfma_ok) {
      // the f64 matrix pipe: 16 rows per block, columns split over KS blocks and their eight waves
      const int qb = (planes ? P * ((d / 32 + 511) / 512) : 0) + (rot.planes ? P * ((d / 8 + 511) / 512) : 0);
      moe_row_extras ex{};
      ex.wx = wx; ex.wx_bf16 = xbf; ex.out_x = out_x;
      ex.tol = tol_out; ex.tol_scale = tol_scale;
      dim3 gx((E + 15) / 16 * KS + (ex.wx || ex.tol ? P : 0) + qb);
      if (parts && KS > 1) {
        *parts = KS;
        ktickets = nullptr;
      }
#define RX_GO(BF, NTT, RD) k_router_mfma<BF, NTT, RD><<<gx, 512, 0, st>>>(W->data, bias, x, P, E, d, logits, planes, meta, planes_natural, KS, kpart, ktickets, ex, rot)
      const int nit = (d / 16 + 8 * KS - 1) / (8 * KS);  // ring steps a wave walks, at most
      if (nit <= 3) {
        if (P <= 16) { if (bf) RX_GO(true, 1, 3); else RX_GO(false, 1, 3); }
        else { if (bf) RX_GO(true, 2, 3); else RX_GO(false, 2, 3); }
      } else {
        if (P <= 16) { if (bf) RX_GO(true, 1, 12); else RX_GO(false, 1, 12); }
        else { if (bf) RX_GO(true, 2, 12); else RX_GO(false, 2, 12); }
      }
#undef RX_GO
      MOE_LAUNCH_CHECK();
      return MOE_OK;
    }
#define RMD_GO(BF, PM) k_router_mid<BF, PM><<<g, 256, 0, st>>>(W->data, bias, wx, xbf, x, P, E, d, logits, out_x, nrows, planes, meta, planes_natural, rot)
    if (P <= 8) { if (bf) RMD_GO(true, 8); else RMD_GO(false, 8); }
    else if (P <= 16) { if (bf) RMD_GO(true, 16); else RMD_GO(false, 16); }
    else { if (bf) RMD_GO(true, 24); else RMD_GO(false, 24); }  // P <= 24 (larger batches were split above)
#undef RMD_GO
  }
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_router_topk_small(const float* logits, int* ids, float* ws, int P, int E, int k, int id_stride,
                                 const moe_rfix* rf, hipStream_t st) {
  const moe_rfix R = rf ? *rf : moe_rfix{};
  if (E <= 512) k_router_topk_block<8><<<P, 256, 0, st>>>(logits, ids, ws, E, k, id_stride, R);
  else k_router_topk_block<16><<<P, 256, 0, st>>>(logits, ids, ws, E, k, id_stride, R);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_router_row_norm_max(const moe_wview* W, float* scratch, float* out_host) {
  if (!W || !W->data || !scratch || !out_host) return MOE_E_INVALID;
  MOE_HIP(hipMemset(scratch, 0, 4));
  k_row_norm_max<<<(unsigned)((W->rows + 3) / 4), 256, 0, nullptr>>>(W->data, W->dtype == MOE_DT_BF16 ? 1 : 0, (int)W->rows,
                                                                     (int)W->cols, (unsigned*)scratch);
  MOE_LAUNCH_CHECK();
  MOE_HIP(hipMemcpy(out_host, scratch, 4, hipMemcpyDeviceToHost));
  return MOE_OK;
}

MOE_API int moe_router_topk(const float* logits, int* ids, float* ws, int P, int E, int k,
                            int id_stride, moe_stream_t st) {
  if (!logits || !ids || !ws) return MOE_E_INVALID;
  if (P < 0 || E < 1 || k < 1 || k > E || k > 64 || id_stride < k) return MOE_E_INVALID;
  if (E > 1024) return MOE_E_UNSUPPORTED;
  if (P == 0) return MOE_OK;
  if (P <= 32)  // few tokens: a block per token, the fp64 exps spread over its threads
    return moe_launch_router_topk_small(logits, ids, ws, P, E, k, id_stride, nullptr, moe_s(st));
  dim3 g((P + 3) / 4);
  if (E <= 512) k_router_topk<8><<<g, 256, 0, moe_s(st)>>>(logits, ids, ws, P, E, k, id_stride);
  else k_router_topk<16><<<g, 256, 0, moe_s(st)>>>(logits, ids, ws, P, E, k, id_stride);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}
