// Router of middle-sized batches (33 .. MOE_ROUTER_CAND_MIN - 1 tokens, up to MOE_ROUTER_SPLIT_MAX where the candidate selection
// does not apply): fp64 logits on the f64 matrix pipe with the columns
// split over the waves of a block and over blocks, then one selecting block per token.  Two launches.
// (reference arithmetic: src/ref.cpp:68-77,565-594)
//
// The candidate selection of router_cand.hip pays off once its third launch, a chain of 15 .. 20 us, is small against the
// fp64 work it saves.  At 130 tokens it is not: all 130 x 512 sums are 0.2 G fp64 FMAs, 5 us of the chip's f64
// matrix rate.  What that needs is enough waves, so columns are dealt out: a block is 32 tokens x 32 experts x one of KS
// column shares, its eight waves take an eighth of the share each and their partial tiles are added in wave order through
// LDS; the KS shares' fp64 partial sums go to memory and the selecting block of a token adds them in share order.  Every
// order is fixed, so results do not depend on timing.
// As in the other parallel orders (router.hip) the sums can differ from the reference's sequential ones in the last fp64
// bits; the selecting block makes the ids certain.
//
// The launch's spare blocks read x anyway, so they leave what else a batch needs from it: the f16 copy in the grouped
// GEMM's order, the mean square (f16 range guard), |x| as the selection's error bound and the shared expert's gate logit.
// Measured (512 experts, d = 3072, bf16 router): 10.7 + 7.6 us at 48 tokens, 25 + 7.7 us at 130 (f32), 53 + 7.2 us at 515; the
// dense fp64 launch that such layers took before (the router and its gate vector of different types) 395 us, the others
// 150 us in the candidate selection of then.
#include "common.h"
#include "internal.h"
#include "router_chain.h"
#include "rowx.h"

namespace {

typedef double double4v __attribute__((ext_vector_type(4)));
constexpr int SP_T = 32, SP_E = 32, SP_W = 8;  // tokens, experts, waves (= column parts) of a block
constexpr int SP_RD = 3;                       // 16-column steps in flight per wave

template <bool BF16>
__global__ void __launch_bounds__(512, 2) k_router_split(const void* __restrict__ W, const float* __restrict__ x, int P, int E,
                                                         int d, int KS, int nrg, int ntg, double* __restrict__ gpart,
                                                         moe_row_extras R) {
  __shared__ double part[SP_W][4 * 4 * 64];  // [wave][tile (token half, expert half)][r][lane]
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nmm = nrg * ntg * KS;
  if ((int)blockIdx.x >= nmm) {
    // a block per token: with a wave per token the row's six dependent trips to memory were the launch's longest path
    const int t = (int)blockIdx.x - nmm;
    float acc;
    double gate;
    row_extras_part(x, t, d, tid, 512, R, acc, gate);
    acc = wave_sum(acc);
    gate = wave_sum(gate);
    if (lane == 0) {
      part[0][2 * wv] = (double)acc;
      part[0][2 * wv + 1] = gate;
    }
    __syncthreads();
    if (tid == 0) {
      acc = 0.f;
      gate = 0.0;
#pragma unroll
      for (int w = 0; w < SP_W; w++) {
        acc += (float)part[0][2 * w];
        gate += part[0][2 * w + 1];
      }
      row_extras_out(t, d, R, acc, gate);
    }
    return;
  }
  const int rg = (int)blockIdx.x % nrg, tg = (int)blockIdx.x / nrg % ntg, ks = (int)blockIdx.x / (nrg * ntg);
  const int li = lane & 15, lg = lane >> 4;
  const int nst = d / 16, slot = ks * SP_W + wv;
  const int s0 = slot * nst / (SP_W * KS), s1 = (slot + 1) * nst / (SP_W * KS);  // this wave's 16-column steps
  // a lane's row / token pointers (past the end: the last one again, never stored), at its four columns of a step
  const uint8_t* wp[2];
  const float* xp[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int e = rg * SP_E + 16 * i + li, t = tg * SP_T + 16 * i + li;
    wp[i] = (const uint8_t*)W + ((size_t)(e < E ? e : E - 1) * d + 4 * lg) * (BF16 ? 2 : 4);
    xp[i] = x + (size_t)(t < P ? t : P - 1) * d + 4 * lg;
  }
  uint4 wr[SP_RD][2];
  float4 xr[SP_RD][2];
  auto fetch = [&](int j, int s) {
    s = s < s1 ? s : s1 - 1;  // past the end: a repeat that is never used
    s = s > 0 ? s : 0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      if (BF16) {
        const uint2 u = *(const uint2*)(wp[i] + (size_t)s * 32);
        wr[j][i].x = u.x; wr[j][i].y = u.y;
      } else {
        wr[j][i] = *(const uint4*)(wp[i] + (size_t)s * 64);
      }
      xr[j][i] = *(const float4*)(xp[i] + (size_t)s * 16);
    }
  };
  double4v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = double4v{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < SP_RD; j++) fetch(j, s0 + j);
  for (int sb = s0; sb < s1; sb += SP_RD) {
#pragma unroll
    for (int j = 0; j < SP_RD; j++) {
      if (sb + j < s1) {  // wave-uniform
        float w[2][4], xv[2][4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          if (BF16) {
            w[i][0] = __uint_as_float(wr[j][i].x << 16); w[i][1] = __uint_as_float(wr[j][i].x & 0xffff0000u);
            w[i][2] = __uint_as_float(wr[j][i].y << 16); w[i][3] = __uint_as_float(wr[j][i].y & 0xffff0000u);
          } else {
            w[i][0] = __uint_as_float(wr[j][i].x); w[i][1] = __uint_as_float(wr[j][i].y);
            w[i][2] = __uint_as_float(wr[j][i].z); w[i][3] = __uint_as_float(wr[j][i].w);
          }
          xv[i][0] = xr[j][i].x; xv[i][1] = xr[j][i].y; xv[i][2] = xr[j][i].z; xv[i][3] = xr[j][i].w;
        }
        fetch(j, sb + j + SP_RD);
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const double a0 = (double)xv[0][q], a1 = (double)xv[1][q], b0 = (double)w[0][q], b1 = (double)w[1][q];
          acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
          acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
          acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
          acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) part[wv][((2 * i + j) * 4 + r) * 64 + lane] = acc[i][j][r];
  __syncthreads();
  // D value r of lane l of a tile = [token 4r + l/16][expert l%16]
#pragma unroll
  for (int n = 0; n < SP_T * SP_E / 512; n++) {
    const int i = tid + 512 * n, tl = i >> 5, el = i & 31;
    const int src = (((tl >> 4) * 2 + (el >> 4)) * 4 + ((tl & 15) >> 2)) * 64 + (tl & 3) * 16 + (el & 15);
    double sum = part[0][src];
#pragma unroll
    for (int w = 1; w < SP_W; w++) sum += part[w][src];
    const int t = tg * SP_T + tl, e = rg * SP_E + el;
    if (t < P && e < E) gpart[((size_t)ks * P + t) * E + e] = sum;
  }
}

// The selecting block of a token (also of 5 .. 32 tokens, behind k_router_mfma's shares): the column shares' sums in share order, + bias, softmax / top-k.
// Its fp64 sums differ from the reference's sequential ones by at most tol; select_listed makes the ids certain.
template <int NPL>
__global__ void __launch_bounds__(256) k_router_split_topk(const double* __restrict__ gpart, int KS, int* __restrict__ ids,
                                                           float* __restrict__ ws, int P, int E, int k, int id_stride,
                                                           moe_rfix RF) {
  constexpr int NV = (64 * NPL + 255) / 256;
  __shared__ __attribute__((aligned(16))) float lg[64 * NPL];
  __shared__ int sel_ids[64];
  __shared__ float sel_ws[64];
  __shared__ __attribute__((aligned(16))) double chain[4][512];
  __shared__ int list[64 * NPL], nlist;
  const int t = blockIdx.x, tid = threadIdx.x;
  if (tid == 0) nlist = 0;
  __syncthreads();
  const float tol = RF.tol[t];
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int e = tid + 256 * j;
    if (e < E) {
      const double* p = gpart + (size_t)t * E + e;
      double v[MOE_ROUTER_SPLIT_KS];
#pragma unroll
      for (int s = 0; s < MOE_ROUTER_SPLIT_KS; s++) v[s] = s < KS ? p[(size_t)s * P * E] : 0.0;  // (KS is uniform)
      double sum = v[0];
#pragma unroll
      for (int s = 1; s < MOE_ROUTER_SPLIT_KS; s++) sum += v[s];
      if (logit_doubtful(sum, tol)) list[atomicAdd(&nlist, 1)] = e;
      lg[e] = (float)sum + (RF.bias ? RF.bias[e] : 0.f);
    }
  }
  __syncthreads();
  select_listed<NPL>(lg, list, nlist, tol, RF, t, E, k, sel_ids, sel_ws, chain);
  if (tid < k) {
    ids[(size_t)t * id_stride + tid] = sel_ids[tid];
    ws[(size_t)t * id_stride + tid] = sel_ws[tid];
  }
}

// Column shares: the number that the following estimate of the first launch is smallest for (microseconds): rounds of
// 512 blocks (two to a CU), each as long as its share of the columns on the f64 pipe and about 3 us of its own, plus the
// partial sums' way to memory and back.
int split_shares(int P, int E, int d) {
  const int tiles = ((E + SP_E - 1) / SP_E) * ((P + SP_T - 1) / SP_T);
  const int most = d / 16 / (SP_W * 3);  // no share of a wave shorter than three 16-column steps
  int best = 1;
  float least = 1e30f;
  for (int ks = 1; ks <= MOE_ROUTER_SPLIT_KS && (ks == 1 || ks <= most); ks++) {
    const float cost = (float)((tiles * ks + 511) / 512) * ((float)d * 0.0133f / (float)ks + 3.f) + (float)ks * P * E * 4e-6f;
    if (cost < least) {
      least = cost;
      best = ks;
    }
  }
  return best;
}

}  // namespace

bool moe_router_split_supported(const moe_wview* W, int P, int k) {
  return P >= 1 && P <= MOE_ROUTER_SPLIT_MAX && W->rows <= 1024 && k <= 63 && W->cols % 32 == 0 && moe_aligned(W->data, 16);
}

size_t moe_router_split_scratch_bytes(int max_tokens, int experts, int d) {
  const int P = max_tokens < MOE_ROUTER_SPLIT_MAX ? max_tokens : MOE_ROUTER_SPLIT_MAX;
  size_t most = 0;
  for (int p = 1; p <= P; p++) {
    const size_t n = (size_t)split_shares(p, experts, d) * p;
    most = n > most ? n : most;
  }
  return most * experts * sizeof(double);
}

int moe_router_batch_split(const moe_wview* W, const float* x, int P, int* ids, float* ws, int k,
                           int id_stride, double* gpart, const moe_row_extras& R, const moe_rfix& RF, hipStream_t st,
                           hipEvent_t after_rows) {
  const int E = (int)W->rows, d = (int)W->cols;
  const int KS = split_shares(P, E, d);
  const int nrg = (E + SP_E - 1) / SP_E, ntg = (P + SP_T - 1) / SP_T;
  const unsigned grid = (unsigned)(nrg * ntg * KS + P);
  if (W->dtype == MOE_DT_BF16) k_router_split<true><<<grid, 512, 0, st>>>(W->data, x, P, E, d, KS, nrg, ntg, gpart, R);
  else k_router_split<false><<<grid, 512, 0, st>>>(W->data, x, P, E, d, KS, nrg, ntg, gpart, R);
  MOE_LAUNCH_CHECK();
  if (after_rows) MOE_HIP(hipEventRecord(after_rows, st));
  return moe_launch_router_split_topk(gpart, KS, ids, ws, P, E, k, id_stride, RF, st);
}

// (also behind k_router_mfma)
int moe_launch_router_split_topk(const double* gpart, int KS, int* ids, float* ws, int P, int E, int k, int id_stride, const moe_rfix& RF,
                                 hipStream_t st) {
  if (KS < 1 || KS > MOE_ROUTER_SPLIT_KS || E > 1024 || !RF.W || !RF.tol) return MOE_E_INVALID;
  if (E <= 512) k_router_split_topk<8><<<P, 256, 0, st>>>(gpart, KS, ids, ws, P, E, k, id_stride, RF);
  else k_router_split_topk<16><<<P, 256, 0, st>>>(gpart, KS, ids, ws, P, E, k, id_stride, RF);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}
