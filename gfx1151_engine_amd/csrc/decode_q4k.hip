// Decode (T <= 32) on raw GGUF Q4_K blocks read in place, integer dot products: the Q4_K twin of
// the q4cp decode kernels.  Unit of work = one 32-byte run of code bytes = 64 weights = two
// 32-element sub-blocks (low nibbles / high nibbles), each with its own 6-bit scale and min:
//   sum_k w_k x_k = d * (sc0 * qA * VA + sc1 * qB * VB) - dmin * (m0 * qA * SA + m1 * qB * SB)
// with V = integer dot product of the codes with the activation group's two 8-bit digit planes
// (natural element order) and q * S = the group's quantised sum.  A lane owns one unit of a row;
// rows of 3072 are 48 units (gate/up deals several rows' units over a wave, ggu_gu_packed), rows of 768 are
// 12 units (four slots per wave).
// (reference: src/gpu/parts/26_kernels_moe_gguf.inc:527-568,693-756,893-939; src/gguf.h:328-336,408-441)
#include <type_traits>

#include "common.h"
#include "internal.h"
#include "iq4.h"
#include "qvec.h"
#include "topk.h"

namespace {

__device__ __forceinline__ float dpp_add_row(float v) {  // sum over each row of 16 lanes, in every lane
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true));
  return v;
}
__device__ __forceinline__ float dpp_max_row(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true)));
  return v;
}
__device__ __forceinline__ float sum64(float v) {
  return rows_total_add(dpp_add_row(v));
}

// activation planes of one unit: two groups (A = low nibbles, B = high nibbles)
struct XU {
  uint32_t a[2][8], b[2][8];
  float qa, qsa, qb, qsb;
};
__device__ __forceinline__ void take_planes(XU& x, const uint4* s) {
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const uint4 a0 = s[2 * p], a1 = s[2 * p + 1], b0 = s[4 + 2 * p], b1 = s[4 + 2 * p + 1];
    x.a[p][0] = a0.x; x.a[p][1] = a0.y; x.a[p][2] = a0.z; x.a[p][3] = a0.w;
    x.a[p][4] = a1.x; x.a[p][5] = a1.y; x.a[p][6] = a1.z; x.a[p][7] = a1.w;
    x.b[p][0] = b0.x; x.b[p][1] = b0.y; x.b[p][2] = b0.z; x.b[p][3] = b0.w;
    x.b[p][4] = b1.x; x.b[p][5] = b1.y; x.b[p][6] = b1.z; x.b[p][7] = b1.w;
  }
}
__device__ __forceinline__ void load_xu(XU& x, const uint32_t* planes, const float2* meta, size_t g0) {
  take_planes(x, (const uint4*)(planes + g0 * QV_GROUP_DW));
  const float2 ma = meta[g0], mb = meta[g0 + 1];
  x.qa = ma.x; x.qsa = ma.y; x.qb = mb.x; x.qsb = mb.y;
}

// gguf scale_min_k4 for sub-blocks 2jj and 2jj+1 of a super-block whose header words are hd
// (hd.x = d | dmin << 16, hd.y/z/w = the 12 packed bytes q[0..11]).  Sub-blocks j < 4 keep their
// 6-bit scale in q[j] and min in q[4+j]; j >= 4 keep 4 bits of each in q[4+j] and the top 2 bits in
// the upper bits of q[j-4] / q[j].  jj differs per lane, so both forms are one sequence of
// bit-field extracts whose source word and widths are per-lane values (a width of 0 extracts 0).
__device__ __forceinline__ void k4_pair(const uint4 hd, int jj, float& a0, float& b0, float& a1, float& b1) {
  union { uint32_t u; __half2 h; } dd;
  dd.u = hd.x;
  const float d = __low2float(dd.h), dmin = __high2float(dd.h);
  const bool lo = jj < 2;
  const uint32_t sh = 16u * (jj & 1), wid = lo ? 6u : 4u, wid2 = lo ? 0u : 2u;
  const uint32_t y = hd.y, z = hd.z, w = hd.w;
  const uint32_t A = lo ? y : w, B = lo ? z : w >> 4;
  const uint32_t sc0 = __builtin_amdgcn_ubfe(A, sh, wid) | (__builtin_amdgcn_ubfe(y, sh + 6, wid2) << 4);
  const uint32_t sc1 = __builtin_amdgcn_ubfe(A, sh + 8, wid) | (__builtin_amdgcn_ubfe(y, sh + 14, wid2) << 4);
  const uint32_t m0 = __builtin_amdgcn_ubfe(B, sh, wid) | (__builtin_amdgcn_ubfe(z, sh + 6, wid2) << 4);
  const uint32_t m1 = __builtin_amdgcn_ubfe(B, sh + 8, wid) | (__builtin_amdgcn_ubfe(z, sh + 14, wid2) << 4);
  a0 = d * (float)sc0;
  a1 = d * (float)sc1;
  b0 = dmin * (float)m0;
  b1 = dmin * (float)m1;
}

// The four lanes that work on one super-block (a quad: units 4b .. 4b+3) each load one dword of its 16-byte
// header and hand the others theirs when the row is computed: 1 register per row in flight instead of 4.
__device__ __forceinline__ uint4 quad_header(uint32_t mine) {
  uint4 hd;
  hd.x = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0x00, 0xf, 0xf, true);  // quad_perm [0,0,0,0]
  hd.y = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0x55, 0xf, 0xf, true);  // [1,1,1,1]
  hd.z = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xAA, 0xf, 0xf, true);  // [2,2,2,2]
  hd.w = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xFF, 0xf, 0xf, true);  // [3,3,3,3]
  return hd;
}

// one unit of one row: c0, c1 = its 32 code bytes, hd = the super-block header
__device__ __forceinline__ float unit_dot(const uint4 c0, const uint4 c1, const uint4 hd, int jj, const XU& x) {
  const uint32_t w[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  int a0 = 0, a1 = 0, b0 = 0, b1 = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int lo = (int)(w[i] & 0x0f0f0f0fu), hi = (int)((w[i] >> 4) & 0x0f0f0f0fu);
    a0 = __builtin_amdgcn_sdot4(lo, (int)x.a[0][i], a0, false);
    a1 = __builtin_amdgcn_sdot4(lo, (int)x.a[1][i], a1, false);
    b0 = __builtin_amdgcn_sdot4(hi, (int)x.b[0][i], b0, false);
    b1 = __builtin_amdgcn_sdot4(hi, (int)x.b[1][i], b1, false);
  }
  // |a0| <= 32 * 15 * 128: the integer sum stays below 2^24 and converts exactly
  const float va = (float)(a0 * 256 + a1);
  const float vb = (float)(b0 * 256 + b1);
  float sa, ma, sb, mb;
  k4_pair(hd, jj, sa, ma, sb, mb);
  return (sa * x.qa * va + sb * x.qb * vb) - (ma * x.qsa + mb * x.qsb);
}

struct Gu4kArgs {
  const uint8_t *gate, *up;        // routed experts [E][mid rows][d/256 blocks]
  const uint8_t *sh_gate, *sh_up;  // shared expert rows (nullptr: none)
};

// grid (mid/32, slots incl. shared, P); block 512.  Wave w: gate rows 4w..4w+3 and the matching up
// rows of this block's 32; lane = unit (d/64 <= 64 units per row).  All 24 loads of a lane (8 rows x
// two code halves + its dword of the header) are in flight together, in under 128 registers: two blocks fit
// a CU, so the grid's 265 blocks are all resident at once (with one block per CU the last nine waited for a
// second round).  For the widths that moe_decgg_passes leaves: k_decgg_gu deals the others' rows over all lanes.
// NPL > 0 (E <= 64*NPL): only the logits are given; the blocks of the routed slots run the softmax /
// top-k of their token themselves and block (0, 0, token) writes ids / weights out for the down
// kernel (as in the q4cp gate/up kernel).
constexpr int G4_ROWS = 32;
template <int NPL>
__global__ void __launch_bounds__(512, 4) k_dec4k_gu(Gu4kArgs A, const uint32_t* __restrict__ xplanes,
                                                     const float2* __restrict__ xmeta,
                                                     const int* __restrict__ ids, int id_stride, int kpt, int d,
                                                     int mid, uint32_t* __restrict__ hplanes,
                                                     float2* __restrict__ hmeta, const float* __restrict__ logits,
                                                     int n_experts, int* __restrict__ ids_out,
                                                     float* __restrict__ ws_out, moe_rfix RF) {
  __shared__ float gs[G4_ROWS], us[G4_ROWS];
  __shared__ uint32_t pk[QV_GROUP_DW];
  __shared__ int sel_ids[64];
  __shared__ float sel_ws[64];
  const int s = blockIdx.y, tok = blockIdx.z, nslots = gridDim.y - (NPL > 0 ? 1 : 0);
  if (NPL > 0 && s == nslots) {
    // one block of the extra grid row: the exact softmax / top-k (ids, renormalised weights) for the down
    // launch, next to the blocks that stream the weights and only need the ids
    if (blockIdx.x == 0) {
      select_certain<NPL ? NPL : 8, 512>(logits + (size_t)tok * n_experts, RF, (int)tok, sel_ids, sel_ws, n_experts, kpt, true);
      __syncthreads();
      if ((int)threadIdx.x < kpt) {
        ids_out[(size_t)tok * id_stride + threadIdx.x] = sel_ids[threadIdx.x];
        ws_out[(size_t)tok * id_stride + threadIdx.x] = sel_ws[threadIdx.x];
      }
    }
    return;
  }
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int U = d / 64;
  const bool shared = s >= kpt;
  const uint64_t rb = (uint64_t)(d / 256) * 144;
  int e = 0;
  if (NPL > 0) {
    if (!shared) {
      // the ids by logit order; the exact selection only when two of the best logits are too close
      const float* lg = logits + (size_t)tok * n_experts;
      if (!select_certain<NPL ? NPL : 8, 512>(lg, RF, (int)tok, sel_ids, sel_ws, n_experts, kpt, false)) __syncthreads();
      e = sel_ids[s];
    }
  } else if (!shared) {
    e = ids[(size_t)tok * id_stride + s];
  }
  e = __builtin_amdgcn_readfirstlane(e);  // (the same in every lane: as a scalar, the offsets below are scalar arithmetic)
  const uint8_t* gbase = shared ? A.sh_gate : A.gate + (uint64_t)e * mid * rb;
  const uint8_t* ubase = shared ? A.sh_up : A.up + (uint64_t)e * mid * rb;
  const int r0 = blockIdx.x * G4_ROWS + 4 * wv;
  // branch-free loads: lanes past the row's units read a unit of the first super-block (their quad then still
  // assembles a real header) and count as zero
  const bool live = lane < U;
  const int ul = live ? lane : (lane & 3);
  const float mlive = live ? 1.f : 0.f;
  const int jj = ul & 3;
  const size_t uoff = (size_t)(ul >> 2) * 144;  // this lane's super-block inside a row
  XU x;
  load_xu(x, xplanes, xmeta, ((size_t)tok * U + ul) * 2);
  uint4 c0[8], c1[8];
  uint32_t hw[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const uint8_t* row = (i < 4 ? gbase : ubase) + (uint64_t)(r0 + (i & 3)) * rb + uoff;
    hw[i] = *(const uint32_t*)(row + 4 * jj);
    c0[i] = *(const uint4*)(row + 16 + jj * 32);
    c1[i] = *(const uint4*)(row + 32 + jj * 32);
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first dot product
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    acc[i] = sum64(unit_dot(c0[i], c1[i], quad_header(hw[i]), jj, x) * mlive);
    if (i & 1) __builtin_amdgcn_sched_barrier(0);  // rows are consumed in arrival order
  }
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      gs[4 * wv + i] = acc[i];
      us[4 * wv + i] = acc[4 + i];
    }
  }
  __syncthreads();
  // SwiGLU on the block's 32 rows = one sub-block of the down projection's input; quantise it
  if (wv == 0) {
    const int j = lane & 31;
    const float g = gs[j], u = us[j];
    const float hv = g / (1.f + expf(-g)) * u;
    float m = dpp_max_row(fabsf(hv));
    m = rows_half_max(m);
    const float inv = m > 0.f ? QV_XMAX / m : 0.f;
    const float q = m * (1.f / QV_XMAX);
    const int X = (int)rintf(hv * inv);
    int p0, p1;
    qv_digits(X, p0, p1);
    float sx = dpp_add_row((float)X);
    sx = rows_half_add(sx);
    if (lane < QV_GROUP_DW) pk[lane] = 0;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    if (lane < 32) {
      const int dw = j >> 2, sh = 8 * (j & 3);  // natural order
      atomicOr(&pk[dw], (uint32_t)(p0 & 0xff) << sh);
      atomicOr(&pk[8 + dw], (uint32_t)(p1 & 0xff) << sh);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    const size_t gi = ((size_t)tok * nslots + s) * (mid / 32) + blockIdx.x;
    if (lane < QV_GROUP_DW) hplanes[gi * QV_GROUP_DW + lane] = pk[lane];
    if (lane == 0) hmeta[gi] = make_float2(q, q * sx);
  }
}

struct Dn4kArgs {
  const uint8_t *down, *sh_down;  // [E][d rows][mid/256 blocks]; shared expert rows (nullptr: none)
  const float* sh_logit;
};

// grid (d/ROWS, P); block = 64 x ceil(slots/4).  A row of 16 lanes = one slot (mid/64 <= 16 units),
// holding that slot's hid planes in registers for all the block's rows.  The weighted combine runs
// afterwards in slot order (descending router probability), then the shared expert.
constexpr int D4_ROWS = 8, D4_MAXSLOTS = 16;
__global__ void __launch_bounds__(256) k_dec4k_dn(Dn4kArgs A, const uint32_t* __restrict__ hplanes,
                                                  const float2* __restrict__ hmeta, const int* __restrict__ ids,
                                                  const float* __restrict__ ws, int id_stride, int kpt, int d,
                                                  int mid, float* __restrict__ out, uint64_t out_stride) {
  __shared__ float part[D4_MAXSLOTS][D4_ROWS];
  __shared__ float wsm[D4_MAXSLOTS];
  const int tok = blockIdx.y;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const bool has_shared = A.sh_down != nullptr;
  const int nslots = kpt + (has_shared ? 1 : 0);
  const int U = mid / 64, u_raw = lane & 15, s_raw = 4 * wv + (lane >> 4);
  const int r0 = blockIdx.x * D4_ROWS;
  const uint64_t rb = (uint64_t)(mid / 256) * 144;
  // combine weights of the token, fetched while the weight rows are in flight
  float wmine = 0.f;
  if ((int)threadIdx.x < nslots)
    wmine = (int)threadIdx.x < kpt ? ws[(size_t)tok * id_stride + threadIdx.x] : A.sh_logit[tok];
  {
    // branch-free loads: lanes past the slots or the row's units read slot 0 / unit 0 and count as zero
    const bool live = s_raw < nslots && u_raw < U;
    const int s = live ? s_raw : 0, u = live ? u_raw : 0;
    const float mlive = live ? 1.f : 0.f;
    const bool shared = has_shared && s == nslots - 1;
    // (an unconditional load: under a per-lane branch the compiler waits for the id before it issues anything else)
    const int e_any = ids[tok * id_stride + (shared ? 0 : s)];
    const uint32_t e = shared ? 0u : (uint32_t)e_any;
    const uint8_t* base = (shared ? A.sh_down : A.down + (uint64_t)(e * (uint32_t)d) * rb) + (uint64_t)r0 * rb + (uint32_t)(u >> 2) * 144;
    const int jj = u & 3;
    XU x;
    load_xu(x, hplanes, hmeta, (((size_t)tok * nslots + s) * U + u) * 2);
    uint4 c0[D4_ROWS], c1[D4_ROWS], hd[D4_ROWS];
#pragma unroll
    for (int r = 0; r < D4_ROWS; r++) {
      const uint8_t* row = base + (uint64_t)r * rb;
      hd[r] = *(const uint4*)row;
      c0[r] = *(const uint4*)(row + 16 + jj * 32);
      c1[r] = *(const uint4*)(row + 32 + jj * 32);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first dot product
#pragma unroll
    for (int r = 0; r < D4_ROWS; r++) {
      const float v = dpp_add_row(unit_dot(c0[r], c1[r], hd[r], jj, x) * mlive);
      if (u_raw == 0 && s_raw < nslots) part[s_raw][r] = v;
      if (r & 1) __builtin_amdgcn_sched_barrier(0);  // rows are consumed in arrival order
    }
  }
  if ((int)threadIdx.x < nslots) wsm[threadIdx.x] = (int)threadIdx.x < kpt ? wmine : sigmoid_f(wmine);
  __syncthreads();
  if (threadIdx.x < D4_ROWS) {
    const int r = threadIdx.x;
    float y = 0.f;
    for (int i = 0; i < kpt; i++) y += wsm[i] * part[i][r];
    if (has_shared) y += wsm[kpt] * part[kpt][r];
    out[(size_t)tok * out_stride + r0 + r] = y;
  }
}

// ---------------------------------------------------------------------------------------------------------------
// The same launches for the other block types of the reference's GGUF checkpoints (Q5_K gate/up, Q5_1 / Q8_0 down,
// a Q8_0 shared expert; src/gpu/parts/30_host_util.inc:399-405, src/gguf_map.h:212-214), any mix of them with Q4_K.
// A lane still owns one unit of 64 weights = two activation groups with their two 8-bit digit planes; what differs
// per type is what a unit's bytes are and how its integer sums are scaled:
//   Q5_K  (176 B / 256): Q4_K plus a fifth bit per code; unit jj of a super-block takes bits 2jj and 2jj+1 of the 32
//         qh bytes; the four lanes of the super-block load 8 qh bytes each and hand them round by DPP
//   Q8_0  (34 B / 32):   two blocks = 68 bytes starting on a 4-byte boundary: fp16 d, 32 int8 codes (2 bytes off the
//         dword grid in the first block: one v_alignbit per word), d, 32 codes; w = d q
//   Q5_1  (24 B / 32):   two blocks = 48 bytes: fp16 d, m, 32 fifth bits, 16 code bytes (low nibbles = elements
//         0..15, high nibbles = 16..31); w = d q + m
//   IQ4_NL (18 B / 32):  two blocks = 36 bytes from a 4-byte boundary: fp16 d, 16 code bytes (2 bytes off the dword
//         grid in the first block), d, 16 code bytes; w = d kv[n] with the 16-entry int8 table of src/gguf.h:376-379,
//         looked up four codes at a time with byte permutes (iq4.h): the table is four registers of constants
//   IQ4_XS (136 B / 256): fp16 d, 8 x 6-bit sub-block scales (scales_h, scales_l), 128 code bytes; a unit = the
//         8-byte header + the 32 code bytes of sub-blocks 2jj, 2jj+1; w = d (ls - 32) kv[n]
// The type of a block (gate/up launch: one slot) or of a wave (down launch: the shared expert has a wave of its
// own) is uniform, so it is one scalar branch outside the loads.  A wave's eight rows are fetched in two batches of
// four.
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <int T> struct GgU;
template <> struct GgU<MOE_GGML_Q4_K> { uint4 c0, c1; uint32_t hw; };
template <> struct GgU<MOE_GGML_Q5_K> { uint4 c0, c1; uint2 qh; uint32_t hw; };
template <> struct GgU<MOE_GGML_Q8_0> { uint32_t w[17]; };
template <> struct GgU<MOE_GGML_Q5_1> { uint4 a, b, c; };
template <> struct GgU<MOE_GGML_IQ4_NL> { uint32_t w[9]; };
template <> struct GgU<MOE_GGML_IQ4_XS> { uint2 hd; uint4 c0, c1; };

__host__ __device__ constexpr uint64_t ggu_row_bytes(int t, uint64_t k) {
  return t == MOE_GGML_Q4_K   ? k / 256 * 144
         : t == MOE_GGML_Q5_K ? k / 256 * 176
         : t == MOE_GGML_Q8_0 ? k / 32 * 34
         : t == MOE_GGML_IQ4_NL ? k / 32 * 18
         : t == MOE_GGML_IQ4_XS ? k / 256 * 136
                                : k / 32 * 24;
}

__device__ __forceinline__ int iq4_lookup4(uint32_t q, int shift) { return (int)moe_iq4_lookup4<0>(q, shift); }
// rows in flight together: four (eight Q4_K rows of nine registers spill next to the kernel's other state and measured
// 1.4 us slower per token than two batches of four)
template <int T> constexpr int ggu_batch() { return 4; }

template <int T>
__device__ __forceinline__ void ggu_fetch(const uint8_t* row, int ul, GgU<T>& o) {
  const int jj = ul & 3;
  if constexpr (T == MOE_GGML_Q4_K) {
    const uint8_t* sb = row + (size_t)(ul >> 2) * 144;
    o.hw = *(const uint32_t*)(sb + 4 * jj);
    o.c0 = *(const uint4*)(sb + 16 + jj * 32);
    o.c1 = *(const uint4*)(sb + 32 + jj * 32);
  } else if constexpr (T == MOE_GGML_Q5_K) {
    const uint8_t* sb = row + (size_t)(ul >> 2) * 176;
    o.hw = *(const uint32_t*)(sb + 4 * jj);
    o.qh = *(const uint2*)(sb + 16 + 8 * jj);
    o.c0 = *(const uint4*)(sb + 48 + jj * 32);
    o.c1 = *(const uint4*)(sb + 64 + jj * 32);
  } else if constexpr (T == MOE_GGML_Q8_0) {
    const uint8_t* p = row + (size_t)ul * 68;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const u32x4_a4 v = *(const u32x4_a4*)(p + 16 * i);
      o.w[4 * i] = v.x; o.w[4 * i + 1] = v.y; o.w[4 * i + 2] = v.z; o.w[4 * i + 3] = v.w;
    }
    o.w[16] = *(const uint32_t*)(p + 64);
  } else if constexpr (T == MOE_GGML_IQ4_NL) {
    const uint32_t* p = (const uint32_t*)(row + (size_t)ul * 36);
    const u32x4_a4 v0 = *(const u32x4_a4*)p, v1 = *(const u32x4_a4*)(p + 4);
    o.w[0] = v0.x; o.w[1] = v0.y; o.w[2] = v0.z; o.w[3] = v0.w;
    o.w[4] = v1.x; o.w[5] = v1.y; o.w[6] = v1.z; o.w[7] = v1.w;
    o.w[8] = p[8];
  } else if constexpr (T == MOE_GGML_IQ4_XS) {
    const uint8_t* sb = row + (size_t)(ul >> 2) * 136;
    o.hd = *(const uint2*)sb;
    const u32x4_a4 v0 = *(const u32x4_a4*)(sb + 8 + jj * 32), v1 = *(const u32x4_a4*)(sb + 24 + jj * 32);
    o.c0 = uint4{v0.x, v0.y, v0.z, v0.w};
    o.c1 = uint4{v1.x, v1.y, v1.z, v1.w};
  } else {
    const uint4* p = (const uint4*)(row + (size_t)ul * 48);
    o.a = p[0]; o.b = p[1]; o.c = p[2];
  }
}

// A unit's activations as they are (layers whose activations stay in f32, moe_decgg_f32_supported): its 64 values and their sums by group.
struct XF {
  float a[32], b[32], sa, sb;
};
__device__ __forceinline__ void take_f32(XF& x, const float4* s) {
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 a = s[i], b = s[8 + i];
    x.a[4 * i] = a.x; x.a[4 * i + 1] = a.y; x.a[4 * i + 2] = a.z; x.a[4 * i + 3] = a.w;
    x.b[4 * i] = b.x; x.b[4 * i + 1] = b.y; x.b[4 * i + 2] = b.z; x.b[4 * i + 3] = b.w;
  }
}
__device__ __forceinline__ void sum_f32(XF& x) {
  float a[4] = {}, b[4] = {};
#pragma unroll
  for (int i = 0; i < 32; i++) {
    a[i & 3] += x.a[i];
    b[i & 3] += x.b[i];
  }
  x.sa = (a[0] + a[1]) + (a[2] + a[3]);
  x.sb = (b[0] + b[1]) + (b[2] + b[3]);
}

// The sum over a group of codes times activations, group A or B (GB) of a unit; codes come four to a word as signed (S) or unsigned bytes.
template <class X> struct Acc;
template <> struct Acc<XU> { int hi = 0, lo = 0; };
template <> struct Acc<XF> { float v = 0.f; };
template <bool GB, bool S>
__device__ __forceinline__ void dot4(Acc<XU>& c, int codes, const XU& x, int i) {
  c.hi = __builtin_amdgcn_sdot4(codes, (int)(GB ? x.b : x.a)[0][i], c.hi, false);
  c.lo = __builtin_amdgcn_sdot4(codes, (int)(GB ? x.b : x.a)[1][i], c.lo, false);
}
template <bool GB, bool S>
__device__ __forceinline__ void dot4(Acc<XF>& c, int codes, const XF& x, int i) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float n = S ? (float)(int8_t)(codes >> (8 * j)) : (float)(((uint32_t)codes >> (8 * j)) & 0xffu);
    c.v = fmaf(n, (GB ? x.b : x.a)[4 * i + j], c.v);
  }
}
// s times that sum.  (digit planes: the integer sums can exceed 2^24 for 5- and 8-bit codes: two exact conversions and one rounded fma
// instead of an integer combine)
template <bool GB>
__device__ __forceinline__ float times(float s, const Acc<XU>& c, const XU& x) { return s * (GB ? x.qb : x.qa) * fmaf((float)c.hi, 256.f, (float)c.lo); }
template <bool GB>
__device__ __forceinline__ float times(float s, const Acc<XF>& c, const XF& x) { return s * c.v; }
// the group's activations, summed
template <bool GB>
__device__ __forceinline__ float total(const XU& x) { return GB ? x.qsb : x.qsa; }
template <bool GB>
__device__ __forceinline__ float total(const XF& x) { return GB ? x.sb : x.sa; }

template <int T, class X>
__device__ __forceinline__ float ggu_dot(const GgU<T>& o, int jj, const X& x) {
  Acc<X> va, vb;
  if constexpr (T == MOE_GGML_Q4_K && std::is_same<X, XU>::value) {
    return unit_dot(o.c0, o.c1, quad_header(o.hw), jj, x);
  } else if constexpr (T == MOE_GGML_Q4_K) {
    const uint32_t w[8] = {o.c0.x, o.c0.y, o.c0.z, o.c0.w, o.c1.x, o.c1.y, o.c1.z, o.c1.w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      dot4<false, false>(va, (int)(w[i] & 0x0f0f0f0fu), x, i);
      dot4<true, false>(vb, (int)((w[i] >> 4) & 0x0f0f0f0fu), x, i);
    }
    float sa, ma, sb, mb;
    k4_pair(quad_header(o.hw), jj, sa, ma, sb, mb);
    return (times<false>(sa, va, x) + times<true>(sb, vb, x)) - (ma * total<false>(x) + mb * total<true>(x));
  } else if constexpr (T == MOE_GGML_Q5_K) {
    const uint4 hd = quad_header(o.hw);
    const uint32_t w[8] = {o.c0.x, o.c0.y, o.c0.z, o.c0.w, o.c1.x, o.c1.y, o.c1.z, o.c1.w};
    const uint32_t to4 = 2u * (uint32_t)jj - 4u, to4h = to4 + 1u;  // (rotations take them modulo 32)
    // qh word i (bytes 4i..4i+3) sits in lane i/2 of the quad, register i%2
    uint32_t qh[8];
    qh[0] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.x, 0x00, 0xf, 0xf, true);
    qh[1] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.y, 0x00, 0xf, 0xf, true);
    qh[2] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.x, 0x55, 0xf, 0xf, true);
    qh[3] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.y, 0x55, 0xf, 0xf, true);
    qh[4] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.x, 0xAA, 0xf, 0xf, true);
    qh[5] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.y, 0xAA, 0xf, 0xf, true);
    qh[6] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.x, 0xFF, 0xf, 0xf, true);
    qh[7] = (uint32_t)__builtin_amdgcn_mov_dpp((int)o.qh.y, 0xFF, 0xf, 0xf, true);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      // (the unit's two bits rotated to bit 4 of each byte: 2 operations of 20 per word less)
      const int lo = (int)((w[i] & 0x0f0f0f0fu) | (__builtin_amdgcn_alignbit(qh[i], qh[i], to4) & 0x10101010u));
      const int hi = (int)(((w[i] >> 4) & 0x0f0f0f0fu) | (__builtin_amdgcn_alignbit(qh[i], qh[i], to4h) & 0x10101010u));
      dot4<false, false>(va, lo, x, i);
      dot4<true, false>(vb, hi, x, i);
    }
    float sa, ma, sb, mb;
    k4_pair(hd, jj, sa, ma, sb, mb);
    return (times<false>(sa, va, x) + times<true>(sb, vb, x)) - (ma * total<false>(x) + mb * total<true>(x));
  } else if constexpr (T == MOE_GGML_Q8_0) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int ca = (int)__builtin_amdgcn_alignbit(o.w[i + 1], o.w[i], 16);  // the first block's codes: 2 bytes off the dword grid
      const int cb = (int)o.w[9 + i];
      dot4<false, true>(va, ca, x, i);
      dot4<true, true>(vb, cb, x, i);
    }
    union { uint16_t u; __half h; } d0, d1;
    d0.u = (uint16_t)(o.w[0] & 0xffffu);
    d1.u = (uint16_t)(o.w[8] >> 16);
    return times<false>(__half2float(d0.h), va, x) + times<true>(__half2float(d1.h), vb, x);
  } else if constexpr (T == MOE_GGML_IQ4_NL || T == MOE_GGML_IQ4_XS) {
    uint32_t qa[4], qb[4];  // the 16 code bytes of the unit's two 32-element blocks
    float da, db;           // their scales
    if constexpr (T == MOE_GGML_IQ4_NL) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        qa[i] = __builtin_amdgcn_alignbit(o.w[i + 1], o.w[i], 16);  // the first block's codes: 2 bytes off the dword grid
        qb[i] = o.w[5 + i];
      }
      union { uint16_t u; __half h; } d0, d1;
      d0.u = (uint16_t)(o.w[0] & 0xffffu);
      d1.u = (uint16_t)(o.w[4] >> 16);
      da = __half2float(d0.h);
      db = __half2float(d1.h);
    } else {
      qa[0] = o.c0.x; qa[1] = o.c0.y; qa[2] = o.c0.z; qa[3] = o.c0.w;
      qb[0] = o.c1.x; qb[1] = o.c1.y; qb[2] = o.c1.z; qb[3] = o.c1.w;
      // sub-blocks 2jj, 2jj+1: 6-bit scales = a nibble of scales_l[jj] | two bits of scales_h << 4, minus 32
      union { uint16_t u; __half h; } dv;
      dv.u = (uint16_t)(o.hd.x & 0xffffu);
      const uint32_t sh = o.hd.x >> 16, sl = (o.hd.y >> (8 * jj)) & 0xffu;
      const int la = (int)((sl & 0xfu) | (((sh >> (4 * jj)) & 3u) << 4)) - 32;
      const int lb = (int)((sl >> 4) | (((sh >> (4 * jj + 2)) & 3u) << 4)) - 32;
      const float dd = __half2float(dv.h);
      da = dd * (float)la;
      db = dd * (float)lb;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int al = iq4_lookup4(qa[i], 0), ah = iq4_lookup4(qa[i], 4);
      const int bl = iq4_lookup4(qb[i], 0), bh = iq4_lookup4(qb[i], 4);
      dot4<false, true>(va, al, x, i);
      dot4<false, true>(va, ah, x, 4 + i);
      dot4<true, true>(vb, bl, x, i);
      dot4<true, true>(vb, bh, x, 4 + i);
    }
    return times<false>(da, va, x) + times<true>(db, vb, x);
  } else {  // Q5_1
    const uint32_t dw[12] = {o.a.x, o.a.y, o.a.z, o.a.w, o.b.x, o.b.y, o.b.z, o.b.w, o.c.x, o.c.y, o.c.z, o.c.w};
    auto block = [&](auto gb, Acc<X>& v) {
      constexpr bool GB = decltype(gb)::value;
      const uint32_t dm = dw[6 * GB], qh = dw[6 * GB + 1];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t q = dw[6 * GB + 2 + i];
        // four fifth bits (elements 4i.. / 16 + 4i..) to bit 4 of the four bytes
        const uint32_t hl = ((((qh >> (4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
        const uint32_t hh = ((((qh >> (16 + 4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
        dot4<GB, false>(v, (int)((q & 0x0f0f0f0fu) | hl), x, i);
        dot4<GB, false>(v, (int)(((q >> 4) & 0x0f0f0f0fu) | hh), x, 4 + i);
      }
      union { uint32_t u; __half2 h; } cv;
      cv.u = dm;
      return times<GB>(__low2float(cv.h), v, x) + __high2float(cv.h) * total<GB>(x);
    };
    return block(std::false_type{}, va) + block(std::true_type{}, vb);
  }
}

// How a wave of the gate/up launch walks its eight rows: as a ring, in which a row that has been multiplied makes place for the one
// four on, or as two batches of four, each waited for.  The ring keeps loads in flight all the time, and its fences keep the
// compiler from interleaving two rows' arithmetic, which Q5_K's, Q8_0's and Q5_1's rows (the longest) need once there are
// tokens enough to hide the loads: the layer at 3072 x 768, us, ring and batches, gate/up / down types, 8, 20 and 32 tokens Q8_0 /
// Q8_0 136.4 134.8, 299.2 292.3, 462.9 451.2; Q5_K / Q8_0 118.3 117.8, 252.3 250.0, 387.0 382.4; Q5_1 / Q8_0 117.2 117.3, 250.3
// 249.1, 382.7 380.7; Q5_K / Q5_K 107.2 106.0, 227.5 225.0, 355.9 353.2.
// Q4_K and IQ4 rows are level or better in the ring (20 tokens, batches and ring: Q4_K 231.0 231.5, IQ4_NL 227.4 226.0, IQ4_XS
// 232.1 231.5; 1 token, four layers: Q4_K 112.8 111.5); one and two tokens of any type are within 1 % either way (FEW).  Down
// rows are better in the ring for every type (ggu_dn_rows; 1 token, four layers: Q5_K / Q8_0 117.5 115.6, Q4_K / Q8_0 111.5
// 107.9, Q8_0 132.5 129.6, Q5_1 112.4 111.4, IQ4_NL 115.4 114.9).
template <int T, bool FEW>
constexpr bool ggu_gu_ring() { return FEW || T == MOE_GGML_Q4_K || T == MOE_GGML_IQ4_NL || T == MOE_GGML_IQ4_XS; }
// eight rows of one wave (gate/up launch: four gate rows and the matching up rows): acc[i] = wave sum of row i
template <int T, bool FEW>
__device__ __forceinline__ void ggu_gu_rows(const uint8_t* gbase, const uint8_t* ubase, int r0, int d, int ul,
                                            float mlive, const XU& x, float (&acc)[8]) {
  constexpr int RB = ggu_batch<T>();
  const uint64_t rb = ggu_row_bytes(T, (uint64_t)d);
  const int jj = ul & 3;
  if constexpr (ggu_gu_ring<T, FEW>()) {
    GgU<T> u[RB];
    auto fetch = [&](int i) { ggu_fetch<T>((i < 4 ? gbase : ubase) + (uint64_t)(r0 + (i & 3)) * rb, ul, u[i % RB]); };
#pragma unroll
    for (int i = 0; i < RB; i++) fetch(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      acc[i] = sum64(ggu_dot<T>(u[i % RB], jj, x) * mlive);
      __builtin_amdgcn_sched_barrier(0);  // rows are consumed in arrival order
      if (i + RB < 8) fetch(i + RB);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int h = 0; h < 8; h += RB) {
      GgU<T> u[RB];
#pragma unroll
      for (int i = 0; i < RB; i++)
        ggu_fetch<T>(((i + h) < 4 ? gbase : ubase) + (uint64_t)(r0 + ((i + h) & 3)) * rb, ul, u[i]);
      __builtin_amdgcn_sched_barrier(0);  // every load of the batch is issued before the first dot product
#pragma unroll
      for (int i = 0; i < RB; i++) {
        acc[i + h] = sum64(ggu_dot<T>(u[i], jj, x) * mlive);
        if (i & 1) __builtin_amdgcn_sched_barrier(0);  // rows are consumed in arrival order
      }
    }
  }
}

// The same eight rows with no lane idle, for rows of U = 8 NP units (NP 4 .. 7): a pass takes one row on lanes 0 .. U - 1, and the
// other 64 - U lanes take the rows behind the first NP, unit by unit (rows follow one another in memory, and the first four are gate
// rows, so what those lanes read is one run of the up tensor): 8 U units in NP passes instead of eight.  A sum of eight lanes lies
// within a row on both sides; part[8 NP] = these sums in the order of the units.  xs: the token's activations in LDS, a unit's 128
// + 16 bytes side by side (the pitch that 16-byte reads of neighbouring units want): lanes of the first kind read theirs once, the
// others a unit's for each pass, which costs LDS a tenth of what the pass's vector instructions cost the SIMD.
// What bounds the launch is those instructions (Q5_K: 145 a pass) from three tokens on, and the loads' latency below.  RB: passes in
// flight; three (with the selection inside the launch, up to four tokens: 1 token, four layers, 100.3 -> 97.8 us; two and a ring of
// five or six, which spills, are slower) or four (20 tokens 223.5, with three 224.1).
// Layers, us, a lane per unit of a row and this (weights from HBM, other inputs each call; four layers, at 20 tokens two): 3072 x 768
// Q5_K / Q8_0 1 token 115 104, 2 168 156, 3 228 208, 4 277 251, 5 318 295, 8 441 402, 20 467 421; Q4_K (k_dec4k_gu, at 1 and 2 tokens with its
// down launch, and this) 1 95.0 85.7, 2 142 127, 3 180 164, 4 225 203, 5 240 224, 8 324 303, 20 330 301; 1 and 20 tokens Q8_0 130 115, 562 529; Q5_1 / Q8_0
// 114 104, 462 439; IQ4_NL 120 105, 410 366; IQ4_XS 124 106, 412 370; Q5_K / Q8_0 2048 wide 99 81, 383 304; 3584 129 119, 530 502; Q4_K 2560
// wide 94 83, 298 268.
constexpr int gx_dw(bool f32) { return f32 ? 68 : 36; }  // dwords of a unit in LDS
__device__ __forceinline__ void lds_x(XU& x, const uint32_t* xs, int unit) {
  const uint4* s = (const uint4*)(xs + unit * gx_dw(false));
  take_planes(x, s);
  const uint4 m = s[8];
  x.qa = __uint_as_float(m.x); x.qsa = __uint_as_float(m.y); x.qb = __uint_as_float(m.z); x.qsb = __uint_as_float(m.w);
}
__device__ __forceinline__ void lds_x(XF& x, const uint32_t* xs, int unit) {
  const float* s = (const float*)(xs + unit * gx_dw(true));
  take_f32(x, (const float4*)s);
  x.sa = s[64];
  x.sb = s[65];
}
// (f32 activations, 66 registers, leave room for two passes)
constexpr int ggu_ring(int npl, bool f32) { return f32 ? 2 : npl > 0 ? 3 : 4; }
__device__ __forceinline__ float sum8(float v) {  // over the eight lanes of an eighth of a wave
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));          // xor 1
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));          // xor 2
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));  // mirror in 8
}
template <int T, int NP, int RB, class X, class Stage>
__device__ __forceinline__ void ggu_gu_packed(const uint8_t* gbase, const uint8_t* ubase, int r0, int lane, const uint32_t* xs, float* part,
                                              Stage&& stage) {
  constexpr int U = 8 * NP, L = 64 - U;
  constexpr uint64_t rb = ggu_row_bytes(T, 64 * U);
  const bool main_lane = lane < U;
  const int u0 = main_lane ? lane : lane - U;
  const uint8_t* const side = ubase + (uint64_t)(r0 + NP - 4) * rb;
  GgU<T> u[RB];
  auto fetch = [&](int p) {
    const uint8_t* const row = (p < 4 ? gbase : ubase) + (uint64_t)(r0 + (p & 3)) * rb;
    ggu_fetch<T>(main_lane ? row : side, main_lane ? u0 : u0 + p * L, u[p % RB]);
  };
#pragma unroll
  for (int p = 0; p < RB; p++) fetch(p);
  __builtin_amdgcn_sched_barrier(0);
  stage();
  X x;
  lds_x(x, xs, u0);
#pragma unroll
  for (int p = 0; p < NP; p++) {
    if (p) {
      const int un = u0 + p * L;
      if (!main_lane) lds_x(x, xs, un % U);
    }
    float v = ggu_dot<T>(u[p % RB], lane & 3, x);
    v = sum8(v);
    if ((lane & 7) == 0) part[main_lane ? p * NP + (u0 >> 3) : NP * NP + ((u0 + p * L) >> 3)] = v;
    __builtin_amdgcn_sched_barrier(0);  // passes are consumed in arrival order
    if (p + RB < NP) fetch(p + RB);
    __builtin_amdgcn_sched_barrier(0);
  }
}

#define GGU_SWITCH(t, CALL)                                                       \
  switch (t) {                                                                    \
    case MOE_GGML_Q4_K: { constexpr int T = MOE_GGML_Q4_K; CALL; } break;          \
    case MOE_GGML_Q5_K: { constexpr int T = MOE_GGML_Q5_K; CALL; } break;          \
    case MOE_GGML_Q8_0: { constexpr int T = MOE_GGML_Q8_0; CALL; } break;          \
    case MOE_GGML_IQ4_NL: { constexpr int T = MOE_GGML_IQ4_NL; CALL; } break;      \
    case MOE_GGML_IQ4_XS: { constexpr int T = MOE_GGML_IQ4_XS; CALL; } break;      \
    default: { constexpr int T = MOE_GGML_Q5_1; CALL; } break;                    \
  }

// (moe_decgg_f32_supported's down rows)
#define GGU_SWITCH_F32(t, CALL)                                                      \
  switch (t) {                                                                    \
    case MOE_GGML_Q8_0: { constexpr int T = MOE_GGML_Q8_0; CALL; } break;          \
    default: { constexpr int T = MOE_GGML_Q5_1; CALL; } break;                    \
  }

struct GuGgArgs {
  const uint8_t *gate, *up, *sh_gate, *sh_up;
  int tgu, tsh;
};

// grid (mid/32, slots incl. shared + the exact top-k row, P); block 512: k_dec4k_gu<NPL> for any of the four types
// NP: rows of 8 NP units, dealt over all lanes (ggu_gu_packed); 0: a lane per unit of a row.
// F32 (with NP): x and hid as they are, x32 and hid32, instead of digit planes
template <int NPL, int NP, bool F32 = false>
__global__ void __launch_bounds__(512, 4) k_decgg_gu(GuGgArgs A, const uint32_t* __restrict__ xplanes,
                                                     const float2* __restrict__ xmeta, int id_stride, int kpt, int d,
                                                     int mid, uint32_t* __restrict__ hplanes,
                                                     float2* __restrict__ hmeta, const float* __restrict__ logits,
                                                     int n_experts, int* __restrict__ ids_out,
                                                     float* __restrict__ ws_out, const int* __restrict__ ids_in, moe_rfix RF,
                                                     const float* __restrict__ x32, float* __restrict__ hid32) {
  static_assert(!F32 || NP, "rows dealt over all lanes");
  // a row's sums: of its eighths of 8 lanes, or of all of it; wave, row, part
  constexpr int PARTS = NP ? NP : 1;
  __shared__ float part[8 * 8 * PARTS];
  __shared__ __attribute__((aligned(16))) uint32_t xs[NP ? 8 * NP * gx_dw(F32) : 4];
  __shared__ uint32_t pk[QV_GROUP_DW];
  __shared__ int sel_ids[64];
  __shared__ float sel_ws[64];
  const int s = blockIdx.y, tok = blockIdx.z, nslots = gridDim.y - (NPL > 0 ? 1 : 0);
  if (NPL > 0 && s == nslots) {  // the extra grid row: exact softmax / top-k for the down launch
    if (blockIdx.x == 0) {
      select_certain<NPL ? NPL : 8, 512>(logits + (size_t)tok * n_experts, RF, (int)tok, sel_ids, sel_ws, n_experts, kpt, true);
      __syncthreads();
      if ((int)threadIdx.x < kpt) {
        ids_out[(size_t)tok * id_stride + threadIdx.x] = sel_ids[threadIdx.x];
        ws_out[(size_t)tok * id_stride + threadIdx.x] = sel_ws[threadIdx.x];
      }
    }
    return;
  }
  const int lane = threadIdx.x & 63, wv = NP ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : (int)(threadIdx.x >> 6);
  const int U = d / 64;
  const bool shared = s >= kpt;
  int e = 0;
  if (!shared) {
    if (NPL > 0) {
      const float* lg = logits + (size_t)tok * n_experts;
      if (!select_certain<NPL ? NPL : 8, 512>(lg, RF, (int)tok, sel_ids, sel_ws, n_experts, kpt, false)) __syncthreads();
      e = sel_ids[s];
    } else {
      e = ids_in[(size_t)tok * id_stride + s];  // (NPL == 0: the ids come from the router's launches)
    }
  }
  e = __builtin_amdgcn_readfirstlane(e);  // (the same in every lane: as a scalar, the offsets below are scalar arithmetic)
  const int t = shared ? A.tsh : A.tgu;
  const uint64_t rb = ggu_row_bytes(t, (uint64_t)d);
  const uint8_t* gbase = shared ? A.sh_gate : A.gate + (uint64_t)e * mid * rb;
  const uint8_t* ubase = shared ? A.sh_up : A.up + (uint64_t)e * mid * rb;
  const int r0 = blockIdx.x * G4_ROWS + 4 * wv;
  if constexpr (NP > 0) {
    // (the activations, requested ahead of the weights, go to LDS behind the weights' requests)
    const int t0 = (int)threadIdx.x;
    constexpr int XP = 8 * NP * (F32 ? 16 : 8);  // 16-byte pieces of the activations
    static_assert(XP <= 1024 && XP % 64 == 0, "two to a thread, whole waves");
    const uint4* const xg = (F32 ? (const uint4*)x32 : (const uint4*)xplanes) + (size_t)tok * XP;
    const uint4 xp = xg[t0 < XP ? t0 : 0], xp2 = XP > 512 ? xg[t0 + 512 < XP ? t0 + 512 : 0] : xp;
    const uint4 xm = F32 ? xp : ((const uint4*)xmeta)[(size_t)tok * (8 * NP) + (t0 < 8 * NP ? t0 : 0)];
    __builtin_amdgcn_sched_barrier(0);
    auto stage = [&]() {
      auto put = [&](int i, const uint4& v) {
        constexpr int PU = F32 ? 16 : 8;  // pieces of a unit
        uint32_t* const u = xs + i / PU * gx_dw(F32);
        if (i < XP) *(uint4*)(u + i % PU * 4) = v;
        if (F32) {  // (a group is the pieces of eight neighbouring lanes)
          float g = (__uint_as_float(v.x) + __uint_as_float(v.y)) + (__uint_as_float(v.z) + __uint_as_float(v.w));
          g = sum8(g);
          if (i < XP && (i & 7) == 0) u[64 + ((i >> 3) & 1)] = __float_as_uint(g);
        }
      };
      put(t0, xp);
      if (XP > 512) put(t0 + 512, xp2);
      if (!F32 && t0 < 8 * NP) *(uint4*)(xs + t0 * gx_dw(false) + 32) = xm;
      moe_lds_barrier();  // (the weights stay in flight)
      __builtin_amdgcn_sched_barrier(0);
    };
    typedef typename std::conditional<F32, XF, XU>::type X;
    GGU_SWITCH(t, (ggu_gu_packed<T, NP, ggu_ring(NPL, F32), X>(gbase, ubase, r0, lane, xs, part + 8 * NP * wv, stage)));
  } else {
    const bool live = lane < U;
    const int ul = live ? lane : (lane & 3);
    const float mlive = live ? 1.f : 0.f;
    XU x;
    load_xu(x, xplanes, xmeta, ((size_t)tok * U + ul) * 2);
    float acc[8];
    GGU_SWITCH(t, (ggu_gu_rows<T, (NPL > 0)>(gbase, ubase, r0, d, ul, mlive, x, acc)));
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < 8; i++) part[8 * wv + i] = acc[i];
    }
  }
  __syncthreads();
  if (wv == 0) {  // SwiGLU on the block's 32 rows = one activation group of the down projection; quantise it
    const int j = lane & 31;
    const float* const pg = part + ((j >> 2) * 8 + (j & 3)) * PARTS;
    float g = pg[0], u = pg[4 * PARTS];
#pragma unroll
    for (int i = 1; i < PARTS; i++) {
      g += pg[i];
      u += pg[4 * PARTS + i];
    }
    const float hv = g / (1.f + expf(-g)) * u;
    if (F32) {
      if (lane < 32) hid32[((size_t)tok * nslots + s) * mid + blockIdx.x * G4_ROWS + j] = hv;
      return;
    }
    float m = dpp_max_row(fabsf(hv));
    m = rows_half_max(m);
    const float inv = m > 0.f ? QV_XMAX / m : 0.f;
    const float q = m * (1.f / QV_XMAX);
    const int X = (int)rintf(hv * inv);
    int p0, p1;
    qv_digits(X, p0, p1);
    float sx = dpp_add_row((float)X);
    sx = rows_half_add(sx);
    if (lane < QV_GROUP_DW) pk[lane] = 0;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    if (lane < 32) {
      const int dw = j >> 2, sh = 8 * (j & 3);
      atomicOr(&pk[dw], (uint32_t)(p0 & 0xff) << sh);
      atomicOr(&pk[8 + dw], (uint32_t)(p1 & 0xff) << sh);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    const size_t gi = ((size_t)tok * nslots + s) * (mid / 32) + blockIdx.x;
    if (lane < QV_GROUP_DW) hplanes[gi * QV_GROUP_DW + lane] = pk[lane];
    if (lane == 0) hmeta[gi] = make_float2(q, q * sx);
  }
}

struct DnGgArgs {
  const uint8_t *down, *sh_down;
  const float* sh_logit;
  int tdn, tsh;
};

// NR output rows of a wave's slots, row j at first + j step of `base`: U lanes of a slot, summed four (QUADS) or two at a time
template <int T, int NR, bool QUADS, class X, class Store>
__device__ __forceinline__ void ggu_dn_rows(const uint8_t* base, int mid, int first, int step, int ul, float mlive, const X& x, Store&& store) {
  constexpr int RB = NR < ggu_batch<T>() ? NR : ggu_batch<T>();
  const uint64_t rb = ggu_row_bytes(T, (uint64_t)mid);
  const int jj = ul & 3;
  GgU<T> u[RB];
  auto fetch = [&](int j) {
    const int r = first + j * step;
    ggu_fetch<T>(base + (uint64_t)(r < D4_ROWS ? r : D4_ROWS - 1) * rb, ul, u[j % RB]);
  };
#pragma unroll
  for (int j = 0; j < RB; j++) fetch(j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NR; j++) {
    float v = ggu_dot<T>(u[j % RB], jj, x) * mlive;
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));  // xor 1
    if (QUADS) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));  // xor 2
    store(first + j * step, v);
    __builtin_amdgcn_sched_barrier(0);
    if (j + RB < NR) fetch(j + RB);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// grid (d/D4_ROWS, P); block = 64 x (ceil(kpt/S) + 1 with a shared expert).  A slot is U = mid / 64 lanes (4, 8, 12 or 16) with a unit
// each, S = 64 / U slots share a wave: waves 0.. hold the routed slots, the last wave the shared expert alone, whose S groups of
// lanes take different rows, so that a wave's block type is uniform.  (Sixteen lanes to a slot whatever its units, and eight rows of the
// shared expert in sixteen lanes of its wave, took four waves for ten slots of twelve units where this takes three, one of them a
// quarter as long.  Q5_K / Q8_0 layers, 3072 x 768, us: 1 token (four layers) 115.0 -> 110.0, 3 (two) 117.6 116.6, 8 120.0 116.4, 20 252 242,
// 32 379 363.  Q4_K layers' own kernel below 32 tokens is faster for them: 1 token 90.7 against 93.2, 20 tokens 175.9, 176.4.)
// U = 2, 6, 10 or 14 (moe_decgg_f32_supported): hid as it is, hid32, instead of digit planes.
template <int U>
__global__ void __launch_bounds__(320) k_decgg_dn(DnGgArgs A, const uint32_t* __restrict__ hplanes,
                                                  const float2* __restrict__ hmeta, const int* __restrict__ ids,
                                                  const float* __restrict__ ws, int id_stride, int kpt, int d,
                                                  float* __restrict__ out, uint64_t out_stride, const float* __restrict__ hid32) {
  constexpr int S = 64 / U, mid = 64 * U, NSH = (D4_ROWS + S - 1) / S, PL = U % 4 ? 2 : 4, NPC = U / PL;
  constexpr bool F32 = PL == 2;
  __shared__ __attribute__((aligned(16))) float part[D4_MAXSLOTS + 1][D4_ROWS][NPC > 4 ? 8 : 4];  // a slot's row: the sums of its quads (pairs) of lanes
  __shared__ float wsm[D4_MAXSLOTS + 1];
  const int tok = blockIdx.y;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool has_shared = A.sh_down != nullptr;
  const int nslots = kpt + (has_shared ? 1 : 0), rw = (kpt + S - 1) / S;  // rw: waves of routed slots
  const int r0 = blockIdx.x * D4_ROWS;
  float wmine = 0.f;
  if ((int)threadIdx.x < nslots)
    wmine = (int)threadIdx.x < kpt ? ws[(size_t)tok * id_stride + threadIdx.x] : A.sh_logit[tok];
  {
    const bool shw = wv >= rw;  // the shared expert's wave
    const int group = lane / U, ul = lane % U, s_raw = shw ? kpt : S * wv + group;
    const bool live = group < S && (shw || s_raw < kpt);
    const int s = live ? s_raw : shw ? kpt : 0;
    const float mlive = live ? 1.f : 0.f;
    const int t = shw ? A.tsh : A.tdn;
    const uint64_t rb = ggu_row_bytes(t, (uint64_t)mid);
    // (an unconditional load: under a per-lane branch the compiler waits for the id before it issues anything else)
    const int e_any = ids[tok * id_stride + (shw ? 0 : s)];
    const uint32_t e = shw ? 0u : (uint32_t)e_any;
    const uint8_t* base = (shw ? A.sh_down : A.down + (uint64_t)(e * (uint32_t)d) * rb) + (uint64_t)r0 * rb;
    typename std::conditional<F32, XF, XU>::type x;
    if constexpr (F32) take_f32(x, (const float4*)(hid32 + (((size_t)tok * nslots + s) * U + ul) * 64));
    else load_xu(x, hplanes, hmeta, (((size_t)tok * nslots + s) * U + ul) * 2);
    auto store = [&](int r, float v) {
      if (live && r < D4_ROWS && ul % PL == 0) part[s][r][ul / PL] = v;
    };
    if constexpr (!F32) {
      if (shw) GGU_SWITCH(t, (ggu_dn_rows<T, NSH, true>(base, mid, group < S ? group : 0, S, ul, mlive, x, store)))
      else GGU_SWITCH(t, (ggu_dn_rows<T, D4_ROWS, true>(base, mid, 0, 1, ul, mlive, x, store)))
    } else {
      sum_f32(x);
      if (shw) GGU_SWITCH_F32(t, (ggu_dn_rows<T, NSH, false>(base, mid, group < S ? group : 0, S, ul, mlive, x, store)))
      else GGU_SWITCH_F32(t, (ggu_dn_rows<T, D4_ROWS, false>(base, mid, 0, 1, ul, mlive, x, store)))
    }
  }
  if ((int)threadIdx.x < nslots) wsm[threadIdx.x] = (int)threadIdx.x < kpt ? wmine : sigmoid_f(wmine);
  __syncthreads();
  if (threadIdx.x < D4_ROWS) {
    const int r = threadIdx.x;
    auto total = [&](int s) {
      float v = part[s][r][0];
#pragma unroll
      for (int i = 1; i < NPC; i++) v += part[s][r][i];
      return v;
    };
    float y = 0.f;
    for (int i = 0; i < kpt; i++) y += wsm[i] * total(i);
    if (has_shared) y += wsm[kpt] * total(kpt);
    out[(size_t)tok * out_stride + r0 + r] = y;
  }
}

// ---- distinct experts of a small batch (verify-size batches: tokens share experts) ----
// The expert-sorted pair lists of the routing permutation, cut into tiles of at most GGQ_PAIRS pairs of one expert
// (the shared expert: expert id >= n_experts, over all tokens): a block fetches its weight rows once and walks the
// tile's pairs, so every distinct expert's bytes are read once per batch instead of once per token
// (reference: the _uq kernels, src/gpu/parts/26_kernels_moe_gguf.inc:758-886).
constexpr int GGQ_PAIRS = 4;  // pairs per tile (the tile lists are built with this cap)
// rows fetched together: two (with a pair's activation planes next to them the kernels stay under 128 registers,
// two blocks per CU; four rows spill)
template <int T>
__device__ __host__ constexpr int ggq_batch() { return T == MOE_GGML_Q8_0 ? 4 : 8; }
template <int T>
__device__ __host__ constexpr int ggq_dn_batch() { return T == MOE_GGML_Q8_0 ? 2 : 4; }
constexpr int GGQ_DR = 4, GGQ_DROWS = 16 * GGQ_DR;  // down: output rows per row of 16 lanes, per block

// eight rows of one wave in batches of GGQ_RB, each batch against every pair of the tile; gs / us: [pair][32] rows of
// the block in LDS, already offset to this wave's four
template <int T>
__device__ __forceinline__ void ggq_gu_rows(const uint8_t* gbase, const uint8_t* ubase, int r0, uint64_t rb, int ul, int jj,
                                            float mlive, const uint32_t* __restrict__ xplanes,
                                            const float2* __restrict__ xmeta, const int (&toks)[GGQ_PAIRS], int npairs,
                                            int U, bool writer, float* gs, float* us) {
  constexpr int RB = ggq_batch<T>();
#pragma unroll
  for (int h = 0; h < 8; h += RB) {
    GgU<T> u[RB];
#pragma unroll
    for (int i = 0; i < RB; i++)
      ggu_fetch<T>(((i + h) < 4 ? gbase : ubase) + (uint64_t)(r0 + ((i + h) & 3)) * rb, ul, u[i]);
    __builtin_amdgcn_sched_barrier(0);  // every load of the batch is issued before the first dot product
#pragma unroll 1
    for (int pi = 0; pi < npairs; pi++) {
      XU x;
      load_xu(x, xplanes, xmeta, ((size_t)toks[pi] * U + ul) * 2);
#pragma unroll
      for (int i = 0; i < RB; i++) {
        const float v = sum64(ggu_dot<T>(u[i], jj, x) * mlive);
        if (writer) {
          if (i + h < 4) gs[pi * G4_ROWS + i + h] = v;
          else us[pi * G4_ROWS + i + h - 4] = v;
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the next batch's loads stay behind this batch's pairs
  }
}

// GGQ_DR output rows of one row of 16 lanes against every pair of the tile; out: pairs + first pair's row + r0
template <int T>
__device__ __forceinline__ void ggq_dn_rows(const uint8_t* base, uint64_t rb, int ul, int jj, float mlive,
                                            const uint32_t* __restrict__ hplanes, const float2* __restrict__ hmeta,
                                            size_t first, int npairs, int U, bool writer, float* out, int d);

// gate/up: grid (mid/32, tiles), block 512 (wave w: gate rows 4w..4w+3 and the matching up rows of the block's 32);
// hid planes go out by pair position, [pair][mid/32 groups]
__global__ void __launch_bounds__(512, 2) k_decgg_gu_uq(GuGgArgs A, const uint32_t* __restrict__ xplanes,
                                                        const float2* __restrict__ xmeta,
                                                        const moe_tile* __restrict__ tiles,
                                                        const int* __restrict__ ntiles, const int* __restrict__ tokidx,
                                                        int n_experts, int d, int mid, uint32_t* __restrict__ hplanes,
                                                        float2* __restrict__ hmeta) {
  __shared__ float gs[GGQ_PAIRS][G4_ROWS], us[GGQ_PAIRS][G4_ROWS];
  __shared__ uint32_t pk[GGQ_PAIRS][QV_GROUP_DW];
  if ((int)blockIdx.y >= ntiles[0]) return;
  const moe_tile tile = tiles[blockIdx.y];
  const bool shared = tile.expert >= n_experts;
  const int npairs = tile.count < GGQ_PAIRS ? tile.count : GGQ_PAIRS;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int U = d / 64;
  const int t = shared ? A.tsh : A.tgu;
  const uint64_t rb = ggu_row_bytes(t, (uint64_t)d);
  const uint8_t* gbase = shared ? A.sh_gate : A.gate + (uint64_t)tile.expert * mid * rb;
  const uint8_t* ubase = shared ? A.sh_up : A.up + (uint64_t)tile.expert * mid * rb;
  const int r0 = blockIdx.x * G4_ROWS + 4 * wv;
  const bool live = lane < U;
  const int ul = live ? lane : (lane & 3);
  const float mlive = live ? 1.f : 0.f;
  const int jj = ul & 3;
  int toks[GGQ_PAIRS];
#pragma unroll
  for (int pi = 0; pi < GGQ_PAIRS; pi++) toks[pi] = tokidx[tile.first + (pi < npairs ? pi : 0)];
  GGU_SWITCH(t, ggq_gu_rows<T>(gbase, ubase, r0, rb, ul, jj, mlive, xplanes, xmeta, toks, npairs, U, lane == 0,
                               &gs[0][4 * wv], &us[0][4 * wv]));
  __syncthreads();
  if (wv < npairs) {  // wave pi: SwiGLU on pair pi's 32 rows = one activation group of the down projection; quantise it
    const int j = lane & 31;
    const float g = gs[wv][j], u = us[wv][j];
    const float hv = g / (1.f + expf(-g)) * u;
    float m = dpp_max_row(fabsf(hv));
    m = rows_half_max(m);
    const float inv = m > 0.f ? QV_XMAX / m : 0.f;
    const float q = m * (1.f / QV_XMAX);
    const int X = (int)rintf(hv * inv);
    int p0, p1;
    qv_digits(X, p0, p1);
    float sx = dpp_add_row((float)X);
    sx = rows_half_add(sx);
    if (lane < QV_GROUP_DW) pk[wv][lane] = 0;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    if (lane < 32) {
      const int dw = j >> 2, sh = 8 * (j & 3);
      atomicOr(&pk[wv][dw], (uint32_t)(p0 & 0xff) << sh);
      atomicOr(&pk[wv][8 + dw], (uint32_t)(p1 & 0xff) << sh);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    const size_t gi = (size_t)(tile.first + wv) * (mid / 32) + blockIdx.x;
    if (lane < QV_GROUP_DW) hplanes[gi * QV_GROUP_DW + lane] = pk[wv][lane];
    if (lane == 0) hmeta[gi] = make_float2(q, q * sx);
  }
}

// down: grid (d/GGQ_DROWS, tiles), block 256 = 16 rows of 16 lanes, each with GGQ_DR output rows; the unweighted row
// results go to pairs[pair][row] (f32) for the weighted combine that follows
template <int T>
__device__ __forceinline__ void ggq_dn_rows(const uint8_t* base, uint64_t rb, int ul, int jj, float mlive,
                                            const uint32_t* __restrict__ hplanes, const float2* __restrict__ hmeta,
                                            size_t first, int npairs, int U, bool writer, float* out, int d) {
  constexpr int RB = ggq_dn_batch<T>();
#pragma unroll
  for (int h = 0; h < GGQ_DR; h += RB) {
    GgU<T> u[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) ggu_fetch<T>(base + (uint64_t)(h + r) * rb, ul, u[r]);
    __builtin_amdgcn_sched_barrier(0);
    for (int pi = 0; pi < npairs; pi++) {
      XU x;
      load_xu(x, hplanes, hmeta, ((first + pi) * U + ul) * 2);
#pragma unroll
      for (int r = 0; r < RB; r++) {
        const float v = dpp_add_row(ggu_dot<T>(u[r], jj, x) * mlive);
        if (writer) out[(size_t)pi * d + h + r] = v;
      }
    }
  }
}

__global__ void __launch_bounds__(256) k_decgg_dn_uq(DnGgArgs A, const uint32_t* __restrict__ hplanes,
                                                     const float2* __restrict__ hmeta,
                                                     const moe_tile* __restrict__ tiles, const int* __restrict__ ntiles,
                                                     int n_experts, int d, int mid, float* __restrict__ pairs) {
  if ((int)blockIdx.y >= ntiles[0]) return;
  const moe_tile tile = tiles[blockIdx.y];
  const bool shared = tile.expert >= n_experts;
  const int npairs = tile.count < GGQ_PAIRS ? tile.count : GGQ_PAIRS;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int U = mid / 64, u_raw = lane & 15;
  const bool live = u_raw < U;
  const int ul = live ? u_raw : (u_raw & 3);
  const float mlive = live ? 1.f : 0.f;
  const int jj = ul & 3;
  const int t = shared ? A.tsh : A.tdn;
  const uint64_t rb = ggu_row_bytes(t, (uint64_t)mid);
  const int r0 = blockIdx.x * GGQ_DROWS + (4 * wv + (lane >> 4)) * GGQ_DR;
  const uint8_t* base = (shared ? A.sh_down : A.down + (uint64_t)tile.expert * d * rb) + (uint64_t)r0 * rb;
  GGU_SWITCH(t, ggq_dn_rows<T>(base, rb, ul, jj, mlive, hplanes, hmeta, (size_t)tile.first, npairs, U, u_raw == 0,
                               pairs + (size_t)tile.first * d + r0, d));
}

}  // namespace

bool moe_dec4k_supported(int d, int mid, int nslots) {
  return d % 256 == 0 && d / 64 <= 64 && mid % 256 == 0 && mid / 64 <= 16 && nslots <= D4_MAXSLOTS &&
         mid % G4_ROWS == 0 && d % D4_ROWS == 0;
}

int moe_launch_dec4k_gu(const uint8_t* gate, const uint8_t* up, const uint8_t* sh_gate, const uint8_t* sh_up,
                        const uint32_t* xplanes, const float2* xmeta, const int* ids, int id_stride, int kpt,
                        int P, int d, int mid, uint32_t* hplanes, float2* hmeta, hipStream_t st) {
  if (!gate || !up || !xplanes || !xmeta || !ids || !hplanes || !hmeta) return MOE_E_INVALID;
  if (!moe_aligned(gate, 16) || !moe_aligned(up, 16) || (sh_gate && (!sh_up || !moe_aligned(sh_gate, 16) || !moe_aligned(sh_up, 16))))
    return MOE_E_INVALID;
  Gu4kArgs A{gate, up, sh_gate, sh_up};
  dim3 grid(mid / G4_ROWS, kpt + (sh_gate ? 1 : 0), P);
  k_dec4k_gu<0><<<grid, 512, 0, st>>>(A, xplanes, xmeta, ids, id_stride, kpt, d, mid, hplanes, hmeta, nullptr, 0,
                                      nullptr, nullptr, moe_rfix{});
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// The same with the softmax / top-k of every token done inside the launch: logits [P][n_experts] in,
// ids / ws rows (id_stride wide) out.
int moe_launch_dec4k_gu_topk(const uint8_t* gate, const uint8_t* up, const uint8_t* sh_gate, const uint8_t* sh_up,
                             const uint32_t* xplanes, const float2* xmeta, const float* logits, int n_experts,
                             int* ids, float* ws, int id_stride, int kpt, int P, int d, int mid,
                             uint32_t* hplanes, float2* hmeta, hipStream_t st, const moe_rfix* rf) {
  const moe_rfix RFV = rf ? *rf : moe_rfix{};
  if (RFV.W && !RFV.tol) return MOE_E_INVALID;
  if (!gate || !up || !xplanes || !xmeta || !logits || !ids || !ws || !hplanes || !hmeta || (!sh_gate != !sh_up))
    return MOE_E_INVALID;
  if (!moe_aligned(gate, 16) || !moe_aligned(up, 16) || (sh_gate && (!moe_aligned(sh_gate, 16) || !moe_aligned(sh_up, 16))))
    return MOE_E_INVALID;
  Gu4kArgs A{gate, up, sh_gate, sh_up};
  dim3 grid(mid / G4_ROWS, kpt + (sh_gate ? 1 : 0) + 1, P);  // + the row of the exact top-k block
  if (n_experts <= 512)
    k_dec4k_gu<8><<<grid, 512, 0, st>>>(A, xplanes, xmeta, nullptr, id_stride, kpt, d, mid, hplanes, hmeta, logits,
                                        n_experts, ids, ws, RFV);
  else
    k_dec4k_gu<16><<<grid, 512, 0, st>>>(A, xplanes, xmeta, nullptr, id_stride, kpt, d, mid, hplanes, hmeta, logits,
                                         n_experts, ids, ws, RFV);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_dec4k_dn(const uint8_t* down, const uint8_t* sh_down, const float* sh_logit,
                        const uint32_t* hplanes, const float2* hmeta, const int* ids, const float* ws,
                        int id_stride, int kpt, int P, int d, int mid, float* out, uint64_t out_stride,
                        hipStream_t st) {
  if (!down || !hplanes || !hmeta || !ids || !ws || !out || (sh_down && !sh_logit)) return MOE_E_INVALID;
  if (!moe_aligned(down, 16) || (sh_down && !moe_aligned(sh_down, 16))) return MOE_E_INVALID;
  Dn4kArgs A{down, sh_down, sh_logit};
  const int nslots = kpt + (sh_down ? 1 : 0);
  dim3 grid(d / D4_ROWS, P);
  k_dec4k_dn<<<grid, 64 * ((nslots + 3) / 4), 0, st>>>(A, hplanes, hmeta, ids, ws, id_stride, kpt, d, mid, out, out_stride);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// ---- any mix of Q4_K / Q5_K / Q8_0 / Q5_1 / IQ4_NL / IQ4_XS (integer-dot kernels above) ----
static bool ggu_type(int t) {
  return t == MOE_GGML_Q4_K || t == MOE_GGML_Q5_K || t == MOE_GGML_Q8_0 || t == MOE_GGML_Q5_1 || t == MOE_GGML_IQ4_NL ||
         t == MOE_GGML_IQ4_XS;
}
bool moe_decgg_supported(int tgu, int tdn, int tsh, bool has_shared, int d, int mid, int kpt, int n_experts) {
  if (!ggu_type(tgu) || !ggu_type(tdn) || (has_shared && !ggu_type(tsh))) return false;
  // (whole 256-element super-blocks in both directions also cover the 64-weight units of the 32-element types)
  return d % 256 == 0 && d / 64 <= 64 && mid % 256 == 0 && mid / 64 <= 16 && kpt + 1 <= D4_MAXSLOTS &&
         mid % G4_ROWS == 0 && d % D4_ROWS == 0 && ((kpt + 3) / 4 + 1) * 64 <= 320 && n_experts <= 1024 && kpt <= 64 &&
         kpt <= n_experts;
}
// Passes of the gate/up launch that deals its rows over all lanes, 0: rows that it does not take -- of 57 units and more, which leave
// hardly a lane idle, of fewer than 32, whose spare lanes would reach into the gate rows, and those that are no whole eights of units,
// whose sums would cross rows.
int moe_decgg_passes(int d) {
  return d % 512 == 0 && d >= 2048 && d <= 3584 ? d / 512 : 0;
}
// Down rows that are no whole super-blocks (2560 x 640): x and hid stay in f32, as on the general kernels (gguf_types.hip), where such layers
// ran before and where tensors that are not aligned for these still do.  (As 24 bits of the group's largest, three digit planes, an
// element 2^16 below it kept 8; that took 10 .. 15 % less time.)  Error against fp64 in the 2-norm at 1, 5 and 20 tokens, on the general kernels and here,
// 1e-7: Q5_K / Q8_0 3.4 8.2 5.7, 2.4 2.0 2.2; Q4_K / Q8_0 4.3 4.6 6.6, 2.5 2.3 2.1; Q8_0 3.9 4.8 4.9, 2.1 2.2 2.3; Q5_1 / Q8_0 6.5 4.7 5.2, 2.4 2.4
// 2.4; IQ4_NL / Q8_0 5.0 5.1 4.9, 2.1 2.2 2.2; IQ4_XS / Q8_0 5.2 6.0 4.9, 2.2 2.3 2.3; Q5_K / Q5_1 3.7 3.4 3.6, 3.2 3.2 3.3.  2560 x 640 Q5_K / Q8_0, us, general
// kernels and here (weights from HBM, other inputs each call): four layers 1 token 221 102, 2 338 143, 4 542 240, 8 990 373; two 20 1126 401, 32 1751 594.
bool moe_decgg_f32_supported(int tgu, int tdn, int tsh, bool has_shared, int d, int mid, int kpt, int n_experts) {
  auto down = [](int t) { return t == MOE_GGML_Q8_0 || t == MOE_GGML_Q5_1; };
  return ggu_type(tgu) && down(tdn) && (!has_shared || down(tsh)) && moe_decgg_passes(d) && mid % 128 == 0 && mid % 256 && mid <= 896 &&
         kpt + 1 <= D4_MAXSLOTS && n_experts <= 1024 && kpt <= n_experts;
}
static size_t ggu_align(int t) { return t == MOE_GGML_Q8_0 || t == MOE_GGML_IQ4_NL ? 4 : 16; }
// Tensors that these launches can read.  The general f32 kernels ask for less (Q8_0 and IQ4_NL 2 bytes, Q5_1 and IQ4_XS 8).
bool moe_decgg_aligned(int tgu, int tdn, int tsh, const uint8_t* gate, const uint8_t* up, const uint8_t* down, const uint8_t* sh_gate,
                       const uint8_t* sh_up, const uint8_t* sh_down) {
  const size_t gu = ggu_align(tgu), sh = ggu_align(tsh);
  return moe_aligned(gate, gu) && moe_aligned(up, gu) && moe_aligned(down, ggu_align(tdn)) &&
         (!sh_gate || (moe_aligned(sh_gate, sh) && moe_aligned(sh_up, sh) && moe_aligned(sh_down, sh)));
}

static bool decgg_gu_ok(bool f32, int tgu, int tsh, bool sh, int d, int mid, int kpt, int n_experts) {
  return f32 ? moe_decgg_f32_supported(tgu, MOE_GGML_Q8_0, tsh, sh, d, mid, kpt, n_experts)
             : moe_decgg_supported(tgu, tgu, tsh, sh, d, mid, kpt, n_experts);
}

int moe_launch_decgg_gu_topk(int tgu, int tsh, const uint8_t* gate, const uint8_t* up, const uint8_t* sh_gate,
                             const uint8_t* sh_up, const uint32_t* xplanes, const float2* xmeta, const float* logits,
                             int n_experts, int* ids, float* ws, int id_stride, int kpt, int P, int d, int mid,
                             uint32_t* hplanes, float2* hmeta, hipStream_t st, const moe_rfix* rf, const moe_dec_f32& f) {
  const moe_rfix RFV = rf ? *rf : moe_rfix{};
  if (RFV.W && !RFV.tol) return MOE_E_INVALID;
  const bool f32 = f.x != nullptr;
  if (!gate || !up || !logits || !ids || !ws || (!sh_gate != !sh_up) || (f32 ? !f.hid || !moe_aligned(f.x, 16) : !xplanes || !xmeta || !hplanes || !hmeta))
    return MOE_E_INVALID;
  if (!decgg_gu_ok(f32, tgu, tsh, sh_gate != nullptr, d, mid, kpt, n_experts)) return MOE_E_UNSUPPORTED;
  if (!moe_aligned(gate, ggu_align(tgu)) || !moe_aligned(up, ggu_align(tgu)) ||
      (sh_gate && (!moe_aligned(sh_gate, ggu_align(tsh)) || !moe_aligned(sh_up, ggu_align(tsh)))))
    return MOE_E_INVALID;
  GuGgArgs A{gate, up, sh_gate, sh_up, tgu, tsh};
  dim3 grid(mid / G4_ROWS, kpt + (sh_gate ? 1 : 0) + 1, P);
#define DECGG_GU(NPL, NP, F32) \
  k_decgg_gu<NPL, NP, F32><<<grid, 512, 0, st>>>(A, xplanes, xmeta, id_stride, kpt, d, mid, hplanes, hmeta, logits, n_experts, ids, ws, nullptr, RFV, f.x, f.hid)
#define DECGG_GU_NP(NPL, F32)                                \
  switch (moe_decgg_passes(d)) {                             \
    case 4: DECGG_GU(NPL, 4, F32); break;                    \
    case 5: DECGG_GU(NPL, 5, F32); break;                    \
    case 6: DECGG_GU(NPL, 6, F32); break;                    \
    case 7: DECGG_GU(NPL, 7, F32); break;                    \
    default: DECGG_GU(NPL, 0, false);                        \
  }
  if (f32 && n_experts <= 512) DECGG_GU_NP(8, true)
  else if (f32) DECGG_GU_NP(16, true)
  else if (n_experts <= 512) DECGG_GU_NP(8, false)
  else DECGG_GU_NP(16, false)
#undef DECGG_GU
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// the same with the ids already there (the router's launches made them)
int moe_launch_decgg_gu(int tgu, int tsh, const uint8_t* gate, const uint8_t* up, const uint8_t* sh_gate,
                        const uint8_t* sh_up, const uint32_t* xplanes, const float2* xmeta, const int* ids, int n_experts,
                        int id_stride, int kpt, int P, int d, int mid, uint32_t* hplanes, float2* hmeta, hipStream_t st,
                        const moe_dec_f32& f) {
  const bool f32 = f.x != nullptr;
  if (!gate || !up || !ids || (!sh_gate != !sh_up) || (f32 ? !f.hid || !moe_aligned(f.x, 16) : !xplanes || !xmeta || !hplanes || !hmeta))
    return MOE_E_INVALID;
  if (!decgg_gu_ok(f32, tgu, tsh, sh_gate != nullptr, d, mid, kpt, n_experts)) return MOE_E_UNSUPPORTED;
  if (!moe_aligned(gate, ggu_align(tgu)) || !moe_aligned(up, ggu_align(tgu)) ||
      (sh_gate && (!moe_aligned(sh_gate, ggu_align(tsh)) || !moe_aligned(sh_up, ggu_align(tsh)))))
    return MOE_E_INVALID;
  GuGgArgs A{gate, up, sh_gate, sh_up, tgu, tsh};
  dim3 grid(mid / G4_ROWS, kpt + (sh_gate ? 1 : 0), P);
#define DECGG_GU(NPL, NP, F32)                                                                                                                \
  k_decgg_gu<NPL, NP, F32><<<grid, 512, 0, st>>>(A, xplanes, xmeta, id_stride, kpt, d, mid, hplanes, hmeta, nullptr, n_experts, nullptr, nullptr, ids, \
                                                 moe_rfix{}, f.x, f.hid)
  if (f32) DECGG_GU_NP(0, true)
  else DECGG_GU_NP(0, false)
#undef DECGG_GU
#undef DECGG_GU_NP
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_decgg_dn(int tdn, int tsh, const uint8_t* down, const uint8_t* sh_down, const float* sh_logit,
                        const uint32_t* hplanes, const float2* hmeta, const int* ids, const float* ws, int id_stride,
                        int kpt, int P, int d, int mid, float* out, uint64_t out_stride, hipStream_t st, const float* hid32) {
  if (!down || (hid32 ? !moe_aligned(hid32, 16) : !hplanes || !hmeta) || !ids || !ws || !out || (sh_down && !sh_logit)) return MOE_E_INVALID;
  if (!moe_aligned(down, ggu_align(tdn)) || (sh_down && !moe_aligned(sh_down, ggu_align(tsh)))) return MOE_E_INVALID;
  DnGgArgs A{down, sh_down, sh_logit, tdn, tsh};
  dim3 grid(d / D4_ROWS, P);
#define DECGG_DN(U) \
  k_decgg_dn<U><<<grid, 64 * ((kpt + 64 / U - 1) / (64 / U) + (sh_down ? 1 : 0)), 0, st>>>(A, hplanes, hmeta, ids, ws, id_stride, kpt, d, out, out_stride, hid32)
  if (mid % 64 || (mid % 256 != 0) != (hid32 != nullptr)) return MOE_E_UNSUPPORTED;
  switch (mid / 64) {  // (moe_decgg_supported, moe_decgg_f32_supported)
    case 4: DECGG_DN(4); break;
    case 8: DECGG_DN(8); break;
    case 12: DECGG_DN(12); break;
    case 16: DECGG_DN(16); break;
    case 2: DECGG_DN(2); break;
    case 6: DECGG_DN(6); break;
    case 10: DECGG_DN(10); break;
    case 14: DECGG_DN(14); break;
    default: return MOE_E_UNSUPPORTED;
  }
#undef DECGG_DN
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// Distinct-expert variants: tiles (at most 4 pairs each; the shared expert as expert id n_experts) / ntiles / tokidx
// from the routing permutation; hplanes / hmeta and pairs are indexed by pair position.
bool moe_decgg_uq_supported(int d) { return d % GGQ_DROWS == 0; }
int moe_decgg_uq_tile_cap() { return GGQ_PAIRS; }

int moe_launch_decgg_gu_uq(int tgu, int tsh, const uint8_t* gate, const uint8_t* up, const uint8_t* sh_gate,
                           const uint8_t* sh_up, const uint32_t* xplanes, const float2* xmeta, const moe_tile* tiles,
                           const int* ntiles, int max_tiles, const int* tokidx, int n_experts, int d, int mid,
                           uint32_t* hplanes, float2* hmeta, hipStream_t st) {
  if (!gate || !up || !xplanes || !xmeta || !tiles || !ntiles || !tokidx || !hplanes || !hmeta || (!sh_gate != !sh_up))
    return MOE_E_INVALID;
  if (!moe_decgg_supported(tgu, tgu, tsh, sh_gate != nullptr, d, mid, 1, n_experts < 1024 ? n_experts : 1024))
    return MOE_E_UNSUPPORTED;
  if (!moe_aligned(gate, ggu_align(tgu)) || !moe_aligned(up, ggu_align(tgu)) ||
      (sh_gate && (!moe_aligned(sh_gate, ggu_align(tsh)) || !moe_aligned(sh_up, ggu_align(tsh)))))
    return MOE_E_INVALID;
  if (max_tiles <= 0) return MOE_OK;
  GuGgArgs A{gate, up, sh_gate, sh_up, tgu, tsh};
  k_decgg_gu_uq<<<dim3(mid / G4_ROWS, max_tiles), 512, 0, st>>>(A, xplanes, xmeta, tiles, ntiles, tokidx, n_experts, d, mid,
                                                                hplanes, hmeta);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_decgg_dn_uq(int tdn, int tsh, const uint8_t* down, const uint8_t* sh_down, const uint32_t* hplanes,
                           const float2* hmeta, const moe_tile* tiles, const int* ntiles, int max_tiles, int n_experts,
                           int d, int mid, float* pairs, hipStream_t st) {
  if (!down || !hplanes || !hmeta || !tiles || !ntiles || !pairs) return MOE_E_INVALID;
  if (!moe_decgg_uq_supported(d) || mid % 256 || mid / 64 > 16) return MOE_E_UNSUPPORTED;
  if (!moe_aligned(down, ggu_align(tdn)) || (sh_down && !moe_aligned(sh_down, ggu_align(tsh))) || !moe_aligned(pairs, 16))
    return MOE_E_INVALID;
  if (max_tiles <= 0) return MOE_OK;
  DnGgArgs A{down, sh_down, nullptr, tdn, tsh};
  k_decgg_dn_uq<<<dim3(d / GGQ_DROWS, max_tiles), 256, 0, st>>>(A, hplanes, hmeta, tiles, ntiles, n_experts, d, mid, pairs);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}
