// Decode (T <= 32): bandwidth-bound expert GEMV on q4cp weights read in place, integer dot products.
// The activation vector is turned once per token into four planes of balanced base-16 digits per
// 32-element group (x ~= q_g * (4096 p3 + 256 p2 + 16 p1 + p0), 15.9 significant bits relative to the
// group maximum), stored in the nibble order of a q4cp code word.  A 16-byte load of 32 codes then
// costs 4 XORs (unsigned code n -> n - 8 in two's complement) and 16 v_dot8_i32_i4 instead of ~100
// float operations: the VALU keeps up with HBM.  Weights stay exact (codes are integers; the group
// scale, the codebook slope / offset and q_g are applied in f32 after the integer sum, the offset
// through the group sum of the activations).
// (reference: src/gpu/parts/20_kernels_gemv.inc:1608-1835 — same contract: per-slot gate/up with
//  SwiGLU, then the down projection with the top-k weighted combine in slot order, no atomics)
#include "common.h"
#include "internal.h"
#include "qvec.h"
#include "topk.h"

namespace {

__device__ __forceinline__ float dpp_max_row(float v) {  // max over each row of 16 lanes
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true)));
  return v;
}
// sum over each half-wave of 32 lanes; every lane of the half gets the result
__device__ __forceinline__ float sum32(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));   // xor 1
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));   // xor 2
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));  // mirror in 8
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true));  // mirror in 16
  return rows_half_add(v);
}
__device__ __forceinline__ float sum64(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true));
  return rows_total_add(v);
}

// Quantise 32 floats held one per lane by lanes [0,32) of a half-wave (j = lane & 31) into the qvec4
// form: returns this lane's four digits, q and q*sum(X).
__device__ __forceinline__ void quant32_lane(float x, int& p0, int& p1, int& p2, int& p3, float& q, float& qsx) {
  float m = dpp_max_row(fabsf(x));
  m = rows_half_max(m);
  const float inv = m > 0.f ? QV4_XMAX / m : 0.f;
  q = m * (1.f / QV4_XMAX);
  const int X = (int)rintf(x * inv);
  qv4_digits(X, p0, p1, p2, p3);
  qsx = q * sum32((float)X);
}

// One thread per group: x (f32, K elements) -> qvec4.  Blocks of 64.
__global__ void __launch_bounds__(64) k_qvec_from_f32(const float* __restrict__ x, uint64_t x_stride,
                                                      int G, uint32_t* __restrict__ planes,
                                                      float2* __restrict__ meta) {
  const int t = blockIdx.y, g = blockIdx.x * 64 + threadIdx.x;
  if (g < G) qvec4_group_from_f32(x, x_stride, G, t, g, planes, meta);
}

struct XG {  // one group's activation planes in registers
  uint32_t p[4][4];
  float q, qsx;
};
__device__ __forceinline__ void load_xg(XG& x, const uint32_t* planes, const float2* meta, size_t gi) {
  const uint4* s = (const uint4*)(planes + gi * QV4_GROUP_DW);
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const uint4 a = s[p];
    x.p[p][0] = a.x; x.p[p][1] = a.y; x.p[p][2] = a.z; x.p[p][3] = a.w;
  }
  const float2 m = meta[gi];
  x.q = m.x;
  x.qsx = m.y;
}

// sum_k cb[n_k] * x_k over one group, cb = a*n + b = a*(n-8) + (8a+b):
//   a * q * (4096 D3 + 256 D2 + 16 D1 + D0) + (8a + b) * q * sum(X),  D_j = sum_k (n_k - 8) * p_j,k
__device__ __forceinline__ float chunk_dot(const uint4 cw, const XG& x, float cb_a, float cb_b8) {
  const uint32_t w[4] = {cw.x ^ 0x88888888u, cw.y ^ 0x88888888u, cw.z ^ 0x88888888u, cw.w ^ 0x88888888u};
  int d0 = 0, d1 = 0, d2 = 0, d3 = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    d0 = __builtin_amdgcn_sdot8((int)w[i], (int)x.p[0][i], d0, false);
    d1 = __builtin_amdgcn_sdot8((int)w[i], (int)x.p[1][i], d1, false);
    d2 = __builtin_amdgcn_sdot8((int)w[i], (int)x.p[2][i], d2, false);
    d3 = __builtin_amdgcn_sdot8((int)w[i], (int)x.p[3][i], d3, false);
  }
  const int D = ((d3 * 16 + d2) * 16 + d1) * 16 + d0;  // |D| < 2^24: exact as f32
  return fmaf(cb_a * x.q, (float)D, cb_b8 * x.qsx);
}

struct DecW {  // one q4cp tensor's planes
  const uint8_t *codes, *scales;
  const float* cb;
  uint64_t ss;
  int gsh;  // 32-element groups per scale = 1 << gsh (q4cp: 0; hgn v2 i4r, one scale per 128 columns: 2)
};

// ---- codebooks that are not a*n + b (the reference converter's fixed non-uniform table, trained tables): the same
// kernels with a look-up instead of the integer dots, all in f32 (no quantised activations: the result differs
// from the f32 GEMV kernels only by the order of the additions).  What bounds them up to about ten tokens is the vector
// instructions of the look-ups, so these are few: the 16 entries lie in LDS 64 times side by side (entry n at byte
// 256 n, a copy per lane: no conflicts, whatever the codes are) at a multiple of the table's size, so that an address is
// bytes put together.  Two masks turn a code word's nibbles into bytes with the table's place in them, and a weight
// costs one byte permute, one LDS read and one FMA, 2.4 vector instructions with its share of the masks (a bit-field extract
// and an address operation per weight, 32 copies: 3).  One layer of 20 tokens, gate/up: 117 -> 104 us; a 256-entry table of
// pairs (64 KB) reads at 6 TB/s there, 95, but gains 1 us at 2 tokens and does not fit beside the selection at 1.
// A lane keeps the 32 activations of the group it is working on in registers.
constexpr int LUT_BYTES = 16 * 256;
typedef float floatx4 __attribute__((ext_vector_type(4)));
// LDS byte address: the first multiple of LUT_BYTES from p on
__device__ __forceinline__ uint32_t lut_at(const void* p) {
  return ((uint32_t)(uintptr_t)p + (LUT_BYTES - 1)) & ~(uint32_t)(LUT_BYTES - 1);
}

struct XF {  // one group's activations
  float v[32];
};
constexpr int XF_PITCH = 36;  // floats between two groups' activations in LDS (see the staging in k_dec_gu)
__device__ __forceinline__ void load_xf(XF& x, const float* src) {  // src: global or LDS, 16-byte aligned
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 f = ((const float4*)src)[i];
    x.v[4 * i] = f.x; x.v[4 * i + 1] = f.y; x.v[4 * i + 2] = f.z; x.v[4 * i + 3] = f.w;
  }
}
// piece i of a table (16 copies of an entry); 256 pieces
__device__ __forceinline__ void lut_put(uint32_t lut, int i, float v) {
  *(__attribute__((address_space(3))) floatx4*)(uintptr_t)(lut + 16u * (uint32_t)i) = floatx4{v, v, v, v};
}
// sum_k cb[n_k] * x_k over one group (16 code bytes, low nibble = the earlier element); lut4 = the table's address >> 8 in
// each byte, lane4 = 4 * lane
__device__ __forceinline__ float lut_dot(const uint4 cw, const XF& x, uint32_t lut4, uint32_t lane4) {
  const uint32_t w[4] = {cw.x, cw.y, cw.z, cw.w};
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    // (an opaque copy of the word, pinned between this step's neighbours: otherwise the compiler works out the
    // addresses of a whole launch's look-ups ahead of the first one and spills hundreds of registers)
    uint32_t wi = w[i];
    asm volatile("" : "+v"(wi));
    const uint32_t lo = (wi & 0x0f0f0f0fu) | lut4, hi = ((wi >> 4) & 0x0f0f0f0fu) | lut4;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t sel = 0x0c0c0000u | (uint32_t)(4 + j) << 8;
      const uint32_t a_lo = __builtin_amdgcn_perm(lo, lane4, sel), a_hi = __builtin_amdgcn_perm(hi, lane4, sel);
      const float t0 = *(const __attribute__((address_space(3))) float*)(uintptr_t)a_lo;
      const float t1 = *(const __attribute__((address_space(3))) float*)(uintptr_t)a_hi;
      a0 = fmaf(t0, x.v[8 * i + 2 * j], a0);
      a1 = fmaf(t1, x.v[8 * i + 2 * j + 1], a1);
    }
    if (i & 1) __builtin_amdgcn_sched_barrier(0);  // sixteen look-ups in flight at a time, not a whole row's
  }
  return a0 + a1;
}

// The same kernels once more for codebooks a*n + b in plain f32 arithmetic (the integer-dot kernels switched off):
// sum_k n_k * x_k over one group -- two masks per code word turn its even and odd nibbles into bytes, then a
// byte-to-float conversion and an FMA per weight; the caller adds b * sum(x).
__device__ __forceinline__ float aff_dot(const uint4 cw, const XF& x) {
  const uint32_t w[4] = {cw.x, cw.y, cw.z, cw.w};
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t lo = w[i] & 0x0f0f0f0fu, hi = (w[i] >> 4) & 0x0f0f0f0fu;
    a0 = fmaf((float)(lo & 0xff), x.v[8 * i], a0);
    a1 = fmaf((float)(hi & 0xff), x.v[8 * i + 1], a1);
    a0 = fmaf((float)((lo >> 8) & 0xff), x.v[8 * i + 2], a0);
    a1 = fmaf((float)((hi >> 8) & 0xff), x.v[8 * i + 3], a1);
    a0 = fmaf((float)((lo >> 16) & 0xff), x.v[8 * i + 4], a0);
    a1 = fmaf((float)((hi >> 16) & 0xff), x.v[8 * i + 5], a1);
    a0 = fmaf((float)(lo >> 24), x.v[8 * i + 6], a0);
    a1 = fmaf((float)(hi >> 24), x.v[8 * i + 7], a1);
  }
  return a0 + a1;
}
__device__ __forceinline__ float xf_sum(const XF& x) {
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int i = 0; i < 32; i += 2) {
    s0 += x.v[i];
    s1 += x.v[i + 1];
  }
  return s0 + s1;
}
// MODE 1: the look-up (any codebook); MODE 2: cb[n] = a n + b0 in f32, sx = the sum of the group's activations
template <int MODE>
__device__ __forceinline__ float f32_dot(const uint4 cw, const XF& x, uint32_t lut4, float a, float b0, float sx) {
  if (MODE == 2) return fmaf(a, aff_dot(cw, x), b0 * sx);
  return lut_dot(cw, x, lut4, 4u * (threadIdx.x & 63));
}

struct GuArgs2 {
  DecW gu;           // fused gate_up [E*2*mid][d]
  DecW shg, shu;     // shared expert gate / up [mid][d] (codes == nullptr: none)
  // hgn v2 rotated experts (not with UQ / LUT): the routed slots read the rotated activations' planes and write
  // their gate | up sums as they are, zraw[token][slot][2 mid] (the rotation back comes before SwiGLU); the shared
  // expert's slot is untouched by this
  float* zraw;
  const uint32_t* xplanes_rot;
  const float2* xmeta_rot;
};

// grid (mid/32, slots incl. shared, P); block 512.  Wave w: gate rows 4w..4w+3 and the matching up
// rows of this block's 32; lane L holds activation groups L and 64 + (L & 31).  Rows are taken two
// at a time with three 16-byte loads per lane: (row0, group L), (row1, group L), and the tail group
// of row0 (lanes < 32) or row1 (lanes >= 32); all twelve loads of a wave are in flight together.
// UQ ("unique experts", verify batches): grid (mid/32, tiles) instead; a tile = one expert with the
// (token, expert) pairs routed to it (expert-sorted lists of the routing permutation; the shared
// expert is the tile with expert id >= n_experts over all tokens).  The block reads its weight rows
// once and walks the tile's pairs; hid planes are then indexed by pair position.
// NPL > 0 (E <= 64*NPL, not with UQ): the router launch only left the logits; every block of a
// routed slot runs the softmax / top-k of its token itself (the same code and therefore the same
// ids and weights in every block; cheaper than a last-block ticket in the router launch plus a
// dependent load of the ids here) and block (0, 0, token) writes ids / weights out for the down
// kernel.  The shared expert's blocks skip it and have the CU to themselves meanwhile.
// LUT = 1 (not with UQ): table look-up arithmetic (above) for any codebook; blocks of 16 or 12 rows; xf32 = the
// tokens' activations [P][d], dynamic LDS = the token's d activations and two tables (gate rows', up rows'), hid goes out as
// f32 only.
// LUT = 2: the same data flow with f32 arithmetic for codebooks a*n + b (no tables).
constexpr int GU2_ROWS = 32;
// (LUT = 1: four waves, 16 rows.  A block is tens of thousands of vector instructions there, and one token's 264 blocks of
// eight waves leave the CUs that get a second one with twice the work: four layers 129 -> 119 us.  With the selection inside, three
// waves and 12 rows.  It is the selection that gains -- probably because a CU's waves go round its SIMDs: of blocks of four waves
// the first ones, which select, would all share a SIMD.  us, out of the last-level cache (from HBM, 3072 x 768, 1 token 117.7 108.1), 16 and 12 rows: 1 token (four layers) 3072 x 768 111.7 104.1, x 512 99.7 85.2, x 1024 127.5 113.5,
// 2560 x 640 108.0 102.9; 2 tokens (two layers) 86.5 76.3 -- with the selection aside, where 16 rows are level or better (4 tokens
// 117.9 120.3, 8 90.5 92.0), 79.7.  The last block's rows past mid are the last rows again and not stored.)
constexpr int gu2_threads(int lut, int npl) { return lut == 1 ? (npl ? 192 : 256) : 512; }
// TL: passes over the groups behind the first 64 of a row, of which a pass takes those of two rows (4 passes: up to 32 groups) or of four
// (2 passes: up to 16), 0 where there are none.  us, four passes throughout and these, weights from HBM: table codebook
// 2560 x 640 1 token 111 106, 3 91 87, 8 86 81, 20 169 158; 2048 x 768 8 90 78; q4cp 2048 x 768 1 81 74, 3 69 65, 8 59 56; q4cp 2560 x 640
// 8 60 59, 20 112 110, and 1 token level at 79: an int kernel with the selection inside keeps four there.
template <bool UQ, int NPL, int LUT, int TL = 4>
__global__ void __launch_bounds__(gu2_threads(LUT, NPL), gu2_threads(LUT, NPL) < 256 ? 3 : 4) k_dec_gu(GuArgs2 A, const uint32_t* __restrict__ xplanes,
                                                const float2* __restrict__ xmeta,
                                                const int* __restrict__ ids, int id_stride, int kpt, int d,
                                                int mid, uint32_t* __restrict__ hplanes,
                                                float2* __restrict__ hmeta, float* __restrict__ hid_f32,
                                                const moe_tile* __restrict__ tiles, const int* __restrict__ ntiles,
                                                const int* __restrict__ tokidx, int n_experts,
                                                const float* __restrict__ logits, int* __restrict__ ids_out,
                                                float* __restrict__ ws_out, const float* __restrict__ xf32, moe_rfix RF) {
  constexpr int NT = gu2_threads(LUT, NPL), ROWS = NT / 16;
  extern __shared__ float lutmem[];
  __shared__ float gs[ROWS], us[ROWS];
  __shared__ uint32_t pk[QV4_GROUP_DW];
  __shared__ int sel_ids[64];
  __shared__ float sel_ws[64];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // (a scalar: see e)
  const int G = d / 32;
  int s = blockIdx.y, nslots = gridDim.y - (NPL > 0 ? 1 : 0), e = 0, first = 0, npairs = 1;
  if (NPL > 0 && s == nslots) {
    // one block of the extra grid row: the exact softmax / top-k (ids, renormalised weights) for the down
    // launch, next to the blocks that stream the weights and only need the ids
    if (blockIdx.x == 0) {
      select_certain<NPL ? NPL : 8, NT>(logits + (size_t)blockIdx.z * n_experts, RF, (int)blockIdx.z, sel_ids, sel_ws, n_experts, kpt, true);
      __syncthreads();
      if ((int)threadIdx.x < kpt) {
        ids_out[(size_t)blockIdx.z * id_stride + threadIdx.x] = sel_ids[threadIdx.x];
        ws_out[(size_t)blockIdx.z * id_stride + threadIdx.x] = sel_ws[threadIdx.x];
      }
    }
    return;
  }
  // Look-up tables and the token's activations: requested here, next to the selection's loads, and put into LDS behind the
  // weights' requests
  const bool sh_blk = !UQ && s >= kpt;
  const float* const cbg = sh_blk ? A.shg.cb : A.gu.cb;
  const float* const cbu = sh_blk ? A.shu.cb : A.gu.cb;
  const bool two_tabs = LUT == 1 && cbu != cbg;  // (block-uniform) the shared expert's up_proj is a tensor with a codebook of its own
  constexpr int XL = (96 * 8 + NT - 1) / NT;  // (d <= 3072)
  static_assert(XL <= 4 && (LUT != 1 || (NT >= 128 && NT <= 256)), "a thread stages at most four pieces of x and two of a table");
  float4 x0, x1, x2, x3;
  float cg0 = 0.f, cu0 = 0.f, cg1 = 0.f, cu1 = 0.f;
  if (LUT) {
    const float4* xr = (const float4*)(xf32 + (size_t)blockIdx.z * d);
    auto ld = [&](int i) {
      const int c = (int)threadIdx.x + NT * i;
      return xr[c < d / 4 ? c : 0];
    };
    x0 = ld(0);
    x1 = ld(1);
    if (XL > 2) x2 = ld(2);
    if (XL > 3) x3 = ld(3);
    if (LUT == 1) {
      cg0 = cbg[threadIdx.x >> 4];
      cu0 = cbu[threadIdx.x >> 4];
      if (NT < 256) {
        cg1 = cbg[(threadIdx.x + NT) >> 4 & 15];
        cu1 = cbu[(threadIdx.x + NT) >> 4 & 15];
      }
    }
  }
  bool shared;
  if (UQ) {
    if ((int)blockIdx.y >= ntiles[0]) return;
    const moe_tile tile = tiles[blockIdx.y];
    shared = tile.expert >= n_experts;
    e = shared ? 0 : tile.expert;
    first = tile.first;
    npairs = tile.count;
  } else if (NPL > 0) {
    shared = s >= kpt;
    if (!shared) {
      // the ids by logit order (no exps, no sums); the exact selection only when two of the best logits
      // are too close for that to be certain
      const float* lg = logits + (size_t)blockIdx.z * n_experts;
      if (!select_certain<NPL ? NPL : 8, NT>(lg, RF, (int)blockIdx.z, sel_ids, sel_ws, n_experts, kpt, false)) __syncthreads();
      e = sel_ids[s];
    }
  } else {
    shared = s >= kpt;
    e = shared ? 0 : ids[(size_t)blockIdx.z * id_stride + s];
  }
  const DecW Wg = shared ? A.shg : A.gu;  // block-uniform choice, by value
  const DecW Wu = shared ? A.shu : A.gu;
  // the expert number is the same in every lane: as a scalar, the row and byte offsets that follow from it are scalar
  // arithmetic instead of 64-bit products per lane (quarter-rate instructions between the selection and the first load)
  e = __builtin_amdgcn_readfirstlane(e);
  const uint32_t lut_g = lut_at(lutmem + d / 32 * XF_PITCH), lut_u = lut_g + (two_tabs ? LUT_BYTES : 0);
  const uint32_t lutg = (lut_g >> 8) * 0x01010101u, lutu = (lut_u >> 8) * 0x01010101u;
  const float* xs = lutmem;
  const uint64_t grow0 = shared ? 0 : (uint64_t)e * 2 * mid;
  const uint64_t urow0 = shared ? 0 : (uint64_t)e * 2 * mid + mid;
  int r0 = blockIdx.x * ROWS + 4 * wv;  // first of this wave's 4 gate rows
  if (NT < 256) r0 = r0 < mid ? r0 : mid - 4;

  // Branch-free loads: a lane whose group lies past the row reads group 0 instead and gets a zero
  // scale.  (Loads inside divergent branches make the compiler wait for each of them where it is
  // issued; in straight-line code all of a wave's loads are in flight together.)
  constexpr int TLANES = TL == 2 ? 16 : 32, TROWS = TL == 2 ? 4 : 2;  // lanes of a row's tail, rows of a pass
  const int tsub = lane / TLANES;            // which of the pass's rows
  const bool vA = lane < G, vB = TL && 64 + (lane & (TLANES - 1)) < G;
  const int gA = vA ? lane : 0, gB = vB ? 64 + (lane & (TLANES - 1)) : 0;
  const float mA = vA ? 1.f : 0.f, mB = vB ? 1.f : 0.f;
  const size_t rb = (size_t)d / 2;
  // the activation planes and codebook constants are requested first: loads return in order, so
  // the dot products of the first row pair can start while the later rows are still in flight
  XG xa, xb;
  const bool raw = !UQ && !LUT && A.zraw && !shared;  // (block-uniform)
  if (!LUT && !UQ) {
    const size_t xbase = (size_t)blockIdx.z * G;
    const uint32_t* xp = raw ? A.xplanes_rot : xplanes;
    const float2* xm = raw ? A.xmeta_rot : xmeta;
    load_xg(xa, xp, xm, xbase + gA);
    if (TL) load_xg(xb, xp, xm, xbase + gB);
  }
  const float ga = Wg.cb[1] - Wg.cb[0], gb = fmaf(8.f, ga, Wg.cb[0]), ua = Wu.cb[1] - Wu.cb[0], ub = fmaf(8.f, ua, Wu.cb[0]);
  // pairs 0,1: gate rows (r0+2p, r0+2p+1); pairs 2,3: the up rows
  uint4 ca[4], cb[4], ct[TL ? TL : 1];
  __half sa[4], sb[4], st[TL ? TL : 1];
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const DecW W = p >= 2 ? Wu : Wg;
    const uint64_t row = (p >= 2 ? urow0 : grow0) + r0 + 2 * (p & 1);
    const uint8_t* c0 = W.codes + row * rb;
    const uint8_t* s0 = W.scales + row * W.ss;
    ca[p] = *(const uint4*)(c0 + (size_t)gA * 16);
    cb[p] = *(const uint4*)(c0 + rb + (size_t)gA * 16);
    sa[p] = *(const __half*)(s0 + (gA >> W.gsh) * 2);
    sb[p] = *(const __half*)(s0 + W.ss + (gA >> W.gsh) * 2);
    if (TL == 4 || (TL == 2 && (p & 1))) {  // (two rows' tails, or those of four: the pair before this one and this)
      const int t = TL == 4 ? p : p >> 1;
      const uint8_t *const ct0 = TL == 4 ? c0 : c0 - 2 * rb, *const st0 = TL == 4 ? s0 : s0 - 2 * W.ss;
      ct[t] = *(const uint4*)(ct0 + (uint64_t)tsub * rb + (size_t)gB * 16);
      st[t] = *(const __half*)(st0 + (uint64_t)tsub * W.ss + (gB >> W.gsh) * 2);
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load above is issued before the first dot product
  if (LUT) {
    // A group's 128 bytes lie at a pitch of 144: lanes read different groups 16 bytes at a time, and at a pitch of
    // 128 every lane of such a read would sit on the same four banks (measured: 6.4 times the LDS time of this pitch).
    auto put = [&](int i, const float4& v) {
      const int c = (int)threadIdx.x + NT * i;
      if (c < d / 4) ((float4*)lutmem)[(c >> 3) * (XF_PITCH / 4) + (c & 7)] = v;
    };
    put(0, x0);
    put(1, x1);
    if (XL > 2) put(2, x2);
    if (XL > 3) put(3, x3);
    if (LUT == 1) {
      lut_put(lut_g, threadIdx.x, cg0);
      if (two_tabs) lut_put(lut_u, threadIdx.x, cu0);
      if (NT < 256 && threadIdx.x + NT < 256) {
        lut_put(lut_g, threadIdx.x + NT, cg1);
        if (two_tabs) lut_put(lut_u, threadIdx.x + NT, cu1);
      }
    }
    moe_lds_barrier();  // (the weights stay in flight)
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int pi = 0; pi < npairs; pi++) {
  const int tok = UQ ? tokidx[first + pi] : (int)blockIdx.z;
  if (UQ) {
    const size_t xbase = (size_t)tok * G;
    load_xg(xa, xplanes, xmeta, xbase + gA);
    load_xg(xb, xplanes, xmeta, xbase + gB);
  }

  float acc[8];
  if (LUT) {
    // group gA of all eight rows first, then the tail group: one group's activations in registers at a time
    XF xf;
    load_xf(xf, xs + (size_t)gA * XF_PITCH);
    const float g0 = Wg.cb[0], u0 = Wu.cb[0];
    float sx = LUT == 2 ? xf_sum(xf) : 0.f;
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const uint32_t lt = p >= 2 ? lutu : lutg;
      const float a = p >= 2 ? ua : ga, b0 = p >= 2 ? u0 : g0;
      acc[2 * p] = __half2float(sa[p]) * mA * f32_dot<LUT>(ca[p], xf, lt, a, b0, sx);
      acc[2 * p + 1] = __half2float(sb[p]) * mA * f32_dot<LUT>(cb[p], xf, lt, a, b0, sx);
    }
    if (TL) load_xf(xf, xs + (size_t)gB * XF_PITCH);
    sx = LUT == 2 ? xf_sum(xf) : 0.f;
#pragma unroll
    for (int t = 0; t < TL; t++) {
      const bool up = 2 * t >= TL;
      const float vt = __half2float(st[t]) * mB * f32_dot<LUT>(ct[t], xf, up ? lutu : lutg, up ? ua : ga, up ? u0 : g0, sx);
#pragma unroll
      for (int i = 0; i < TROWS; i++)
        if (tsub == i) acc[TROWS * t + i] += vt;
    }
  } else {
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const float a = p >= 2 ? ua : ga, b = p >= 2 ? ub : gb;
    // (a multiplication, not a select: a select lets the compiler move the load back under a branch)
    const float fa = __half2float(sa[p]) * mA, fb = __half2float(sb[p]) * mA;
    acc[2 * p] = fa * chunk_dot(ca[p], xa, a, b);
    acc[2 * p + 1] = fb * chunk_dot(cb[p], xa, a, b);
    if (TL == 4 || (TL == 2 && (p & 1))) {
      const int t = TL == 4 ? p : p >> 1;
      const float vt = __half2float(st[t]) * mB * chunk_dot(ct[t], xb, a, b);
#pragma unroll
      for (int i = 0; i < TROWS; i++)
        if (tsub == i) acc[TROWS * t + i] += vt;
    }
    __builtin_amdgcn_sched_barrier(0);  // row pair p is finished before the wait for pair p + 1
  }
  }
#pragma unroll
  for (int i = 0; i < 8; i++) acc[i] = sum64(acc[i]);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      gs[4 * wv + i] = acc[i];
      us[4 * wv + i] = acc[4 + i];
    }
  }
  __syncthreads();
  if (raw) {
    if (threadIdx.x < 32) {
      float* zr = A.zraw + ((size_t)tok * kpt + s) * 2 * mid + blockIdx.x * ROWS + threadIdx.x;
      zr[0] = gs[threadIdx.x];
      zr[mid] = us[threadIdx.x];
    }
    return;
  }
  // SwiGLU on the block's 32 rows = one group of the down projection's input; quantise it
  if (wv == 0) {
    const int j = (lane & 31) < ROWS ? lane & 31 : 0;
    const float g = gs[j], u = us[j];
    const float hv = g / (1.f + expf(-g)) * u;
    const size_t slot = UQ ? (size_t)(first + pi) : (size_t)tok * nslots + s;
    if (hid_f32 && lane < ROWS && (NT >= 256 || (int)blockIdx.x * ROWS + j < mid)) hid_f32[slot * mid + blockIdx.x * ROWS + j] = hv;
    if (LUT) return;  // (the down kernel of this arithmetic reads hid as f32)
    int p0, p1, p2, p3;
    float q, qsx;
    quant32_lane(hv, p0, p1, p2, p3, q, qsx);
    if (lane < QV4_GROUP_DW) pk[lane] = 0;
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    if (lane < 32) {
      const int dw = j >> 3, sh = 4 * (j & 7);
      atomicOr(&pk[dw], (uint32_t)(p0 & 15) << sh);
      atomicOr(&pk[4 + dw], (uint32_t)(p1 & 15) << sh);
      atomicOr(&pk[8 + dw], (uint32_t)(p2 & 15) << sh);
      atomicOr(&pk[12 + dw], (uint32_t)(p3 & 15) << sh);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    const size_t gi = slot * (mid / 32) + blockIdx.x;
    if (lane < QV4_GROUP_DW) hplanes[gi * QV4_GROUP_DW + lane] = pk[lane];
    if (lane == 0) hmeta[gi] = make_float2(q, qsx);
  }
  if (UQ) __syncthreads();  // gs / us / pk are reused by the next pair
  }
}

struct DnArgs2 {
  DecW dn;   // routed down [E*d][mid]
  DecW shd;  // shared expert down [d][mid] (codes == nullptr: none)
  const float* sh_logit;
  float* out_sh;  // != nullptr: the shared expert's gated rows go here instead of into the sum (same strides as out)
};

// grid (d/ROWS, P); block = 64 x ceil(slots/2).  Wave = one slot pair, half-wave = one slot: lane
// (L & 31) holds that slot's activation group (K/32 <= 32 groups) in registers for all the block's
// rows.  The weighted combine runs afterwards in slot order (descending router probability), then
// the shared expert: deterministic, no atomics.
constexpr int DN2_MAXSLOTS = 16;
#ifndef MOE_DN_ROWS
#define MOE_DN_ROWS 6
#endif
// LUT = 1: table look-up arithmetic for any codebook; hid_f32 = [P][slots][mid], dynamic LDS = two tables (the routed
// experts' tensor, the shared expert's).  LUT = 2: f32 arithmetic for codebooks a*n + b, no tables.
template <int ROWS, int LUT>
__global__ void __launch_bounds__(512) k_dec_dn(DnArgs2 A, const uint32_t* __restrict__ hplanes,
                                                const float2* __restrict__ hmeta,
                                                const int* __restrict__ ids, const float* __restrict__ ws,
                                                int id_stride, int kpt, int d, int mid,
                                                float* __restrict__ out, uint64_t out_stride,
                                                const float* __restrict__ hid_f32) {
  extern __shared__ float lutmem[];
  __shared__ float part[DN2_MAXSLOTS][ROWS];
  __shared__ float wsm[DN2_MAXSLOTS];
  const int tok = blockIdx.y;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const bool has_shared = A.shd.codes != nullptr;
  const int nslots = kpt + (has_shared ? 1 : 0);
  const int G = mid / 32, half = lane >> 5;
  const int r0 = blockIdx.x * ROWS;
  const size_t rb = (size_t)mid / 2;
  // (the tables' entries are requested first and written behind the weights' requests)
  const float* const tcb = has_shared ? A.shd.cb : A.dn.cb;
  float c0 = 0.f, c1 = 0.f;
  if (LUT == 1) {
    c0 = A.dn.cb[threadIdx.x >> 4 & 15];
    c1 = tcb[threadIdx.x >> 4 & 15];
  }
  const uint32_t lut_r = lut_at(lutmem), lut_s = lut_r + LUT_BYTES;
  // combine weights of the token, fetched while the weight rows are in flight
  float wmine = 0.f;
  if ((int)threadIdx.x < nslots)
    wmine = (int)threadIdx.x < kpt ? ws[(size_t)tok * id_stride + threadIdx.x] : A.sh_logit[tok];
  {
    // Branch-free loads: lanes past the slots or past the row's groups read slot 0 / group 0 and
    // get a zero factor, so that all of a wave's loads are in flight together.
    const int s_raw = 2 * wv + half, g_raw = lane & 31;
    const bool live = s_raw < nslots && g_raw < G;
    const int s = live ? s_raw : 0, g = live ? g_raw : 0;
    const float m = live ? 1.f : 0.f;
    const bool shared = has_shared && s == nslots - 1;
    // per-lane choice of tensor: pick the members by value (a reference to one of two kernel
    // arguments would be re-read from memory in front of every load)
    const uint8_t* wcodes = shared ? A.shd.codes : A.dn.codes;
    const uint8_t* wscales = shared ? A.shd.scales : A.dn.scales;
    const float* wcb = shared ? A.shd.cb : A.dn.cb;
    const uint64_t wss = shared ? A.shd.ss : A.dn.ss;
    const int wgsh = shared ? A.shd.gsh : A.dn.gsh;
    // (an unconditional load -- the shared expert's lanes read slot 0's id and drop it: under a per-lane branch the
    // compiler waits for the id before it issues anything else.  Indices in 32 bits: a 64-bit product per lane is two
    // quarter-rate instructions.)
    const int e_any = ids[tok * id_stride + (shared ? 0 : s)];
    const uint32_t e = shared ? 0u : (uint32_t)e_any;
    XG x;
    XF xh;
    if (LUT) load_xf(xh, hid_f32 + ((size_t)tok * nslots + s) * mid + (size_t)g * 32);
    else load_xg(x, hplanes, hmeta, (size_t)((tok * nslots + s) * G + g));
    const uint32_t lt = ((shared ? lut_s : lut_r) >> 8) * 0x01010101u;
    const float a = wcb[1] - wcb[0], b = fmaf(8.f, a, wcb[0]);
    const uint32_t row0 = e * (uint32_t)d + (uint32_t)r0;  // < experts * d: the launcher checks that it fits
    const uint8_t* cp = wcodes + (uint64_t)row0 * (uint32_t)rb + (uint32_t)g * 16;
    const uint8_t* sp = wscales + (uint64_t)row0 * (uint32_t)wss + (uint32_t)(g >> wgsh) * 2;
    uint4 cw[ROWS];
    __half sc[ROWS];
    {
      // (row addresses by repeated addition: wss is a per-lane value, and r * wss as a 64-bit product costs two
      // quarter-rate instructions per row)
      const uint8_t *cpr = cp, *spr = sp;
#pragma unroll
      for (int r = 0; r < ROWS; r++) {
        cw[r] = *(const uint4*)cpr;
        sc[r] = *(const __half*)spr;
        cpr += rb;
        spr += wss;
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first dot product
    if (LUT == 1) {
      if (threadIdx.x < 256) {
        lut_put(lut_r, threadIdx.x, c0);
        lut_put(lut_s, threadIdx.x, c1);
      }
      for (int i = threadIdx.x + blockDim.x; i < 256; i += blockDim.x) {  // (blocks of fewer than four waves)
        lut_put(lut_r, i, A.dn.cb[i >> 4]);
        lut_put(lut_s, i, tcb[i >> 4]);
      }
      moe_lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    const float b0 = LUT == 2 ? wcb[0] : 0.f, sxh = LUT == 2 ? xf_sum(xh) : 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      float v = __half2float(sc[r]) * m * (LUT ? f32_dot<LUT>(cw[r], xh, lt, a, b0, sxh) : chunk_dot(cw[r], x, a, b));
      v = sum32(v);
      if (g_raw == 0 && s_raw < nslots) part[s_raw][r] = v;
      if ((r & 1) == 1) __builtin_amdgcn_sched_barrier(0);  // rows are consumed in arrival order
    }
  }
  if ((int)threadIdx.x < nslots) wsm[threadIdx.x] = (int)threadIdx.x < kpt ? wmine : sigmoid_f(wmine);
  __syncthreads();
  if (threadIdx.x < ROWS) {
    const int r = threadIdx.x;
    float y = 0.f;
    for (int s = 0; s < kpt; s++) y += wsm[s] * part[s][r];
    if (has_shared) {
      const float shv = wsm[kpt] * part[kpt][r];
      if (A.out_sh) A.out_sh[(size_t)tok * out_stride + r0 + r] = shv;
      else y += shv;
    }
    out[(size_t)tok * out_stride + r0 + r] = y;
  }
}

// The same for rows of 16, 20 or 24 groups, which leave lanes of a half-wave without one: a wave takes four slots, and its lanes the
// 4 G (slot, group) units of a row one after the other -- the first 64, then the R = 4 G - 64 that are left, those of 64 / R rows
// at a time (24 groups: two rows in three passes instead of four, 20: four rows in five instead of eight, 16: a row in one
// instead of two).  A lane keeps the activations of its two units for all rows.  Units of a slot start at multiples of 8 (20
// groups: 4) lanes, so a row's sums are taken over as many lanes in registers, the rest from LDS.
// grid (d / ROWS, P), block 64 ceil(slots / 4).
// What bounds the launch from a few tokens on is vector instructions: half-waves of 24, 20 or 16 busy lanes of 32 take 31 for a
// row and slot, 24 groups packed 19.  Layers, us, half-waves and packed (rows of a block that are fastest): 3072 x 768 4 tokens (two
// layers) 95.2 92.9, 12 102.8 100.9, 20 (local) 146.4 140.4, rotated experts 11 91.8 88.6; 2560 x 640 1 (four layers) 73.9 71.3, 20 124.1 118.7;
// 3072 x 512 1 69.9 68.1, 20 119.3 106.1; table codebooks 3072 x 768 2 87.0 78.4, 5 78.1 67.8, 2560 x 640 3 96.9 83.8, 3072 x 512 5 68.2 51.7.
// With 24 groups one token waits for latency, not instructions, and half as many waves are slower: one token 79.8 and 80 .. 82,
// table 112.5 and 114 .. 119; three tokens 74.5 either way.  Rows: more share a lane's activations, fewer leave more blocks and waves
// (20 tokens, 4, 8, 12, 16 and 24 rows of 24 groups: 152, 142, 140, 141 and 142; 20 groups 8 and 16: 122 and 119; one token 4 and 8: 71.3, 72.2).
// 16, 20 and 24 groups are the widths that this dealing fits: what is left of four slots' units after 64 has to divide 64 (17 and 18
// would too, but their sums are no whole quads of lanes; narrower rows would want more slots to a wave).  All other widths stay on
// half-waves, with the lanes past their groups idle.
template <int G, int ROWS, bool LUT>
__global__ void __launch_bounds__(256) k_dec_dn_packed(DnArgs2 A, const uint32_t* __restrict__ hplanes, const float2* __restrict__ hmeta,
                                                       const int* __restrict__ ids, const float* __restrict__ ws, int id_stride, int kpt,
                                                       int d, float* __restrict__ out, uint64_t out_stride,
                                                       const float* __restrict__ hid_f32) {
  constexpr int R = 4 * G - 64, RS = R ? 64 / R : 1, NB = R ? ROWS / RS : 0;
  static_assert(R >= 0 && R < 64 && (R == 0 || 64 % R == 0) && ROWS % RS == 0, "");
  constexpr int PL = G % 8 ? 4 : 8, NPC = G / PL, PCP = NPC > 4 ? 8 : 4;  // lanes of a sum, sums of a row, floats of them in LDS
  constexpr int SETS = R ? 2 : 1;
  extern __shared__ float lutmem[];
  __shared__ __attribute__((aligned(16))) float part[DN2_MAXSLOTS][ROWS][PCP];
  __shared__ float wsm[DN2_MAXSLOTS];
  const int tok = blockIdx.y, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const bool has_shared = A.shd.codes != nullptr;
  const int nslots = kpt + (has_shared ? 1 : 0), r0 = blockIdx.x * ROWS;
  constexpr uint32_t rb = 16u * G;
  const float* const tcb = has_shared ? A.shd.cb : A.dn.cb;
  float c0 = 0.f, c1 = 0.f, c2 = 0.f, c3 = 0.f;
  const int t2 = (int)(threadIdx.x + blockDim.x);
  if (LUT) {  // (a thread's first two pieces of each table)
    c0 = A.dn.cb[threadIdx.x >> 4 & 15];
    c1 = tcb[threadIdx.x >> 4 & 15];
    c2 = A.dn.cb[t2 >> 4 & 15];
    c3 = tcb[t2 >> 4 & 15];
  }
  float wmine = 0.f;
  if ((int)threadIdx.x < nslots)
    wmine = (int)threadIdx.x < kpt ? ws[(size_t)tok * id_stride + threadIdx.x] : A.sh_logit[tok];
  // (branch-free loads, as above: a unit without a slot reads slot 0 and counts nothing)
  int slot[SETS], grp[SETS];
  float m[SETS], ca[SETS], cb[SETS];
  const uint8_t *cp[SETS], *sp[SETS];
  uint64_t wss[SETS];
  uint32_t lt[SETS];
  XG x[LUT ? 1 : SETS];
  XF xh[LUT ? SETS : 1];
  const uint32_t lut_r = LUT ? lut_at(lutmem) : 0u, lut_s = lut_r + LUT_BYTES;
#pragma unroll
  for (int i = 0; i < SETS; i++) {
    const int u = i ? 64 + lane % (R ? R : 1) : lane;
    grp[i] = u % G;
    slot[i] = 4 * wv + u / G;
    const bool live = slot[i] < nslots, shared = has_shared && slot[i] == nslots - 1;
    const int s = live ? slot[i] : 0;
    m[i] = live ? 1.f : 0.f;
    const uint8_t* const codes = shared ? A.shd.codes : A.dn.codes;
    const uint8_t* const scales = shared ? A.shd.scales : A.dn.scales;
    const float* const wcb = shared ? A.shd.cb : A.dn.cb;
    wss[i] = shared ? A.shd.ss : A.dn.ss;
    const int gsh = shared ? A.shd.gsh : A.dn.gsh;
    const int e_any = ids[tok * id_stride + (shared ? 0 : s)];
    const uint32_t row0 = (shared ? 0u : (uint32_t)e_any) * (uint32_t)d + (uint32_t)(r0 + (i ? lane / (R ? R : 1) : 0));
    if (LUT) load_xf(xh[LUT ? i : 0], hid_f32 + ((size_t)(tok * nslots + s) * G + grp[i]) * 32);
    else load_xg(x[LUT ? 0 : i], hplanes, hmeta, (size_t)((tok * nslots + s) * G + grp[i]));
    lt[i] = ((shared ? lut_s : lut_r) >> 8) * 0x01010101u;
    ca[i] = wcb[1] - wcb[0];
    cb[i] = fmaf(8.f, ca[i], wcb[0]);
    cp[i] = codes + (uint64_t)row0 * rb + (uint32_t)grp[i] * 16;
    sp[i] = scales + (uint64_t)row0 * (uint32_t)wss[i] + (uint32_t)(grp[i] >> gsh) * 2;
  }
  uint4 cw[ROWS], cwb[NB ? NB : 1];
  __half sc[ROWS], scb[NB ? NB : 1];
  {
    const uint8_t *c = cp[0], *q = sp[0];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      cw[r] = *(const uint4*)c;
      sc[r] = *(const __half*)q;
      c += rb;
      q += wss[0];
    }
  }
  if constexpr (R > 0) {
    const uint8_t *c = cp[1], *q = sp[1];
#pragma unroll
    for (int r = 0; r < NB; r++) {
      cwb[r] = *(const uint4*)c;
      scb[r] = *(const __half*)q;
      c += RS * rb;
      q += RS * wss[1];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first dot product
  if (LUT) {
    if (threadIdx.x < 256) {
      lut_put(lut_r, threadIdx.x, c0);
      lut_put(lut_s, threadIdx.x, c1);
    }
    if (t2 < 256) {
      lut_put(lut_r, t2, c2);
      lut_put(lut_s, t2, c3);
    }
    for (int i = t2 + (int)blockDim.x; i < 256; i += blockDim.x) {  // (one wave)
      lut_put(lut_r, i, A.dn.cb[i >> 4]);
      lut_put(lut_s, i, tcb[i >> 4]);
    }
    moe_lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
  auto dot = [&](int i, const uint4& c, __half s, int row) {
    float v;
    if (LUT) v = f32_dot<1>(c, xh[LUT ? i : 0], lt[i], 0.f, 0.f, 0.f);
    else v = chunk_dot(c, x[LUT ? 0 : i], ca[i], cb[i]);
    v *= __half2float(s) * m[i];
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));  // xor 1
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));  // xor 2
    if (PL == 8) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true));  // mirror in 8
    if (lane % PL == 0) part[slot[i]][row][grp[i] / PL] = v;
  };
#pragma unroll
  for (int r = 0; r < ROWS; r++) {
    dot(0, cw[r], sc[r], r);
    if (r & 1) __builtin_amdgcn_sched_barrier(0);  // rows are consumed in arrival order
  }
  if constexpr (R > 0) {
#pragma unroll
    for (int r = 0; r < NB; r++) {
      dot(1, cwb[r], scb[r], RS * r + lane / R);
      if (r & 1) __builtin_amdgcn_sched_barrier(0);
    }
  }
  if ((int)threadIdx.x < nslots) wsm[threadIdx.x] = (int)threadIdx.x < kpt ? wmine : sigmoid_f(wmine);
  __syncthreads();
  if (threadIdx.x < ROWS) {
    const int r = threadIdx.x;
    auto total = [&](int s) {
      float v = part[s][r][0];
#pragma unroll
      for (int i = 1; i < NPC; i++) v += part[s][r][i];
      return v;
    };
    float y = 0.f;
    for (int s = 0; s < kpt; s++) y += wsm[s] * total(s);
    if (has_shared) {
      const float shv = wsm[kpt] * total(kpt);
      if (A.out_sh) A.out_sh[(size_t)tok * out_stride + r0 + r] = shv;
      else y += shv;
    }
    out[(size_t)tok * out_stride + r0 + r] = y;
  }
}

// Down projection of the unique-expert path: grid (d/DU_ROWS, tiles), block 256 = 8 half-waves of
// DU_HW rows.  Lane g of a half-wave holds group g of its weight rows and walks the tile's pairs; the
// unweighted row results go to pairs[pair][row] (f32) for the weighted combine that follows.
// All loads are unconditional (a lane past the last group reads group 0 and contributes 0) and are
// requested before the first is used: activation planes of the first pair, then the rows.
constexpr int DU_HW = 8, DU_ROWS = 8 * DU_HW;
__global__ void __launch_bounds__(256) k_dec_dn_uq(DnArgs2 A, const uint32_t* __restrict__ hplanes,
                                                   const float2* __restrict__ hmeta,
                                                   const moe_tile* __restrict__ tiles,
                                                   const int* __restrict__ ntiles, int n_experts, int d, int mid,
                                                   float* __restrict__ pairs) {
  if ((int)blockIdx.y >= ntiles[0]) return;
  const moe_tile tile = tiles[blockIdx.y];
  const bool shared = tile.expert >= n_experts;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int G = mid / 32, g_raw = lane & 31, hw = 2 * wv + (lane >> 5);
  const int g = g_raw < G ? g_raw : 0;
  const float live = g_raw < G ? 1.f : 0.f;
  const size_t rb = (size_t)mid / 2;
  const DecW W = shared ? A.shd : A.dn;  // block-uniform, by value
  const int r0 = blockIdx.x * DU_ROWS + DU_HW * hw;
  const uint64_t row0 = (shared ? 0 : (uint64_t)tile.expert * d) + r0;
  const uint8_t* cp = W.codes + row0 * rb + (size_t)g * 16;
  const uint8_t* sp = W.scales + row0 * W.ss + (g >> W.gsh) * 2;
  XG x;
  load_xg(x, hplanes, hmeta, (size_t)tile.first * G + g);
  const float c0 = W.cb[0], c1 = W.cb[1];
  uint4 cw[DU_HW];
  uint16_t sr[DU_HW];
#pragma unroll
  for (int r = 0; r < DU_HW; r++) {
    cw[r] = *(const uint4*)(cp + r * rb);
    sr[r] = *(const uint16_t*)(sp + r * W.ss);
  }
  __builtin_amdgcn_sched_barrier(0);
  const float a = c1 - c0, b = fmaf(8.f, a, c0);
  for (int pi = 0; pi < tile.count; pi++) {
    const size_t pr = (size_t)tile.first + pi;
    XG xn;  // the next pair's planes are requested before this pair's dot products (the last pair repeats itself)
    load_xg(xn, hplanes, hmeta, (pr + (pi + 1 < tile.count ? 1 : 0)) * G + g);
    float v[DU_HW];
#pragma unroll
    for (int r = 0; r < DU_HW; r++)
      v[r] = sum32(live * __half2float(__ushort_as_half(sr[r])) * chunk_dot(cw[r], x, a, b));
    if (g_raw == 0) {
      float4* o = (float4*)(pairs + pr * d + r0);
#pragma unroll
      for (int r = 0; r < DU_HW; r += 4) o[r / 4] = make_float4(v[r], v[r + 1], v[r + 2], v[r + 3]);
    }
    x = xn;
  }
}

DecW decw(const moe_wview* w) {
  DecW o{};
  if (w && w->dtype == MOE_DT_I4R) {  // codes, then one fp16 scale per 128 columns, rows unpadded; codebook n - 8
    o.codes = w->data;
    o.scales = w->data + w->rows * w->cols / 2;
    o.cb = moe_i4r_codebook();
    o.ss = w->cols / 128 * 2;
    o.gsh = 2;
  } else if (w) {
    Q4cpOps q = q4cp_ops(w);
    o.codes = q.codes; o.scales = q.scales; o.cb = q.cb; o.ss = q.scale_stride;
  }
  return o;
}

}  // namespace

size_t moe_qvec_plane_bytes(int K) { return (size_t)(K / 32) * QV_GROUP_DW * 4; }
size_t moe_qvec_meta_bytes(int K) { return (size_t)(K / 32) * sizeof(float2); }

// Supported shapes of the integer-dot decode kernels (otherwise the caller uses the f32 kernels).
bool moe_dec_supported(int d, int mid, int nslots) {
  return d % 32 == 0 && d / 32 <= 96 && mid % 32 == 0 && mid / 32 <= 32 && nslots <= DN2_MAXSLOTS &&
         mid % GU2_ROWS == 0;  // (d % 32 == 0 covers the 8-row down blocks)
}
// the unique-expert kernels on top of that: whole row blocks of the down kernel
bool moe_dec_uq_supported(int d) { return d % DU_ROWS == 0; }

int moe_launch_qvec(const float* x, uint64_t x_stride, int P, int K, uint32_t* planes, float2* meta,
                    hipStream_t st) {
  const int G = K / 32;
  dim3 grid((G + 63) / 64, P);
  k_qvec_from_f32<<<grid, 64, 0, st>>>(x, x_stride, G, planes, meta);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// (TL of k_dec_gu by the row's groups)
#define DEC_GU_TAILS(GO)            \
  do {                              \
    if (d <= 64 * 32) GO(0);        \
    else if (d <= 80 * 32) GO(2);   \
    else GO(4);                     \
  } while (0)
int moe_launch_dec_gu(const moe_wview* gu, const moe_wview* sh_gate, const moe_wview* sh_up,
                      const uint32_t* xplanes, const float2* xmeta, const int* ids, int id_stride, int kpt,
                      int P, int d, int mid, uint32_t* hplanes, float2* hmeta, float* hid_f32,
                      hipStream_t st, const moe_dec_v2* v2) {
  GuArgs2 A{};
  A.gu = decw(gu);
  A.shg = decw(sh_gate);
  A.shu = decw(sh_up);
  if (v2) {
    if (!v2->zraw || !v2->xplanes_rot || !v2->xmeta_rot) return MOE_E_INVALID;
    A.zraw = v2->zraw;
    A.xplanes_rot = v2->xplanes_rot;
    A.xmeta_rot = v2->xmeta_rot;
  }
  if (!A.gu.cb) return MOE_E_STATE;
  dim3 grid(mid / GU2_ROWS, kpt + (sh_gate ? 1 : 0), P);
#define DEC_GU(TL)                                                                                                                   \
  k_dec_gu<false, 0, 0, TL><<<grid, 512, 0, st>>>(A, xplanes, xmeta, ids, id_stride, kpt, d, mid, hplanes, hmeta, hid_f32, nullptr, nullptr, \
                                                  nullptr, 0, nullptr, nullptr, nullptr, nullptr, moe_rfix{})
  DEC_GU_TAILS(DEC_GU);
#undef DEC_GU
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// The same with the softmax / top-k of every token done inside the launch: logits [P][n_experts] in,
// ids / ws rows (id_stride wide) out.
bool moe_dec_gu_topk_supported(int n_experts, int kpt) { return n_experts <= 1024 && kpt <= 64 && kpt <= n_experts; }
int moe_launch_dec_gu_topk(const moe_wview* gu, const moe_wview* sh_gate, const moe_wview* sh_up,
                           const uint32_t* xplanes, const float2* xmeta, const float* logits, int n_experts,
                           int* ids, float* ws, int id_stride, int kpt, int P, int d, int mid,
                           uint32_t* hplanes, float2* hmeta, float* hid_f32, hipStream_t st, const moe_dec_v2* v2,
                           const moe_rfix* rf) {
  const moe_rfix RFV = rf ? *rf : moe_rfix{};
  if (RFV.W && !RFV.tol) return MOE_E_INVALID;
  GuArgs2 A{};
  A.gu = decw(gu);
  A.shg = decw(sh_gate);
  A.shu = decw(sh_up);
  if (v2) {
    if (!v2->zraw || !v2->xplanes_rot || !v2->xmeta_rot) return MOE_E_INVALID;
    A.zraw = v2->zraw;
    A.xplanes_rot = v2->xplanes_rot;
    A.xmeta_rot = v2->xmeta_rot;
  }
  if (!A.gu.cb) return MOE_E_STATE;
  dim3 grid(mid / GU2_ROWS, kpt + (sh_gate ? 1 : 0) + 1, P);  // + the row of the exact top-k block
#define DEC_GU(TL)                                                                                                                      \
  k_dec_gu<false, 8, 0, TL><<<grid, 512, 0, st>>>(A, xplanes, xmeta, nullptr, id_stride, kpt, d, mid, hplanes, hmeta, hid_f32, nullptr, nullptr, \
                                                  nullptr, n_experts, logits, ids, ws, nullptr, RFV)
  if (n_experts <= 512 && d <= 64 * 32) DEC_GU(0);
  else if (n_experts <= 512) DEC_GU(4);
#undef DEC_GU
  else
    k_dec_gu<false, 16, 0><<<grid, 512, 0, st>>>(A, xplanes, xmeta, nullptr, id_stride, kpt, d, mid, hplanes, hmeta,
                                                     hid_f32, nullptr, nullptr, nullptr, n_experts, logits, ids, ws, nullptr, RFV);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// The look-up kernels (any codebook): x f32 [P][d] in, hid f32 [P][kpt + shared][mid] out; softmax / top-k inside
// the launch as above.
// (affine: every codebook involved is a*n + b -- the f32 arithmetic instead of the look-up.  logits == nullptr: the
//  ids are given and no selection runs inside the launch.)
int moe_launch_dec_gu_lut(const moe_wview* gu, const moe_wview* sh_gate, const moe_wview* sh_up, const float* x,
                          const float* logits, int n_experts, int* ids, float* ws, int id_stride, int kpt, int P, int d,
                          int mid, float* hid_f32, hipStream_t st, const moe_rfix* rf, bool affine) {
  if (!x || !hid_f32 || !ids || (logits && !moe_dec_gu_topk_supported(n_experts, kpt))) return MOE_E_INVALID;
  const moe_rfix RFV = rf ? *rf : moe_rfix{};
  if (logits && RFV.W && !RFV.tol) return MOE_E_INVALID;
  GuArgs2 A{};
  A.gu = decw(gu);
  A.shg = decw(sh_gate);
  A.shu = decw(sh_up);
  if (d > 3072) return MOE_E_UNSUPPORTED;
  const int nt = gu2_threads(affine ? 2 : 1, logits != nullptr);
  dim3 grid((mid + nt / 16 - 1) / (nt / 16), kpt + (sh_gate ? 1 : 0) + (logits ? 1 : 0), P);
  const int lds = (affine ? 0 : 3 * LUT_BYTES) + d / 32 * XF_PITCH * 4;  // (a table's worth for the tables' alignment)
#define DEC_GU_F32(NPL, MODE, ...)                                                                                     \
  k_dec_gu<false, NPL, MODE, ##__VA_ARGS__><<<grid, nt, lds, st>>>(A, nullptr, nullptr, NPL ? nullptr : ids, id_stride, kpt, d, mid, nullptr, \
                                                     nullptr, hid_f32, nullptr, nullptr, nullptr, n_experts, logits, ids, ws, x, RFV)
  if (!logits) {
#define DEC_GU(TL) DEC_GU_F32(0, 1, TL)
    if (affine) DEC_GU_F32(0, 2);
    else DEC_GU_TAILS(DEC_GU);
#undef DEC_GU
  } else if (n_experts <= 512) {
#define DEC_GU(TL) DEC_GU_F32(8, 1, TL)
    if (affine) DEC_GU_F32(8, 2);
    else DEC_GU_TAILS(DEC_GU);
#undef DEC_GU
  } else {
    if (affine) DEC_GU_F32(16, 2);
    else DEC_GU_F32(16, 1);
  }
#undef DEC_GU_F32
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_dec_dn_lut(const moe_wview* dn, const moe_wview* sh_down, const float* sh_logit, const float* hid_f32,
                          const int* ids, const float* ws, int id_stride, int kpt, int P, int d, int mid, float* out,
                          uint64_t out_stride, hipStream_t st, bool affine) {
  DnArgs2 A{};
  A.dn = decw(dn);
  A.shd = decw(sh_down);
  A.sh_logit = sh_logit;
  if (dn->rows > 0xffffffffull) return MOE_E_UNSUPPORTED;  // (row numbers are 32-bit in the kernel)
  const int nslots = kpt + (sh_down ? 1 : 0), bs = 64 * ((nslots + 1) / 2);
  constexpr int lds = 3 * LUT_BYTES;  // (one for the tables' alignment)
#define DEC_DN_F32(ROWS, MODE)                                                                                          \
  k_dec_dn<ROWS, MODE><<<dim3(d / ROWS, P), bs, MODE == 1 ? lds : 0, st>>>(A, nullptr, nullptr, ids, ws, id_stride, kpt, d, mid, \
                                                                           out, out_stride, hid_f32)
  if (!affine) {
    const int bs4 = 64 * ((nslots + 3) / 4);
#define DEC_DN_PACKED(G, ROWS)                                                                                                       \
  k_dec_dn_packed<G, ROWS, true><<<dim3(d / ROWS, P), bs4, lds, st>>>(A, nullptr, nullptr, ids, ws, id_stride, kpt, d, out, out_stride, hid_f32)
    bool taken = true;
    if (mid == 768 && P > 1) DEC_DN_PACKED(24, 8);
    else if (mid == 640 && P > 1) DEC_DN_PACKED(20, 8);
    else if (mid == 640) DEC_DN_PACKED(20, 4);
    else if (mid == 512 && P > 1) DEC_DN_PACKED(16, 8);
    else if (mid == 512) DEC_DN_PACKED(16, 4);
    else taken = false;
#undef DEC_DN_PACKED
    if (taken) {
      MOE_LAUNCH_CHECK();
      return MOE_OK;
    }
  }
  if (d % MOE_DN_ROWS == 0) {
    if (affine) DEC_DN_F32(MOE_DN_ROWS, 2);
    else DEC_DN_F32(MOE_DN_ROWS, 1);
  } else {
    if (affine) DEC_DN_F32(8, 2);
    else DEC_DN_F32(8, 1);
  }
#undef DEC_DN_F32
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// Unique-expert variants: tiles / ntiles / tokidx from the routing permutation (tiles of <= 32 pairs,
// the shared expert as expert id n_experts); hplanes / hmeta and pairs are indexed by pair position.
int moe_launch_dec_gu_uq(const moe_wview* gu, const moe_wview* sh_gate, const moe_wview* sh_up,
                         const uint32_t* xplanes, const float2* xmeta, const moe_tile* tiles, const int* ntiles,
                         int max_tiles, const int* tokidx, int n_experts, int d, int mid, uint32_t* hplanes,
                         float2* hmeta, hipStream_t st) {
  GuArgs2 A{};
  A.gu = decw(gu);
  A.shg = decw(sh_gate);
  A.shu = decw(sh_up);
  if (max_tiles <= 0) return MOE_OK;
  dim3 grid(mid / GU2_ROWS, max_tiles);
  k_dec_gu<true, 0, 0><<<grid, 512, 0, st>>>(A, xplanes, xmeta, nullptr, 0, 0, d, mid, hplanes, hmeta, nullptr, tiles,
                                                 ntiles, tokidx, n_experts, nullptr, nullptr, nullptr, nullptr, moe_rfix{});
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_dec_dn_uq(const moe_wview* dn, const moe_wview* sh_down, const uint32_t* hplanes,
                         const float2* hmeta, const moe_tile* tiles, const int* ntiles, int max_tiles,
                         int n_experts, int d, int mid, float* pairs, hipStream_t st) {
  DnArgs2 A{};
  A.dn = decw(dn);
  A.shd = decw(sh_down);
  if (max_tiles <= 0) return MOE_OK;
  dim3 grid(d / DU_ROWS, max_tiles);
  k_dec_dn_uq<<<grid, 256, 0, st>>>(A, hplanes, hmeta, tiles, ntiles, n_experts, d, mid, pairs);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

int moe_launch_dec_dn(const moe_wview* dn, const moe_wview* sh_down, const float* sh_logit,
                      const uint32_t* hplanes, const float2* hmeta, const int* ids, const float* ws,
                      int id_stride, int kpt, int P, int d, int mid, float* out, uint64_t out_stride,
                      hipStream_t st, float* out_sh) {
  DnArgs2 A{};
  A.dn = decw(dn);
  A.shd = decw(sh_down);
  A.sh_logit = sh_logit;
  A.out_sh = out_sh;
  if (!A.dn.cb) return MOE_E_STATE;
  if (dn->rows > 0xffffffffull) return MOE_E_UNSUPPORTED;  // (row numbers are 32-bit in the kernel)
  const int nslots = kpt + (sh_down ? 1 : 0), bs = 64 * ((nslots + 1) / 2);
  const int bs4 = 64 * ((nslots + 3) / 4);
#define DEC_DN_PACKED(G, ROWS)                                                                                                       \
  k_dec_dn_packed<G, ROWS, false><<<dim3(d / ROWS, P), bs4, 0, st>>>(A, hplanes, hmeta, ids, ws, id_stride, kpt, d, out, out_stride, nullptr)
  bool taken = true;
  if (mid == 768 && P > 3 && d % 12 == 0) DEC_DN_PACKED(24, 12);
  else if (mid == 768 && P > 3) DEC_DN_PACKED(24, 8);
  else if (mid == 640 && P == 1) DEC_DN_PACKED(20, 4);
  else if (mid == 640 && P > 8 && d % 16 == 0) DEC_DN_PACKED(20, 16);
  else if (mid == 640) DEC_DN_PACKED(20, 8);
  else if (mid == 512 && P > 8 && d % 16 == 0) DEC_DN_PACKED(16, 16);
  else if (mid == 512) DEC_DN_PACKED(16, 8);
  else taken = false;
#undef DEC_DN_PACKED
  if (taken) {
    MOE_LAUNCH_CHECK();
    return MOE_OK;
  }
  // MOE_DN_ROWS rows per block where that divides d (d = 3072: 512 blocks, two per CU), else 8
  if (d % MOE_DN_ROWS == 0)
    k_dec_dn<MOE_DN_ROWS, 0><<<dim3(d / MOE_DN_ROWS, P), bs, 0, st>>>(A, hplanes, hmeta, ids, ws, id_stride, kpt, d, mid, out, out_stride, nullptr);
  else
    k_dec_dn<8, 0><<<dim3(d / 8, P), bs, 0, st>>>(A, hplanes, hmeta, ids, ws, id_stride, kpt, d, mid, out, out_stride, nullptr);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}
