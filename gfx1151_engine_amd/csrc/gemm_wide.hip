// Grouped expert GEMM for 8-bit codes: Q8_0 tensors of GGUF layers, q8g32 shared experts of overlay files.
// (same contract as gguf_types.hip's general kernel: src/gpu/parts/26_kernels_moe_gguf.inc:81-386; weights are f16(code * scale),
// one rounding, f32 sums)
//
// A block (four waves) multiplies a tile of up to 128 pairs with 256 weight rows (gate/up: 128 gate rows and the 128 up rows that
// match, SwiGLU on the accumulators); a wave owns 64 of them.  The general kernel dequantises into LDS and reads both operands
// back; here the codes go from memory into the registers of the lane that multiplies them -- v_mfma_f32_32x32x16_f16 takes the
// weights as A, lane (n, h) = row n, and which columns a lane half takes is free as long as the activations agree: half h
// takes 64 columns in a row (two 34-byte blocks, 68 bytes from a 4-byte boundary) -- and only the activations pass through LDS,
// 128 columns at a time, double-buffered.  An MFMA occupies the matrix pipe for 32 cycles and the vector pipe for 8, which
// leaves room for six vector operations; dequantisation takes 30 per step of 2 .. 8 MFMAs.  The order of a step is fixed by hand:
// an item of two MFMAs reads one activation operand two items ahead and dequantises a part of the next step's weights.
// Two blocks to a CU (65 KB of LDS, 256 registers): their barriers, prologues and epilogues are independent.
// us, general kernel and this one (3072 x 768, 512 experts): routed Q8_0 down, 2000 tokens 541 and 423, 4096 (skewed) 656 and 538,
// 8192 (skewed / even) 938 / 1065 and 767 / 806; the Q8_0 shared expert's two launches beside the router's, 4096 tokens 92 + 66 and 84
// + 45, 8192 219 + 87 and 137 + 120; layers with a q8g32 shared expert, 2560 x 640 2000 tokens 614 and 594, 3072 x 768 of 64 experts
// 130 tokens 219 and 155; all-Q8_0 layers 130 tokens 1460 and 1062, 2000 1755 and 1323, 8192 3600 and 2727.  What bounds it is the
// loads: 16 bytes of every row and half per lane are 100 cycles of the address unit each (busy 85 % of the launch), and rows are
// visited 136 bytes at a time, 1.6 times the lines that they have.  (Few blocks: moe_wide_takes.)
// (All of a stage's loads in a row instead of half of them half a stage later, so that a line's second load finds it in L1:
// 466 -> 427; two stages in registers instead of one, by itself: no change.)
#include <type_traits>

#include "common.h"
#include "dense.h"
#include "half.h"
#include "internal.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

enum { W_Q80, W_G32 };

struct WideW {
  const uint8_t *w, *w_up;
  uint64_t sc;  // q8g32: byte offset of the scale plane
};

constexpr int XROW = 256;              // bytes of a stage (128 columns) of one pair row
constexpr int XBUF = 128 * XROW;       // of a tile
constexpr int PROW = 128 + 16;         // down: bytes of a pair row in a wave's patch of results (64 f16 and padding)
constexpr int SMEM = 2 * XBUF + 1024;  // + row scales and gate/up's row offsets
constexpr int SMEM_DN = 2 * XBUF + 4 * 16 * PROW;

// LX: order of the activations (moe_f32_to_f16's layouts); MF: groups of 32 pairs
template <int FMT, bool UP, int LX, int MF>
__device__ __forceinline__ void wide_tile(uint8_t* smem, const WideW& L, int e, const moe_tile tile, int nb, int npass,
                                          const __half* __restrict__ x, const int* __restrict__ tokidx, __half* __restrict__ out,
                                          int M, int K, const moe_hscale& hs, moe_cmag cmag) {
  float* const rowscale = (float*)(smem + 2 * XBUF);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int NS = K >> 7, total = npass * NS;
  const uint32_t RB = FMT == W_Q80 ? (uint32_t)(K / 32 * 34) : (uint32_t)K;
  // ---- weights: MFMA row n of fragment f.  D row 8 a + 4 h + b is register 4 a + b of lane half h: these rows make a lane's results
  // neighbours (down: 32 of the wave's 64 rows, gate/up: 16 of its 32) ----
  constexpr int WR = UP ? 32 : 64;  // (gate) rows of a wave
  const int hn = (n >> 2) & 1, i4 = 4 * (n >> 3) + (n & 3);
  auto row0 = [&](int p) {
    const int r = (nb + p) * 4 * WR + WR * wv;
    return r < M ? r : 0;  // (loaded, never stored)
  };
  const uint32_t lrow = (uint32_t)(UP ? 16 * hn + i4 : 32 * hn + i4), lo = lrow * RB + (FMT == W_G32 ? 64u : 68u) * (uint32_t)h;
  // stages of codes in registers: as parts are used up, those of NB stages on take their place
  constexpr int NB = MF < 4 ? 2 : 1;
  uint4 c[NB][2][4];     // the lane's 64 columns: Q8_0 dwords 0 .. 15 of 17, q8g32 the codes
  uint32_t last[NB][2];  // Q8_0 dword 16; q8g32 both scales
  constexpr bool G32 = FMT == W_G32;
  // part 0: what steps 0 .. 3 need, part 1: the rest
  auto load = [&](auto part, int nst, auto slot) {
    constexpr int S = decltype(slot)::value;
    nst = nst < total ? nst : total - 1;
    const int p = UP ? 0 : nst / NS, s = UP ? nst : nst - p * NS;
    const size_t first = (size_t)e * M + row0(p);
#pragma unroll
    for (int f = 0; f < 2; f++) {
      // (down's second fragment: sixteen rows on)
      const size_t fr = first + (UP || !f ? 0 : 16);
      const uint8_t* const b = (UP && f ? L.w_up : L.w) + fr * RB + (G32 ? 128 : 136) * (size_t)s;
      auto ld = [&](int k) {
        const uint32_t* d = (const uint32_t*)(b + 16 * k + lo);
        c[S][f][k] = make_uint4(d[0], d[1], d[2], d[3]);
      };
      if (decltype(part)::value == 0) {
        ld(0);
        ld(LX == 2 ? 2 : 1);
        if (G32)
          last[S][f] = *(const uint32_t*)((UP && f ? L.w_up : L.w) + L.sc +
                                          ((fr * (size_t)(K >> 5) + 4 * s) * 2 + (lrow * (uint32_t)(K >> 5) + 2u * (uint32_t)h) * 2u));
      } else {
        ld(LX == 2 ? 1 : 2);
        ld(3);
        if (!G32) last[S][f] = *(const uint32_t*)(b + 64 + lo);
      }
    }
  };
  constexpr std::integral_constant<int, 0> P0{};
  constexpr std::integral_constant<int, 1> P1{};
  load(P0, 0, P0);
  load(P1, 0, P0);
  if constexpr (NB == 2) {
    load(P0, 1, P1);
    load(P1, 1, P1);
  }
  // ---- activations: thread = chunk tid % 16 of pair rows tid / 16 + 16 l, half of the rows at a time ----
  // (rows past the tile's pairs repeat its last one.  Offsets in 16-byte pieces; gate/up's, which tokidx gives, wait in LDS)
  constexpr int XL = 2 * MF;
  const int xc = tid & 15, xt = tid >> 4, lastp = tile.count - 1;
  uint32_t* const rowoff = (uint32_t*)(rowscale + 128);
  if constexpr (UP) {
    if (tid < 32 * MF) {
      const int row = tokidx[tile.first + (tid < lastp ? tid : lastp)];
      rowoff[tid] = (uint32_t)row * (uint32_t)(K >> 3);
      rowscale[tid] = hs.xms ? moe_hid_scale(cmag, hs.xms[row]) : 1.f;
    }
    moe_lds_barrier();
  }
  auto x_at = [&](int l) -> uint32_t {
    const int m = 16 * l + xt;
    if constexpr (UP) return rowoff[m] + (uint32_t)xc;
    return (uint32_t)(tile.first + (m < lastp ? m : lastp)) * (uint32_t)(K >> 3) + (uint32_t)xc;
  };
  // the next stage's activations go to LDS in NP parts of XP loads
  constexpr int NP = MF == 4 ? 4 : 2, XP = XL / NP;
  static_assert(XP * NP == XL && XP <= 3, "named registers");
  uint4 xv0, xv1, xv2;  // (named: an array here ends up in scratch memory)
  auto fetch_x = [&](int nst, auto part) {
    constexpr int l = XP * decltype(part)::value;
    nst = nst < total ? nst : total - 1;
    const uint4* const b = (const uint4*)x + 16 * (size_t)(UP ? nst : nst % NS);
    xv0 = b[x_at(l)];
    if constexpr (XP > 1) xv1 = b[x_at(l + 1)];
    if constexpr (XP > 2) xv2 = b[x_at(l + 2)];
  };
  auto put_x = [&](int buf, auto part) {
    auto put = [&](int l, const uint4& v) {
      const int m = 16 * l + xt;
      *(uint4*)(smem + buf * XBUF + m * XROW + ((xc ^ (m & 15)) << 4)) = v;
    };
    constexpr int l = XP * decltype(part)::value;
    put(l, xv0);
    if constexpr (XP > 1) put(l + 1, xv1);
    if constexpr (XP > 2) put(l + 2, xv2);
  };
  // between parts p and p + 1 of a stage (0, ..., NP - 1)
  auto turn_x = [&](int buf, int nst, auto part) {
    constexpr int p = decltype(part)::value;
    put_x(buf, part);
    if constexpr (p + 1 < NP) fetch_x(nst, std::integral_constant<int, p + 1>{});
  };
  constexpr std::integral_constant<int, 2> P2{};
  constexpr std::integral_constant<int, 3> P3{};
  fetch_x(0, P0);
  turn_x(0, 0, P0);
  turn_x(0, 0, P1);
  if constexpr (NP == 4) {
    turn_x(0, 0, P2);
    turn_x(0, 0, P3);
  }
  // chunk 8 h + w of pair row n; rows of a read's sixteen lanes differ in their low four bits (0-3, 12-15 and 20-27; ...)
  const uint32_t xa0 = (uint32_t)(n * XROW + (((8 * h) ^ (n & 15)) << 4));

  half2v sA[2], sB[2];  // scales of the lane's two blocks
  uint32_t d8[2];       // Q8_0: dword 8 has the first block's last codes beside the second's scale
  auto dw = [&](int S, int f, int k) { return k == 16 ? last[S][f] : word(c[S][f][k >> 2], k & 3); };
  auto code = [&](int S, int f, int blk, int k) -> uint32_t {  // four codes + 128
    if (G32) return dw(S, f, 8 * blk + k) ^ 0x80808080u;
    if (blk) return dw(S, f, 9 + k) ^ 0x80808080u;
    return __builtin_amdgcn_alignbyte(k == 7 ? d8[f] : dw(S, f, k + 1), dw(S, f, k), 2) ^ 0x80808080u;
  };
  auto scale_a = [&](int S, int f) {
    if (!G32) sA[f] = h2(__builtin_amdgcn_perm(c[S][f][0].x, c[S][f][0].x, 0x01000100u));
    else sA[f] = h2(__builtin_amdgcn_perm(last[S][f], last[S][f], 0x01000100u));
  };
  auto scale_b = [&](int S, int f) {
    if (!G32) sB[f] = h2(__builtin_amdgcn_perm(c[S][f][2].x, c[S][f][2].x, 0x03020302u));
    else sB[f] = h2(__builtin_amdgcn_perm(last[S][f], last[S][f], 0x03020302u));
    d8[f] = c[S][f][2].x;
  };
  H8 a[2][2];
  const half2v k1152 = {(_Float16)1152.f, (_Float16)1152.f};  // 1024 + u with u = code + 128
  auto unit = [&](int S, int w, int u) {  // a pair of step w's weights
    const int f = u >> 2, b = u & 3;
    uint32_t t;
    int blk;
    if (LX == 2) {  // chunk w = columns 4w, 4w+2, 32+4w, 32+4w+2, 4w+1, 4w+3, 32+4w+1, 32+4w+3
      blk = b & 1;
      t = __builtin_amdgcn_perm(0x64646464u, code(S, f, blk, w), b & 2 ? 0x04030401u : 0x04020400u);
    } else if (LX == 0) {
      blk = w >> 2;
      t = __builtin_amdgcn_perm(0x64646464u, code(S, f, blk, 2 * (w & 3) + (b >> 1)), b & 1 ? 0x04030402u : 0x04010400u);
    } else {  // columns 0, 4, 1, 5, 2, 6, 3, 7 of the chunk
      blk = w >> 2;
      t = __builtin_amdgcn_perm(code(S, f, blk, 2 * (w & 3) + 1), code(S, f, blk, 2 * (w & 3)),
                                0x0c040c00u + 0x00010001u * (uint32_t)b) | 0x64006400u;
    }
    a[w & 1][f].h[b] = (h2(t) - k1152) * (blk ? sB[f] : sA[f]);
  };
  floatx16 acc[2][MF];
  auto zero = [&]() {
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int mf = 0; mf < MF; mf++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[f][mf][i] = 0.f;
  };
  zero();
#pragma unroll
  for (int f = 0; f < 2; f++) {
    scale_a(0, f);
    scale_b(0, f);
  }
#pragma unroll
  for (int u = 0; u < 8; u++) unit(0, 0, u);

  constexpr int AHEAD = 2, N = 8 * MF;
  auto stage = [&](auto bc, int nst) {
    constexpr int B = decltype(bc)::value, CUR = NB == 2 ? B : 0, NEXT = NB == 2 ? B ^ 1 : 0;
    constexpr std::integral_constant<int, CUR> SLOT{};
    moe_lds_barrier();  // this stage's activations are in LDS; the other buffer has been read
    fetch_x(nst + 1, P0);
    half8 xf[AHEAD + 1];
    auto ldx = [&](int t) {
      xf[t % (AHEAD + 1)] = *(const half8*)(smem + (xa0 ^ (uint32_t)(t / MF << 4)) + (B * XBUF + 32 * (t % MF) * XROW));
    };
#pragma unroll
    for (int t = 0; t < AHEAD; t++) ldx(t);
#pragma unroll
    for (int t = 0; t < N; t++) {
      const int w = t / MF, mf = t % MF;
      if (NP == 4 && mf == 0 && w == 2) turn_x(B ^ 1, nst + 1, P0);
      if (mf == 0 && w == 4) {
        if constexpr (NP == 4) turn_x(B ^ 1, nst + 1, P1);
        else turn_x(B ^ 1, nst + 1, P0);
        if constexpr (NB == 1) load(P0, nst + NB, SLOT);  // (the first half of the codes is used up)
      }
      if constexpr (NP == 4) {
        if (mf == 0 && w == 6) turn_x(B ^ 1, nst + 1, P2);
      }
      if (mf == 0 && w == (LX == 2 ? 7 : 3)) {
        // (LX 2: both blocks' scales come with the next stage's part 0; else the second block's with this stage's part 1)
#pragma unroll
        for (int f = 0; f < 2; f++) scale_b(LX == 2 ? NEXT : CUR, f);
      }
      if (mf == 0 && w == 7) {
#pragma unroll
        for (int f = 0; f < 2; f++) scale_a(NEXT, f);
      }
      if (LX != 2 && !G32 && mf == 0 && w == 0) {
#pragma unroll
        for (int f = 0; f < 2; f++) d8[f] = c[CUR][f][2].x;
      }
      if (t + AHEAD < N) ldx(t + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < 2; f++) {
        acc[f][mf] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[w & 1][f].v, xf[t % (AHEAD + 1)], acc[f][mf], 0, 0, 0);
        const int slot = 2 * mf + f;
#pragma unroll
        for (int u = slot * 4 / MF; u < (slot + 1) * 4 / MF; u++) unit(w == 7 ? NEXT : CUR, (w + 1) & 7, u);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (NP == 4) turn_x(B ^ 1, nst + 1, P3);
    else turn_x(B ^ 1, nst + 1, P1);
    // (two stages in registers: the whole of a stage's columns at once, while its cache lines are in L1)
    if constexpr (NB == 2) load(P0, nst + NB, SLOT);
    load(P1, nst + NB, SLOT);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto finish = [&](int p) {
    const int r0 = (nb + p) * 4 * WR + WR * wv;
    if (r0 >= M) return;
    auto pack8 = [&](const float* v) {
      union { __half2 h[4]; uint4 q; } u;
#pragma unroll
      for (int k = 0; k < 4; k++) u.h[k] = __floats2half2_rn(v[2 * k], v[2 * k + 1]);
      return u.q;
    };
    if constexpr (!UP) {
      // sixteen pairs at a time through the wave's patch, so that eight lanes store a line: as 16-byte pieces of 64 lines the
      // stores took the address unit 64 cycles each (8192 tokens, even, 835 -> 814 us; 4096, skewed, level)
      uint32_t ln = lane;
      asm volatile("" : "+v"(ln));  // (opaque: addresses made here instead of held through the stages)
      uint8_t* const patch = smem + 2 * XBUF + wv * 16 * PROW;
      const uint32_t wr = (ln & 15) * PROW + 64 * (ln >> 5), rd = (ln >> 3) * PROW + 16 * (ln & 7);
      const uint32_t low = ln & 16;
      int m = (int)(ln >> 3);
      __half* o = out + (size_t)(tile.first + m) * M + r0 + 8 * (ln & 7);
#pragma unroll
      for (int mf = 0; mf < MF; mf++) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
          if ((low != 0) == (q != 0)) {
#pragma unroll
            for (int f = 0; f < 2; f++)
#pragma unroll
              for (int k = 0; k < 2; k++) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; i++) v[i] = acc[f][mf][8 * k + i];
                *(uint4*)(patch + wr + 32 * f + 16 * k) = pack8(v);
              }
          }
          __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the patch is the wave's own
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int j = 0; j < 2; j++) {
            const uint4 v = *(const uint4*)(patch + rd + 8 * j * PROW);
            if (m < tile.count) *(uint4*)o = v;
            m += 8;
            o += 8 * (size_t)M;
            asm volatile("" : "+v"(m), "+v"(o));
          }
          __builtin_amdgcn_s_waitcnt(0xC07F);
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      return;
    }
#pragma unroll
    for (int mf = 0; mf < MF; mf++) {
      const int m = 32 * mf + n;
      if (m >= tile.count) continue;
      __half* const o = out + (size_t)(tile.first + m) * M + r0 + 16 * h;
#pragma unroll
      for (int k = 0; k < 2; k++) {
        float v[8];
        const float rs = rowscale[m];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const float gv = acc[0][mf][8 * k + i], uv = acc[1][mf][8 * k + i];
          v[i] = gv / (1.f + __expf(-gv)) * uv * rs;
        }
        *(uint4*)(o + 8 * k) = pack8(v);
      }
    }
  };
  // the stages of all passes are one pipeline: a pass ends between two of them
  int p = 0, left = NS;
  auto end = [&]() {
    if (--left) return;
    finish(p++);
    zero();
    left = NS;
  };
  for (int nst = 0;; nst += 2) {
    stage(P0, nst);
    end();
    if (nst + 1 >= total) break;
    stage(P1, nst + 1);
    end();
    if (nst + 2 >= total) break;
  }
}

template <int FMT, bool UP, int LX>
__global__ void __launch_bounds__(256, 2)
k_moe_wide(WideW R, WideW Sh, int n_experts, const __half* __restrict__ x, const int* __restrict__ tokidx,
           const moe_tile* __restrict__ tiles, const int* __restrict__ ntiles, __half* __restrict__ out, int M, int K, int nblk,
           int npass, moe_hscale hs) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // consecutive workgroup ids go round-robin over the XCDs: each takes a contiguous run of tiles (gemm_q4cp.hip).  With no more
  // tiles than XCDs their blocks are dealt out one by one instead: all of a shared expert's on the first XCD, beside the routed
  // experts' launches, slowed that XCD's share of those (512 experts, 3072 x 768 Q5_K / Q8_0, 33 tokens 377 -> 368 us, 96 631 -> 622;
  // 2560 x 640 q4cp with a q8g32 shared expert 33 237 -> 226, 130 380 -> 371; 128 experts, 3072 x 768, 33 253 -> 239.  Up to 31 or 63
  // tiles dealt out: up to 14 % slower, blocks of a tile fetch its activations through every L2)
  const int nt = ntiles[0], per = (nt + 7) >> 3;
  const bool spread = nt <= 8;
  const int xcd = blockIdx.x & 7, j = spread ? blockIdx.x : blockIdx.x >> 3, tl = j / nblk, ti = spread ? tl : xcd * per + tl;
  if ((!spread && tl >= per) || ti >= nt) return;
  const moe_tile tile = tiles[ti];
  const bool shared = tile.expert >= n_experts;
  WideW L;
  L.w = shared ? Sh.w : R.w;
  L.w_up = shared ? Sh.w_up : R.w_up;
  L.sc = shared ? Sh.sc : R.sc;
  const int e = shared ? 0 : tile.expert, nb = (j - tl * nblk) * npass;
  const moe_cmag cmag = shared ? hs.c_shared : hs.c_routed;
  const int mfn = (tile.count + 31) >> 5;
#define WD_GO(MF) wide_tile<FMT, UP, LX, MF>(smem, L, e, tile, nb, npass, x, tokidx, out, M, K, hs, cmag)
  if (mfn <= 1) WD_GO(1);
  else if (mfn == 2) WD_GO(2);
  else if (mfn == 3) WD_GO(3);
  else WD_GO(4);
#undef WD_GO
}

template <int FMT, bool UP, int LX>
int launch(const WideW& R, const WideW& S, int n_experts, const __half* x, const int* tokidx, const moe_tile* tiles, const int* ntiles,
           int max_tiles, __half* out, int m, int k, moe_hscale hs, hipStream_t st) {
  constexpr int LDS = UP ? SMEM : SMEM_DN;
  static moe_dev_once once;
  int dev;
  if (moe_dev_pending(once, &dev)) {
    MOE_HIP(hipFuncSetAttribute((const void*)k_moe_wide<FMT, UP, LX>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS));
    moe_dev_done(once, dev);
  }
  const int rows = UP ? 128 : 256;
  int nblk = (m + rows - 1) / rows, npass = 1;
  // down: a block walks up to three neighbouring groups of rows while that leaves four blocks per CU
  if (!UP)
    for (int w = 2; w <= 3; w++)
      if (nblk % w == 0 && (int64_t)max_tiles * (nblk / w) >= 1024) npass = w;
  nblk /= npass;
  const int per = (max_tiles + 7) / 8;
  k_moe_wide<FMT, UP, LX><<<(unsigned)(per * nblk * 8), 256, LDS, st>>>(R, S, n_experts, x, tokidx, tiles, ntiles, out, m, k, nblk,
                                                                        npass, hs);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

}  // namespace

// The launches of moe_launch_gemm_gg that k_moe_wide takes: every tensor Q8_0 or every tensor q8g32, whole stages of 128
// columns, whole waves of rows.  each: pairs that an expert has on average; alone: the launch is the shared expert's
bool moe_wide_takes(bool up, int type, const uint8_t* w, const uint8_t* w_up, int tsh, const uint8_t* sh_w, const uint8_t* sh_w_up,
                    int m, int k, int a_layout, int n_experts, int max_tiles, int each, bool alone) {
  if (type != MOE_GGML_Q8_0 && type != MOE_T_Q8G32) return false;
  if (sh_w && tsh != type) return false;
  const size_t al = type == MOE_GGML_Q8_0 ? 4 : 16;
  for (const uint8_t* p : {w, up ? w_up : w, sh_w ? sh_w : w, sh_w && up ? sh_w_up : w})
    if (!moe_aligned(p, al)) return false;
  if (k % 128 || m % (up ? 32 : 64)) return false;
  // Q8_0 on few blocks: the launch takes as long as a block does, and the general kernel's have half the rows.  (q8g32: it has no
  // pipelined form for that, a layer takes up to 45 % longer with it and is level at best.)  us of a layer, here and there, Q5_K /
  // Q8_0 with a Q8_0 shared expert:
  //   up to four tiles of more than 64 tokens   3072 x 768 of 16 experts 130 138 125, 300 155 130, 400 163 141, 515 (five) 154 149; of
  //     32 130 150 135, 400 181 161, 700 (six) 214 221; of 64 256 216 190, 700 243 274; of 128 400 340 333, 1000 (eight) 381 397
  //   one tile of at most 64, next to a launch of many weights   3072 x 768 of 64 (151 M) 33 185 167, 64 189 171; 2048 x 1536 of 64 191
  //     185; 2560 x 640 of 64 (105 M) 144 138; of 512 experts level; with fewer weights the shared expert is waited for, and is done
  //     sooner here: 3072 x 768 of 32 (75 M) 48 127 132; 1024 x 768 of 64 93 99
  //   routed gate/up, more than 64 pairs, fewer than 128 blocks   all Q8_0, top-2 of 8, 2560 x 640 1000 tokens 141 120, 4096 x 1024 400
  //     194 187, 700 (152 blocks) 154 162
  if (type == MOE_GGML_Q8_0) {
    if (each <= 64) {
      if (alone && (int64_t)m * k * n_experts >= (int64_t)3 << 25) return false;
    } else if (alone ? max_tiles <= 4 : up && max_tiles * ((m + 127) / 128) < 128) {
      return false;
    }
  }
  return a_layout == 0 || (type == MOE_GGML_Q8_0 && a_layout == 2) || (type == MOE_T_Q8G32 && up && a_layout == 1);
}
int moe_launch_wide(bool up, int type, const uint8_t* w, const uint8_t* w_up, const uint8_t* sh_w, const uint8_t* sh_w_up, int n_experts,
                    const __half* x, const int* tokidx, const moe_tile* tiles, const int* ntiles,
                    int max_tiles, __half* out, int m, int k, moe_hscale hs, hipStream_t st, int a_layout) {
  const uint64_t sc = (uint64_t)m * (uint64_t)k;  // (q8g32 tensors are one expert's)
  const WideW R{w, w_up, sc}, S{sh_w ? sh_w : w, sh_w ? sh_w_up : w_up, sc};
#define WD(F, U, LX) return launch<F, U, LX>(R, S, n_experts, x, tokidx, tiles, ntiles, max_tiles, out, m, k, hs, st)
  if (type == MOE_GGML_Q8_0) {
    if (up && a_layout == 2) WD(W_Q80, true, 2);
    if (up) WD(W_Q80, true, 0);
    if (a_layout == 2) WD(W_Q80, false, 2);
    WD(W_Q80, false, 0);
  }
  if (up && a_layout == 1) WD(W_G32, true, 1);
  if (up) WD(W_G32, true, 0);
  WD(W_G32, false, 0);
#undef WD
}
