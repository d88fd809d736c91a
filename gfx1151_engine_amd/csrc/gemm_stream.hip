// Grouped expert GEMM for tiles of few pairs: the weights stream from memory straight into registers.
// (same contract as gemm_q4cp.hip: src/gpu/parts/27_kernels_moe_lut.inc:660-821, 26_kernels_moe_gguf.inc:456-485)
//
// From a few dozen to about two thousand tokens every expert is read and none has many pairs: what bounds a launch is the
// experts' bytes (1.4 / 0.7 GB per layer for gate/up / down).  gemm_q4cp.hip, made for 128-pair tiles, moves them through
// LDS in 32-byte pieces of 256 rows, two 64-column stages ahead, and reaches 3.5 TB/s of the 6.3 that plain loads reach
// on this chip (a load of 16 rows x 64 bytes per wave instruction, four or more in flight per wave; 32 rows x 32 bytes:
// 4.4 .. 5.3).  Here:
//   - a wave owns 16 weight rows twice (gate/up: 16 gate rows and their 16 up rows; down: 32 rows) and walks K, any multiple of
//     128 (K-quants and i4r: 256), in lines of 256 columns.  v_mfma_f32_16x16x32_f16 takes the weights as A: lane (n, g) = row
//     n, 16-byte chunks g and g + 4 of the line's 128 code bytes, so a load instruction covers 64 contiguous bytes of 16 rows
//     and a chunk is one lane's operand for four MFMAs.  Which columns a lane group multiplies is free as long as the
//     activations agree; a chunk is one scale group of 32 columns (q4cp), half of a 64-column run (Q4_K, Q5_K), a lane group's
//     run (Q8_0).
//   - gate/up keeps two lines per wave in flight, line by line; down requests a fragment's whole rows at once where they are
//     three lines, else two lines at a time.  q4cp rows start 64 bytes off the 128-byte cache lines (the codebook heads the
//     tensor), and what one visit leaves of a cache line is gone from L2 before the next; so whole rows at once brought down
//     from 6.9 to 5.3 M cache lines (of 5.0), and gate/up turns its lines by half a line, the last of a row ending with the row's
//     first 64 bytes (up_rotates).
//   - activations (16 pairs per MFMA, up to 64 per tile) go through LDS: gate/up one line at a time, double-buffered, one
//     LDS-only barrier per line; down, where they are short, once per block, which then runs without barriers.
//   - no branch stands around a load of the loops: the compiler counts outstanding loads exactly only along straight code
//     (with branches every wait drained the pipeline: 332 against 270 us).
// The weights' f16 values are those of gemm_q4cp.hip's form of the same name (scaled, plain, table, K-quant) bit for bit; the sums
// run over the same columns in f32.  Q4_K and Q5_K layers that gemm_q4cp.hip does not take (widths that are no multiples of
// 256) go to the general kernel of gguf_types.hip otherwise, which rounds a weight once, from its exact value; so does
// their form here (F_Q4E, F_Q5E: three instructions for two weights where the packed f16 arithmetic of F_Q4K and F_Q5K, which
// rounds d * sc and dmin * m as well, takes two.  Error of a 2560 x 640 layer's output against fp64 4.9e-4, with the packed
// arithmetic 5.5e-4; 130 / 515 / 1500 tokens 544 / 612 / 796 us, with it 522 / 581 / 760, on the general kernel 1855 / 1968 /
// 2060).
// Pairs per tile: 16, 32 or 64 by the batch's average (moe_stream_tile_cap): a block's work is the weights whatever the
// tile holds, so tiles should hold an expert's pairs as a rule, and larger ones cost LDS and registers.
// Measured (512 experts, top-10, 3072 x 768, gate/up + down, us; in brackets the 128-pair kernels):
//   130 tokens q4cp 240 + 135 (354 + 178)      48 table 175 + 102 (298 + 170)    515 Q4_K 337 + 167 (431 + 234)
//   200 Q5_K / Q8_0 396 + 282 (487 + 357)     200 i4r 266 + 135 (369 + 191)      2048 q4cp 357 + 206 (444 + 239)
// (130 and 48 tokens behind a router launch with a redone logit, of which the chip comes back rested; else 253 + 138 and 195 + 107)
// The layer at other widths (with q4cp and table rows as they lie, see up_rotates: up to 515 tokens 4 .. 10 % more than now), us (128-pair
// kernels in brackets), 48 / 515 / 1200 tokens, d = 3072: mid 256 q4cp 162 / 258 / 331 (207 / 307 /
// 361), Q5_K / Q8_0 214 / 343 / 437 (261 / 409 / 461); 512 q4cp 245 / 401 / 474 (312 / 491 / 549), table 272 / 434 / 535 (392 / 610 / 639),
// Q4_K 257 / 428 / 513 (339 / 544 / 602), i4r 245 / 378 / 467 (318 / 478 / 542); 1024 q4cp 429 / 719 / 827 (520 / 851 / 942), table 471 /
// 781 / 930 (645 / 1074 / 1143); d = 2048: 1536 q4cp 419 / 759 / 891 (518 / 833 / 896), 2048 545 / 969 / 1083 (669 / 1083 / 1148).
#include <type_traits>

#include "common.h"
#include "half.h"
#include "hv2.h"
#include "internal.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// F_DN: affine q4cp codebooks whose experts all have a power of two for the scaled dequantisation (gemm_q4cp.hip, DN)
// F_Q4E, F_Q5E: Q4_K and Q5_K weights rounded to f16 once, from their exact values
// F_I4D: i4r with codes read as denormals and no power of two (gemm_q4cp.hip, DN), layers whose experts all have scales below 2^-4
// (3001 skewed tokens, gate/up 495 -> 474 us, down 271 -> 261; 130: 248 -> 236, 128 -> 124; the weights are F_I4R's bit for bit).
// Q4_K gained half a per cent of a layer with it and Q5_K lost 15 at 1200 tokens, both short of registers.)
enum { F_DN, F_AFF, F_TAB, F_I4R, F_Q4K, F_Q5K, F_Q80, F_Q4E, F_Q5E, F_I4D };
constexpr bool q4(int FMT) { return FMT == F_Q4K || FMT == F_Q4E; }
constexpr bool q5(int FMT) { return FMT == F_Q5K || FMT == F_Q5E; }
constexpr bool i4(int FMT) { return FMT == F_I4D || FMT == F_I4R; }
constexpr bool once_rounded(int FMT) { return FMT == F_Q4E || FMT == F_Q5E; }
constexpr bool scale_plane(int FMT) { return FMT <= F_I4R || FMT == F_I4D; }
// order of activations and hid (moe_f32_to_f16's layouts)
constexpr int x_layout(int FMT) { return FMT == F_TAB ? 0 : scale_plane(FMT) ? 1 : 2; }

constexpr int XROW = 512;  // bytes of a line of one pair row (256 f16)
constexpr size_t LDS_MOST = 160 * 1024;  // of a CU
// copies of a pair table: lanes eight (four) apart share one.  Gate/up: what lets four blocks of up to 32 pairs, two of 64, share
// a CU's LDS, with two tables as well (smem_bytes; 515 tokens, 32 pairs, eight copies and four 346 -> 340 us; 2048, 64 pairs,
// four and eight 324 -> 317; 16 pairs have room for sixteen, which take longer to fill than they save: 197 -> 208); down with
// 64 pairs: four for the registers (246 us with eight copies, 237 with four at 2048 tokens)
constexpr int tab_copies(bool UP, int MFX) { return MFX == 4 ? (UP ? 8 : 4) : UP && MFX == 2 ? 4 : 8; }

struct SW {
  const uint8_t *w, *w_up, *sc, *sc_up;
  const float *cb, *cb_up;
  int sstride, e_rows, up_off;
  const int8_t* pexp;
};

// (v & mask) | bits.  An instruction reads one scalar, and left to itself the compiler makes two instructions of this rather than keep
// `bits` in a register: 64 of the 335 that a line of two Q4_K fragments took.  Layers, us: Q4_K 40 tokens 305.0 -> 300.7, 130 494 489,
// 515 569.6 565.1, 1500 711.5 706.8, 2500 879 875; Q4_K / Q8_0 300 678.7 677.0.  (Not FUSED: down with 64 pairs, which has no
// registers left.)
template <bool FUSED>
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t bits) {
  if (!FUSED) return (v & mask) | bits;
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(bits));
  return r;
}
__device__ __forceinline__ half2v both(float f) { return half2v{(_Float16)f, (_Float16)f}; }

template <int FMT>
__device__ __forceinline__ uint32_t row_bytes(int K) {
  return q4(FMT) ? K / 256 * 144 : q5(FMT) ? K / 256 * 176 : FMT == F_Q80 ? K / 32 * 34 : K / 2;
}
constexpr int line_bytes(int FMT) { return q4(FMT) ? 144 : q5(FMT) ? 176 : FMT == F_Q80 ? 272 : 128; }

// element of a group of 16 NW rows that output position 16 wv + i holds: the order the down launch reads hid in (layout 2
// runs over 64-element blocks, four waves' groups)
template <int LAYOUT>
__device__ __forceinline__ int pos_elem(int wv, int i) {
  if (LAYOUT == 1) return 16 * wv + (i & 8) + (((i & 1) << 2) | ((i & 7) >> 1));
  if (LAYOUT == 2) {
    const int p = 16 * (wv & 3) + i, w = p >> 3, r = p & 7;
    return 64 * (wv >> 2) + 4 * w + ((r & 2) << 4) + ((r & 1) << 1) + (r >> 2);
  }
  return 16 * wv + i;
}

// ---- one line of one weight fragment (16 rows) in registers ----
// SPLIT: a K-quant's header and fifth bits in parts (gather4)
constexpr bool split_head(int MFX) { return MFX < 4; }
template <int FMT, bool SPLIT>
struct Line {
  uint4 c[FMT == F_Q80 ? 4 : 2];  // codes
  typename std::conditional<SPLIT, uint32_t, uint4>::type hd;  // K-quants: word g of the block's header, or all of it
  uint2 qh;                       // Q5_K: half of the fifth bits of lane groups g and g ^ 2
  uint32_t last;                  // Q8_0: the 17th word
};
// b: wave-uniform address of the line's first row, o: this lane's row offset, half: the second half does not exist; second: where
// the codes' second half lies behind the first, 64 bytes as a rule
template <int FMT, bool SPLIT>
__device__ __forceinline__ void load_line(Line<FMT, SPLIT>& q, const uint8_t* b, uint32_t o, int g, bool half, ptrdiff_t second = 64) {
  if constexpr (FMT == F_Q80) {
    // lane group g = columns 64 g .. of the line: two blocks, 68 bytes (4-byte aligned)
    const uint8_t* s = b + (o + 68u * (half ? (uint32_t)(g & 1) : (uint32_t)g));
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t* d = (const uint32_t*)(s + 16 * k);
      q.c[k] = make_uint4(d[0], d[1], d[2], d[3]);
    }
    q.last = *(const uint32_t*)(s + 64);
  } else {
    constexpr uint32_t C0 = q4(FMT) ? 16 : q5(FMT) ? 48 : 0;
    if constexpr (q4(FMT) || q5(FMT)) q.hd = *(const decltype(q.hd)*)(b + (o + (SPLIT ? 4u * (uint32_t)g : 0u)));
    if (q5(FMT)) q.qh = *(const uint2*)(b + (o + 16u + 16u * (uint32_t)(g & 1) + 8u * (uint32_t)(g >> 1)));
    q.c[0] = *(const uint4*)(b + (o + C0 + 16u * (uint32_t)g));
    const uint8_t* b1 = b + (half ? 0 : second);
    q.c[1] = *(const uint4*)(b1 + (o + C0 + 16u * (uint32_t)g));
  }
}

// A K-quant's header and fifth bits are the same for all (two) lane groups of a row, and a load costs the address unit 64 cycles
// for 16 bytes of every lane, 16 for 4: each group fetches its part, and these hand the others' over.  us of the layer, whole and in
// parts: Q4_K 130 tokens 490 487, 515 573.5 570; Q5_K / Q8_0 300 768 763, 800 844 830, 1300 954 937, 2560 x 640 3000 1147 1127.  (Tiles of
// 64 pairs, Q4_K, where the vector port counts for more: 1300 tokens 694 698, 2500 898 901; they fetch it whole.)
// word g of lane group g -> all four words
__device__ __forceinline__ uint4 gather4(uint32_t v) {
  const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  const auto a = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false), b = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
  return make_uint4(a[0], b[0], a[1], b[1]);
}
// words 2 (g / 2), 2 (g / 2) + 1 of lane groups g and g ^ 2 -> all four
__device__ __forceinline__ uint4 gather2(uint2 v) {
  const auto a = __builtin_amdgcn_permlane32_swap(v.x, v.x, false, false), b = __builtin_amdgcn_permlane32_swap(v.y, v.y, false, false);
  return make_uint4(a[0], b[0], a[1], b[1]);
}

// What dequantisation needs beside the codes: per fragment the codebook's slope and offset or its pair table
struct Consts {
  float cb_a[2], cb_b[2];
  const uint8_t* tabs;  // LDS
  uint32_t tabo[2];
  uint32_t selb;        // K-quants: this lane's two sub-blocks of four
  int g;
};

// acc[f][mf] += line of fragment f x the line's activations.  f0: fragment 0's index into the constants; sw: this lane's two
// scales of the line (scale planes); xb: the activations' line in LDS; xa: this lane's operand addresses of four steps
// (Q8_0: eight)
// FUSED: and_or as one instruction
template <int FMT, int F, int MF, int XP, int TABC, bool FUSED = true, bool SPLIT>
__device__ __forceinline__ void line_mma(const Line<FMT, SPLIT> (&q)[F], const uint32_t (&sw)[F], const Consts& C, int f0,
                                         const uint8_t* xb, const uint32_t* xa, bool half, floatx4 (&acc)[F][MF]) {
  auto mma = [&](uint32_t xo, const H8 (&w)[F]) {
#pragma unroll
    for (int mf = 0; mf < MF; mf++) {
      const half8 xf = *(const half8*)(xb + xo + 16 * mf * XP);
#pragma unroll
      for (int f = 0; f < F; f++) acc[f][mf] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[f].v, xf, acc[f][mf], 0, 0, 0);
    }
  };
  if constexpr (FMT == F_Q80) {
    half2v sc[F][2];
    uint32_t cw[F][16];
#pragma unroll
    for (int f = 0; f < F; f++) {
      const uint32_t w[17] = {q[f].c[0].x, q[f].c[0].y, q[f].c[0].z, q[f].c[0].w, q[f].c[1].x, q[f].c[1].y, q[f].c[1].z, q[f].c[1].w,
                              q[f].c[2].x, q[f].c[2].y, q[f].c[2].z, q[f].c[2].w, q[f].c[3].x, q[f].c[3].y, q[f].c[3].z, q[f].c[3].w,
                              q[f].last};
      // bytes 0-1 the first block's scale, 2-33 its codes, 34-35 the second's scale, 36-67 its codes
      sc[f][0] = h2(__builtin_amdgcn_perm(w[0], w[0], 0x01000100u));
      sc[f][1] = h2(__builtin_amdgcn_perm(w[8], w[8], 0x03020302u));
#pragma unroll
      for (int k = 0; k < 8; k++) {
        cw[f][k] = __builtin_amdgcn_alignbyte(w[k + 1], w[k], 2) ^ 0x80808080u;
        cw[f][8 + k] = w[9 + k] ^ 0x80808080u;
      }
      if (half && C.g >= 2) {  // (runs past K)
        sc[f][0] = sc[f][1] = both(0.f);
      }
    }
    // layout 2: chunk w of a run = columns 4w, 4w+2, 32+4w, 32+4w+2, 4w+1, 4w+3, 32+4w+1, 32+4w+3
    const half2v k1152 = both(1152.f);  // 1024 + u with u = code + 128
#pragma unroll
    for (int w = 0; w < 8; w++) {
      H8 a[F];
#pragma unroll
      for (int f = 0; f < F; f++) {
        const uint32_t lo = cw[f][w], hi = cw[f][8 + w];
        a[f].h[0] = (h2(__builtin_amdgcn_perm(0x64646464u, lo, 0x04020400u)) - k1152) * sc[f][0];
        a[f].h[1] = (h2(__builtin_amdgcn_perm(0x64646464u, hi, 0x04020400u)) - k1152) * sc[f][1];
        a[f].h[2] = (h2(__builtin_amdgcn_perm(0x64646464u, lo, 0x04030401u)) - k1152) * sc[f][0];
        a[f].h[3] = (h2(__builtin_amdgcn_perm(0x64646464u, hi, 0x04030401u)) - k1152) * sc[f][1];
      }
      mma(xa[w], a);
    }
    return;
  } else {
    uint4 head[F], fifth[F];
    if constexpr (q4(FMT) || q5(FMT)) {
#pragma unroll
      for (int f = 0; f < F; f++) {
        if constexpr (SPLIT) head[f] = gather4(q[f].hd);
        else head[f] = q[f].hd;
        if (q5(FMT)) fifth[f] = gather2(q[f].qh);
      }
    }
    auto part = [&](auto ec) {
      constexpr int E_ = decltype(ec)::value;
      half2v as[F][2], bs[F][2];
      float ka[F][2], kb[F][2];
      constexpr bool ONCE = once_rounded(FMT);
#pragma unroll
      for (int f = 0; f < F; f++) {
        if (q4(FMT) || q5(FMT)) {
          // 6-bit (scale, min) fields of sub-blocks 0-3 (E_ = 0) or 4-7 as bytes, gguf scale_min_k4
          const uint4 hd = head[f];
          const uint32_t sc = E_ ? (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u) : hd.y & 0x3f3f3f3fu;
          const uint32_t mn = E_ ? ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3f3f3f3fu;
          const half2v k1024 = both(1024.f);
          const half2v s2 = h2(__builtin_amdgcn_perm(0x64646464u, sc, C.selb)) - k1024;
          const half2v m2 = h2(__builtin_amdgcn_perm(0x64646464u, mn, C.selb)) - k1024;
          if (ONCE) {
            // (codes are read as denormals, below: n 2^-24, Q4_K's high ones n 2^-20.  d * sc, dmin * m and n times the slope are exact in
            // f32, so that the addition alone rounds.  With codes as 1024 + n and 1024 times the slope in the constant 0.8 .. 1.6 % of the
            // weights were not the nearest f16, and 2560 x 640 of Q5_K / Q8_0 took 1100 us at 3000 tokens, now 1072; level below 1000)
            const half2v dd = h2(hd.x);
            ka[f][0] = (float)s2.x * ((float)dd.x * 0x1p24f);
            ka[f][1] = (float)s2.y * ((float)dd.x * (q5(FMT) ? 0x1p24f : 0x1p20f));
            kb[f][0] = -((float)m2.x * (float)dd.y);
            kb[f][1] = -((float)m2.y * (float)dd.y);
          } else {  // d * sc and dmin * m as packed f16 products of exact integers
            const half2v dd = h2(__builtin_amdgcn_perm(hd.x, hd.x, 0x01000100u));
            const half2v dm = h2(__builtin_amdgcn_perm(hd.x, hd.x, 0x03020302u) ^ 0x80008000u);
            const half2v a = s2 * dd, b = m2 * dm;
            as[f][0] = half2v{a.x, a.x}; as[f][1] = half2v{a.y, a.y};
            bs[f][0] = half2v{b.x, b.x}; bs[f][1] = half2v{b.y, b.y};
          }
        } else {
          const half2v s2 = h2(__builtin_amdgcn_perm(sw[f], sw[f], E_ ? 0x03020302u : 0x01000100u));
          if (FMT == F_TAB) {
            as[f][0] = s2;
          } else {
            const float s = (float)s2.x;
            as[f][0] = both(C.cb_a[f0 + f] * s);
            bs[f][0] = bs[f][1] = FMT == F_I4D ? as[f][0] * both(-0x1p-17f) : both(C.cb_b[f0 + f] * s);  // (i4r: -8 * s, exact)
            as[f][1] = FMT == F_DN ? as[f][0] * both(0.0625f) : as[f][0];
          }
        }
      }
#pragma unroll
      for (int s = 0; s < 4; s++) {
        H8 a[F];
#pragma unroll
        for (int f = 0; f < F; f++) {
          const uint4 cq = q[f].c[E_];
          const uint32_t w = s == 0 ? cq.x : s == 1 ? cq.y : s == 2 ? cq.z : cq.w;
          if (FMT == F_TAB) {
            // one look-up gives a code byte's two weights before scaling
#pragma unroll
            for (int b = 0; b < 4; b++)
              a[f].h[b] = h2(*(const uint32_t*)(C.tabs + (((w >> (8 * b)) & 0xffu) * (4u * TABC) + C.tabo[f0 + f]))) * as[f][0];
            continue;
          }
          const uint32_t w8 = w >> 8;
          if (FMT == F_I4D) {  // codes read as f16 denormals, n * 2^-20
            a[f].h[0] = h2((w << 4) & 0x00f000f0u) * as[f][0] + bs[f][0];
            a[f].h[1] = h2(w & 0x00f000f0u) * as[f][0] + bs[f][0];
            a[f].h[2] = h2((w >> 4) & 0x00f000f0u) * as[f][0] + bs[f][0];
            a[f].h[3] = h2(w8 & 0x00f000f0u) * as[f][0] + bs[f][0];
          } else if (FMT == F_DN) {  // n * 2^-24, n * 2^-20
            a[f].h[0] = h2(w & 0x000f000fu) * as[f][0] + bs[f][0];
            a[f].h[1] = h2(w & 0x00f000f0u) * as[f][1] + bs[f][0];
            a[f].h[2] = h2(w8 & 0x000f000fu) * as[f][0] + bs[f][0];
            a[f].h[3] = h2(w8 & 0x00f000f0u) * as[f][1] + bs[f][0];
          } else {  // 0x6400 | n is the f16 1024 + n, 0x5400 | n << 4 is 64 + n; ONCE: n by itself is the denormal n 2^-24
            constexpr float HI = q5(FMT) ? 1024.f : 64.f;
            uint32_t t0, t1, t2, t3;
            if (q5(FMT)) {
              // fifth bits: bit 2 jj (low nibbles) and 2 jj + 1 (high) of the qh byte, jj = g / 2 + 2 E_, rotated to bit 4 of the
              // codes' bytes; two bytes are a pair of 1024 + n: 19 operations for eight weights where bits put into the four pairs
              // of the other formats' form took 22.  Q5_K / Q8_0 layers, us: 40 tokens 422 -> 415, 130 693 -> 680, 300 754 -> 742, 1400
              // 953 -> 941
              const uint4 qq = fifth[f];
              const uint32_t qw = s == 0 ? qq.x : s == 1 ? qq.y : s == 2 ? qq.z : qq.w;
              const uint32_t lo = (w & 0x0f0f0f0fu) | (__builtin_amdgcn_alignbit(qw, qw, (uint32_t)((C.g & 2) + 4 * E_ + 28) & 31u) & 0x10101010u);
              const uint32_t hi = ((w >> 4) & 0x0f0f0f0fu) | (__builtin_amdgcn_alignbit(qw, qw, (uint32_t)((C.g & 2) + 4 * E_ + 29) & 31u) & 0x10101010u);
              // (selector 0x0c is a byte of zeros)
              t0 = __builtin_amdgcn_perm(0x64646464u, lo, ONCE ? 0x0c020c00u : 0x04020400u);
              t1 = __builtin_amdgcn_perm(0x64646464u, hi, ONCE ? 0x0c020c00u : 0x04020400u);
              t2 = __builtin_amdgcn_perm(0x64646464u, lo, ONCE ? 0x0c030c01u : 0x04030401u);
              t3 = __builtin_amdgcn_perm(0x64646464u, hi, ONCE ? 0x0c030c01u : 0x04030401u);
            } else if (ONCE) {
              t0 = w & 0x000f000fu; t1 = w & 0x00f000f0u;
              t2 = w8 & 0x000f000fu; t3 = w8 & 0x00f000f0u;
            } else {
              t0 = and_or<FUSED>(w, 0x000f000fu, 0x64006400u); t1 = and_or<FUSED>(w, 0x00f000f0u, 0x54005400u);
              t2 = and_or<FUSED>(w8, 0x000f000fu, 0x64006400u); t3 = and_or<FUSED>(w8, 0x00f000f0u, 0x54005400u);
            }
            if (ONCE) {
              auto once = [&](uint32_t t, int i) {
                const half2v n = h2(t);
                return half2v{(_Float16)fmaf((float)n.x, ka[f][i], kb[f][i]), (_Float16)fmaf((float)n.y, ka[f][i], kb[f][i])};
              };
              a[f].h[0] = once(t0, 0);
              a[f].h[1] = once(t1, 1);
              a[f].h[2] = once(t2, 0);
              a[f].h[3] = once(t3, 1);
              continue;
            }
            const half2v k1024 = both(1024.f), khi = both(HI);
            a[f].h[0] = (h2(t0) - k1024) * as[f][0] + bs[f][0];
            a[f].h[1] = (h2(t1) - khi) * as[f][1] + bs[f][1];
            a[f].h[2] = (h2(t2) - k1024) * as[f][0] + bs[f][0];
            a[f].h[3] = (h2(t3) - khi) * as[f][1] + bs[f][1];
          }
        }
        mma(xa[s] + E_ * 256, a);
      }
    };
    part(std::integral_constant<int, 0>{});
    if (!half) part(std::integral_constant<int, 1>{});
  }
}

// ---- half a line (128 columns) of F q4cp fragments ----
// slopes and offsets of half E_'s scale
template <int F>
struct Deq {
  half2v as[F][2], bs[F];
};
template <int FMT, int F, int E_>
__device__ __forceinline__ Deq<F> make_deq(const uint32_t (&sw)[F], const Consts& C) {
  static_assert(FMT == F_DN || FMT == F_AFF || FMT == F_TAB, "");
  Deq<F> D;
#pragma unroll
  for (int f = 0; f < F; f++) {
    const half2v s2 = h2(__builtin_amdgcn_perm(sw[f], sw[f], E_ ? 0x03020302u : 0x01000100u));
    if (FMT == F_TAB) {
      D.as[f][0] = s2;
    } else {
      const float s = (float)s2.x;
      D.as[f][0] = both(C.cb_a[f] * s);
      D.bs[f] = both(C.cb_b[f] * s);
      D.as[f][1] = FMT == F_DN ? D.as[f][0] * both(0.0625f) : D.as[f][0];
    }
  }
  return D;
}

// acc[f][mf] += half line E_ of fragment f x the line's activations (line_mma's arguments and its sums, in its order).
// A step's MFMAs run while the next step's operands are made: every (step, 16 pairs) is an item of F MFMAs, one activation
// operand is read two items ahead, and the next step's weights are dequantised in equal parts next to the step's items.
// The fences keep that order: left alone the compiler reads every activation operand into the same four registers and
// waits a trip through LDS for each, and puts a step's dequantisation into one clump (a SIMD takes eight 16x16x32 MFMAs and 32
// vector operations in 199 cycles side by side, in 219 clump behind clump).
template <int FMT, int F, int MF, int XP, int TABC, int E_>
__device__ __forceinline__ void half_mma(const uint4 (&c)[F], const Deq<F>& D, const Consts& C, const uint8_t* xb, const uint32_t* xa,
                                         floatx4 (&acc)[F][MF]) {
  constexpr int N = 4 * MF, AHEAD = 2;
  half8 xf[AHEAD + 1];
  auto ldx = [&](int t) { xf[t % (AHEAD + 1)] = *(const half8*)(xb + xa[t / MF] + E_ * 256 + 16 * (t % MF) * XP); };
  H8 a[2][F];
  uint32_t lut[4 * F];
  auto look = [&](int s) {  // table codebooks: the two weights of every code byte before scaling
#pragma unroll
    for (int u = 0; u < 4 * F; u++)
      lut[u] = *(const uint32_t*)(C.tabs + (((word(c[u >> 2], s) >> (8 * (u & 3))) & 0xffu) * (4u * TABC) + C.tabo[u >> 2]));
  };
  auto unit = [&](int s, int u) {  // a pair of step s's weights (line_mma's forms)
    const int f = u >> 2, b = u & 3, i = b & 1;
    H8& o = a[s & 1][f];
    if constexpr (FMT == F_TAB) {
      o.h[b] = h2(lut[u]) * D.as[f][0];
    } else {
      const uint32_t w = word(c[f], s), n = (b & 2 ? w >> 8 : w) & (i ? 0x00f000f0u : 0x000f000fu);
      if constexpr (FMT == F_DN) o.h[b] = h2(n) * D.as[f][i] + D.bs[f];
      else o.h[b] = (h2(and_or<true>(b & 2 ? w >> 8 : w, i ? 0x00f000f0u : 0x000f000fu, i ? 0x54005400u : 0x64006400u)) -
                     both(i ? 64.f : 1024.f)) * D.as[f][i] + D.bs[f];
    }
  };
#pragma unroll
  for (int t = 0; t < AHEAD; t++) ldx(t);
  if constexpr (FMT == F_TAB) look(0);
#pragma unroll
  for (int u = 0; u < 4 * F; u++) unit(0, u);
#pragma unroll
  for (int t = 0; t < N; t++) {
    const int st = t / MF, mf = t % MF;
    if constexpr (FMT == F_TAB) {
      if (mf == 0 && st < 3) look(st + 1);
    }
    if (t + AHEAD < N) ldx(t + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < F; f++) {
      acc[f][mf] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[st & 1][f].v, xf[t % (AHEAD + 1)], acc[f][mf], 0, 0, 0);
      if (st < 3) {
        const int slot = F * mf + f;
#pragma unroll
        for (int u = slot * 4 / MF; u < (slot + 1) * 4 / MF; u++) unit(st + 1, u);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Scales of four lines of a row (64 bytes, i4r: 16) from line `first` on: lane group i fetches line first + i's, the exchange
// below then hands every lane one word per line with its own two scales.  (Past the row's end: one address for all lanes.)
// ro: bytes of codes by which the lines are rotated (up_tile); last: the line whose second half is then the row's first 64 bytes
template <int FMT>
struct Raw { uint4 v; };
template <int FMT>
__device__ __forceinline__ Raw<FMT> load_scales(const uint8_t* b, uint32_t o, int first, int g, int sstride, uint32_t ro = 0, int last = -1) {
  Raw<FMT> r;
  if (i4(FMT)) {  // one word per line: both scales, the same for all lane groups
    const uint32_t p = 4u * (uint32_t)(first + g);
    r.v.x = *(const uint32_t*)(b + (p < (uint32_t)sstride ? o + p : 0u));
  } else if (last < 0) {
    const uint32_t p = 16u * (uint32_t)(first + g);
    r.v = *(const uint4*)(b + (p < (uint32_t)sstride ? o + p : 0u));
  } else {
    const uint32_t p = 16u * (uint32_t)(first + g) + (ro >> 3), p1 = ro && first + g == last ? 0u : p + 8u;
    const bool past = first + g > last;
    const uint2 u = *(const uint2*)(b + (past ? 0u : o + p)), v = *(const uint2*)(b + (past ? 0u : o + p1));
    r.v = make_uint4(u.x, u.y, v.x, v.y);
  }
  return r;
}
template <int FMT>
__device__ __forceinline__ void take_scales(const Raw<FMT>& r, uint32_t (&sq)[4]) {
  uint32_t p0 = r.v.x, p1 = p0, p2 = p0, p3 = p0;
  if (!i4(FMT)) {  // word k: (scale k, scale 4 + k), lane group k's chunks k and k + 4
    p0 = __builtin_amdgcn_perm(r.v.z, r.v.x, 0x05040100u); p1 = __builtin_amdgcn_perm(r.v.z, r.v.x, 0x07060302u);
    p2 = __builtin_amdgcn_perm(r.v.w, r.v.y, 0x05040100u); p3 = __builtin_amdgcn_perm(r.v.w, r.v.y, 0x07060302u);
  }
  // 4 x 4 transposition between lane groups and words
  auto a = __builtin_amdgcn_permlane32_swap(p0, p2, false, false);
  auto b = __builtin_amdgcn_permlane32_swap(p1, p3, false, false);
  auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  sq[0] = c[0]; sq[1] = c[1]; sq[2] = d[0]; sq[3] = d[1];
}

// Pair tables: a thread's entry of each, as f32.  Requested before the first weights -- loads come back in order -- and written
// (make_consts) when the activations are, four copies at a time.  Entries that were fetched one copy at a time behind the
// weights kept a block from its first line: 48 tokens, gate/up 215 -> 196 and down 115 -> 105 us one by one, the layer, whose
// launches overlap less, 353.5 -> 350.5; 300 tokens of 2560 x 640 418 -> 411, 515 599 -> 589.
struct TabEntry {
  float lo[2], hi[2];
};
template <int NT, int TABC>
constexpr int tab_pieces() { return 64 * TABC > NT ? 64 * TABC / NT : 1; }  // 16-byte pieces (four copies) of a thread
template <int NT, int TABC>
__device__ __forceinline__ int tab_index(int tid) { return tid * tab_pieces<NT, TABC>() / (TABC / 4); }
template <int FMT, bool UP, int NT, int TABC>
__device__ __forceinline__ TabEntry load_entry(const SW& L, int tid) {
  TabEntry t{};
  if (FMT == F_TAB) {
    static_assert(tab_pieces<NT, TABC>() <= TABC / 4, "one entry per thread");
    const int b = tab_index<NT, TABC>(tid) & 255;
    t.lo[0] = L.cb[b & 15]; t.hi[0] = L.cb[b >> 4];
    if (UP) { t.lo[1] = L.cb_up[b & 15]; t.hi[1] = L.cb_up[b >> 4]; }
  }
  return t;
}
template <int FMT, bool UP, int NT, int TABC>
__device__ __forceinline__ Consts make_consts(const SW& L, int pexp, const TabEntry& te, uint8_t* tabs, int tid, float& oscale) {
  Consts C;
  C.g = (tid & 63) >> 4;
  C.selb = (C.g & 2) ? 0x04030402u : 0x04010400u;
  C.cb_a[0] = C.cb_a[1] = 1.f;
  C.cb_b[0] = C.cb_b[1] = -8.f;  // (i4r)
  C.tabs = tabs;
  C.tabo[0] = C.tabo[1] = 0u;
  oscale = 1.f;
  if (FMT == F_I4D) {
    C.cb_a[0] = C.cb_a[1] = 0x1p20f;
  } else if (FMT == F_AFF || FMT == F_DN) {
    C.cb_a[0] = L.cb[1] - L.cb[0]; C.cb_b[0] = L.cb[0];
    C.cb_a[1] = UP ? L.cb_up[1] - L.cb_up[0] : C.cb_a[0]; C.cb_b[1] = UP ? L.cb_up[0] : C.cb_b[0];
    if (FMT == F_DN) {  // in units of 2^pexp; slopes for codes read as f16 denormals
      const float s24 = __builtin_ldexpf(1.f, 24 + pexp), sp = __builtin_ldexpf(1.f, pexp);
      C.cb_a[0] *= s24; C.cb_a[1] *= s24; C.cb_b[0] *= sp; C.cb_b[1] *= sp;
      oscale = __builtin_ldexpf(1.f, -pexp);
      // (the same in every lane: as scalars they leave the down launches of 64 pairs their registers.  The layer, us: 2048 tokens q4cp 701
      // 696, 3001 skewed i4r 882 871)
      auto scalar = [](float& f) { f = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(f))); };
      scalar(C.cb_a[0]); scalar(C.cb_a[1]); scalar(C.cb_b[0]); scalar(C.cb_b[1]); scalar(oscale);
    }
  } else if (FMT == F_TAB) {
    // TABC copies side by side: lanes that differ in their low bits never meet on a bank (with one copy the look-ups of a
    // wave run into 3.5-way conflicts on average)
    const bool two = UP && L.cb_up != L.cb;
    constexpr int PT = tab_pieces<NT, TABC>();
    if (64 * TABC >= NT || tid < 64 * TABC) {
#pragma unroll
      for (int t = 0; t < 2; t++) {
        if (t && !two) break;
        const uint32_t v = u2(half2v{(_Float16)te.lo[t], (_Float16)te.hi[t]});
#pragma unroll
        for (int i = 0; i < PT; i++) ((uint4*)tabs)[64 * TABC * t + PT * tid + i] = make_uint4(v, v, v, v);
      }
    }
    C.tabo[0] = (uint32_t)(tid & (TABC - 1)) * 4u;
    C.tabo[1] = C.tabo[0] + (two ? 256u * TABC * 4u : 0u);
  }
  return C;
}

// Where a pair row's line has its 16-byte chunk c (16 e + 4 g + q: lane group g's step q of half e; Q8_0: 8 g + q) in LDS: the
// bits of q above those of g, the low four XORed with the row.  A 128-bit read goes through the 64 banks sixteen lanes at
// a time, lanes 0-3, 12-15 and 20-27 first: rows 4-11 come from the next lane group there, so a group bit may not meet the
// rows' bits 2 and 3 (with chunks in order, g at bit 2, every read took twice as long).
template <int FMT>
__device__ __forceinline__ int x_slot(int c, int row) {
  const int lo = FMT == F_Q80 ? ((c & 7) << 1) | ((c >> 3) & 1) : ((c & 3) << 2) | ((c >> 2) & 3);
  return (c & 16) | (lo ^ (row & 15));
}
// this lane's operand address of step q of pair row n
template <int FMT, int XP>
__device__ __forceinline__ void x_addrs(int n, int g, uint32_t (&xa)[8]) {
#pragma unroll
  for (int q = 0; q < 8; q++) xa[q] = (uint32_t)(n * XP + (x_slot<FMT>((FMT == F_Q80 ? 8 : 4) * g + q, n) << 4));
}

// ---- gate/up ----
// HALVES (64 pairs of q4cp codes): the codes go through registers in half lines, the next line's activations in two parts, and
// half_mma orders the rest.  Else whole lines, one ahead of the line worked on, in the compiler's order.  What either is
// bound by with 64 pairs is traffic first: 16.6 M cache lines for the 10.6 M that 2048 tokens' gate/up rows and scales have (q4cp; rows are
// visited a line, their scales four lines at a time), 345 us of 386 at the 6.15 TB/s that plain loads reach; half lines need 15.2 M.  us of the launch, whole lines and
// halves: 2048 tokens q4cp 386 371, table 483 432; but 515 q4cp (32 pairs) 312 320, 1500 Q4_K 404 425, 2048 i4r 401 406.
// Tried beside it: a row's scales all at once (registers: spills at 64 pairs), non-temporal loads (21 M cache lines), 32 gate and 32 up rows to
// a wave with two waves per SIMD (half the LDS reads, +12 us), and x in registers with the waves of a block splitting K, which
// reads 9.8 M cache lines for 9.75 M at 130 tokens but leaves two waves per SIMD whose arithmetic does not hide (280 us for 268).
// (Straight code of two lines, where K is known to be whole pairs of lines, gave the compiler room to move loads and operands
// further and cost 20 us of 390 at 64 pairs (spills: up to 150): the branches around half and last lines stay.)
constexpr bool up_halves(int FMT, int MFX) { return MFX == 4 && FMT <= F_TAB; }
// Bytes of LDS for the tile's row scales.  None beside two pair tables: those and the activations fill half of a CU's LDS (64
// pairs) or a quarter (32) to the byte, so the epilogue reads the scales' sources again.  us of the layer, table codebook with a
// shared expert of its own tables, 64 experts, top-8, with the scales behind them (one block fewer per CU) and without: 3072 x 768
// 100 tokens (32 pairs) 128.3 126.6, 200 (64 pairs) 143.0 135.7, 256 146.4 140.7; 2560 x 640 200 123.5 116.2.  With one table there
// is room, and reading again costs: 200 tokens without a shared expert 126.6 127.9
constexpr size_t up_scales(int FMT, int tabs) { return FMT == F_TAB && tabs == 2 ? 0 : 256; }
// Tiles of 16 and 32 pairs of q4cp codes: lines that begin where the cache lines do, where the rows of both tensors start in the
// middle of one (up_tile's ro; activations and scales follow), and the scales of twelve (eight) lines requested together.
// 130 tokens, gate/up: 13.3 M cache lines of 128 bytes for 9.8 M -> 9.9 M, 282 -> 265 us; the lines alone 262, of the scales alone 253.
// us of the layer, before and after: q4cp 40 tokens 283 266, 130 457 429, 515 540 509, 800 585 560, 2560 x 640 200 362 330; table 40 313
// 301, 515 588 562.  Not for tiles of 64, whose half lines come half a stage apart: 1200 tokens 623 -> 635, 2048 706 -> 711; nor
// is there room for more scales (32 pairs, twelve lines' instead of eight: up to 9 registers in scratch, 515 tokens 512).
constexpr bool up_rotates(int FMT, int MFX) { return FMT <= F_TAB && MFX < 4; }
constexpr int up_scale_groups(int FMT, int MFX) { return FMT > F_TAB || MFX == 4 ? 1 : MFX == 2 ? 2 : 3; }
template <int FMT, int MFX, int MF, bool ROT, int NW>
__device__ __forceinline__ void up_tile(uint8_t* smem, const SW& L, int e, const moe_tile tile, int nb, const __half* __restrict__ x,
                                        const int* __restrict__ tokidx, __half* __restrict__ out, int M, int K, int pexp,
                                        const moe_hscale& hs, moe_cmag cmag, const moe_rotv& rot, bool two_tabs) {
  constexpr int LAYOUT = x_layout(FMT), LB = line_bytes(FMT), NT = 64 * NW, UPR = 16 * NW;
  constexpr int XBUF = MFX * 16 * XROW;
  constexpr bool HALVES = up_halves(FMT, MFX);
  constexpr int DB = HALVES ? 1 : 2;  // lines of codes in registers
  float* const rowscale = (float*)(smem + 2 * XBUF);
  const bool scales = !(FMT == F_TAB && two_tabs);  // (up_scales)
  uint8_t* const tabs = smem + 2 * XBUF + up_scales(FMT, scales ? 1 : 2);
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const uint32_t RB = row_bytes<FMT>(K);
  const int nline = (K + 255) >> 8;
  const bool tail = (K & 128) != 0;  // the last line is half a line

  int r = nb * UPR + pos_elem<LAYOUT>(wv, n);
  r = r < M ? r : M - 1;  // (loaded, never stored)
  const uint8_t* wb[2];   // wave-uniform: the expert's gate and up rows
  const uint8_t* sb[2];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const size_t first = (size_t)e * L.e_rows + (f ? L.up_off : 0);
    wb[f] = (f ? L.w_up : L.w) + first * RB;
    sb[f] = scale_plane(FMT) ? (f ? L.sc_up : L.sc) + first * (size_t)L.sstride : nullptr;
  }
  const uint32_t wo = (uint32_t)r * RB, so = (uint32_t)r * (uint32_t)L.sstride;
  const uint32_t ro = up_rotates(FMT, MFX) && (K & 255) == 0 && ((uintptr_t)wb[0] & 127) == 64 && ((uintptr_t)wb[1] & 127) == 64 ? 64u : 0u;
  typedef Line<FMT, split_head(MFX)> Ln;
  Ln ln[HALVES ? 1 : DB][2];
  uint4 cd[HALVES ? DB : 1][2][2];  // line, half, fragment
  // (past the last line: one address for all lanes instead of a branch around the load)
  auto load = [&](Ln(&q)[2], int i) {
#pragma unroll
    for (int f = 0; f < 2; f++) {
      const bool past = i >= nline;
      load_line(q[f], wb[f] + (past ? (size_t)0 : (size_t)i * LB + ro), past ? 0u : wo, past ? 0 : g, tail && i >= nline - 1,
                     ro && i == nline - 1 ? (ptrdiff_t)64 - (ptrdiff_t)RB : (ptrdiff_t)64);
    }
  };
  auto load_half = [&](uint4(&q)[2], int i, int E) {
    const bool past = i >= nline;
    const size_t at = past ? (size_t)0 : (size_t)i * LB + (E && !(tail && i == nline - 1) ? 64 : 0);
#pragma unroll
    for (int f = 0; f < 2; f++) q[f] = *(const uint4*)(wb[f] + at + (past ? 0u : wo + 16u * (uint32_t)g));
  };
  // ---- the pipeline's first requests.  Loads come back in order: the tile's row indices, which the activations' addresses wait
  // for, go ahead of the weights (after them 0.4 .. 0.7 % slower with both timed in turn -- 130 tokens i4r 436.5 433.5 us, 300 Q5_K 770 766,
  // 515 Q4_K 578 575.5 --, little more than two runs differ) ----
  constexpr int XL = MF * 16 * 32 / NT, XS = NT / 32;  // loads per thread and line, rows per load
  constexpr int XH = HALVES ? (XL + 1) / 2 : XL;       // loads of a part of the line
  static_assert(XL >= 1 && XL * NT == MF * 16 * 32 && XH <= 4, "whole loads, named registers below");
  const int xc = tid & 31, xt = tid >> 5;
  int xrow[XL];
  auto load_rows = [&]() {
#pragma unroll
    for (int l = 0; l < XL; l++) {
      const int m = XS * l + xt;
      xrow[l] = tokidx[tile.first + (m < tile.count ? m : 0)];
    }
  };
  if constexpr (MFX < 4) {
    load_rows();
    __builtin_amdgcn_sched_barrier(0);
  }
  TabEntry te;
  if constexpr (MFX < 4) te = load_entry<FMT, true, NT, tab_copies(true, MFX)>(L, tid);
  constexpr int SD = up_scale_groups(FMT, MFX);  // groups of four lines whose scales are in registers
  Raw<FMT> raw[2][SD];
  uint32_t sq[2][4];
  auto scales_of = [&](int f, int i) { return load_scales<FMT>(sb[f], so, i, g, L.sstride, ro, up_rotates(FMT, MFX) ? nline - 1 : -1); };
  if (scale_plane(FMT)) {
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int k = 0; k < SD; k++) raw[f][k] = scales_of(f, 4 * k);
  }
#pragma unroll
  for (int b = 0; b < DB; b++) {
    if constexpr (HALVES) {
      load_half(cd[b][0], b, 0);
      load_half(cd[b][1], b, 1);
    } else {
      load(ln[b], b);
    }
  }
  // ---- activations: thread = 16-byte chunk tid % 32 of pair rows tid / 32 + (NT / 32) l ----
  // (rows past the tile's pairs repeat its first one: no branch around a load, and the lines are in L1)
  uint32_t xr[XL];  // (32-bit byte offsets: moe_launch_stream)
  if constexpr (MFX == 4) load_rows();  // (no registers for them any earlier)
#pragma unroll
  for (int l = 0; l < XL; l++) {
    const int m = XS * l + xt;
    const int row = xrow[l];
    xr[l] = ((uint32_t)row * (uint32_t)K + 8u * (uint32_t)xc) * 2u;
    if (scales && xc == 0) rowscale[m] = hs.xms ? moe_hid_scale(cmag, hs.xms[row]) : 1.f;
  }
  uint4 xv0, xv1, xv2, xv3;  // (named: an array here ends up in scratch memory)
  auto fetch_x = [&](int i, auto part) {
    constexpr int h = XH * decltype(part)::value;
    i = i < nline ? i : nline - 1;
    // (the last line: half of it repeated where the row has none, the row's first columns where the lines are rotated)
    const bool end = i == nline - 1 && xc >= 16;
    const uint8_t* const xb = (const uint8_t*)x + (up_rotates(FMT, MFX) ? (size_t)0 : 512 * (size_t)i);
    const uint32_t at = up_rotates(FMT, MFX) ? 512u * (uint32_t)i + 4u * ro - (!end ? 0u : tail ? 256u : ro ? 2u * (uint32_t)K : 0u)
                                             : end && tail ? 0u - 256u : 0u;
    if constexpr (h < XL) xv0 = *(const uint4*)(xb + (xr[h] + at));
    if constexpr (XH > 1 && h + 1 < XL) xv1 = *(const uint4*)(xb + (xr[h + 1] + at));
    if constexpr (XH > 2 && h + 2 < XL) xv2 = *(const uint4*)(xb + (xr[h + 2] + at));
    if constexpr (XH > 3 && h + 3 < XL) xv3 = *(const uint4*)(xb + (xr[h + 3] + at));
  };
  auto put_x = [&](int buf, auto part) {
    constexpr int h = XH * decltype(part)::value;
    auto put = [&](int l, const uint4& v) {
      const int m = XS * l + xt;
      *(uint4*)(smem + buf * XBUF + m * XROW + (x_slot<FMT>(xc, m) << 4)) = v;
    };
    if constexpr (h < XL) put(h, xv0);
    if constexpr (XH > 1 && h + 1 < XL) put(h + 1, xv1);
    if constexpr (XH > 2 && h + 2 < XL) put(h + 2, xv2);
    if constexpr (XH > 3 && h + 3 < XL) put(h + 3, xv3);
  };
  constexpr std::integral_constant<int, 0> P0{};
  constexpr std::integral_constant<int, 1> P1{};
  fetch_x(0, P0);
  if constexpr (HALVES) {
    put_x(0, P0);
    fetch_x(0, P1);
  }
  float oscale;
  if constexpr (MFX == 4) te = load_entry<FMT, true, NT, tab_copies(true, MFX)>(L, tid);  // (no registers for it any earlier)
  const Consts C = make_consts<FMT, true, NT, tab_copies(true, MFX)>(L, pexp, te, tabs, tid, oscale);
  uint32_t xa[8];
  x_addrs<FMT, XROW>(n, g, xa);
  floatx4 acc[2][MF];
#pragma unroll
  for (int f = 0; f < 2; f++)
#pragma unroll
    for (int mf = 0; mf < MF; mf++) acc[f][mf] = floatx4{0.f, 0.f, 0.f, 0.f};
  if constexpr (HALVES) put_x(0, P1);
  else put_x(0, P0);

  // stage V (mod 4): line i
  auto stage = [&](auto vc, int i) {
    constexpr int V = decltype(vc)::value, B = V & 1, S = V % DB;
    moe_lds_barrier();  // this line's activations are in LDS; the other buffer has been read
    fetch_x(i + 1, P0);
    if constexpr (HALVES) {
      __builtin_amdgcn_sched_barrier(0);
      if (V == 0) {
#pragma unroll
        for (int f = 0; f < 2; f++) take_scales<FMT>(raw[f][0], sq[f]);
      }
      const uint32_t sw[2] = {sq[0][V], sq[1][V]};
      half_mma<FMT, 2, MF, XROW, tab_copies(true, MFX), 0>(cd[S][0], make_deq<FMT, 2, 0>(sw, C), C, smem + B * XBUF, xa, acc);
      const Deq<2> d1 = make_deq<FMT, 2, 1>(sw, C);
      put_x(B ^ 1, P0);
      fetch_x(i + 1, P1);
      load_half(cd[S][0], i + DB, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (!(tail && i == nline - 1))
        half_mma<FMT, 2, MF, XROW, tab_copies(true, MFX), 1>(cd[S][1], d1, C, smem + B * XBUF, xa, acc);
      __builtin_amdgcn_sched_barrier(0);
      put_x(B ^ 1, P1);
      load_half(cd[S][1], i + DB, 1);
      if (V == 2) {  // (the next four lines')
#pragma unroll
        for (int f = 0; f < 2; f++) raw[f][0] = scales_of(f, i + 2);
      }
      __builtin_amdgcn_sched_barrier(0);
    } else {
      const uint32_t sw[2] = {sq[0][V], sq[1][V]};
      line_mma<FMT, 2, MF, XROW, tab_copies(true, MFX)>(ln[S], sw, C, 0, smem + B * XBUF, xa, tail && i == nline - 1, acc);
      load(ln[S], i + DB);
      put_x(B ^ 1, P0);
    }
  };
  for (int i = 0;; i += 4) {
    if (scale_plane(FMT) && !HALVES) {
#pragma unroll
      for (int f = 0; f < 2; f++) {
        take_scales<FMT>(raw[f][0], sq[f]);
#pragma unroll
        for (int k = 0; k + 1 < SD; k++) raw[f][k] = raw[f][k + 1];
        raw[f][SD - 1] = scales_of(f, i + 4 * SD);
      }
    }
    stage(std::integral_constant<int, 0>{}, i);
    if (i + 1 >= nline) break;
    stage(std::integral_constant<int, 1>{}, i + 1);
    if (i + 2 >= nline) break;
    stage(std::integral_constant<int, 2>{}, i + 2);
    if (i + 3 >= nline) break;
    stage(std::integral_constant<int, 3>{}, i + 3);
    if (i + 4 >= nline) break;
  }

  if constexpr (ROT) {
    // hgn v2: the slot-wise middle on the block's 128 gate and 128 up sums of every pair (gemm_q4cp.hip, ROT)
    static_assert(UPR == 128, "whole 128-blocks");
    constexpr int BP = 2 * UPR * 2 + 16;
    static_assert(MFX * 16 * BP <= 2 * XBUF, "the row scales stay");
    moe_lds_barrier();
    uint8_t* const patch = smem;  // (over the activations, which every wave has read)
#pragma unroll
    for (int mf = 0; mf < MF; mf++)
#pragma unroll
      for (int f = 0; f < 2; f++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
          const int c = pos_elem<LAYOUT>(wv, 4 * g + r4);
          *(__half*)(patch + (16 * mf + n) * BP + f * UPR * 2 + c * 2) = __float2half(acc[f][mf][r4]);
        }
    __syncthreads();
    const int j = tid & 15, c = nb * UPR + 8 * j;
    float fg[8], fu[8], sd[8];
    {
      const int cc = c < M ? c : 0;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        fg[k] = rot.svh_gu[cc + k];
        fu[k] = rot.svh_gu[M + cc + k];
        sd[k] = rot.suh_dn[cc + k];
      }
    }
    for (int m = tid >> 4; m < 16 * MF; m += NT / 16) {
      const uint4 gq = *(const uint4*)(patch + m * BP + j * 16), uq = *(const uint4*)(patch + m * BP + UPR * 2 + j * 16);
      const __half2* gh = (const __half2*)&gq;
      const __half2* uh = (const __half2*)&uq;
      float gv8[8], uv8[8], hv[8];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const float2 a = __half22float2(gh[k]), b = __half22float2(uh[k]);
        gv8[2 * k] = a.x; gv8[2 * k + 1] = a.y; uv8[2 * k] = b.x; uv8[2 * k + 1] = b.y;
      }
      moe_fwht128_r8(gv8, lane);
      moe_fwht128_r8(uv8, lane);
      const float rs = rowscale[m];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const float gg = gv8[k] * MOE_RS128 * fg[k], uu = uv8[k] * MOE_RS128 * fu[k];
        hv[k] = gg * __builtin_amdgcn_rcpf(1.f + __expf(-gg)) * uu * (sd[k] * rs);
      }
      moe_fwht128_r8(hv, lane);
#pragma unroll
      for (int k = 0; k < 8; k++) hv[k] *= MOE_RS128;
      if (m < tile.count && c < M) moe_st8_f16_ilv(out + (size_t)(tile.first + m) * M + c, hv);
    }
  } else {
    const int col = nb * UPR + 16 * wv + 4 * g;
    float rsv[MF];
#pragma unroll
    for (int mf = 0; mf < MF; mf++) {
      const int m = 16 * mf + n;
      if (scales) rsv[mf] = rowscale[m];
      else rsv[mf] = hs.xms ? hs.xms[tokidx[tile.first + (m < tile.count ? m : 0)]] : 0.f;
    }
#pragma unroll
    for (int mf = 0; mf < MF; mf++) {
      const int m = 16 * mf + n;
      if (m < tile.count && col < M) {
        const float rs = scales ? rsv[mf] : hs.xms ? moe_hid_scale(cmag, rsv[mf]) : 1.f;
        float h4[4];
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
          const float gv = acc[0][mf][r4] * oscale, uv = acc[1][mf][r4] * oscale;
          h4[r4] = gv * __builtin_amdgcn_rcpf(1.f + __expf(-gv)) * uv * rs;
        }
        const __half2 a = __floats2half2_rn(h4[0], h4[1]), b = __floats2half2_rn(h4[2], h4[3]);
        *(uint2*)(out + (size_t)(tile.first + m) * M + col) = make_uint2(*(const uint32_t*)&a, *(const uint32_t*)&b);
      }
    }
  }
}

// ---- down.  The tile's hid rows lie in LDS for the whole block (ONE: row by row, else line by line: strides the compiler knows);
// a wave takes 32 rows at a time, a piece of LN
// lines of both fragments in registers, and requests a fragment's next piece as soon as this one is used up; no barrier after
// the first.  Rows of three lines are one piece (ONE: neighbouring rows then share their boundary cache lines as well); rows of
// any other length go two lines at a time. ----
template <int FMT, int MFX, int MF, int NW, int LN, bool ONE>
__device__ __forceinline__ void dn_tile(uint8_t* smem, const SW& L, int e, const moe_tile tile, int nb, int npass,
                                        const __half* __restrict__ x, __half* __restrict__ out, int M, int K, int pexp) {
  constexpr int LB = line_bytes(FMT), NT = 64 * NW, DNR = 32 * NW, XP = ONE ? LN * XROW : XROW, XLINE = ONE ? XROW : MFX * 16 * XROW;
  const int nline = ONE ? LN : (K + 255) >> 8, np = ONE ? 1 : (nline + LN - 1) / LN;
  uint8_t* const tabs = smem + nline * MFX * 16 * XROW;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const uint32_t RB = row_bytes<FMT>(K);
  const bool tail = (K & 128) != 0;
  const uint8_t* const wb = L.w + (size_t)e * L.e_rows * RB;
  const uint8_t* const sb = scale_plane(FMT) ? L.sc + (size_t)e * L.e_rows * (size_t)L.sstride : nullptr;
  // fragment f, MFMA row i = weight row 8 (i / 4) + 4 f + i % 4 of the wave's 32: a lane's eight results are neighbours
  typedef Line<FMT, split_head(MFX)> Ln;
  Ln ln[2][LN];
  Raw<FMT> raw[2];
  auto first_row = [&](int p) {
    const int r = (nb + p) * DNR + 32 * wv;
    return r < M ? r : M - 32;  // (loaded, never stored)
  };
  // fragment f, pass p, piece q (past the end: the last rows again)
  auto load = [&](int f, int p, int q) {
    const int row0 = first_row(p < npass ? p : npass - 1);
    const int r = 8 * (n >> 2) + 4 * f + (n & 3);
    if (scale_plane(FMT)) raw[f] = load_scales<FMT>(sb + (size_t)row0 * L.sstride, (uint32_t)r * (uint32_t)L.sstride, q * LN, g, L.sstride);
#pragma unroll
    for (int i = 0; i < LN; i++) {
      const int l = ONE || q * LN + i < nline ? q * LN + i : nline - 1;
      load_line(ln[f][i], wb + ((size_t)row0 * RB + l * LB), (uint32_t)r * RB, g, tail && l == nline - 1);
    }
  };
  TabEntry te;
  if constexpr (MFX < 4) te = load_entry<FMT, false, NT, tab_copies(false, MFX)>(L, tid);
  load(0, 0, 0);
  load(1, 0, 0);
  for (int l = 0; l < nline; l++)
    for (int c = tid; c < 16 * MF * 32; c += NT) {
      const int m = c >> 5, k = 32 * l + (c & 31);
      const int kk = 8 * k < K ? k : 0;  // (a half line's second half: never multiplied)
      const uint4 v = *(const uint4*)(x + (size_t)(tile.first + (m < tile.count ? m : 0)) * K + 8 * kk);
      *(uint4*)(smem + l * XLINE + m * XP + (x_slot<FMT>(c & 31, m) << 4)) = v;
    }
  float oscale;
  if constexpr (MFX == 4) te = load_entry<FMT, false, NT, tab_copies(false, MFX)>(L, tid);
  const Consts C = make_consts<FMT, false, NT, tab_copies(false, MFX)>(L, pexp, te, tabs, tid, oscale);
  uint32_t xa[8];
  x_addrs<FMT, XP>(n, g, xa);
  moe_lds_barrier();
  for (int p = 0; p < npass; p++) {
    floatx4 acc[2][MF];
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int mf = 0; mf < MF; mf++) acc[f][mf] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < np; q++) {
      const int pn = q + 1 < np ? p : p + 1, qn = q + 1 < np ? q + 1 : 0;  // the piece after this one
      if constexpr (MFX < 4) {
#pragma unroll
        for (int f = 0; f < 2; f++) {
          asm volatile("" ::: "memory");  // (the activations are the same for all rows: hoisted out of the loop they would fill the registers)
          uint32_t sq[4] = {0u, 0u, 0u, 0u};
          if (scale_plane(FMT)) take_scales<FMT>(raw[f], sq);
          floatx4 a1[1][MF];
#pragma unroll
          for (int mf = 0; mf < MF; mf++) a1[0][mf] = acc[f][mf];
#pragma unroll
          for (int i = 0; i < LN; i++) {
            const int l = q * LN + i;
            if (!ONE && l >= nline) break;
            const Ln q1[1] = {ln[f][i]};
            const uint32_t sw[1] = {sq[i]};
            line_mma<FMT, 1, MF, XP, tab_copies(false, MFX)>(q1, sw, C, 0, smem + l * XLINE, xa, tail && l == nline - 1, a1);
          }
#pragma unroll
          for (int mf = 0; mf < MF; mf++) acc[f][mf] = a1[0][mf];
          load(f, pn, qn);
        }
      } else {  // (64 pairs: both fragments share an activation operand's trip out of LDS)
        asm volatile("" ::: "memory");
        uint32_t sq[2][4];
        if (scale_plane(FMT)) {
#pragma unroll
          for (int f = 0; f < 2; f++) take_scales<FMT>(raw[f], sq[f]);
        }
#pragma unroll
        for (int i = 0; i < LN; i++) {
          const int l = q * LN + i;
          if (!ONE && l >= nline) break;
          const Ln q2[2] = {ln[0][i], ln[1][i]};
          const uint32_t sw[2] = {sq[0][i], sq[1][i]};
          line_mma<FMT, 2, MF, XP, tab_copies(false, MFX), false>(q2, sw, C, 0, smem + l * XLINE, xa, tail && l == nline - 1, acc);
        }
        load(0, pn, qn);
        load(1, pn, qn);
      }
    }
    const int row0 = (nb + p) * DNR + 32 * wv, col = row0 + 8 * g;
#pragma unroll
    for (int mf = 0; mf < MF; mf++) {
      const int m = 16 * mf + n;
      if (m < tile.count && row0 < M) {
        uint4 o;
        __half2 h[4];
#pragma unroll
        for (int k = 0; k < 4; k++) h[k] = __floats2half2_rn(oscale * acc[k >> 1][mf][2 * (k & 1)], oscale * acc[k >> 1][mf][2 * (k & 1) + 1]);
        o.x = *(uint32_t*)&h[0]; o.y = *(uint32_t*)&h[1]; o.z = *(uint32_t*)&h[2]; o.w = *(uint32_t*)&h[3];
        *(uint4*)(out + (size_t)(tile.first + m) * M + col) = o;
      }
    }
  }
}

// Waves of a block.  Four: several blocks to a CU pass their prologues, barriers and epilogues independently.  Eight for
// rotated experts' gate/up, whose epilogue works on 128 rows; more as well where a tile's activations leave a CU's LDS to one or
// two blocks (64 pairs: gate/up eight, down sixteen; down with 32 pairs and rows of more than four lines: sixteen, Q8_0 with its
// registers eight.  us of a layer with
// four, eight and sixteen there, q4cp, 2048 x 1536: 130 tokens 585, 620, 621, with 32 pairs to a tile 515 tokens 779, 749, 740, 800
// 880, 805, 792; 3072 x 512: 515 tokens 401, 404, 435).
constexpr int DN_ONE = 3;  // lines of the rows that a wave takes whole
constexpr int up_waves(int FMT, int MFX) { return MFX == 4 || i4(FMT) ? 8 : 4; }
// waves per SIMD asked for: what the registers of the lines in flight leave.  (Gate/up with Q5_K rounded once, 32 pairs: three; with
// four 21 registers went to scratch inside the loop, 757 us for 702 at 1200 tokens of 2560 x 640.  One kernel keeps four
// registers of its prologue in scratch until the epilogue: down F_TAB with 64 pairs.  F_Q5K with 32 and three waves is no faster: 808 us
// for 799 at 515 tokens, 1159 for 1152 at 1700.)
constexpr int simd_waves(int FMT, bool UP, int MFX, int NW) {
  if (UP) return FMT == F_Q5E && MFX == 2 ? 3 : 4;
  return NW == 16 ? 4 : FMT == F_Q80 || FMT == F_Q4K ? 3 : 4;
}
// tabs: pair tables (gate/up: two where an up tensor has a codebook of its own)
constexpr size_t smem_bytes(int FMT, bool UP, int MFX, int nline, int tabs) {
  const size_t tab = FMT == F_TAB ? (size_t)tabs * 256 * tab_copies(UP, MFX) * 4 : 0;
  return UP ? (size_t)2 * MFX * 16 * XROW + up_scales(FMT, tabs) + tab : (size_t)MFX * 16 * XROW * nline + tab;
}
// (gate/up keeps with two tables the blocks that a CU has with one)
static_assert(2 * smem_bytes(F_TAB, true, 4, 0, 2) <= LDS_MOST && 4 * smem_bytes(F_TAB, true, 2, 0, 2) <= LDS_MOST &&
              4 * smem_bytes(F_TAB, true, 1, 0, 2) <= LDS_MOST, "blocks per CU");

// LN: lines of a piece (down)
template <int FMT, bool UP, int MFX, int LN, int NW>
__global__ void __launch_bounds__(64 * NW, simd_waves(FMT, UP, MFX, NW))
k_moe_stream(SW R, SW Sh, int n_experts, const __half* __restrict__ x, const int* __restrict__ tokidx,
             const moe_tile* __restrict__ tiles, const int* __restrict__ ntiles, __half* __restrict__ out, int M, int K,
             int nblk_n, int split, int npass, moe_hscale hs, moe_rotv rot) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // XCD-aware order as in gemm_q4cp.hip: consecutive workgroup ids go round-robin over the XCDs; each takes a contiguous
  // run of tiles, routed and shared ones dealt separately
  const int nt = ntiles[0], nr = split ? ntiles[1] : nt;
  const int wg = blockIdx.x, xcd = wg & 7, j = wg >> 3;
  const int per_r = (nr + 7) >> 3, per_s = (nt - nr + 7) >> 3;
  const int tl = j / nblk_n, nb = (j - tl * nblk_n) * npass;
  int ti;
  if (tl < per_r) {
    ti = xcd * per_r + tl;
    if (ti >= nr) return;
  } else {
    const int k2 = tl - per_r;
    ti = nr + xcd * per_s + k2;
    if (k2 >= per_s || ti >= nt) return;
  }
  const moe_tile tile = tiles[ti];
  const bool shared = tile.expert >= n_experts;
  SW L;
  L.w = shared ? Sh.w : R.w;
  L.w_up = shared ? Sh.w_up : R.w_up;
  L.sc = shared ? Sh.sc : R.sc;
  L.sc_up = shared ? Sh.sc_up : R.sc_up;
  L.cb = shared ? Sh.cb : R.cb;
  L.cb_up = shared ? Sh.cb_up : R.cb_up;
  L.sstride = shared ? Sh.sstride : R.sstride;
  L.e_rows = shared ? Sh.e_rows : R.e_rows;
  L.up_off = shared ? Sh.up_off : R.up_off;
  L.pexp = shared ? Sh.pexp : R.pexp;
  const int e = shared ? 0 : tile.expert;
  const int pexp = FMT == F_DN ? (int)L.pexp[e] : 0;
  const moe_cmag cmag = shared ? hs.c_shared : hs.c_routed;
  const int mfn = (tile.count + 15) >> 4;
  const bool two_tabs = R.cb != R.cb_up || Sh.cb != Sh.cb_up;  // (launch)
#define ST_GO(MF)                                                                                              \
  do {                                                                                                         \
    if constexpr (UP) up_tile<FMT, MFX, MF, i4(FMT), NW>(smem, L, e, tile, nb, x, tokidx, out, M, K, pexp, hs, cmag, rot, two_tabs); \
    else dn_tile<FMT, MFX, MF, NW, LN, LN == DN_ONE>(smem, L, e, tile, nb, npass, x, out, M, K, pexp);                           \
  } while (0)
  // (33 .. 48 pairs as three groups instead of four: 2048 tokens q4cp, 755 -> 720 us a layer)
  if (MFX == 1 || mfn <= 1) ST_GO(1);
  else if (MFX == 2 || mfn <= 2) ST_GO(2);
  else if constexpr (MFX > 2) {
    if (mfn <= 3) ST_GO(3);
    else ST_GO(4);
  }
#undef ST_GO
}

SW to_dev(const moe_lutw* p, const float* cb_up, const int8_t* pexp) {
  SW d{};
  d.pexp = pexp;
  if (p) {
    d.w = p->w; d.w_up = p->w_up; d.sc = p->sc; d.sc_up = p->sc_up; d.cb = p->cb;
    d.cb_up = cb_up ? cb_up : p->cb;
    d.sstride = p->sstride; d.e_rows = p->e_rows; d.up_off = p->up_off;
  }
  return d;
}

template <int FMT, bool UP, int MFX, int LN, int NW>
int launch(const SW& R, const SW& S, int n_experts, const __half* x, const int* tokidx, const moe_tile* tiles,
           const int* ntiles, int max_tiles, __half* out, int m, int k, int split, moe_hscale hs, const moe_rotv* rot,
           hipStream_t st) {
  const size_t lds = smem_bytes(FMT, UP, MFX, (k + 255) / 256, UP && (R.cb != R.cb_up || S.cb != S.cb_up) ? 2 : 1);
  static moe_dev_once once;
  int dev;
  if (moe_dev_pending(once, &dev)) {
    MOE_HIP(hipFuncSetAttribute((const void*)k_moe_stream<FMT, UP, MFX, LN, NW>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(LN == 0 || LN == DN_ONE ? (UP ? smem_bytes(FMT, UP, MFX, 0, 2) : lds) : LDS_MOST)));
    moe_dev_done(once, dev);
  }
  int nblk = UP ? (m + 16 * NW - 1) / (16 * NW) : (m + 32 * NW - 1) / (32 * NW), npass = 1;
  // Down: a block walks several groups of rows behind one staging of the activations; the longest walk that leaves ten blocks
  // per CU, Q8_0 rows eight (64 pairs: two.  Staging is most of a short walk there: 2048 tokens i4r 205 us, with six blocks 223, with
  // twelve 300).  That is of the tile list's places, all that the host knows: it has one for every expert, so that with a pair to an
  // expert a third of them, and of the ten blocks, have nothing to do, and with half a pair three in five.  With these instead of twelve
  // throughout, us of the layer: 512 experts Q5_K / Q8_0 48 tokens 452 -> 441, 100 615 602, 300 743 737, 800 818 805, 2560 x 640 60 399 377; q4cp
  // 2560 x 640 60 239 235, 3072 x 768 300 486 486; Q4_K 300 543 540.  192 experts Q5_K / Q8_0 62 353 314, 2560 x 640 (four slots) 273 280 256, q4cp (eight
  // slots) 49 193 180; 256 experts table 2048 x 768 (eight) 464 281 259, Q4_K / Q8_0 2048 x 768 87 298 264; 128 experts q4cp 128 168 155, Q4_K 250
  // 214 200; with 16 to 64 experts a block has one group of rows either way.  With eight for all, whose longer walks end raggedly where tiles
  // are few, from ten: 512 experts q4cp 48 282 280 but 36 247 248, 52 295 298, 300 486 491; Q4_K 48 317 315 but 40 290 292; 1000 experts q4cp and Q4_K 33
  // 270 276, 303 312
  constexpr int LEAVE = MFX == 4 ? 512 : FMT == F_Q80 ? 2048 : 2560;
  if (!UP)
    for (int c = 1; c <= nblk; c++)
      if (nblk % c == 0 && (int64_t)max_tiles * (nblk / c) >= LEAVE) npass = c;
  nblk /= npass;
  const int per_xcd = (max_tiles + 7) / 8 + 1;
  k_moe_stream<FMT, UP, MFX, LN, NW><<<(unsigned)(per_xcd * nblk * 8), 64 * NW, lds, st>>>(
      R, S, n_experts, x, tokidx, tiles, ntiles, out, m, k, nblk, split, npass, hs, rot ? *rot : moe_rotv{nullptr, nullptr});
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

}  // namespace

// Pairs per tile for a batch of P tokens, 0 = the batch belongs to the 128-pair kernels.
// An expert's pairs spread by about the root of their mean, so tiles of 16 and 32 hold nearly all experts in one up to averages of 10
// and 22; 64-pair tiles at an average of 25 against 32-pair ones: 797 -> 779 us per layer (q4cp), 740 -> 738 (i4r).  Above, more
// and more experts take a second tile and the 128-pair kernels draw level; the line lies where they do, for each kind of
// layer with its own kernels, at even and at Zipf-skewed routing.  Layers, us, 128-pair kernels and these (3072 x 768):
//   average pairs        51, even / skewed            56, table 60               62, table 66           66, table 70
//   q4cp                 889 819 / 921 834            914 850 / 959 870          961 923 / 1013 927     996 1006 / 1050 953
//   Q4_K                 966 927 / 1012 950           1005 995 / 1062 982 (55)   1043 1053 / 1115 1058
//   i4r                  866 794 / 896 824            890 841 / 933 862          952 918 / 999 921      986 995 / 1032 951
//   table                                             1142 1021 / 1193 1043      1194 1163 / 1262 1102  1239 1234 / 1300 1182
// (i4r's line was found while its weights took an instruction more on either side, and lies a few pairs short of that.)
// That is of layers whose weights are many.  With fewer the 128-pair kernels draw level earlier: a launch is then one or two rounds
// of blocks, and a second tile of some experts is a round more.  d x mid x experts tells the layers apart better than either
// width or the number of experts does.  q4cp, even / skewed, averages of 50, 56 and 62 (change against the 128-pair kernels, %):
//   3072 x 768 of 384 (906 M)  -9 / -11, -8, 0 / -6      of 256 (604 M)  -7 / -8, -6, -3 / -7       of 128 (302 M)  -6 / -6, 0, +1 / -2
//   4096 x 1024 of 128 (537 M) -6 / -9, -3, -1 / -4      2048 x 1024 of 256 (537 M) -3 / -4, -2, +2 / -3
//   1024 x 512 of 1000 (524 M) -3 / -4, -3, 0 / -3       2048 x 768 of 256 (403 M)  0 / -4, 0, +2 / -4
//   1024 x 768 of 512 (403 M)  0 / -5, +1, +3 / -1       3072 x 768 of 64 (151 M)   +9 / -1, +10, +15 / -3
// (i4r, even / skewed, 46, 50, 56 and 62: of 256 -8 / -6, -4 / -6, -3 / -5, 0 / -7; of 128 -6 / -8, -6 / -10, -5 / -10, +3 / -6.  Q4_K 1 .. 2 % less
// throughout; table codebooks 2048 x 768 of 256 at 62 and 70 -3, 0, 3072 x 768 of 256 -3, +2.)  The
// line between many and few lies between 403 and 524 M.
constexpr int64_t MANY_WEIGHTS = (int64_t)7 << 26;
// Q8_0 down rows beside Q4_K or Q5_K: the 128-pair kernels are k_moe_wide's, 32-pair tiles are the largest here.  Averages of 25, 28, 31
// and 34, %, Q4_K | Q5_K gate/up: 3072 x 768 of 512 -9 -6 -1 +3 | (29) -3, (33) +5; of 384 -9 -5 -1 +3 | -7 -2 +2 +7; of 256 -11
// -7 -2 0 | -9 -4 +1 +3; of 192 (453 M) -13 -9 -4 -3 | -10 -6 -1 -1; 2048 x 768 of 512 -8 -4 0 +4 | -4 -1 +5 +8; of 256 (403 M) -6 -3
// +3 +5 | -3 0 +6 +10; 4096 x 1024 of 256 -8 -4 -1 +4 | -5 0 +2 +7; skewed, 28: -3 .. -10 | +2 .. -7.  With fewer weights, 22, 25, 28
// and 31: 3072 x 768 of 128 0 +1 +1 +8 | -1 +2 +2 +9; of 64 +1 +1 +1 +4 | +2 +4 +2 +7; 2048 x 768 of 128 (201 M) +2 +1 +6 +8 | +2 +1
// +7 +10; 1024 x 512 of 128 (67 M) -1 -3 -2 +3 | +3 -1 +1 +6; 4096 x 1024 of 32 +1 +1 +1 +5 | +5 +4 +2 +5.  Below 34 M the two are
// level at any average up to 38 (16 .. 64 experts of 512 x 256 .. 1024 x 768: 75 .. 95 us either way), and the line lies where
// it did with slower 128-pair kernels.
// Rows of more than four lines of hid (mid > 1024) leave no LDS for 64 pairs: 32-pair tiles as well, level earlier (2048 x 1536 of 512, even /
// skewed: q4cp 23 882 869 / 920 909, 25 891 877 / 922 933, 27 899 908 / 940 962, 29 914 959 / 953 982; 2048 x 2048 of 256 25 608 587 / 636 623, 27
// 613 594 / 643 639, 29 628 635 / 644 656; Q4_K 23 956 895 / 1010 986, 25 963 926 / 1012 1012, 27 978 963 / 1027 1047; table 29 1149 1054 / 1210
// 1113, 33 1212 1188 / 1260 1207, 37 1263 1312 / 1280 1295: its line was found before tiles of 32 turned their lines (1149 1139 at 29, 1248 1409
// at 37) and lies short of where both are level now).  Beside Q8_0, averages of 23,
// 26, 29 and 32, Q4_K | Q5_K: 512 experts -5 -4 +2 +6 | -2 0 +6 +11; 128 0 +2 +9 +11 | +2 +5 +12 +16; 64 -4 -5 -3 +1 | -1 -1 +1 +9;
// 16 -7 -4 +1 +5 | -8 -5 -4 +2.
// (Q5_K with Q4_K down rows: 25, 28 and 31 3072 x 768 of 512 -7 -6 +1, of 256 -9 -5 0, 2048 x 768 of 256 -4 0 +8, 3072 x 768 of 64 -1 +1
// +13: the same lines.)
// Layers that go to the general kernel otherwise (F_Q4E, F_Q5E): as far as was measured (2560 x 640 of 512, Q5_K / Q8_0: 60 1912 1273; 100
// 2220 1869 / 2541 1863; 160 3676 2688; Q4_K / Q8_0: 100 2154 1646 / 2464 1636; 160 3562 2390; of 64, Q5_K: 60 367 236, 160 578 413; of
// 16: 179 126, 198 169).
constexpr float ONCE_LINE = 160.f;
int moe_stream_tile_cap(int P, int k, int experts, int fmt_up, int fmt_dn, int d, int mid) {
  const float avg = (float)P * (float)k / (float)experts;
  const int64_t weights = (int64_t)d * mid * experts;
  const bool small = q5(fmt_up) || fmt_dn == F_Q80, lone = mid > 1024, big = weights >= MANY_WEIGHTS, five = q5(fmt_up);
  float line;
  if (once_rounded(fmt_up)) line = ONCE_LINE;
  else if (small && lone) line = !five ? 28.f : experts >= 64 ? 26.f : 32.f;
  else if (small && weights >= (int64_t)3 << 27) line = five ? 29.f : 31.f;
  else if (small && weights >= 1 << 25) line = five ? 22.f : 26.f;
  else if (small) line = five && experts >= 64 ? 31.f : 38.f;
  else if (fmt_up == F_TAB) line = lone ? 29.f : big ? 70.f : 60.f;
  else line = lone ? 25.f : !big ? 50.f : fmt_up == F_DN || fmt_up == F_AFF ? 62.f : 60.f;
  if (avg <= 10.f) return 16;
  return avg > line ? 0 : small || lone || avg <= 22.f ? 32 : 64;
}
// The smallest that any layer takes (0 above the last line): what the tile list is sized for.
int moe_stream_tile_cap_least(int P, int k, int experts) {
  const float avg = (float)P * (float)k / (float)experts;
  return avg <= 10.f ? 16 : avg <= ONCE_LINE ? 32 : 0;
}

// fmt: MOE_STREAM_*; the views as for moe_launch_gemm_q4cp; x_rows: rows of x.  max_tiles == 0: checks only.
int moe_launch_stream(int fmt, bool up, int cap, const moe_lutw* routed, const moe_lutw* sh, int n_experts, const __half* x, int x_rows,
                      const int* tokidx, const moe_tile* tiles, const int* ntiles, int max_tiles, __half* out, int m, int k,
                      moe_hscale hs, hipStream_t st, const float* sh_cb_up, const int8_t* pexp_routed,
                      const int8_t* pexp_sh, const moe_rotv* rot) {
  if (!x || !tiles || !ntiles || !out || max_tiles < 0 || !routed || (up && !tokidx)) return MOE_E_INVALID;
  const bool plane = scale_plane(fmt);
  auto ok = [&](const moe_lutw* p) {
    if (!p->w || (up && !p->w_up)) return false;
    if (!moe_aligned(p->w, fmt == F_Q80 ? 4 : 16) || (up && !moe_aligned(p->w_up, 16))) return false;
    if (plane) {
      const int a = i4(fmt) ? 4 : 16;
      if (!p->sc || !p->cb || !moe_aligned(p->sc, a) || p->sstride % a || p->sstride < k / (i4(fmt) ? 128 : 32) * 2) return false;
      if (up && (!p->sc_up || !moe_aligned(p->sc_up, a))) return false;
    }
    return true;
  };
  if (!ok(routed) || (sh && !ok(sh))) return MOE_E_UNSUPPORTED;
  if (k % 128 || ((q4(fmt) || q5(fmt) || i4(fmt)) && k % 256)) return MOE_E_UNSUPPORTED;
  // (down: groups of 32 rows, and a tile's hid rows in LDS)
  if (up && (uint64_t)x_rows * (uint64_t)k * 2 >= 1ull << 32) return MOE_E_UNSUPPORTED;  // (32-bit byte offsets into x)
  if (up ? k < 256 : k < 128 || m % 32 || smem_bytes(fmt, false, cap / 16, (k + 255) / 256, 1) > LDS_MOST) return MOE_E_UNSUPPORTED;
  if (up && (m % 16 || (!plane && m % 64) || (i4(fmt) && m % 128))) return MOE_E_UNSUPPORTED;
  if ((up && fmt == F_Q80) || (!up && (q5(fmt) || once_rounded(fmt))) || (cap > 32 && (q5(fmt) || fmt == F_Q80))) return MOE_E_UNSUPPORTED;
  if (i4(fmt) && up != (rot != nullptr)) return MOE_E_INVALID;
  if (rot && (!rot->svh_gu || !rot->suh_dn)) return MOE_E_INVALID;
  if (fmt == F_DN && (!pexp_routed || (sh && !pexp_sh))) return MOE_E_INVALID;
  if (!moe_aligned(x, 16) || !moe_aligned(out, 16)) return MOE_E_INVALID;
  if (max_tiles == 0) return MOE_OK;
  const SW R = to_dev(routed, nullptr, pexp_routed), S = to_dev(sh ? sh : routed, sh ? sh_cb_up : nullptr, sh ? pexp_sh : pexp_routed);
  const int split = sh ? 1 : 0;
#define ST_ARGS R, S, n_experts, x, tokidx, tiles, ntiles, max_tiles, out, m, k, split, hs, rot, st
#define ST_UP(F)                                                                        \
  do {                                                                                  \
    if (cap == 16) return launch<F, true, 1, 0, up_waves(F, 1)>(ST_ARGS);               \
    if (cap == 32) return launch<F, true, 2, 0, up_waves(F, 2)>(ST_ARGS);               \
    if constexpr (!q5(F) && !once_rounded(F)) return launch<F, true, 4, 0, up_waves(F, 4)>(ST_ARGS); \
    return MOE_E_UNSUPPORTED;                                                           \
  } while (0)
  // (Q4_K with 64 pairs has no registers for whole rows of three lines: 21 in scratch, and 743 us for 733 at 1500 tokens, 815
  //  for 805 at 2000; the other formats lose 1 .. 2 % with pieces of two)
  const int nline = (k + 255) / 256;
#define ST_DN(F)                                                                        \
  do {                                                                                  \
    if (nline == DN_ONE && !(F == F_Q4K && cap > 32)) {                                 \
      if (cap == 16) return launch<F, false, 1, DN_ONE, 4>(ST_ARGS);                    \
      if (cap == 32) return launch<F, false, 2, DN_ONE, 4>(ST_ARGS);                    \
      if constexpr (F != F_Q80 && F != F_Q4K) return launch<F, false, 4, DN_ONE, 16>(ST_ARGS); \
      return MOE_E_UNSUPPORTED;                                                         \
    }                                                                                   \
    if (cap == 16) return launch<F, false, 1, 2, 4>(ST_ARGS);                           \
    if (cap == 32 && nline <= 4) return launch<F, false, 2, 2, 4>(ST_ARGS);             \
    if (cap == 32) return launch<F, false, 2, 2, F == F_Q80 ? 8 : 16>(ST_ARGS);         \
    if constexpr (F != F_Q80) return launch<F, false, 4, 2, 16>(ST_ARGS);               \
    return MOE_E_UNSUPPORTED;                                                           \
  } while (0)
#define ST_DIR(F)      \
  do {                 \
    if (up) ST_UP(F);  \
    ST_DN(F);          \
  } while (0)
  switch (fmt) {
    case F_DN: ST_DIR(F_DN);
    case F_AFF: ST_DIR(F_AFF);
    case F_TAB: ST_DIR(F_TAB);
    case F_I4D: ST_DIR(F_I4D);
    case F_I4R: ST_DIR(F_I4R);
    case F_Q4K: ST_DIR(F_Q4K);
    case F_Q5K: ST_UP(F_Q5K);
    case F_Q4E: ST_UP(F_Q4E);
    case F_Q5E: ST_UP(F_Q5E);
    case F_Q80: ST_DN(F_Q80);
    default: return MOE_E_INVALID;
  }
#undef ST_ARGS
#undef ST_UP
#undef ST_DN
#undef ST_DIR
}
