// Expert-sorted token permutation: one membership bit per token and expert in LDS masks, popcounts of those masks give
// counts and ranks, prefix sums over waves / blocks / experts give every pair its slot.  Stable: inside an expert pairs
// are in ascending token order, exactly what the reference's stable radix sort yields.
// (reference: src/gpu/parts/10_ple_io.inc:784-861)
#include <mutex>
#include <new>

#include "common.h"
#include "internal.h"

struct moe_routing {
  int capacity_pairs, experts;
  int* blockcnt;  // [blocks of tokens][experts] pairs of a block that go to an expert
};

namespace {
constexpr int RT_MAXE = 1024;

// The permutation, a thread per token.  A wave's 64 tokens leave one membership bit each in an LDS mask per expert
// (masks[wave][expert]), so a pair's place inside its expert is the count of the earlier waves' bits plus the lower bits
// of its own wave's mask: stable without a sort, and every step is one parallel pass over the block's tokens or experts.
//   ROUTE_ONE    the whole batch in one block: permutation and (with tiles) the tile list in one launch
//   ROUTE_COUNT  larger batches, first launch: pairs per block and expert
//   ROUTE_PLACE  second launch: every block adds the counts of all blocks up for itself (no scan launch in between)
// (Counting, a one-block scan, a scatter and a tile launch, each with ballots over the key bits or one expert's counts at
//  a time, took 45 us from 128 to 4096 tokens, most of it dependent round trips, and 56 us at 16384; now 8 us at 48 tokens, 10 us at 515, 6 + 10 us at 4096 and 6 + 12 us
//  at 16384)
// KV: a token's picks as KV 16-byte loads (k <= 4 KV, rows of ids aligned for it); 0 = any k, read one by one.
enum { ROUTE_ONE, ROUTE_COUNT, ROUTE_PLACE };
constexpr int route_block_tokens(int E) { return E <= 512 ? 1024 : 512; }  // tokens of a block: the masks fit its LDS
constexpr size_t route_lds_bytes(int E, int waves) { return (size_t)waves * E * 10 + (size_t)E * 4; }
// the most a launch asks for (1024 experts, 512 tokens: 86016 bytes; 512 experts, 1024 tokens: 83968)
constexpr size_t route_lds_most() {
  size_t most = 0;
  for (int E = 1; E <= RT_MAXE; E++) {
    const size_t n = route_lds_bytes(E, route_block_tokens(E) / 64);
    most = n > most ? n : most;
  }
  return most;
}
constexpr size_t ROUTE_LDS_MOST = route_lds_most();
static_assert(ROUTE_LDS_MOST + 4096 <= 160 * 1024, "a CU's LDS");
// A block writes the pairs of an eighth of its tokens only (RT_SUB blocks per token block, each building the same masks):
// the scattered stores are single lanes' cache lines, 1024 tokens' worth of them kept one CU busy for 17 us.
constexpr int RT_SUB = 8;
template <int KV, int MODE>
__global__ void __launch_bounds__(RT_MAXE) k_route(const int* __restrict__ ids, const float* __restrict__ ws, int P, int k, int E,
                                                   int id_stride, int tpb, int* __restrict__ blockcnt, int* __restrict__ tokidx,
                                                   float* __restrict__ pw, int* __restrict__ eoff, int* __restrict__ pairids,
                                                   moe_tile* __restrict__ tiles, int* __restrict__ total, int cap, int sh_first) {
  extern __shared__ __attribute__((aligned(16))) uint8_t rsm[];
  __shared__ int wsum[RT_MAXE / 64], tsum[RT_MAXE / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int blk = MODE == ROUTE_COUNT ? blockIdx.x : blockIdx.x / RT_SUB, sub = MODE == ROUTE_COUNT ? 0 : blockIdx.x % RT_SUB;
  const int nblk = MODE == ROUTE_COUNT ? gridDim.x : gridDim.x / RT_SUB;
  const int t0 = blk * tpb, nt_blk = P - t0 < tpb ? P - t0 : tpb, nw = (nt_blk + 63) >> 6;
  unsigned long long* const masks = (unsigned long long*)rsm;        // [nw][E]
  int* const eo = (int*)(masks + (size_t)nw * E);                    // [E]
  uint16_t* const pre = (uint16_t*)(eo + E);                         // [nw][E] bits of the earlier waves
  for (int i = tid; i < nw * E; i += RT_MAXE) masks[i] = 0ull;
  const int t = t0 + tid;
  const bool live = tid < nt_blk;
  int u[KV > 0 ? 4 * KV : 1];
  if (KV > 0 && live) {
    const int4* r = (const int4*)(ids + (size_t)t * id_stride);
#pragma unroll
    for (int i = 0; i < KV; i++) {
      const int4 q = r[i];
      u[4 * i] = q.x; u[4 * i + 1] = q.y; u[4 * i + 2] = q.z; u[4 * i + 3] = q.w;
    }
  }
  // (the weights of the tokens whose pairs this block writes, requested next to the picks: they are needed last.  Requested where
  // they are needed the launch took 8.3 us for 7.5 at 48 tokens, 12.8 for 8.6 at 515, the second of two 10.5 for 9.6 at 4096)
  const bool writes = MODE != ROUTE_COUNT && live && tid / ((tpb + RT_SUB - 1) / RT_SUB) == sub;
  float wt[KV > 0 ? 4 * KV : 1];
  if (KV > 0 && writes) {
    const float4* r = (const float4*)(ws + (size_t)t * id_stride);
#pragma unroll
    for (int i = 0; i < KV; i++) {
      const float4 q = r[i];
      wt[4 * i] = q.x; wt[4 * i + 1] = q.y; wt[4 * i + 2] = q.z; wt[4 * i + 3] = q.w;
    }
  }
  auto pick = [&](int s) -> int {
    const int id = KV > 0 ? u[s] : ids[(size_t)t * id_stride + s];
    return id >= 0 && id < E ? id : -1;
  };
  auto slots = [&](auto&& f) {
    if (KV > 0) {
#pragma unroll
      for (int s = 0; s < 4 * KV; s++)
        if (s < k) f(s);
    } else {
      for (int s = 0; s < k; s++) f(s);
    }
  };
  __syncthreads();
  if (live)
    slots([&](int s) {
      const int key = pick(s);
      if (key >= 0) atomicOr(&masks[w * E + key], 1ull << lane);
    });
  __syncthreads();
  const int e = tid;
  int here = 0;
  if (e < E)
    for (int i = 0; i < nw; i++) {
      pre[i * E + e] = (uint16_t)here;
      here += __popcll(masks[i * E + e]);
    }
  if (MODE == ROUTE_COUNT) {
    if (e < E) blockcnt[(size_t)blk * E + e] = here;
    return;
  }
  int ne = here, before = 0;
  if (MODE == ROUTE_PLACE) {
    ne = 0;
    if (e < E)
      for (int b0 = 0; b0 < nblk; b0 += 8) {  // eight counts requested together
        int c[8];
#pragma unroll
        for (int i = 0; i < 8; i++) c[i] = b0 + i < nblk ? blockcnt[(size_t)(b0 + i) * E + e] : 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
          before += b0 + i < blk ? c[i] : 0;
          ne += c[i];
        }
      }
  }
  const int nt = tiles && e < E ? (ne + cap - 1) / cap : 0;
  int inc = ne, inct = nt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int a = __shfl_up(inc, o, 64), b = __shfl_up(inct, o, 64);
    if (lane >= o) {
      inc += a;
      inct += b;
    }
  }
  if (lane == 63) {
    wsum[w] = inc;
    tsum[w] = inct;
  }
  __syncthreads();
  int base = 0, baset = 0, allt = 0;
#pragma unroll
  for (int i = 0; i < RT_MAXE / 64; i++) {
    base += i < w ? wsum[i] : 0;
    baset += i < w ? tsum[i] : 0;
    allt += tsum[i];
  }
  const int first = base + inc - ne, begin = baset + inct - nt;
  if (e < E) {
    eo[e] = first + before;
    if (blockIdx.x == 0) {
      eoff[e] = first;
      if (e == E - 1) eoff[E] = first + ne;
      for (int j = 0; j < nt; j++) {
        moe_tile q;
        q.expert = e;
        q.first = first + j * cap;
        q.count = min(cap, ne - j * cap);
        tiles[begin + j] = q;
      }
    }
  }
  if (tiles) {  // the shared expert's tiles behind the routed ones, its pairs' tokens
    if (blockIdx.x == 0) {
      const int nsh = sh_first >= 0 ? (P + cap - 1) / cap : 0;
      for (int j = tid; j < nsh; j += RT_MAXE) {
        moe_tile q;
        q.expert = E;
        q.first = sh_first + j * cap;
        q.count = min(cap, P - j * cap);
        tiles[allt + j] = q;
      }
      if (tid == 0) {
        total[0] = allt + nsh;
        total[1] = allt;
      }
    }
    if (sh_first >= 0 && live && sub == 0) tokidx[sh_first + t] = t;
  }
  __syncthreads();
  if (!writes) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  slots([&](int s) {
    const int key = pick(s);
    if (key < 0) return;
    const int pos = eo[key] + (int)pre[w * E + key] + __popcll(masks[w * E + key] & below);
    tokidx[pos] = t;
    pw[pos] = KV > 0 ? wt[s] : ws[(size_t)t * id_stride + s];
    if (pairids) {
      int rank = 0;
      slots([&](int r) { rank += (KV > 0 ? u[r] : ids[(size_t)t * id_stride + r]) < key; });
      pairids[(size_t)t * k + rank] = pos;
    }
  });
}

// Tiles in expert order: thread e owns expert e, LDS scan of the per-expert tile counts.
__global__ void __launch_bounds__(RT_MAXE) k_tiles(const int* __restrict__ eoff,
                                                   moe_tile* __restrict__ tiles,
                                                   int* __restrict__ total, int E, int cap) {
  __shared__ int wsum[RT_MAXE / 64];
  const int e = threadIdx.x, lane = e & 63, w = e >> 6;
  const int first = e < E ? eoff[e] : 0;
  const int ne = e < E ? eoff[e + 1] - first : 0;
  const int count = (ne + cap - 1) / cap;
  int inc = count;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int base = 0;
  for (int i = 0; i < w; i++) base += wsum[i];
  const int begin = base + inc - count;
  if (e == RT_MAXE - 1) *total = begin + count;
  for (int j = 0; j < count; j++) {
    moe_tile t;
    t.expert = e;
    t.first = first + j * cap;
    t.count = min(cap, ne - j * cap);
    tiles[begin + j] = t;
  }
}
}  // namespace

template <int KV, int MODE>
static int route_launch(unsigned grid, size_t lds, hipStream_t st, const int* ids, const float* ws, int P, int k, int E,
                        int id_stride, int tpb, int* blockcnt, int* tokidx, float* pw, int* eoff, int* pairids, moe_tile* tiles,
                        int* total, int cap, int sh_first) {
  static moe_dev_once once;
  int dev;
  if (moe_dev_pending(once, &dev)) {
    MOE_HIP(hipFuncSetAttribute((const void*)k_route<KV, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ROUTE_LDS_MOST));
    moe_dev_done(once, dev);
  }
  k_route<KV, MODE><<<grid, RT_MAXE, lds, st>>>(ids, ws, P, k, E, id_stride, tpb, blockcnt, tokidx, pw, eoff, pairids, tiles,
                                                total, cap, sh_first);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}

// Internal: permutation (and, with tiles != nullptr, the tile list incl. the shared expert's) of any batch.
// blockcnt: [ceil(P / 512)][experts] ints, untouched (may be null) where one block takes the whole batch.
int moe_launch_route(int* blockcnt, const int* ids, const float* ws, int* tokidx, float* pw, int* eoff, int* pairids, int P,
                     int k, int experts, int id_stride, moe_tile* tiles, int* ntiles, int cap, int sh_first, hipStream_t st) {
  if (!eoff || (P > 0 && (!ids || !ws || !tokidx || !pw)) || (tiles && (!ntiles || cap < 1))) return MOE_E_INVALID;
  if (experts < 1 || experts > RT_MAXE || k < 1 || id_stride < k) return MOE_E_UNSUPPORTED;
  const int tpb = route_block_tokens(experts), nblk = P > 0 ? (P + tpb - 1) / tpb : 1;
  if (nblk > 1 && !blockcnt) return MOE_E_INVALID;
  const size_t lds = route_lds_bytes(experts, ((P < tpb ? P : tpb) + 63) / 64);
  // (one block of tokens: as many of its RT_SUB writers as there are tokens for)
  const int per = (tpb + RT_SUB - 1) / RT_SUB, nsub = P > per ? (P + per - 1) / per : 1;
  const bool wide = id_stride % 4 == 0 && moe_aligned(ids, 16) && moe_aligned(ws, 16) && id_stride >= (k + 3) / 4 * 4;
#define RT_ARGS lds, st, ids, ws, P, k, experts, id_stride, tpb, blockcnt, tokidx, pw, eoff, pairids, tiles, ntiles, cap, sh_first
#define RT_GO(KV)                                                           \
  do {                                                                      \
    if (nblk == 1) return route_launch<KV, ROUTE_ONE>((unsigned)nsub, RT_ARGS);             \
    const int rc = route_launch<KV, ROUTE_COUNT>((unsigned)nblk, RT_ARGS);                  \
    return rc ? rc : route_launch<KV, ROUTE_PLACE>((unsigned)(nblk * RT_SUB), RT_ARGS);                \
  } while (0)
  if (wide && k <= 8) RT_GO(2);
  if (wide && k <= 12) RT_GO(3);
  if (wide && k <= 16) RT_GO(4);
  RT_GO(0);
#undef RT_GO
#undef RT_ARGS
}

int* moe_routing_blockcnt(moe_routing* r) { return r->blockcnt; }

MOE_API int moe_routing_create(int capacity_pairs, int experts, moe_routing** out) {
  if (!out || capacity_pairs < 1 || experts < 1) return MOE_E_INVALID;
  if (experts > RT_MAXE) return MOE_E_UNSUPPORTED;
  moe_routing* r = new (std::nothrow) moe_routing();
  if (!r) return (int)hipErrorOutOfMemory;
  r->capacity_pairs = capacity_pairs;
  r->experts = experts;
  r->blockcnt = nullptr;
  const int tpb = route_block_tokens(experts);
  const size_t blocks = ((size_t)capacity_pairs + tpb - 1) / tpb;  // enough for any k >= 1
  const hipError_t e = hipMalloc(&r->blockcnt, blocks * experts * sizeof(int));
  if (e != hipSuccess) {
    delete r;
    return (int)e;
  }
  *out = r;
  return MOE_OK;
}

MOE_API int moe_routing_destroy(moe_routing* r) {
  if (!r) return MOE_OK;
  const hipError_t e = hipFree(r->blockcnt);
  delete r;
  return (int)e;
}

MOE_API int moe_routing_run(moe_routing* r, const int* ids, const float* ws, int* tokidx, float* pw,
                            int* eoff, int* pairids, int P, int k, int experts, int id_stride,
                            moe_stream_t st) {
  if (!r || !eoff || (P > 0 && (!ids || !ws || !tokidx || !pw))) return MOE_E_INVALID;
  if (P < 0 || k < 1 || id_stride < k || experts != r->experts) return MOE_E_INVALID;
  if ((int64_t)P * k > r->capacity_pairs) return MOE_E_STATE;
  return moe_launch_route(r->blockcnt, ids, ws, tokidx, pw, eoff, pairids, P, k, experts, id_stride, nullptr, nullptr, 0, -1,
                          moe_s(st));
}

// ---- the permutation for callers that cannot allocate ----
// The per-block counts of batches over one block live in a file-scope device array instead of a moe_routing object's
// allocation, one copy per GPU, held until the process ends.  Every call writes the part of the array it later reads
// (nothing has to start at zero), and every call on a GPU uses the same array: calls that overlap on one GPU (two
// streams, two threads) race.
namespace {
constexpr int RT_MAX_DEVICES = 64;
}  // namespace
static __device__ __align__(256) int scratch[MOE_ROUTING_STATIC_MAX_TOKENS / 512 * RT_MAXE];
static int* g_scratch_ptr[RT_MAX_DEVICES];  // device address of `scratch` on each GPU (its name is no address on the host)
static std::mutex g_scratch_mu;

// The address of this GPU's copy of `scratch`, looked up once per device with that device current.
static int scratch_of_current_device(int** out) {
  int dev = -1;
  MOE_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= RT_MAX_DEVICES) return MOE_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int* p = nullptr;
    MOE_HIP(hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch)));
    if (!p) return (int)hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return MOE_OK;
}

MOE_API int moe_routing_run_static(const int* ids, const float* ws, int* tokidx, float* pw, int* eoff, int* pairids,
                                   int P, int k, int experts, int id_stride, moe_stream_t st) {
  if (!eoff || (P > 0 && (!ids || !ws || !tokidx || !pw))) return MOE_E_INVALID;
  if (P < 0 || k < 1 || id_stride < k || experts < 1) return MOE_E_INVALID;
  if (experts > RT_MAXE) return MOE_E_UNSUPPORTED;
  if (P > MOE_ROUTING_STATIC_MAX_TOKENS) return MOE_E_STATE;  // beyond the fixed scratch: use moe_routing_create / run
  // (the look-up comes first, whatever the batch size: any call made outside a capture, P = 0 included, sets the
  //  device up for later calls inside one)
  int* base = nullptr;
  const int rc = scratch_of_current_device(&base);
  if (rc) return rc;
  return moe_launch_route(base, ids, ws, tokidx, pw, eoff, pairids, P, k, experts, id_stride, nullptr, nullptr, 0, -1, moe_s(st));
}

MOE_API int moe_tiles(const int* eoff, moe_tile* tiles, int* ntiles, int experts, int cap,
                      moe_stream_t st) {
  if (!eoff || !tiles || !ntiles || cap < 1 || experts < 1) return MOE_E_INVALID;
  if (experts > RT_MAXE) return MOE_E_UNSUPPORTED;
  k_tiles<<<1, RT_MAXE, 0, moe_s(st)>>>(eoff, tiles, ntiles, experts, cap);
  MOE_LAUNCH_CHECK();
  return MOE_OK;
}
