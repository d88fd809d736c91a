"""The calls of the routed-expert MoE layer that are timed when its kernels or their launches change.

A case is one pass of `capi.Moe.forward` -- the call that stands in for the engine's GpuModel::moe / moe_b -- over a
batch of `tokens` rows, through `layers` consecutive layers of one context.  The cases follow what an engine does with
such a layer: decode steps of one request, of a few concurrent requests and of speculative verification, short prompts
and small concurrent batches, prefill chunks up to the largest, in every weight format the engine loads, with the
batch sizes it happens to get (odd and ragged ones too).

  format   q4cp: zero-point-8 codebook; table: q4cp with the fixed non-uniform codebook of the reference's converter;
           q4k: GGUF Q4_K throughout; ggmix: the type mix of the GGUF checkpoints (Q5_K gate/up, Q8_0 down and shared
           expert); i4r: hgn v2 rotated experts
  router   dtype of the router matrix (checkpoints hold bf16, the benchmark's layer f32)
  shared   "same": the shared expert in the layer's own format; "q8g32": as the quality overlay files store it
  skew     True: a Zipf(1.1) bias on the router logits makes the hottest expert about 12 times as busy as the mean
  local    True: three tenths of the tokens pick the same experts, as drafted tokens do
  layers   decode steps go through several layers, each with its own weights and input row: one layer's experts for
           one token would stay in the last-level cache between passes, which a model's 48 layers never do
"""
import functools
import math

import torch

from gfx1151_engine_amd import capi
from gfx1151_engine_amd import workloads as W

EXPERTS, TOPK = 512, 10
ROUTER_STD = 0.02    # what workloads.DeviceLayer draws the router matrix with
ZIPF, BETA = 1.1, 0.27


def _case(name, format, tokens, d=3072, mid=768, router="f32", shared="same", skew=False, local=False, layers=1):
    c = {"format": format, "tokens": tokens, "d": d, "mid": mid, "router": router, "shared": shared, "skew": skew,
         "local": local, "layers": layers}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one request decoding: the smallest call, bound by latency and by the experts' bytes
        _case("decode_q4cp_1", "q4cp", 1, layers=4),
        # the same with the codebook that the converter writes
        _case("decode_table_1", "table", 1, router="bf16", layers=4),
        # three requests decoding together on a GGUF checkpoint
        _case("decode_ggmix_3", "ggmix", 3, router="bf16", layers=2),
        # speculative verification on a small draft, hgn v2 checkpoint
        _case("verify_i4r_11", "i4r", 11, local=True),
        # speculative verification of four requests with four drafted tokens each
        _case("verify_q4cp_20", "q4cp", 20, local=True),
        # many concurrent requests decoding together
        _case("batch_table_48", "table", 48, router="bf16"),
        # a short prompt
        _case("prompt_q4cp_130", "q4cp", 130),
        # a prompt of middle length on a GGUF checkpoint
        _case("prompt_q4k_515", "q4k", 515, router="bf16"),
        # a prefill chunk of the reference's default size, its other layer shape, with the quality overlay's shared expert
        _case("chunk_table_2048", "table", 2048, d=2560, mid=640, router="bf16", shared="q8g32", skew=True),
        # the ragged last chunk of a long prompt, hgn v2
        _case("chunk_i4r_3001", "i4r", 3001, skew=True),
        # a large chunk on a GGUF checkpoint
        _case("chunk_ggmix_4096", "ggmix", 4096, router="bf16", skew=True),
        # the largest prefill chunk
        _case("chunk_q4cp_16384", "q4cp", 16384, skew=True),
    ]


def draw(rng):
    fmt = rng.choice(["q4cp", "table", "q4k", "ggmix", "i4r"])
    most = 16384 if fmt == "q4cp" else 8192
    tokens = min(most, int(math.exp(rng.uniform(0.0, math.log(most + 1)))))
    # (Q4_K rows come in blocks of 256 columns, and rotated experts want both widths to be multiples of 256)
    small = fmt in ("q4cp", "table", "ggmix") and rng.random() < 0.3
    d, mid = (2560, 640) if small else (3072, 768)
    shared = "q8g32" if fmt in ("q4cp", "table") and rng.random() < 0.2 else "same"
    return _case(None, fmt, tokens, d=d, mid=mid, router=rng.choice(["f32", "bf16"]), shared=shared,
                 skew=tokens > 256 and rng.random() < 0.5, local=4 < tokens <= 32 and rng.random() < 0.5,
                 layers=4 if tokens == 1 else 2 if tokens <= 4 else 1)


def _zipf_bias():
    return -BETA * ZIPF * torch.log(torch.arange(1, EXPERTS + 1, dtype=torch.float32, device="cuda"))


def _layer(case, seed):
    fmt = {"table": "q4cp", "ggmix": "q4k"}.get(case["format"], case["format"])
    return W.DeviceLayer(seed, case["d"], case["mid"], EXPERTS, TOPK, fmt,
                         gg_types=(13, 8, 8) if case["format"] == "ggmix" else (12, 12, 12),
                         codebook="universal" if case["format"] == "table" else "zp8")


def _q8g32(g, rows, cols):
    codes = torch.randint(0, 256, (rows * cols,), dtype=torch.uint8, device="cuda", generator=g)
    scales = (torch.randn((rows * cols // 32,), device="cuda", generator=g).abs() * (0.01 / 16)).to(torch.float16)
    return torch.cat([codes, scales.view(torch.uint8)])


def prepare(case, seed):
    d, mid, T = case["d"], case["mid"], case["tokens"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + 15)
    m = capi.Moe(d, mid, EXPERTS, TOPK, layers=case["layers"], max_tokens=T)
    weights, xs = [], []
    for l in range(case["layers"]):
        L = _layer(case, seed * 16 + l)
        if case["skew"]:
            L.bias = _zipf_bias()[torch.randperm(EXPERTS, device="cuda", generator=g)].contiguous()
        L.register(m, l)
        if case["router"] == "bf16":
            L.router = L.router.to(torch.bfloat16)
            m.set_router(l, capi.wview(L.router, capi.BF16, EXPERTS, d), L.bias)
        if case["shared"] == "q8g32":
            L.sh = [_q8g32(g, mid, d), _q8g32(g, mid, d), _q8g32(g, d, mid)]
            m.set_shared(l, capi.wview(L.sh[0], capi.Q8G32, mid, d), capi.wview(L.sh[1], capi.Q8G32, mid, d),
                         capi.wview(L.sh[2], capi.Q8G32, d, mid), capi.wview(L.sh_sg, capi.F32, 1, d))
        x = torch.randn((T, d), device="cuda", generator=g)
        if case["local"]:
            n = max(1, round(0.3 * T))
            x[1:n] = x[0] + 1e-3 * torch.randn((n - 1, d), device="cuda", generator=g)
        weights.append(L)
        xs.append(x.to(torch.bfloat16).to(torch.float32))  # the engine's residual stream is bf16
    return {"moe": m, "weights": weights, "x": xs, "y": [torch.empty_like(x) for x in xs]}


def run(state):
    for l, (x, y) in enumerate(zip(state["x"], state["y"])):
        state["moe"].forward(l, x, y)
    return state["y"]


@functools.lru_cache(maxsize=None)
def _pick_rates(d, skew):
    """How often a token picks each expert: Gaussian logits of the router's spread plus the bias, the top k of them."""
    sd = ROUTER_STD * math.sqrt(d)
    bias = [-BETA * ZIPF * math.log(r) if skew else 0.0 for r in range(1, EXPERTS + 1)]
    lo, hi = -20.0, 20.0
    for _ in range(60):
        cut = 0.5 * (lo + hi)
        p = [0.5 * math.erfc((cut - b) / (sd * math.sqrt(2.0))) for b in bias]
        lo, hi = (cut, hi) if sum(p) > TOPK else (lo, cut)
    return p


def work(case):
    d, mid, T = case["d"], case["mid"], case["tokens"]
    different = T - max(1, round(0.3 * T)) + 1 if case["local"] else T
    experts = sum(1.0 - (1.0 - p) ** different for p in _pick_rates(d, case["skew"]))
    row = {"q4cp": lambda c: c // 2 + c // 16, "table": lambda c: c // 2 + c // 16, "i4r": lambda c: c // 2 + c // 64,
           "q4k": lambda c: W.gg_row_bytes(12, c)}
    gate_up, down = row.get(case["format"], lambda c: W.gg_row_bytes(13, c)), row.get(case["format"], lambda c: W.gg_row_bytes(8, c))
    sh = (lambda c: c + c // 16) if case["shared"] == "q8g32" or case["format"] == "ggmix" else row[
        "q4cp" if case["format"] == "i4r" else case["format"]]
    weights = experts * (2 * mid * gate_up(d) + d * down(mid)) + 2 * mid * sh(d) + d * sh(mid)
    router = (EXPERTS + 1) * d * (2 if case["router"] == "bf16" else 4)
    return {"bytes": case["layers"] * (weights + router + 2 * T * d * 4),
            "flops": case["layers"] * T * (6.0 * (TOPK + 1) * d * mid + 2.0 * EXPERTS * d)}


def tolerance(case):
    # batches over 32 tokens: f16 operands, f16 hidden rows and f16 expert outputs, f32 sums; up to 32 tokens:
    # activations of 16 significant bits per 32 columns (integer-dot kernels), or f32 throughout (table codebooks)
    return {"rel": 1e-3 if case["tokens"] > 32 else 1e-5 if case["format"] == "table" else 1e-4}
