"""Batches between the in-place kernels and the largest prefill chunks: the sizes at which the router, the permutation
and the grouped GEMM change kernels, against the oracle."""
import numpy as np
import pytest

from helpers import HostLayer, max_abs_rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gfx1151_engine_amd import capi as m
    return m


def gpu(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# ---------- permutation: one block of tokens, its writers, several blocks ----------
@pytest.mark.parametrize("P,E,k,stride", [(64, 512, 10, 16), (128, 512, 10, 16), (129, 64, 4, 16), (1024, 512, 10, 16),
                                          (1025, 512, 10, 16), (2049, 8, 3, 4), (512, 1000, 12, 16), (513, 1000, 13, 16),
                                          (512, 1024, 10, 16), (600, 1024, 15, 16), (1024, 513, 10, 16),
                                          (700, 30, 17, 20), (1100, 30, 17, 17)])
def test_routing_block_edges(capi, oracle, P, E, k, stride):
    rng = np.random.default_rng(P + E)
    ids = np.zeros((P, stride), np.int32)
    ws = rng.random((P, stride)).astype(np.float32)
    pr = 1.0 / (np.arange(E) + 1.0)
    pr /= pr.sum()
    for t in range(P):
        ids[t, :k] = rng.choice(E, k, replace=False, p=pr)
    to, po, eo, qo = oracle.route(ids, ws, k, E)
    r = capi.Routing(P * k, E)
    for got in (r.run(gpu(ids), gpu(ws), k), capi.routing_run_static(gpu(ids), gpu(ws), k, E)):
        tokidx, pw, eoff, pairids = (a.cpu().numpy() for a in got)
        assert (eoff == eo).all() and (tokidx == to).all() and (pw == po).all() and (pairids == qo).all()
    r.close()


# ---------- router of 1 .. 4 tokens: rows of less than a column step, of ragged steps, of more than one pass over the columns ----------
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("P,E,d", [(1, 33, 4), (2, 9, 252), (3, 512, 2560), (4, 40, 3076), (1, 17, 6400), (3, 8, 3072)])
def test_router_rows_of_a_few_tokens(capi, oracle, P, E, d, dt):
    from gfx1151_engine_amd import synth as S
    rng = np.random.default_rng(100 * P + d)
    W = rng.standard_normal((E, d), dtype=np.float32) * 0.02
    x = rng.standard_normal((P, d), dtype=np.float32)
    if dt == "bf16":
        W = S.f32_to_bf16_bits(W)
    lo, _, _ = oracle.router(oracle.Mat(oracle.BF16 if dt == "bf16" else oracle.F32, W, E, d), x, 4)
    lg = capi.router_logits(capi.wview(gpu(W.view(np.int16) if dt == "bf16" else W), capi.BF16 if dt == "bf16" else capi.F32, E, d),
                            gpu(x), None, 0).cpu().numpy()
    assert np.abs(lg - lo).max() <= 2.4e-7 * np.abs(lo).max()  # fp64 sums in another order: at most the last f32 bit


@pytest.mark.parametrize("T", [1, 2, 3, 4])
def test_router_and_gate_vector_of_two_types(capi, oracle, T):
    rng = np.random.default_rng(T)
    hl = HostLayer(rng, 768, 256, 33, 5, router_dtype="bf16")  # (the gate vector is f32)
    x = rng.standard_normal((T, 768), dtype=np.float32)
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids = m.last_routing(T)[0].cpu().numpy()[:, :5]
    m.close()
    assert (ids == io[:, :5]).all()
    assert max_abs_rel(y, yo) <= 2e-3


# The launches of 5 .. 32 tokens: a gate vector of the matrix's own type and one of the other type (off any alignment) meet in
# the same kernel, so layers that differ in nothing but the type their equal values are stored in give equal results.
@pytest.mark.parametrize("T,E,d", [(5, 512, 3072), (16, 33, 768), (17, 520, 2560), (24, 48, 128), (25, 33, 640), (32, 512, 3072)])
def test_gate_vector_of_the_other_type(capi, oracle, T, E, d):
    import torch
    rng = np.random.default_rng(T)
    hl = HostLayer(rng, d, 256, E, 5, router_dtype="bf16")
    x = rng.standard_normal((T, d), dtype=np.float32)
    m, dev = hl.to_gpu(max_tokens=T)
    bits = dev["router"].view(torch.bfloat16).reshape(E, d)
    gate = dev["shsg"].reshape(-1).to(torch.bfloat16)
    got = {}
    for rt in (torch.bfloat16, torch.float32):
        r = bits.to(rt).contiguous()
        m.set_router(0, capi.wview(r, capi.BF16 if rt == torch.bfloat16 else capi.F32, E, d))
        for gt in (torch.bfloat16, torch.float32):
            room = torch.zeros(d + 8, dtype=gt, device="cuda")
            room[1:1 + d] = gate
            m.set_shared(0, *(capi.wview(dev[n], capi.Q4CP, a, b) for n, a, b in (("shg", 256, d), ("shu", 256, d), ("shd", d, 256))),
                         capi.wview(room[1:], capi.BF16 if gt == torch.bfloat16 else capi.F32, 1, d))
            got[rt, gt] = m.forward(0, gpu(x)).cpu()
    ids = m.last_routing(T)[0].cpu().numpy()[:, :5]
    m.close()
    lo, io, _ = oracle.router(hl.oracle_layer().router, x, 5)
    assert (ids == io[:, :5]).all()
    ref = got[torch.float32, torch.float32]
    for y in got.values():
        assert torch.equal(y, ref)


# ---------- the shared expert's gate vector may start at any element, whatever router a batch takes ----------
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("T,candidates", [(1, 1), (4, 1), (6, 1), (20, 1), (32, 1), (40, 1), (256, 1), (300, 1), (40, 0), (300, 0)])
def test_gate_vector_at_any_element(capi, T, candidates, dt):
    import torch
    rng = np.random.default_rng(T)
    d, mid = 512, 256
    hl = HostLayer(rng, d, mid, 32, 4, router_dtype=dt)
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_ROUTER_CANDIDATES, candidates)
    gate = dev["shsg"].reshape(-1).to(torch.bfloat16 if dt == "bf16" else torch.float32)
    x = gpu(rng.standard_normal((T, d), dtype=np.float32))
    ys = []
    for off in (0, 1, 3):
        room = torch.zeros(d + 8, dtype=gate.dtype, device="cuda")
        room[off:off + d] = gate
        m.set_shared(0, *(capi.wview(dev[n], capi.Q4CP, r, c) for n, r, c in (("shg", mid, d), ("shu", mid, d), ("shd", d, mid))),
                     capi.wview(room[off:], capi.BF16 if dt == "bf16" else capi.F32, 1, d))
        ys.append(m.forward(0, x).cpu())
    m.close()
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])


# ---------- router: edges of its token and expert tiles, the last batch it takes and the first it does not ----------
@pytest.mark.parametrize("T,E,k,d,dt", [(33, 512, 10, 3072, "bf16"), (64, 33, 5, 256, "f32"), (65, 512, 10, 2560, "f32"),
                                        (515, 512, 10, 768, "bf16"), (1024, 520, 10, 384, "f32"), (1025, 512, 10, 384, "bf16")])
def test_router_tiles(capi, oracle, T, E, k, d, dt):
    rng = np.random.default_rng(T)
    hl = HostLayer(rng, d, 256, E, k, router_dtype=dt)  # (the gate vector is f32 beside either type)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[T // 2] = x[0]
    lo, io, wo = oracle.router(hl.oracle_layer().router, x, k)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    ids, ws = (a.cpu().numpy()[:, :k] for a in m.last_routing(T))
    m.close()
    assert (ids == io[:, :k]).all()
    assert np.abs(ws - wo[:, :k]).max() <= 2.5e-7
    sel = np.r_[0, T // 2, T - 1]
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x[sel])
    assert max_abs_rel(y[sel], yo) <= 2e-3


def test_router_ties_above_the_middle(capi, oracle):
    """Tokens that the candidate selection lists, at a size only it takes: tied and nearly tied rows, a zero token."""
    rng = np.random.default_rng(11)
    E, k, d, T = 128, 10, 512, 1200
    hl = HostLayer(rng, d, 256, E, k, shared=False)
    hl.router[7] = hl.router[3]
    hl.router[16] = hl.router[5] * np.float32(1 + 2 ** -22)
    for zeros in (2, T - 30):  # few tokens to redo; most of them (padding: their sums are known)
        x = rng.standard_normal((T, d), dtype=np.float32)
        x[:zeros] = 0.0
        lo, io, wo = oracle.router(hl.oracle_layer().router, x, k)
        m, dev = hl.to_gpu(max_tokens=T)
        m.forward(0, gpu(x))
        ids, ws = (a.cpu().numpy()[:, :k] for a in m.last_routing(T))
        m.close()
        assert (ids == io[:, :k]).all()
        assert np.abs(ws - wo[:, :k]).max() <= 2.5e-7


# ---------- router, candidate selection: tiles and column shares of its f16 launch, ragged experts, ties, doubt, padding ----------
@pytest.mark.parametrize("T,E,k,d,dt,fmt", [(513, 512, 10, 3072, "bf16", "q4cp"), (600, 500, 10, 512, "f32", "q4cp"), (700, 43, 15, 256, "f32", "q4cp"),
                                            (777, 128, 4, 320, "f32", "q8_0"), (2600, 512, 10, 256, "bf16", "q4cp"), (2689, 510, 8, 384, "f32", "q4cp")])
def test_router_candidates(capi, oracle, T, E, k, d, dt, fmt):
    rng = np.random.default_rng(T)
    kw = dict(fmt="q4k", gg_types=(8, 8, 8)) if fmt == "q8_0" else {}
    hl = HostLayer(rng, d, 256, E, k, router_dtype=dt, shared=False, **kw)
    hl.router[E - 1] = hl.router[2]          # a tie for every token, in and out of the selection
    if dt == "f32":
        hl.router[E // 2] = hl.router[1] * np.float32(1 + 2 ** -22)  # logits an ulp apart: tokens for the redo
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[5] = 0.0                               # padding, a value past f16's range, a spread that underflows probabilities
    x[T - 1] = 0.0
    x[6, 3] = 1e6
    x[7] *= 300.0
    lo, io, wo = oracle.router(hl.oracle_layer().router, x, k)
    m, dev = hl.to_gpu(max_tokens=T)
    m.forward(0, gpu(x))
    assert m.last_path() == capi.PATH_BATCH
    ids, ws = (a.cpu().numpy()[:, :k] for a in m.last_routing(T))
    m.close()
    assert (ids == io[:, :k]).all()
    assert np.abs(ws - wo[:, :k]).max() <= 2.5e-7


# ... at the sizes where four waves share a token: the smallest and largest, rows of fewer runs than waves, uneven shares, a
# second pass over the candidates (many close logits)
@pytest.mark.parametrize("T,E,k,d,dt,fmt,std", [(257, 512, 10, 3072, "f32", "q4cp", 0.02), (258, 43, 15, 192, "bf16", "q8_0", 0.02),
                                                (300, 512, 10, 320, "f32", "q8_0", 0.02), (301, 300, 15, 512, "bf16", "q4cp", 0.0005),
                                                (1024, 128, 4, 128, "f32", "q8_0", 0.02), (1025, 128, 4, 128, "f32", "q8_0", 0.02)])
def test_router_candidates_of_small_batches(capi, oracle, T, E, k, d, dt, fmt, std):
    rng = np.random.default_rng(T)
    kw = dict(fmt="q4k", gg_types=(8, 8, 8)) if fmt == "q8_0" else {}
    hl = HostLayer(rng, d, 256, E, k, router_dtype=dt, router_std=std, shared=False, **kw)
    hl.router[E - 1] = hl.router[2]
    if dt == "f32":
        hl.router[E // 2] = hl.router[1] * np.float32(1 + 2 ** -22)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[5] = 0.0
    x[6, 3] = 1e6
    x[7] *= 300.0
    x[T - 1] = x[0]
    lo, io, wo = oracle.router(hl.oracle_layer().router, x, k)
    m, dev = hl.to_gpu(max_tokens=T)
    m.forward(0, gpu(x))
    assert m.last_path() == capi.PATH_BATCH
    ids, ws = (a.cpu().numpy()[:, :k] for a in m.last_routing(T))
    m.close()
    assert (ids == io[:, :k]).all()
    assert np.abs(ws - wo[:, :k]).max() <= 2.5e-7


# ... and at the widths of the exact dot products' panels (three, four and five pieces of 256 columns, whole and cut short, one
# panel and several), on both sides of the line between four waves and one, with odd numbers of candidates and with more
# than one pass of sixteen takes; weights that are zero or subnormal (the products are widened by shifting)
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("T,E,k,d,std", [(768, 512, 10, 3072, 0.02), (769, 512, 10, 3072, 0.02), (300, 512, 9, 2560, 0.02), (770, 512, 9, 2560, 0.02),
                                         (771, 300, 15, 832, 0.0005), (900, 128, 4, 1280, 0.02), (800, 64, 5, 64, 0.02), (780, 40, 11, 1600, 0.02)])
def test_router_candidates_exact_products(capi, oracle, T, E, k, d, std, dt):
    rng = np.random.default_rng(T + d)
    kw = dict(fmt="q4k", gg_types=(8, 8, 8)) if d % 128 else {}
    hl = HostLayer(rng, d, 256, E, k, router_dtype=dt, router_std=std, shared=False, **kw)
    w = hl.router
    w[:, ::7] = 0
    w[1, ::3] = np.float32(1e-40) if dt == "f32" else w.dtype.type(1)  # (the smallest bf16)
    w[2, 1::5] = np.float32(-1e-41) if dt == "f32" else w.dtype.type(0x8001)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[::2] = x[::2].astype(np.float16)       # exact in f16 (no rounding error to bound), and not
    x[8] = 0.0
    x[9, 0] = 3e4
    lo, io, wo = oracle.router(hl.oracle_layer().router, x, k)
    m, dev = hl.to_gpu(max_tokens=T)
    m.forward(0, gpu(x))
    assert m.last_path() == capi.PATH_BATCH
    ids, ws = (a.cpu().numpy()[:, :k] for a in m.last_routing(T))
    m.close()
    assert (ids == io[:, :k]).all()
    assert np.abs(ws - wo[:, :k]).max() <= 2.5e-7


# ---------- routers of 33 tokens and more: tokens that the fast selection cannot settle, few and many of them ----------
def route_and_compare(capi, oracle, hl, x, k):
    T = len(x)
    _, io, wo = oracle.router(hl.oracle_layer().router, x, k, bias=hl.bias)
    m, dev = hl.to_gpu(max_tokens=T)
    m.profile(True)
    xg = gpu(x)
    ms = []
    for _ in range(4):
        m.forward(0, xg)
        ms.append(m.profile_read()["router"])
    assert m.last_path() == capi.PATH_BATCH
    ids, ws = (a.cpu().numpy()[:, :k] for a in m.last_routing(T))
    m.close()
    assert (ids == io[:, :k]).all(), np.where((ids != io[:, :k]).any(1))
    wo = wo[:, :k]
    ok = np.isfinite(wo)
    assert (np.isfinite(ws) == ok).all()
    assert np.abs(ws[ok] - wo[ok]).max(initial=0.0) <= 2.5e-7
    return min(ms)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("T,E,d", [(130, 512, 512), (300, 512, 512), (1200, 500, 384), (2600, 128, 256), (2700, 500, 256)])
@pytest.mark.parametrize("kind", ["one off", "most off", "all but k off", "too many off", "wide", "some wide", "a nan", "infinities"])
def test_tokens_the_selection_cannot_settle(capi, oracle, kind, T, E, d, dt):
    rng = np.random.default_rng(T)
    k = 10
    bias = None
    x = rng.standard_normal((T, d), dtype=np.float32)
    if "off" in kind:  # experts switched off by a bias of minus infinity (too many: k reaches into them)
        n = {"one off": 1, "most off": E - 40, "all but k off": E - k, "too many off": E - k + 3}[kind]
        bias = rng.standard_normal(E).astype(np.float32) * 0.1
        bias[rng.permutation(E)[:n]] = -np.inf
    elif kind == "wide":        # probabilities underflow: every token has to be redone
        x *= 400.0
    elif kind == "some wide":   # a part of the batch, a ragged last group, padding between them
        x[::4] *= 400.0
        x[1::8] = 0.0
    elif kind == "a nan":
        x[T // 2, 3] = np.nan
    else:
        x[5, 7] = np.inf
        x[::9, 1] = -np.inf
        x[9, 2] = np.inf
    hl = HostLayer(rng, d, 256, E, k, router_dtype=dt, shared=False, bias=bias)
    route_and_compare(capi, oracle, hl, x, k)


# ... and what they cost: a batch of ordinary tokens and the same with an expert off, with one NaN, with nothing but tokens to
# redo.  Measured at 2048 tokens of 3072 columns: 0.08 ms ordinary and with an expert off, 0.16 with one NaN, 0.35 with all
# tokens to redo; with each of them redone by its own block 0.8, 9.7 and 1.3 .. 41 ms.
@pytest.mark.parametrize("T", [130, 2048])
def test_cost_of_tokens_the_selection_cannot_settle(capi, oracle, T):
    rng = np.random.default_rng(5)
    E, d, k = 512, 1024, 10
    hl = HostLayer(rng, d, 256, E, k, shared=False)
    x = rng.standard_normal((T, d), dtype=np.float32)
    plain = route_and_compare(capi, oracle, hl, x, k)
    hl.bias = np.zeros(E, np.float32)
    hl.bias[17] = -np.inf
    assert route_and_compare(capi, oracle, hl, x, k) <= 1.5 * plain + 0.06
    hl.bias = None
    nan = x.copy()
    nan[T // 2, 3] = np.nan
    assert route_and_compare(capi, oracle, hl, nan, k) <= 1.5 * plain + 0.2
    nan[:, 3] = np.nan
    assert route_and_compare(capi, oracle, hl, nan, k) <= 1.5 * plain + 0.4
    assert route_and_compare(capi, oracle, hl, x * np.float32(300.0), k) <= 1.5 * plain + 0.4


# ---------- grouped GEMM over tiles of few pairs: every format, tile size and side of a line between them ----------
TABLE = np.array([-1.0, -0.7, -0.53, -0.4, -0.28, -0.18, -0.09, 0.0, 0.08, 0.16, 0.25, 0.34, 0.44, 0.56, 0.72, 1.0], np.float32)


@pytest.mark.parametrize("T", [33, 40, 41, 88, 89, 152, 153, 176, 177])
@pytest.mark.parametrize("kind,kw,d,mid", [
    ("q4cp", dict(fmt="q4cp"), 512, 640), ("q4cp-affine", dict(fmt="q4cp"), 1024, 768),
    ("q4cp-table", dict(fmt="q4cp", codebook=TABLE), 512, 640),
    ("q4cp-tables", dict(fmt="q4cp", codebook=TABLE, shared_codebooks=[TABLE, TABLE[::-1].copy(), TABLE * 0.5]), 1024, 768),
    ("i4r", dict(fmt="i4r"), 512, 768), ("q4k", dict(fmt="q4k"), 512, 768), ("q4k-alone", dict(fmt="q4k", shared=False), 1024, 768),
    ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 13)), 512, 768), ("q4k-q8_0", dict(fmt="q4k", gg_types=(12, 8, 8)), 1024, 768)])
def test_tiles_of_few_pairs(capi, oracle, kind, kw, d, mid, T):
    rng = np.random.default_rng(T + d)
    E, k = 16, 4  # (averages of 10, 22, 38 and 44 pairs per expert at 40, 88, 152 and 176 tokens)
    hl = HostLayer(rng, d, mid, E, k, bias=np.linspace(0, 0.5, E, dtype=np.float32), **kw)
    if kind == "q4cp-affine":  # one expert's row with a scale 2^6 below its others: no scaled dequantisation
        sc = hl.gate_up[64 + E * 2 * mid * d // 2:].view(np.float16).reshape(E * 2 * mid, -1)
        sc[3, :] = np.float16(np.abs(sc).max() / 128)
    x = rng.standard_normal((T, d), dtype=np.float32)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(x)).cpu().numpy()
    again = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert (y == again).all()
    sel = np.r_[0, 1, T // 2, T - 2, T - 1]
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x[sel])
    assert max_abs_rel(y[sel], yo) <= 2e-3


# ---------- ... against the 128-pair kernels ----------
STREAM_KINDS = [("q4cp", dict(fmt="q4cp"), 512, 640), ("q4cp-affine", dict(fmt="q4cp"), 512, 768),
                ("q4cp-table", dict(fmt="q4cp", codebook=TABLE), 512, 640), ("q4k", dict(fmt="q4k"), 512, 768),
                ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 768), ("q4k-q8_0", dict(fmt="q4k", gg_types=(12, 8, 8)), 512, 768)]


def both_kernels(capi, hl, x):
    m, dev = hl.to_gpu(max_tokens=len(x))
    ys = []
    for on in (1, 0):
        m.set_option(capi.OPT_STREAM_GEMM, on)
        ys.append(m.forward(0, gpu(x)).cpu().numpy())
        assert m.last_path() == capi.PATH_BATCH
    m.close()
    return ys


@pytest.mark.parametrize("T", [40, 88, 152])
@pytest.mark.parametrize("kind,kw,d,mid", STREAM_KINDS)
def test_few_pair_tiles_multiply_the_same_weights(capi, kind, kw, d, mid, T):
    """Tokens with one column, experts with one row of up_proj: every sum has one term, so that both kernels' results are
    products of the same f16 weights, bit for bit."""
    rng = np.random.default_rng(T + mid)
    E, k = 16, 4
    hl = HostLayer(rng, d, mid, E, k, shared=False, bias=np.linspace(0, 0.5, E, dtype=np.float32), **kw)
    keep = np.r_[0, 1, 31, 32, 33, 100, 127, 128, 191, 255, 256, 300, 383, 511, mid - 129, mid - 1]  # row of expert 0, 1, ...
    if hl.fmt == "q4cp":
        up = hl.gate_up[64:64 + E * 2 * mid * d // 2].reshape(E, 2, mid, d // 2)[:, 1]
        zero = 0x77 if "table" in kind else 0x88
        if kind == "q4cp-affine":  # every expert has a row with scales 2^6 below the others: no scaled dequantisation
            hl.gate_up[64 + E * 2 * mid * d // 2:].view(np.float16).reshape(E, 2 * mid, -1)[:, 3, :] = np.float16(1e-5)
    else:
        up = hl.up.reshape(E, mid, -1)
        zero = 0
    for e in range(E):
        row = up[e, keep[e]].copy()
        up[e] = zero
        up[e, keep[e]] = row
    x = np.zeros((T, d), np.float32)
    x[np.arange(T), rng.integers(0, d, T)] = rng.choice([-2.0, 1.0, 0.5], T) * 16
    y1, y0 = both_kernels(capi, hl, x)
    assert np.abs(y0).max() > 0
    assert (y1 == y0).all()


@pytest.mark.parametrize("fused", [1, 0])
@pytest.mark.parametrize("T", [40, 88, 152])
@pytest.mark.parametrize("kind", ["i4r", "i4r-mixed"])
def test_few_pair_tiles_multiply_the_same_rotated_weights(capi, kind, T, fused):
    """Tokens that the rotation turns into one column, down_proj of one column: every sum over the weights has one term here too.
    In a layer with one expert of larger scales the streaming launches give all experts the plain form, the 128-pair ones that expert."""
    rng = np.random.default_rng(T)
    d, mid, E, k = 512, 768, 16, 4
    hl = HostLayer(rng, d, mid, E, k, fmt="i4r", shared=False, bias=np.linspace(0, 0.5, E, dtype=np.float32))
    hl.planes = [np.ones_like(p) for p in hl.planes]
    for w, n, cols in ((hl.gate_up, 2 * mid, d), (hl.down, d, mid)):
        sc = w[E * n * cols // 2:].view(np.float16).reshape(E, n, cols // 128)
        sc[:, :, 1] *= np.float16(2.0 ** -7)  # (weights that would be subnormal in units of an expert's largest scale)
        if kind == "i4r-mixed":
            sc[7, 3] = np.float16(0.25)
    dn = hl.down[:E * d * mid // 2].reshape(E, d, mid // 2)
    for e in range(E):
        col = dn[e, :, 23 * e].copy()
        dn[e] = 0x88
        dn[e, :, 23 * e] = (col & 15) | 0x80
    had = np.ones((1, 1), np.float32)
    while len(had) < 128:
        had = np.block([[had, had], [had, -had]])
    x = np.zeros((T, d // 128, 128), np.float32)
    x[np.arange(T), rng.integers(0, d // 128, T)] = had[rng.integers(0, 128, T)] * rng.choice([-2.0, 1.0, 0.5], (T, 1)).astype(np.float32)
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_V2_FUSED_MIDDLE, fused)
    ys = []
    for on in (1, 0):
        m.set_option(capi.OPT_STREAM_GEMM, on)
        ys.append(m.forward(0, gpu(x.reshape(T, d))).cpu().numpy())
        assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert np.abs(ys[1]).max() > 0
    assert (ys[0] == ys[1]).all()


# where the code planes lie against the cache lines (a blob's codes start 64 bytes behind it): the streaming GEMM turns its lines by half
# a line where rows start in the middle of one -- in one tensor of a launch, in both, in none; rows of one line, of more
# scales than are fetched at once (twelve lines) and of half a line more; tiles of 16, 32 and 64 pairs
@pytest.mark.parametrize("kind", ["q4cp", "table"])
@pytest.mark.parametrize("d,T", [(256, 33), (512, 64), (2560, 40), (3072, 64), (3328, 33), (640, 40), (3328, 70), (512, 130)])
def test_lines_against_cache_lines(capi, oracle, kind, d, T):
    import torch
    rng = np.random.default_rng(d + T)
    E, k, mid = 16, 4, 256
    cb = None if kind == "q4cp" else np.sort(rng.standard_normal(16)).astype(np.float32)
    hl = HostLayer(rng, d, mid, E, k, codebook=cb)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)

    def at(name, offset):  # the blob moved by `offset` bytes inside an allocation
        t = dev[name]
        buf = torch.zeros(t.numel() + 256, dtype=torch.uint8, device="cuda")
        buf[offset:offset + t.numel()] = t
        dev[name + str(offset)] = buf
        return buf[offset:offset + t.numel()]
    ys = []
    for experts, shared in ((0, 0), (64, 64), (64, 0), (0, 64), (16, 48)):
        m.set_experts_q4cp(0, capi.wview(at("gate_up", experts), capi.Q4CP, E * 2 * mid, d),
                           capi.wview(at("down", experts), capi.Q4CP, E * d, mid))
        m.set_shared(0, capi.wview(at("shg", 0), capi.Q4CP, mid, d), capi.wview(at("shu", shared), capi.Q4CP, mid, d),
                     capi.wview(at("shd", shared), capi.Q4CP, d, mid), capi.wview(dev["shsg"], capi.F32, 1, d))
        ys.append(m.forward(0, gpu(x)).cpu().numpy())
        assert m.last_path() == capi.PATH_BATCH
        assert max_abs_rel(ys[-1], yo) <= 2e-3  # (as the other whole-layer tests of batches: f16 operands and intermediates)
    m.close()
    # against one another: the order of f32 sums of d terms, and f16 roundings of hid and pairs that it tips over (2^-11 each)
    assert max(max_abs_rel(y, ys[0]) for y in ys[1:]) <= 2 * 2.0 ** -11


# rows of hid of one line to eight, with and without a half line at the end; rows of d that are no whole blocks of sixteen waves
STREAM_WIDTHS = [("q4cp", dict(fmt="q4cp"), 640, 256), ("q4cp", dict(fmt="q4cp"), 896, 384), ("q4cp", dict(fmt="q4cp"), 512, 1152),
                 ("q4cp", dict(fmt="q4cp"), 384, 2048), ("q4cp", dict(fmt="q4cp"), 256, 2560), ("q4cp-table", dict(fmt="q4cp", codebook=TABLE), 640, 512),
                 ("q4cp-table", dict(fmt="q4cp", codebook=TABLE), 256, 1024), ("q4cp-table", dict(fmt="q4cp", codebook=TABLE), 384, 1408),
                 ("q4k", dict(fmt="q4k"), 768, 256), ("q4k", dict(fmt="q4k"), 256, 1024), ("q4k", dict(fmt="q4k"), 512, 1536),
                 ("i4r", dict(fmt="i4r"), 768, 256), ("i4r", dict(fmt="i4r"), 256, 1024),
                 ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 768, 384), ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 256, 896),
                 ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 1280), ("q4k-q8_0", dict(fmt="q4k", gg_types=(12, 8, 8)), 256, 512)]


@pytest.mark.parametrize("T", [40, 88, 152])
@pytest.mark.parametrize("kind,kw,d,mid", STREAM_KINDS + STREAM_WIDTHS + [("i4r", dict(fmt="i4r"), 512, 768),
                                                          ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 640),
                                                          ("q4k-q8_0", dict(fmt="q4k", gg_types=(12, 8, 8)), 512, 640)])
def test_few_pair_tiles_are_no_less_exact(capi, oracle, kind, kw, d, mid, T):
    """All rows, dense activations: the 2-norm error against the oracle is that of the 128-pair kernel the layer would take
    otherwise (roundings of x, hid and pairs to f16 and of the weights, 3 .. 6e-4; another order of the f32 sums moves it
    by less than a hundredth).  Q5_K and Q4_K beside Q8_0 with widths that are no multiples of 256 take
    the general kernel there, which rounds a weight once."""
    rng = np.random.default_rng(T + mid)
    hl = HostLayer(rng, d, mid, 16, 4, bias=np.linspace(0, 0.5, 16, dtype=np.float32), **kw)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo = oracle.moe_layer(hl.oracle_layer(), x)[0].astype(np.float64)
    y1, y0 = both_kernels(capi, hl, x)
    e1, e0 = (np.linalg.norm(y - yo) / np.linalg.norm(yo) for y in (y1, y0))
    assert e1 <= 1.02 * e0 <= 1e-3, (e1, e0)
    assert (y1 != y0).any() or (mid > 1024 and T > 100)  # (two kernels; longer rows leave them earlier)


def k4_scale_bytes(sc, mn):
    """The 12 bytes of eight 6-bit scales and minima."""
    b = np.empty(sc.shape[:-1] + (12,), np.uint8)
    b[..., 0:4] = sc[..., 0:4] | (sc[..., 4:8] >> 4) << 6
    b[..., 4:8] = mn[..., 0:4] | (mn[..., 4:8] >> 4) << 6
    b[..., 8:12] = (sc[..., 4:8] & 15) | (mn[..., 4:8] & 15) << 4
    return b


@pytest.mark.parametrize("ratio", [1.0, 0.125])
@pytest.mark.parametrize("tgu", [12, 13])
def test_few_pair_tiles_round_weights_beside_q8_0_rows_once(capi, tgu, ratio):
    """Q4_K / Q5_K gate/up weights themselves: a token is one column of ones, gate rows are all 32 (silu(32) = 32 in f32), a down row picks one hid
    column, one expert a token: y is 32 times a weight as the kernel has it.  It is the f16 nearest to d * sc * n - dmin * m, unless its
    f32 value was rounded onto the middle between two, one of 2^13 places, from the other side: 2^-14 of the weights at most."""
    rng = np.random.default_rng(tgu)
    d, mid, E, T = 512, 640, 16, 512
    hl = HostLayer(rng, d, mid, E, 1, fmt="q4k", gg_types=(tgu, 8, 8), shared=False)
    nb, five = d // 256, tgu == 13
    size, most = (176, 31) if five else (144, 15)

    def rows(dd, dmin, sc, mn, n):  # n: codes [E, mid, nb, 4 pairs of sub-blocks, 2, 32]
        b = np.zeros((E, mid, nb, size), np.uint8)
        b[..., 0:2] = dd[..., None].view(np.uint8)
        b[..., 2:4] = dmin[..., None].view(np.uint8)
        b[..., 4:16] = k4_scale_bytes(sc, mn)
        b[..., size - 128:] = ((n[..., 0, :] & 15) | (n[..., 1, :] & 15) << 4).reshape(E, mid, nb, 128)
        if five:
            for j in range(8):
                b[..., 16:48] |= (n[..., j // 2, j % 2, :] >> 4) << j
        return b.reshape(-1)
    one = np.ones((E, mid, nb), np.float16)
    full = lambda v: np.full((E, mid, nb, 8), v, np.uint8)
    hl.gate = rows(one, 0 * one, full(32), full(0), np.ones((E, mid, nb, 4, 2, 32), np.uint8))
    dd = (np.abs(rng.standard_normal((E, mid, nb))) * 0.01 + 0.002).astype(np.float16)
    dmin = (dd.astype(np.float32) * ratio * rng.uniform(0.5, 2, dd.shape)).astype(np.float16)
    sc, mn = (rng.integers(0, 64, (E, mid, nb, 8)).astype(np.uint8) for _ in range(2))
    n = rng.integers(0, most + 1, (E, mid, nb, 4, 2, 32)).astype(np.uint8)
    hl.up = rows(dd, dmin, sc, mn, n)
    dn = np.zeros((E, d, mid // 32, 34), np.uint8)
    dn[..., 0:2] = np.ones(1, np.float16).view(np.uint8)
    pick = (5 * np.arange(d)[None] + np.arange(E)[:, None]) % mid
    ee, rr = np.meshgrid(np.arange(E), np.arange(d), indexing="ij")
    dn[ee, rr, pick // 32, 2 + pick % 32] = 1
    hl.down = dn.reshape(-1)
    w = (dd.astype(np.float64)[..., None] * sc)[..., None] * n.reshape(E, mid, nb, 8, 32)
    w = (w - (dmin.astype(np.float64)[..., None] * mn)[..., None]).reshape(E, mid, d)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(np.eye(T, d, dtype=np.float32))).cpu().numpy()
    e = m.last_routing(T)[0].cpu().numpy()[:, 0]
    m.close()
    want = w[e[:, None], pick[e], np.arange(T)[:, None]].astype(np.float16)
    far = np.abs(want) >= 0.03  # (32 of these are no f16 denormals, whatever the power of two that hid is kept at)
    got = (y / 32).astype(np.float16)
    assert far.mean() > 0.9 and np.abs(got[far].view(np.int16).astype(int) - want[far].view(np.int16)).max() <= 1
    assert (got != want)[far].mean() <= 2.0 ** -14 + 4 * (2.0 ** -14 / far.sum()) ** 0.5


@pytest.mark.parametrize("kind,kw,d,mid,last", [("q4cp", dict(fmt="q4cp"), 512, 640, 50), ("q4cp", dict(fmt="q4cp"), 384, 1152, 25),
                                                ("table", dict(fmt="q4cp", codebook=TABLE), 512, 768, 60), ("i4r", dict(fmt="i4r"), 512, 768, 50),
                                                ("table", dict(fmt="q4cp", codebook=TABLE), 384, 1152, 29), ("q4k", dict(fmt="q4k"), 512, 768, 50),
                                                ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 768, 38),
                                                ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 1280, 32),
                                                ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 640, 160)])
def test_where_the_few_pair_tiles_end(capi, oracle, kind, kw, d, mid, last):
    """The largest batch that each kind of layer runs on them, and the next one on the 128-pair kernels."""
    E, k = 16, 4
    T = last * E // k
    rng = np.random.default_rng(T + mid)
    hl = HostLayer(rng, d, mid, E, k, **kw)
    x = rng.standard_normal((T + 1, d), dtype=np.float32)
    sel = np.r_[0, T // 2, T - 1]
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x[sel])
    y1, y0 = both_kernels(capi, hl, x[:T])
    assert (y1 != y0).any()
    assert max_abs_rel(y1[sel], yo) <= 2e-3
    y1, y0 = both_kernels(capi, hl, x)
    assert (y1 == y0).all()


@pytest.mark.parametrize("E,last", [(63, 38), (64, 31)])
def test_where_the_few_pair_tiles_of_many_q5k_experts_end(capi, oracle, E, last):
    """Q5_K / Q8_0: with experts that fill the chip in 128-pair tiles the line lies lower."""
    k, d, mid = 3, 512, 256
    T = last * E // k
    rng = np.random.default_rng(E)
    hl = HostLayer(rng, d, mid, E, k, fmt="q4k", gg_types=(13, 8, 8))
    x = rng.standard_normal((T + 1, d), dtype=np.float32)
    sel = np.r_[0, T // 2, T]
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x[sel])
    y1, y0 = both_kernels(capi, hl, x[:T])
    assert (y1 != y0).any()
    y1, y0 = both_kernels(capi, hl, x)
    assert (y1 == y0).all()
    assert max_abs_rel(y1[sel], yo) <= 2e-3


@pytest.mark.parametrize("fmt,codebook,last", [("q4cp", "zp8", 62), ("q4cp", "universal", 70), ("q4k", "zp8", 60), ("i4r", "zp8", 60)])
def test_where_the_few_pair_tiles_of_many_weights_end(capi, fmt, codebook, last):
    """512 experts of 2048 x 768: the lines of layers whose weights are many.  The two kernels' outputs are each within 6e-4 of
    the exact ones in the 2-norm (test_few_pair_tiles_are_no_less_exact)."""
    import torch
    from gfx1151_engine_amd import workloads as W
    d, mid, E, k = 2048, 768, 512, 10
    T = last * E // k
    L = W.DeviceLayer(5, d, mid, E, k, fmt, codebook=codebook)
    m = capi.Moe(d, mid, E, k, max_tokens=T + 1)
    L.register(m, 0)
    x = torch.randn((T + 1, d), device="cuda", generator=torch.Generator(device="cuda").manual_seed(T))
    for n, same in ((T, False), (T + 1, True)):
        ys = []
        for on in (1, 0):
            m.set_option(capi.OPT_STREAM_GEMM, on)
            ys.append(m.forward(0, x[:n].contiguous()).double())
        assert torch.equal(ys[0], ys[1]) == same
        assert float((ys[0] - ys[1]).norm() / ys[1].norm()) <= 1.2e-3
    m.close()


def ends_at(capi, L, d, mid, E, k, T):
    """T tokens are the largest batch of layer L on the few-pair tiles.  The two kernels' outputs are each within 6e-4 of the exact
    ones in the 2-norm (test_few_pair_tiles_are_no_less_exact)."""
    import torch
    m = capi.Moe(d, mid, E, k, max_tokens=T + 1)
    L.register(m, 0)
    x = torch.randn((T + 1, d), device="cuda", generator=torch.Generator(device="cuda").manual_seed(T))
    for n, same in ((T, False), (T + 1, True)):
        ys = []
        for on in (1, 0):
            m.set_option(capi.OPT_STREAM_GEMM, on)
            ys.append(m.forward(0, x[:n].contiguous()).double())
        assert torch.equal(ys[0], ys[1]) == same
        assert float((ys[0] - ys[1]).norm() / ys[1].norm()) <= 1.2e-3
    m.close()


@pytest.mark.parametrize("fmt,codebook,d,mid,E,last", [("q4cp", "zp8", 3072, 768, 256, 62), ("q4cp", "zp8", 2048, 768, 256, 50),
                                                       ("q4cp", "universal", 1024, 512, 1000, 70), ("q4cp", "universal", 1024, 768, 256, 60),
                                                       ("q4k", "zp8", 2048, 1024, 256, 60), ("i4r", "zp8", 3072, 768, 192, 50)])
def test_which_layers_have_many_weights(capi, fmt, codebook, d, mid, E, last):
    from gfx1151_engine_amd import workloads as W
    ends_at(capi, W.DeviceLayer(6, d, mid, E, 8, fmt, codebook=codebook), d, mid, E, 8, last * E // 8)


@pytest.mark.parametrize("types,d,mid,E,last", [((12, 8, 8), 2048, 768, 256, 31), ((13, 8, 8), 2048, 768, 256, 29), ((12, 8, 8), 1024, 768, 64, 26),
                                                ((13, 8, 12), 1024, 768, 64, 22), ((12, 8, 8), 512, 512, 32, 38), ((13, 8, 8), 512, 512, 32, 38),
                                                ((12, 8, 8), 768, 1536, 64, 28), ((13, 8, 8), 768, 1536, 64, 26)])
def test_where_the_few_pair_tiles_beside_8_bit_down_rows_end(capi, types, d, mid, E, last):
    from gfx1151_engine_amd import workloads as W
    ends_at(capi, W.DeviceLayer(7, d, mid, E, 8, "q4k", gg_types=types), d, mid, E, 8, last * E // 8)


@pytest.mark.parametrize("fmt,T", [("q4cp", 40), ("q4cp", 300), ("q4k", 300), ("q4cp", 1100)])
def test_the_callers_f16_copy_at_every_router(capi, fmt, T):
    """moe_forward_x16 against moe_forward, bit for bit; the router of 257 tokens and more makes its own copy all the same."""
    rng = np.random.default_rng(T)
    hl = HostLayer(rng, 512, 256, 16, 4, fmt=fmt)
    m, dev = hl.to_gpu(max_tokens=T)
    x = gpu(rng.standard_normal((T, 512), dtype=np.float32))
    y0 = m.forward(0, x).cpu().numpy()
    i0 = m.last_routing(T)[0].cpu().numpy()
    y1 = m.forward_x16(0, x, capi.f32_to_f16(x, layout=m.x16_layout(0))).cpu().numpy()
    assert (y0 == y1).all() and (m.last_routing(T)[0].cpu().numpy() == i0).all()
    m.close()


@pytest.mark.parametrize("pairs", [(33, 33), (32, 48), (49, 47), (48, 16), (63, 17), (64, 33), (65, 31)])
@pytest.mark.parametrize("kind,kw,d,mid", [("q4cp", dict(fmt="q4cp"), 1152, 640), ("q4cp-affine", dict(fmt="q4cp"), 512, 256),
                                           ("q4cp-table", dict(fmt="q4cp", codebook=TABLE), 640, 640), ("i4r", dict(fmt="i4r"), 512, 256),
                                           ("q4k", dict(fmt="q4k"), 768, 256)])
def test_tiles_of_33_to_64_pairs(capi, oracle, kind, kw, d, mid, pairs):
    """Whole tiles and the edges of their 16-pair groups, lines of d that are four, one more, and half of one: two experts
    that share the batch by the sign of one column.  All rows against the oracle, the grouped GEMM's tolerance."""
    rng = np.random.default_rng(sum(pairs) + d)
    hl = HostLayer(rng, d, mid, 4, 1, shared=False, bias=np.float32([0, 0, -90, -90]), **kw)
    hl.router[:] = 0
    hl.router[0, 0], hl.router[1, 0] = 40, -40
    if kind == "q4cp-affine":  # no scaled dequantisation
        hl.gate_up[64 + 8 * mid * d // 2:].view(np.float16).reshape(4, 2 * mid, -1)[:, 3, :] = np.float16(1e-5)
    x = rng.standard_normal((sum(pairs), d), dtype=np.float32)
    x[:, 0] = rng.permutation(np.repeat(np.float32([1, -1]), pairs))
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    assert np.bincount(io[:, 0]).tolist() == list(pairs)
    y1, y0 = both_kernels(capi, hl, x)
    assert max_abs_rel(y1, yo) <= 2e-3
    assert (y1 != y0).any()  # (its own kernel)


@pytest.mark.parametrize("T", [40, 88, 152])
@pytest.mark.parametrize("shared", ["its own tables", "the same values", "none"])
def test_row_scales_beside_one_table_and_two(capi, oracle, shared, T):
    """Table codebooks, tiles of 16, 32 and 64 pairs: with two pair tables the row scales of hid are read in the epilogue, with one
    they wait in LDS.  Rows of a thousandth to three hundred times the usual size, so that a tile's scales differ; every row against
    the oracle by its own size, the layer's tolerance."""
    rng = np.random.default_rng(T)
    kw = {"its own tables": dict(shared_codebooks=[TABLE, TABLE[::-1].copy(), TABLE * 0.5]), "the same values": {}, "none": dict(shared=False)}
    hl = HostLayer(rng, 512, 384, 16, 4, fmt="q4cp", codebook=TABLE, **kw[shared])
    x = rng.standard_normal((T, 512), dtype=np.float32) * np.float32(10) ** rng.uniform(-3, 2.5, (T, 1)).astype(np.float32)
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert (np.abs(y - yo).max(1) <= 2e-3 * np.abs(yo).max(1)).all()


# ---------- 8-bit codes from memory into registers (gemm_wide.hip): tiles of 1 .. 128 pairs, stages of 128 columns ----------
@pytest.mark.parametrize("pairs", [(1, 32), (33, 64), (65, 96), (97, 128), (129, 31)])
@pytest.mark.parametrize("kind,kw,d,mid", [
    ("q5k-q8_0", dict(fmt="q4k", gg_types=(13, 8, 8)), 512, 768), ("q8_0", dict(fmt="q4k", gg_types=(8, 8, 8)), 384, 128),
    ("q8_0-narrow", dict(fmt="q4k", gg_types=(8, 8, 8)), 640, 320), ("q4k-q8_0", dict(fmt="q4k", gg_types=(12, 8, 8)), 512, 640),
    ("q8g32", dict(fmt="q4cp", shared_dense="q8g32"), 512, 640), ("q8g32-table", dict(fmt="q4cp", codebook=TABLE, shared_dense="q8g32"), 384, 256),
    ("q8g32-i4r", dict(fmt="i4r", shared_dense="q8g32"), 256, 768)])
def test_8_bit_codes_in_tiles_of_every_size(capi, oracle, kind, kw, d, mid, pairs):
    """Two experts that share the batch by the sign of one column (the shared expert has all of it), groups of 32 pairs and
    one more or less; columns of one stage to six, rows that are no whole blocks; widths that the general kernel keeps (320).
    Tolerance: that of the grouped GEMMs."""
    rng = np.random.default_rng(sum(pairs) + d)
    hl = HostLayer(rng, d, mid, 4, 1, bias=np.float32([0, 0, -90, -90]), **kw)
    hl.router[:] = 0
    hl.router[0, 0], hl.router[1, 0] = 40, -40
    T = sum(pairs)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[:, 0] = rng.permutation(np.repeat(np.float32([1, -1]), pairs))
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    assert np.bincount(io[:, 0]).tolist() == list(pairs)
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_STREAM_GEMM, 0)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert max_abs_rel(y, yo) <= 2e-3


@pytest.mark.parametrize("E", [5, 7, 8, 16, 17])
def test_8_bit_codes_on_few_tiles_and_more(capi, oracle, E):
    """Six tiles to eighteen, the shared expert's among them: up to eight are dealt out to the XCDs block by block."""
    rng = np.random.default_rng(E)
    hl = HostLayer(rng, 512, 384, E, E // 2, fmt="q4k", gg_types=(8, 8, 8))
    x = rng.standard_normal((60, 512), dtype=np.float32)
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    assert (np.bincount(io[:, :E // 2].ravel(), minlength=E) > 0).all()
    m, dev = hl.to_gpu(max_tokens=60)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert max_abs_rel(y, yo) <= 2e-3


@pytest.mark.parametrize("d,mid,E", [(2560, 128, 205), (2560, 256, 205), (1536, 128, 512)])
def test_8_bit_down_blocks_of_several_row_groups(capi, oracle, d, mid, E):
    """Down blocks that walk two neighbouring groups of 256 rows (of ten) and three (of six), one stage of columns to a pass and two:
    what a pass leaves behind for the next one."""
    rng = np.random.default_rng(d + mid)
    hl = HostLayer(rng, d, mid, E, 4, fmt="q4k", gg_types=(8, 8, 8))
    x = rng.standard_normal((33, d), dtype=np.float32)
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=33)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert max_abs_rel(y, yo) <= 2e-3


@pytest.mark.parametrize("types,T", [((13, 8, 8), 64), ((13, 8, 8), 65), ((13, 8, 8), 512), ((13, 8, 8), 513), ((8, 8, 8), 257), ((8, 8, 8), 520)])
def test_8_bit_shared_experts_alone(capi, oracle, types, T):
    """A shared expert's own launches on either side of the line between the kernels (one tile of 64, five of 128), and all-Q8_0 layers
    whose routed gate/up has few blocks."""
    rng = np.random.default_rng(T)
    hl = HostLayer(rng, 512, 256, 4, 2, fmt="q4k", gg_types=types)
    x = rng.standard_normal((T, 512), dtype=np.float32)
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert max_abs_rel(y, yo) <= 2e-3


# ---------- Q5_K in 128-pair tiles: rows that end inside a block, one super-block and several, tiles of every size ----------
@pytest.mark.parametrize("d,mid,E,T", [(256, 320, 8, 40), (512, 192, 2, 150), (768, 64, 3, 200), (1024, 960, 4, 70)])
def test_fifth_bits_of_part_filled_row_blocks(capi, oracle, d, mid, E, T):
    rng = np.random.default_rng(d + mid)
    hl = HostLayer(rng, d, mid, E, 2, fmt="q4k", gg_types=(13, 8, 8))
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_STREAM_GEMM, 0)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.last_path() == capi.PATH_BATCH
    m.close()
    assert max_abs_rel(y, yo) <= 2e-3
