"""GPU parity of the whole layer through moe_forward against the oracle (the restated
src/ref.cpp Model::moe): router ids bit-exact, y within max-abs-rel 2e-3 (the small-batch f32
kernels are held to 1e-4, the integer-dot kernels to 2e-4 (q4cp) and 5e-4 (Q4_K))."""
import zlib

import numpy as np
import pytest

from gfx1151_engine_amd import synth as S

from helpers import HostLayer, bits, max_abs_rel

pytestmark = pytest.mark.gpu

TOL_LAYER = 2e-3   # stated tolerance for the layer (f16/bf16 MFMA path)
TOL_GEMV = 1e-4    # small-batch GEMV path, f32 kernels
TOL_INT_Q4CP = 2e-4  # integer-dot kernels, q4cp: activations as four 4-bit digit planes per 32-group (worst of
                     # 60 seeds at one token: 7.8e-5)
TOL_INT_Q4K = 5e-4  # integer-dot kernels on raw Q4_K blocks: activations as two 8-bit digit planes per
                    # 32-group; the unsigned codes (w = d*sc*n - dmin*m, n in 0..15) double the weight of
                    # the activations' rounding against the zero-centred q4cp codes (worst of 80 seeds: 2.4e-4)


def tol_small(fmt):
    return TOL_INT_Q4K if fmt == "q4k" else TOL_INT_Q4CP


def gpu(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def run_layer(hl, x, max_tokens=None):
    m, dev = hl.to_gpu(max_tokens=max_tokens or max(32, x.shape[0]))
    y = m.forward(0, gpu(x))
    ids, ws = m.last_routing(x.shape[0])
    out = y.cpu().numpy(), ids.cpu().numpy(), ws.cpu().numpy()
    m.close()
    return out


@pytest.mark.parametrize("fmt,d,mid,E,k,T,cb", [
    ("q4cp", 3072, 768, 32, 10, 1, None), ("q4cp", 3072, 768, 32, 10, 20, None),
    ("q4cp", 640, 160, 16, 4, 7, "random"), ("q4k", 3072, 768, 24, 10, 1, None),
    ("q4k", 3072, 768, 24, 10, 20, None), ("q4k", 256, 256, 8, 3, 5, None)])
def test_small_batch_layer(oracle, fmt, d, mid, E, k, T, cb):
    rng = np.random.default_rng(zlib.crc32(f"{fmt}-{d}-{T}".encode()))  # (hash() of a str changes per process)
    codebook = rng.uniform(-2, 2, 16).astype(np.float32) if cb == "random" else None
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt, codebook=codebook)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all(), "router ids must be bit-exact"
    assert np.abs(ws[:, :k] - wo[:, :k]).max() <= 1e-6
    assert max_abs_rel(y, yo) <= tol_small(fmt), max_abs_rel(y, yo)


TOL_LUT = 2e-5  # look-up kernels for codebooks that are not a*n + b: f32 throughout (f32 sums against the
                # reference's fp64 ones; the order of the additions is the only difference from the f32 GEMV kernels)


@pytest.mark.parametrize("T", [1, 2, 5, 6, 20, 32])
@pytest.mark.parametrize("kind", ["universal", "random"])
def test_small_batch_table_codebooks(oracle, T, kind):
    """The reference converter's fixed non-uniform table (tools/flashnext2hgn.py:530-531) in every routed-expert
    tensor, and a table of its own in each of the shared expert's tensors (:164-187): the look-up decode kernels
    against the oracle, and the plain f32 kernels (MOE_OPT_INT_DECODE = 0) as a second opinion."""
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(500 + T)
    d, mid, E, k = 3072, 768, 24, 10
    cb = S.UNIVERSAL_CODEBOOK if kind == "universal" else np.sort(rng.standard_normal(16)).astype(np.float32)
    scb = [np.sort(rng.standard_normal(16)).astype(np.float32) * (0.5 + i) for i in range(3)]
    hl = HostLayer(rng, d, mid, E, k, codebook=cb, shared_codebooks=scb, scale_std=0.05)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[0] *= 300.0  # (each 32-group of activations is rescaled by a power of two on its way to f16)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=32)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids, ws = m.last_routing(T)
    assert (ids.cpu().numpy()[:, :k] == io[:, :k]).all()
    assert np.abs(ws.cpu().numpy()[:, :k] - wo[:, :k]).max() <= 1e-6
    err = max(max_abs_rel(y[t], yo[t]) for t in range(T))  # per token: token 0 is 300 times larger
    assert err <= TOL_LUT, err  # (up to 5 tokens the look-up kernels, beyond that the plain f32 kernels)
    m.set_option(capi.OPT_INT_DECODE, 0)
    y2 = m.forward(0, gpu(x)).cpu().numpy()
    assert max(max_abs_rel(y2[t], yo[t]) for t in range(T)) <= TOL_GEMV
    m.close()


@pytest.mark.parametrize("T", [1, 3, 6])
@pytest.mark.parametrize("d", [2016, 2048, 2080, 2304, 2560, 2592, 3072])
@pytest.mark.parametrize("kind", ["q4cp", "table"])
def test_small_batch_gate_up_rows_of_64_groups_and_more(oracle, kind, d, T):
    """Gate/up rows of 63 to 96 groups: none behind the first 64, up to 16 (four rows' to a pass) and more (two rows')."""
    rng = np.random.default_rng(d + T)
    cb = np.sort(rng.standard_normal(16)).astype(np.float32) if kind == "table" else None
    hl = HostLayer(rng, d, 64, 12, 4, codebook=cb, scale_std=0.05)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :4] == io[:, :4]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= (TOL_LUT if kind == "table" else TOL_INT_Q4CP)


@pytest.mark.parametrize("most", [0, 32])
@pytest.mark.parametrize("T", [1, 2, 4])
@pytest.mark.parametrize("d,mid,E", [(256, 32, 20), (512, 96, 20), (384, 160, 600), (768, 352, 20), (3072, 1024, 12)])
def test_small_batch_table_gate_up_rows_of_a_block(oracle, d, mid, E, T, most):
    """Gate/up blocks of twelve rows (the selection inside) and of sixteen (ids given): widths that are and are no multiples of
    twelve, the last block with rows past mid, more than 512 experts."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(d + mid + T)
    hl = HostLayer(rng, d, mid, E, 4, codebook=np.sort(rng.standard_normal(16)).astype(np.float32), scale_std=0.05,
                   shared_codebooks=[np.sort(rng.standard_normal(16)).astype(np.float32) for _ in range(3)])
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_GU_TOPK_MAX_TOKENS, most)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids, _ = m.last_routing(T)
    m.close()
    assert (ids.cpu().numpy()[:, :4] == io[:, :4]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_LUT


@pytest.mark.parametrize("T", [1, 3, 6])
@pytest.mark.parametrize("mid", [256, 512, 768, 1024])
@pytest.mark.parametrize("types,k,shared", [((13, 8, 8), 1, True), ((13, 8, 8), 10, True), ((12, 8, 12), 5, True), ((13, 13, 8), 15, True),
                                            ((13, 8, 8), 6, False), ((8, 7, 12), 13, True)])
def test_small_batch_gguf_rows_of_packed_units(oracle, types, k, shared, mid, T):
    """Down rows of 4 to 16 units of 64 columns: one slot to fifteen, the last wave full and not, the shared expert's rows in its groups of
    lanes, its type the routed experts' and another."""
    rng = np.random.default_rng(mid + 10 * T + k)
    hl = HostLayer(rng, 256, mid, 20, k, fmt="q4k", gg_types=types, shared=shared)
    x = rng.standard_normal((T, 256), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_INT_Q4K


@pytest.mark.parametrize("T", [1, 3, 4, 5, 9])
@pytest.mark.parametrize("d,mid", [(768, 768), (512, 768), (384, 640), (544, 640), (768, 512), (544, 512)])
@pytest.mark.parametrize("kind,k,shared", [("q4cp", 1, False), ("q4cp", 10, True), ("q4cp", 15, True), ("table", 3, True), ("table", 10, True), ("table", 12, False)])
def test_small_batch_rows_of_packed_groups(oracle, kind, k, shared, d, mid, T):
    """Down rows of 16, 20 and 24 groups, which four slots to a wave share: one slot to sixteen (waves with slots left over), widths
    that are and are not whole blocks of 12 and 16 rows, the shared expert with codebooks and scale strides of its own."""
    rng = np.random.default_rng(d + mid + 10 * T + k)
    cb = np.sort(rng.standard_normal(16)).astype(np.float32) if kind == "table" else None
    scb = [np.sort(rng.standard_normal(16)).astype(np.float32) for _ in range(3)] if kind == "table" else None
    hl = HostLayer(rng, d, mid, 20, k, codebook=cb, shared_codebooks=scb, shared=shared, scale_std=0.05)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= (TOL_LUT if kind == "table" else TOL_INT_Q4CP)


@pytest.mark.parametrize("limit", [0, 3, 32])
@pytest.mark.parametrize("codebook", ["affine", "universal"])
def test_f32_decode_token_limit(oracle, limit, codebook):
    """MOE_OPT_F32_DECODE_MAX_TOKENS moves the batch size at which the f32 path's down launch changes from the
    register-resident kernel to the plain one: every setting gives the oracle's ids and meets the f32 bar at 2, 4 and
    20 tokens (affine codebook with the integer-dot kernels off; the converter's table with them on)."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(9100 + limit)
    d, mid, E, k = 3072, 768, 24, 10
    hl = HostLayer(rng, d, mid, E, k, codebook=S.UNIVERSAL_CODEBOOK, scale_std=0.05) if codebook == "universal" else \
        HostLayer(rng, d, mid, E, k)
    m, dev = hl.to_gpu(max_tokens=32)
    if codebook == "affine":
        m.set_option(capi.OPT_INT_DECODE, 0)
    m.set_option(capi.OPT_F32_DECODE_MAX_TOKENS, limit)
    for T in (2, 4, 20):
        x = rng.standard_normal((T, d), dtype=np.float32)
        yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
        y = m.forward(0, gpu(x)).cpu().numpy()
        ids, ws = m.last_routing(T)
        assert (ids.cpu().numpy()[:, :k] == io[:, :k]).all(), T
        assert np.abs(ws.cpu().numpy()[:, :k] - wo[:, :k]).max() <= 1e-6
        assert max_abs_rel(y, yo) <= TOL_GEMV, (T, max_abs_rel(y, yo))
    with pytest.raises(capi.MoeError):
        m.set_option(capi.OPT_F32_DECODE_MAX_TOKENS, 33)
    m.close()


@pytest.mark.parametrize("fmt,T,rdt", [("q4cp", 3, "f32"), ("q4cp", 32, "f32"), ("q4k", 27, "f32"), ("q4k", 2, "f32"),
                                        ("q4cp", 1, "bf16"), ("q4cp", 4, "bf16"), ("q4cp", 5, "f32"), ("q4cp", 11, "f32"), ("q4cp", 12, "bf16"), ("q4cp", 17, "f32"),
                                        ("q4k", 30, "bf16")])
def test_small_batch_sizes_and_router_dtypes(oracle, fmt, T, rdt):
    """The token counts at which the small path changes kernels (1 / 2-4 / 5-24 / 25-32: the logits
    launch differs, above 24 tokens it is split in two) with f32 and bf16 router matrices."""
    rng = np.random.default_rng(4242 + 7 * T + (rdt == "bf16"))
    d, mid, E, k = 3072, 768, 24, 10
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt, router_dtype=rdt)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all(), "router ids must be bit-exact"
    assert np.abs(ws[:, :k] - wo[:, :k]).max() <= 1e-6
    assert max_abs_rel(y, yo) <= tol_small(fmt), max_abs_rel(y, yo)


@pytest.mark.parametrize("T", [3, 6, 12, 21, 30])
@pytest.mark.parametrize("rdt", ["f32", "bf16"])
def test_small_batch_router_without_gate_vector_and_ragged_rows(oracle, T, rdt):
    """A layer without a shared expert (no gate vector beside the router matrix) whose expert count is not a multiple
    of the router launch's rows per block, at a width where 5..24 tokens take the row-per-wave launch (d not a
    multiple of 256): the padding rows of the last block read the router matrix, never the absent gate vector."""
    rng = np.random.default_rng(3300 + T + (rdt == "bf16"))
    d, mid, E, k = 320, 256, 33, 4
    hl = HostLayer(rng, d, mid, E, k, router_dtype=rdt, shared=False,
                   bias=rng.standard_normal(E).astype(np.float32) * 0.1)
    x = rng.standard_normal((T, d), dtype=np.float32) * 3
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all(), "router ids must be bit-exact"
    assert np.abs(ws[:, :k] - wo[:, :k]).max() <= 1e-6
    assert max_abs_rel(y, yo) <= TOL_INT_Q4CP, max_abs_rel(y, yo)


@pytest.mark.parametrize("fmt,T", [("q4cp", 1), ("q4cp", 3), ("q4cp", 5), ("q4cp", 6), ("q4cp", 9), ("q4cp", 32),
                                   ("q4k", 1), ("q4k", 9)])
def test_int_decode_switch(oracle, fmt, T):
    """MOE_OPT_INT_DECODE 1 (integer-dot kernels, default) and 0 (f32 kernels) both meet the GEMV bar
    and select the same experts.  (q4cp with the switch at 0: up to 4 tokens the register-resident f32 kernels with
    the top-k inside the gate/up launch, at 5 with the ids from the router's launches, from 6 on the plain f32 down
    kernel behind the register-resident gate/up launch.)"""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(77 + T)
    d, mid, E, k = 3072, 768, 16, 10
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=32)
    ys = []
    for opt in (1, 0):
        m.set_option(capi.OPT_INT_DECODE, opt)
        y = m.forward(0, gpu(x)).cpu().numpy()
        ids, _ = m.last_routing(T)
        assert (ids.cpu().numpy()[:, :k] == io[:, :k]).all()
        assert max_abs_rel(y, yo) <= (tol_small(fmt) if opt else TOL_GEMV), (opt, max_abs_rel(y, yo))
        ys.append(y)
    assert not (ys[0] == ys[1]).all(), "the two paths are different kernels (digit planes vs f32)"
    m.close()


@pytest.mark.parametrize("fmt,T", [("q4cp", 1), ("q4cp", 6), ("q4k", 1), ("q4k", 3)])
def test_decode_topk_near_ties(oracle, fmt, T):
    """The decode gate/up kernels rank the experts by logit and fall back to the exact softmax selection when two
    of the k + 1 best logits are closer than 1e-6.  Router rows repeated (equal logits: the lower index must come
    first, and a copy may sit on the rank k / k + 1 boundary) and rows that differ in the last bits force that
    fallback; ids and order must still be the oracle's."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(17 + T)
    d, mid, E, k = (3072, 768, 24, 10) if fmt == "q4cp" else (512, 256, 24, 10)
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt)
    hl.router[7] = hl.router[3]
    hl.router[20] = hl.router[3]
    hl.router[11] = hl.router[5]
    hl.router[16] = hl.router[5] * np.float32(1 + 2 ** -22)
    hl.router[2] = hl.router[9]
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=8)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids, ws = m.last_routing(T)
    ids, ws = ids.cpu().numpy(), ws.cpu().numpy()
    assert (ids[:, :k] == io[:, :k]).all(), (ids[:, :k], io[:, :k])
    assert np.abs(ws[:, :k] - wo[:, :k]).max() <= 1e-6
    assert max_abs_rel(y, yo) <= tol_small(fmt), max_abs_rel(y, yo)
    m.close()


@pytest.mark.parametrize("fmt", ["q4cp", "q4k"])
def test_decode_topk_wide_logit_range(oracle, fmt):
    """Router rows scaled so that the logits span hundreds: below the best few, the reference's f32 probabilities
    go subnormal or to zero and tie, and ties are ordered by expert index.  The gate/up launch of the decode path
    (which ranks by logit) and the down launch (which takes the ids of the exact selection) must still agree with
    each other and with the oracle: a slot that ran gate/up for one expert and down for another shows in y."""
    rng = np.random.default_rng(29)
    d, mid, E, k = (3072, 768, 24, 10) if fmt == "q4cp" else (512, 256, 24, 10)
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt)
    # rows in descending-logit order that runs AGAINST the index order: ties between underflowed probabilities
    # then come out by index, i.e. opposite to the logits
    x = rng.standard_normal((3, d), dtype=np.float32)
    u = x[0] / np.linalg.norm(x[0])
    hl.router[:] = 1e-3 * rng.standard_normal((E, d), dtype=np.float32)
    hl.router += np.outer(np.linspace(-9.0, 3.0, E), u).astype(np.float32)  # token 0: logits ~ 55 * (-9 .. 3)
    x[2] = 0.0                                                                # token 2: all logits equal
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    lg = oracle.router(hl.oracle_layer().router, x, k)[0]
    assert lg[0].max() - np.sort(lg[0])[-k] > 90, "the k-th logit of token 0 must lie in the underflow range"
    m, dev = hl.to_gpu(max_tokens=8)
    for T in (1, 3):
        y = m.forward(0, gpu(x[:T])).cpu().numpy()
        ids, ws = m.last_routing(T)
        ids, ws = ids.cpu().numpy(), ws.cpu().numpy()
        assert (ids[:, :k] == io[:T, :k]).all(), (T, ids[:, :k], io[:T, :k])
        assert np.abs(ws[:, :k] - wo[:T, :k]).max() <= 1e-6
        assert max_abs_rel(y, yo[:T]) <= tol_small(fmt), (T, max_abs_rel(y, yo[:T]))
    m.close()


@pytest.mark.parametrize("tgu,tdn,tsh,T", [(13, 8, 12, 1), (12, 7, 12, 5), (13, 7, 8, 3), (12, 8, 13, 40), (23, 20, 12, 2),
                                            (20, 23, 23, 7), (13, 8, 8, 1), (13, 8, 8, 20), (12, 7, 7, 32), (8, 13, 7, 2),
                                            (20, 20, 20, 1), (23, 23, 23, 4), (23, 20, 8, 19), (12, 23, 20, 30)])
def test_gguf_mixed_types(oracle, tgu, tdn, tsh, T):
    """GGUF layers in the type mix of the reference's checkpoints (Q4_K / Q5_K gate and up, Q5_1 / Q8_0 down, a Q8_0
    shared expert; src/gpu/parts/30_host_util.inc:399-405, src/gguf_map.h:212-214) and in the IQ4_NL / IQ4_XS types
    (src/gguf.h:376-407): every mix takes the integer-dot decode kernels (and, with MOE_OPT_INT_DECODE = 0, the general
    f32 GEMV kernels); ids bit-exact; T = 40 is a batch for the general grouped GEMM."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(tgu * 100 + tdn * 10 + T)
    d, mid, E, k = 512, 256, 12, 4
    hl = HostLayer(rng, d, mid, E, k, fmt="q4k", gg_types=(tgu, tdn, tsh))
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=64)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids, ws = m.last_routing(T)
    assert (ids.cpu().numpy()[:, :k] == io[:, :k]).all()
    assert np.abs(ws.cpu().numpy()[:, :k] - wo[:, :k]).max() <= 1e-6
    # batches over 32 tokens take the general grouped GEMM (f16 MFMA operands): the batch tolerance
    tol = 2e-3 if T > 32 else TOL_INT_Q4K
    assert max_abs_rel(y, yo) <= tol, max_abs_rel(y, yo)
    if T <= 32:
        m.set_option(capi.OPT_INT_DECODE, 0)
        y2 = m.forward(0, gpu(x)).cpu().numpy()
        assert max_abs_rel(y2, yo) <= TOL_GEMV, max_abs_rel(y2, yo)
    m.close()


@pytest.mark.parametrize("T", [1, 2, 4, 5, 9])
@pytest.mark.parametrize("types,d", [((12, 12, 12), 2048), ((12, 12, 12), 2560), ((12, 12, 12), 3072), ((12, 12, 12), 3584),
                                     ((13, 8, 8), 2048), ((13, 8, 8), 2560), ((13, 8, 8), 3072), ((13, 8, 8), 3584), ((8, 8, 13), 2560),
                                     ((7, 7, 12), 3072), ((20, 20, 23), 2560), ((23, 20, 20), 3584), ((13, 13, 7), 1792), ((12, 12, 12), 4096)])
def test_small_batch_gguf_gate_up_rows_dealt_over_a_wave(oracle, types, d, T):
    """Gate/up rows of 32, 40, 48 and 56 units, whose idle lanes take other rows (and of 28 and 64, which go a row at a time); the
    selection inside the launch and ahead of it; the shared expert of the experts' type and of another."""
    rng = np.random.default_rng(d + 10 * T + types[0])
    hl = HostLayer(rng, d, 256, 10, 3, fmt="q4k", gg_types=types)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :3] == io[:, :3]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_INT_Q4K


# f32 throughout: chains of 32 products (2^-24 of what has been added at each), up to 112 groups' sums in trees, two projections one behind the
# other: 2 .. 4e-7 in the 2-norm (worst of eight mixes of types, 1 .. 20 tokens: 4.5e-7), and an output four times its typical error off
# lies four times below the token's largest
TOL_F32 = 1e-6


@pytest.mark.parametrize("T", [1, 4, 5, 9, 20, 32])
@pytest.mark.parametrize("types,k,shared,d,mid", [((13, 8, 8), 3, True, 2560, 640), ((12, 8, 8), 10, True, 2560, 640), ((13, 7, 8), 6, True, 3072, 640),
                                                  ((8, 8, 7), 7, True, 2048, 384), ((13, 8, 8), 15, True, 2048, 896), ((7, 8, 8), 1, False, 3584, 128),
                                                  ((20, 7, 7), 5, False, 2560, 896), ((23, 8, 8), 2, True, 3072, 128)])
def test_small_batch_gguf_down_rows_of_no_whole_super_blocks(oracle, types, k, shared, d, mid, T):
    """Down rows of 2, 6, 10 and 14 units of 64 columns, one slot to fifteen, on activations in f32."""
    rng = np.random.default_rng(d + mid + 10 * T + k)
    hl = HostLayer(rng, d, mid, 16, k, fmt="q4k", gg_types=types, shared=shared)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[0, 40:72] *= 1e-6  # (a group whose elements are of two sizes, and one that is small throughout)
    x[T - 1] *= 1e4
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_F32


def gg_bytes(t, cols):
    return {12: cols // 256 * 144, 13: cols // 256 * 176, 8: cols // 32 * 34, 7: cols // 32 * 24}[t]


def without_column(t, rows, col):
    """The rows with weight 0 in column `col` of every 32 (minima and offsets of all blocks 0)."""
    size = {12: 144, 13: 176, 8: 34, 7: 24}[t]
    b = rows.reshape(-1, size).copy()
    if t in (12, 13):
        b[:, 2:4] = 0
        b[:, size - 128 + col::32] = 0
        if t == 13:
            b[:, 16 + col] = 0
    elif t == 8:
        b[:, 2 + col] = 0
    else:  # (column col < 16: the low nibble of byte col)
        b[:, 2:4] = 0
        b[:, 4 + col // 8] &= 255 - (1 << col % 8)
        b[:, 8 + col] &= 0xf0
    return b.reshape(-1)


@pytest.mark.parametrize("T", [1, 4, 9])
@pytest.mark.parametrize("types", [(13, 8, 8), (12, 8, 7), (8, 7, 8), (7, 7, 7)])
def test_small_batch_gguf_activations_of_many_sizes_in_a_group(oracle, types, T):
    """Down rows of no whole super-blocks: x with elements 2^16 times their group's others, hid with elements 2^9 times theirs, all of them
    where every weight is 0: the others keep their 24 bits."""
    rng = np.random.default_rng(T + types[0])
    d, mid, E, k, col = 2560, 640, 12, 4, 7
    hl = HostLayer(rng, d, mid, E, k, fmt="q4k", gg_types=types)

    def larger(t, rows):  # the rows that make hid's columns `col`
        b = rows.reshape(-1, 32, gg_bytes(t, d)).copy()
        size = {12: 144, 13: 176, 8: 34, 7: 24}[t]
        f = b[:, col].reshape(-1, size)
        f[:, 0:2] = (f[:, 0:2].copy().view(np.float16) * np.float16(512)).view(np.uint8)
        b[:, col] = f.reshape(b[:, col].shape)
        return b.reshape(-1)
    hl.gate = without_column(types[0], hl.gate, col)
    hl.up = larger(types[0], without_column(types[0], hl.up, col))
    hl.down = without_column(types[1], hl.down, col)
    hl.shared[0] = without_column(types[2], hl.shared[0], col)
    hl.shared[1] = larger(types[2], without_column(types[2], hl.shared[1], col))
    hl.shared[2] = without_column(types[2], hl.shared[2], col)
    hl.router[:, col::32] = 0
    hl.shared[3][:, col::32] = 0
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[:, col::32] *= 2.0 ** 16
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :k] == io[:, :k]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_F32


@pytest.mark.parametrize("T", [1, 3])
@pytest.mark.parametrize("scale", [1e-17, 1e-18, 3e-19])
def test_small_batch_gguf_hid_far_below_one(oracle, scale, T):
    """hid above and below 2^-104: an element keeps its 24 bits down to 2^-126, and a block's scale of 2^-24 takes none of them in products
    that are added up before they are scaled."""
    rng = np.random.default_rng(T)
    hl = HostLayer(rng, 2560, 640, 16, 4, fmt="q4k", gg_types=(13, 8, 8))
    x = rng.standard_normal((T, 2560), dtype=np.float32) * np.float32(scale)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    assert np.abs(yo).max() > 1e-33
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :4] == io[:, :4]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_F32


@pytest.mark.parametrize("T", [1, 4, 20, 40])
@pytest.mark.parametrize("types,d,mid", [((13, 8, 8), 2560, 640), ((8, 7, 7), 2048, 128), ((20, 8, 7), 2048, 384), ((23, 7, 8), 2048, 128)])
@pytest.mark.parametrize("moved", ["gate_up", "down", "shared"])
def test_gguf_tensors_that_begin_where_their_blocks_may(oracle, types, d, mid, T, moved):
    """Tensors two bytes (Q8_0, IQ4_NL) and eight bytes (Q5_1, IQ4_XS) off the alignment of the fastest kernels."""
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(d + mid + T)
    hl = HostLayer(rng, d, mid, 6, 3, fmt="q4k", gg_types=types)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)

    def at(name, t, off):
        n = {8: 2, 20: 2, 7: 8, 23: 8}.get(t, 0) if off else 0
        buf = torch.zeros(dev[name].numel() + n, dtype=torch.uint8, device="cuda")
        buf[n:] = dev[name].reshape(-1)
        dev[name + "_moved"] = buf
        return buf[n:]
    m.set_experts_gguf(0, at("gate", types[0], moved == "gate_up"), at("up", types[0], moved == "gate_up"), at("down", types[1], moved == "down"),
                       types[0], types[1])
    sh = [at(n, types[2], moved == "shared") for n in ("shg", "shu", "shd")]
    m.set_shared(0, capi.wview(sh[0], 0, mid, d), capi.wview(sh[1], 0, mid, d), capi.wview(sh[2], 0, d, mid), capi.wview(dev["shsg"], capi.F32, 1, d),
                 types[2])
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids = m.last_routing(T)[0].cpu().numpy()
    m.close()
    assert (ids[:, :3] == io[:, :3]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= (TOL_GEMV if T <= 32 else TOL_LAYER)


@pytest.mark.parametrize("T", [5, 16, 17, 25, 32])
@pytest.mark.parametrize("E,d,router,shared", [(17, 1024, "f32", True), (32, 2048, "bf16", True), (513, 1024, "f32", False), (20, 768, "bf16", True),
                                               (1000, 256, "f32", True), (16, 384, "f32", True), (40, 640, "f32", True), (33, 2304, "bf16", True), (18, 128, "f32", False)])
def test_small_batch_router_in_column_shares(oracle, E, d, router, shared, T):
    """5 .. 32 tokens: one and two tiles of tokens, row groups with rows left over, one to eight column shares, equal and not; the shared expert's
    gate logit and the selection's bound beside them.  One token's best logits are equal in pairs, another's are a tie in f32
    only, so that the selection needs the bound."""
    rng = np.random.default_rng(E + d + T)
    hl = HostLayer(rng, d, 256, E, 6, router_dtype=router, shared=shared, scale_std=0.02)
    if router == "f32":
        hl.router[1] = hl.router[0]
        hl.router[3] = hl.router[2]
        hl.router[3, ::2] *= np.float32(1.0 + 2.0 ** -23)
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[1] = 30 * hl.router[0].astype(np.float32) if router == "f32" else x[1]
    x[2] = 30 * hl.router[2].astype(np.float32) if router == "f32" else x[2]
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    y, ids, ws = run_layer(hl, x)
    assert (ids[:, :6] == io[:, :6]).all()
    assert np.abs(ws[:, :6] - wo[:, :6]).max() <= 1e-6
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_INT_Q4CP


@pytest.mark.parametrize("T", [1, 3])
@pytest.mark.parametrize("types,d,mid", [((13, 8, 8), 2048, 256), ((13, 8, 8), 2560, 256), ((12, 12, 12), 3072, 256), ((8, 13, 8), 3584, 256),
                                         ((13, 8, 8), 2560, 640), ((13, 7, 8), 2048, 128), ((20, 8, 7), 3072, 384), ((12, 8, 8), 3584, 128)])
def test_gguf_gate_up_selects_among_more_than_512_experts(types, d, mid, T):
    """The selection inside the gate/up launch and the router's own give the same ids, and the rows' sums do not depend on it."""
    import torch
    from gfx1151_engine_amd import capi, workloads as W
    L = W.DeviceLayer(1, d, mid, 520, 8, "q4k", gg_types=types)
    m = capi.Moe(d, mid, 520, 8, layers=1, max_tokens=T)
    L.register(m, 0)
    x = torch.randn((T, d), device="cuda")
    m.set_option(capi.OPT_GU_TOPK_MAX_TOKENS, 32)
    y = m.forward(0, x).clone()
    m.set_option(capi.OPT_GU_TOPK_MAX_TOKENS, 0)
    assert torch.equal(y, m.forward(0, x))
    m.close()


@pytest.mark.parametrize("tgu", [12, 13, 7, 8, 20, 23])
def test_gguf_gate_up_rows_in_both_orders(oracle, tgu):
    """Every gate/up type (the shared expert's as well) in the launch that selects the experts itself, whose waves take their rows
    as a ring, and in the one that is given them, where longer rows go in two batches: the same sums, bit for bit."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(tgu)
    T, d, mid = 5, 768, 256
    hl = HostLayer(rng, d, mid, 12, 4, fmt="q4k", gg_types=(tgu, 8, tgu))
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    ys = []
    for most in (T, 0):
        m.set_option(capi.OPT_GU_TOPK_MAX_TOKENS, most)
        ys.append(m.forward(0, gpu(x)).cpu().numpy())
    m.close()
    assert (ys[0] == ys[1]).all()
    assert max_abs_rel(ys[0], yo) <= TOL_INT_Q4K


@pytest.mark.parametrize("share", [0.3, 1.0])
def test_unique_expert_path(oracle, share):
    """MOE_OPT_UNIQUE_MIN_TOKENS: a verify-size batch through the expert-sorted pair lists (every distinct
    expert read once) gives the same experts and, within the GEMV bar, the same output."""
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(91)
    d, mid, E, k, T = 3072, 768, 24, 10, 20
    hl = HostLayer(rng, d, mid, E, k)
    x = rng.standard_normal((T, d), dtype=np.float32)
    n = int(round(share * T))
    for i in range(1, n):  # drafted tokens that reproduce the template token's routing
        x[i] = x[0] + 1e-3 * rng.standard_normal(d).astype(np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=32)
    m.set_option(capi.OPT_UNIQUE_MIN_TOKENS, 8)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids, _ = m.last_routing(T)
    assert (ids.cpu().numpy()[:, :k] == io[:, :k]).all()
    assert max_abs_rel(y, yo) <= TOL_INT_Q4CP, max_abs_rel(y, yo)
    m.set_option(capi.OPT_UNIQUE_MIN_TOKENS, 0)
    y2 = m.forward(0, gpu(x)).cpu().numpy()
    assert max_abs_rel(y2, yo) <= TOL_INT_Q4CP
    m.close()


@pytest.mark.parametrize("types,T,share,shared", [((12, 12, 12), 20, 0.3, True), ((13, 8, 8), 20, 1.0, True),
                                                  ((12, 7, 13), 12, 0.3, True), ((13, 8, 8), 32, 0.5, False),
                                                  ((8, 13, 7), 17, 0.0, True)])
def test_unique_expert_path_gguf(oracle, types, T, share, shared):
    """The distinct-expert kernels for GGUF layers (any mix of Q4_K / Q5_K / Q8_0 / Q5_1): a verify-size batch through
    the expert-sorted pair lists, tiles of at most four pairs, against the oracle and against the per-token kernels."""
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(92 + T)
    d, mid, E, k = 3072, 768, 24, 10
    hl = HostLayer(rng, d, mid, E, k, fmt="q4k", gg_types=types, shared=shared)
    x = rng.standard_normal((T, d), dtype=np.float32)
    for i in range(1, int(round(share * T))):
        x[i] = x[0] + 1e-3 * rng.standard_normal(d).astype(np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=32)
    m.set_option(capi.OPT_UNIQUE_MIN_TOKENS, 8)
    m.set_option(capi.OPT_UNIQUE_GGUF, 1)
    m.profile(True)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert m.profile_read()["reduce"] > 0, "the distinct-expert path ends in a combine launch"
    m.profile(False)
    ids, ws = m.last_routing(T)
    assert (ids.cpu().numpy()[:, :k] == io[:, :k]).all()
    assert np.abs(ws.cpu().numpy()[:, :k] - wo[:, :k]).max() <= 1e-6
    assert max_abs_rel(y, yo) <= TOL_INT_Q4K, max_abs_rel(y, yo)
    m.set_option(capi.OPT_UNIQUE_GGUF, 0)
    y2 = m.forward(0, gpu(x)).cpu().numpy()
    assert max_abs_rel(y2, yo) <= TOL_INT_Q4K
    assert max_abs_rel(y, y2) <= 1e-5, "the same integer sums per pair: only the order of the combine's additions differs"
    m.close()


@pytest.mark.parametrize("i", [0, 1, 2, 3])
def test_golden_layers_from_reference(oracle, golden, i):
    """Inputs and outputs of the reference's own Model::moe (tests/golden/moe_layer.npz): four layers, two of them
    with a bf16 shared expert, one with a q8g64 one."""
    import torch
    from gfx1151_engine_amd import capi
    g = golden("moe_layer.npz")
    assert int(g["n"]) == 4
    d, mid, E, k, sh_dt = (int(v) for v in g[f"cfg{i}"])
    m = capi.Moe(d, mid, E, k)
    sh16 = sh_dt == oracle.BF16  # bf16 matrices are stored as uint16 bit patterns
    shv = [g[f"shg{i}"], g[f"shu{i}"], g[f"shd{i}"]]
    keep = [gpu(g[f"router{i}"].view(np.int16)), gpu(g[f"gu{i}"]), gpu(g[f"dn{i}"])] + \
           [gpu(a.view(np.int16) if sh16 else a) for a in shv] + [gpu(g[f"sg{i}"].view(np.int16))]
    wt = {oracle.BF16: capi.BF16, oracle.Q4CP: capi.Q4CP, oracle.Q8G64: capi.Q8G64}[sh_dt]
    m.set_router(0, capi.wview(keep[0], capi.BF16, E, d))
    m.set_experts_q4cp(0, capi.wview(keep[1], capi.Q4CP, E * 2 * mid, d), capi.wview(keep[2], capi.Q4CP, E * d, mid))
    m.set_shared(0, capi.wview(keep[3], wt, mid, d), capi.wview(keep[4], wt, mid, d),
                 capi.wview(keep[5], wt, d, mid), capi.wview(keep[6], capi.BF16, 1, d))
    x = g[f"x{i}"]
    want = g[f"ybits{i}"].view(np.float32)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert max_abs_rel(y, want) <= TOL_INT_Q4CP, i  # integer-dot decode kernels where the codebook is affine
    m.set_option(capi.OPT_INT_DECODE, 0)
    y = m.forward(0, gpu(x)).cpu().numpy()
    assert max_abs_rel(y, want) <= 5e-6, i          # f32 kernels: f32 against the reference's fp64 sums
    m.close()


def test_forward_errors(oracle):
    import torch
    from gfx1151_engine_amd import capi
    m = capi.Moe(256, 64, 8, 2, max_tokens=4)
    x = torch.zeros((2, 256), device="cuda")
    with pytest.raises(capi.MoeError):  # no weights registered
        m.forward(0, x)
    with pytest.raises(capi.MoeError):  # bad layer index
        m.forward(3, x)
    m.close()
    with pytest.raises(capi.MoeError):  # d not a multiple of 32
        capi.Moe(100, 64, 8, 2)


def test_stage_skipping_is_not_in_the_default_build_and_guarded_in_the_timing_twin():
    """MOE_OPT_TIMING_SKIP_STAGE makes a call return wrong results: the default library refuses it outright; the
    benchmark's timing twin takes it only once a complete call of that size has filled the scratch that the stages
    behind the skipped one index with."""
    import os
    import torch
    from gfx1151_engine_amd import LIB_TIMING, capi
    rng = np.random.default_rng(11)
    hl = HostLayer(rng, 1024, 256, 16, 4)
    m, dev = hl.to_gpu(max_tokens=8)
    with pytest.raises(capi.MoeError, match="unsupported"):
        m.set_option(capi.OPT_TIMING_SKIP_STAGE, 3)
    m.close()
    if not os.path.exists(LIB_TIMING):
        pytest.skip("timing twin of the library not built")
    twin = capi.second_binding(LIB_TIMING)
    mt, dev2 = hl.to_gpu(max_tokens=8, binding=twin)
    with pytest.raises(twin.MoeError, match="not ready"):
        mt.set_option(capi.OPT_TIMING_SKIP_STAGE, 3)  # fresh context: nothing has run yet
    x1 = torch.from_numpy(rng.standard_normal((1, 1024), dtype=np.float32)).cuda()
    x2 = torch.from_numpy(rng.standard_normal((2, 1024), dtype=np.float32)).cuda()
    y_full = mt.forward(0, x1).clone()
    mt.set_option(capi.OPT_TIMING_SKIP_STAGE, 3)
    mt.forward(0, x1)                       # runs (on the scratch of the complete call)
    with pytest.raises(twin.MoeError, match="not ready"):
        mt.forward(0, x2)                   # no complete call of two tokens yet
    mt.set_option(capi.OPT_TIMING_SKIP_STAGE, 0)
    assert torch.equal(mt.forward(0, x1), y_full)
    torch.cuda.synchronize()
    mt.close()


@pytest.mark.parametrize("fmt,T,int_decode", [("q4cp", 1, 1), ("q4cp", 3, 1), ("q4cp", 7, 1), ("q4cp", 20, 1),
                                               ("q4cp", 2, 0), ("q4k", 1, 1), ("q4k", 6, 1)])
def test_small_batch_ids_when_summation_orders_disagree(oracle, fmt, T, int_decode):
    """The small-batch router sums a logit's products lane-parallel, the reference one after the other
    (src/ref.cpp:70-77); the two fp64 sums can differ, and with them the f32 logits.  Here they differ by far more
    than an ulp: token activations with +-2^36 in two columns that cancel in one expert's row, so that the order of
    the additions decides what is left of the small terms.  A ladder of experts whose logits are pure biases, 1e-5
    apart, brackets that expert's sequential logit; wherever the parallel sum lands, its rank in the ladder is not
    the reference's.  The library must notice that the gaps are within what the two orders can differ by (a bound
    from the norms of the operands), recompute the logits in the reference's order and return the oracle's ids."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(101 + T)
    d, mid, E, k = 1024, 256, 64, 8
    bias = np.full(E, -30.0, np.float32)
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt, bias=bias)
    A = 61                                     # the expert with the ill-conditioned sum (a high index: ties go to lower ones)
    hl.router[:] = 0.0
    hl.router[A] = rng.standard_normal(d).astype(np.float32) * np.float32(0.05)
    hl.router[A, 0] = 1.0
    hl.router[A, d - 1] = 1.0
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[:, 0] = np.float32(2.0 ** 36)
    x[:, d - 1] = -np.float32(2.0 ** 36)
    bias[A] = 0.0
    # the sequential logit of A for token 0, then the ladder around it (every token sees the same ladder; the
    # tokens' own values of A differ, so A's rank differs from token to token)
    lgA = oracle.router(hl.oracle_layer().router, x, k, bias=bias)[0][:, A]
    ladder = [e for e in range(E) if e != A][:40]
    for j, e in enumerate(ladder):
        bias[e] = np.float32(np.float64(lgA[0]) + (3.5 - j) * 1e-5)  # four rungs above A's logit, the others below
    hl.bias = bias
    ol = hl.oracle_layer()
    lg, io, wo = oracle.router(ol.router, x, k, bias=bias)
    # the parallel-order logits of the stateless entry point (the forward call's launches use other splits of the
    # sum, with other roundings): they must not agree with the sequential ones, or the test tests nothing
    import torch
    Wd = torch.from_numpy(hl.router).cuda()
    lt = capi.router_logits(capi.wview(Wd, capi.F32, E, d), torch.from_numpy(x).cuda(), torch.from_numpy(bias).cuda(), mode=0).cpu().numpy()
    assert np.abs(lt[:, A].astype(np.float64) - lg[:, A]).max() > 2e-5, "the two summation orders (nearly) agree on this input: nothing to test"
    m, dev = hl.to_gpu(max_tokens=32)
    m.set_option(capi.OPT_INT_DECODE, int_decode)
    y = m.forward(0, torch.from_numpy(x).cuda())
    ids, ws = m.last_routing(T)
    torch.cuda.synchronize()
    ids = ids.cpu().numpy()
    assert (ids[:, :k] == io[:, :k]).all(), (ids[:, :k], io[:, :k])
    assert np.isfinite(y.cpu().numpy()).all()
    m.close()


@pytest.mark.parametrize("T", [1, 3, 7, 20, 32])
@pytest.mark.parametrize("fmt,d,E", [("q4cp", 1024, 64), ("q4cp", 1056, 64), ("table", 640, 64), ("q4k", 2304, 64), ("q4k", 2560, 64), ("ggmix", 1024, 64),
                                     ("ggmix", 3072, 64), ("i4r", 1024, 64), ("q4cp", 1024, 62), ("q4cp", 1056, 520), ("table", 640, 520), ("q4k", 512, 513),
                                     ("q4k", 2048, 63), ("ggmix", 2560, 62), ("i4r", 512, 520), ("f32", 640, 520), ("q4k", 512, 62)])
def test_all_blocks_of_a_launch_select_by_one_bound(oracle, fmt, d, E, T):
    """The ladder of test_small_batch_ids_when_summation_orders_disagree with MOE_OPT_GU_TOPK_MAX_TOKENS = 32: the blocks that only rank must judge
    a token's gaps by the bound of the block that writes the ids, or a slot's gate/up rows and its down rows are two experts'.  The
    selection aside gives the same result but for the last bits of the weights, whose normaliser has terms of logits that are not redone:
    two steps of 2^-23 of experts' outputs that are up to some hundred times their sum; another expert's output is of its size.  (1056 columns: the router launch leaves no bounds above four tokens; 62, 63 and more than 512
    experts: rows that cannot be ranked by logit.)"""
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(d + T)
    mid, k = 256, 8
    bias = np.full(E, -30.0, np.float32)
    cb = np.sort(rng.standard_normal(16)).astype(np.float32) if fmt == "table" else None
    hl = HostLayer(rng, d, mid, E, k, fmt={"table": "q4cp", "ggmix": "q4k", "f32": "q4cp"}.get(fmt, fmt), bias=bias, codebook=cb, scale_std=0.05,
                   gg_types=(13, 8, 8) if fmt == "ggmix" else (12, 12, 12))
    hl.router[:] = 0.0
    A = 61
    hl.router[A] = rng.standard_normal(d).astype(np.float32) * np.float32(0.05)
    hl.router[A, [0, d - 1]] = 1.0
    x = rng.standard_normal((T, d), dtype=np.float32)
    x[:, 0], x[:, d - 1] = 2.0 ** 36, -2.0 ** 36
    bias[A] = 0.0
    lgA = oracle.router(hl.oracle_layer().router, x, k, bias=bias)[0][:, A]
    for j in range(40):
        bias[j] = np.float32(np.float64(lgA[0]) + (3.5 - j) * 1e-5)
    hl.bias = bias
    io = oracle.router(hl.oracle_layer().router, x, k, bias=bias)[1]
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_INT_DECODE, fmt != "f32")
    ys = []
    for most in (32, 0):
        m.set_option(capi.OPT_GU_TOPK_MAX_TOKENS, most)
        ys.append(m.forward(0, gpu(x)).cpu().numpy())
        assert (m.last_routing(T)[0].cpu().numpy()[:, :k] == io[:, :k]).all()
    m.close()
    assert np.isfinite(ys[0]).all()
    assert max(max_abs_rel(ys[0][t], ys[1][t]) for t in range(T)) <= 1e-4


@pytest.mark.parametrize("T", [5, 17, 32])
@pytest.mark.parametrize("E,d,router", [(40, 640, "f32"), (40, 2304, "bf16"), (24, 2560, "f32"), (100, 384, "f32"), (18, 128, "f32"), (20, 1024, "bf16")])
def test_small_batch_router_shares_added_by_the_last_block(oracle, E, d, router, T):
    """The selection inside the gate/up launch at more than four tokens: the column shares are handed over by tickets.  One and two tiles of
    tokens, several row groups, one with rows left over, equal and unequal shares."""
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(E + d + T)
    hl = HostLayer(rng, d, 256, E, 6, router_dtype=router, scale_std=0.02)
    if router == "f32":
        hl.router[1] = hl.router[0]
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, wo = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    m.set_option(capi.OPT_GU_TOPK_MAX_TOKENS, 32)
    for _ in range(3):  # (the tickets rest at 0 between launches)
        y = m.forward(0, gpu(x)).cpu().numpy()
        ids, ws = (a.cpu().numpy()[:, :6] for a in m.last_routing(T))
        assert (ids == io[:, :6]).all() and np.abs(ws - wo[:, :6]).max() <= 1e-6
        assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_INT_Q4CP
    m.close()


# ---------- few tokens, codebooks by look-up: where its blocks, tables and selection end ----------
# (one slot: a down block of a single wave fills the tables in four turns; 1000 experts: the selection keeps twice the LDS;
# a gate codebook and an up codebook of the shared expert: two tables; groups past the lanes of a row: d = 3072)
@pytest.mark.parametrize("d,mid,E,k,shared,T", [(3072, 64, 20, 10, "own", 1), (32, 32, 8, 1, None, 1), (64, 32, 8, 1, "same", 3),
                                                (2080, 96, 1000, 4, "own", 1), (1024, 992, 24, 14, "own", 2), (96, 64, 40, 7, None, 5),
                                                (3072, 96, 530, 2, "same", 4), (2048, 32, 16, 3, "own", 6)])
def test_look_up_blocks(oracle, d, mid, E, k, shared, T):
    rng = np.random.default_rng(d + mid + T)
    own = [np.sort(rng.uniform(-2, 2, 16)).astype(np.float32) for _ in range(3)]
    hl = HostLayer(rng, d, mid, E, k, codebook=rng.uniform(-2, 2, 16).astype(np.float32), shared=shared is not None,
                   shared_codebooks=own if shared == "own" else None, scale_std=0.05)
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    m, dev = hl.to_gpu(max_tokens=T)
    y = m.forward(0, gpu(x)).cpu().numpy()
    ids = m.last_routing(T)[0].cpu().numpy()[:, :k]
    m.close()
    assert (ids == io[:, :k]).all()
    assert max(max_abs_rel(y[t], yo[t]) for t in range(T)) <= TOL_LUT


@pytest.mark.parametrize("what", ["experts", "shared", "gguf"])
def test_a_refused_registration_leaves_the_layer_as_it_was(what):
    """Blobs off their alignment are refused after their codebooks have been looked at: the layer's own weights, of the other kind of
    codebook, go on as before, in the integer-dot and the look-up decode kernels and in batches."""
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(3)
    d, mid, E, k = 512, 256, 8, 2
    cb = None if what == "shared" else np.sort(rng.standard_normal(16)).astype(np.float32)
    hl = HostLayer(rng, d, mid, E, k, codebook=cb, scale_std=0.05)
    m, dev = hl.to_gpu(max_tokens=64)
    xs = [gpu(rng.standard_normal((T, d), dtype=np.float32)) for T in (1, 20, 64)]
    before = [m.forward(0, x).cpu().numpy() for x in xs]

    def off(a):
        t = torch.zeros(a.nbytes + 16, dtype=torch.uint8, device="cuda")
        t[2:2 + a.nbytes] = gpu(a.view(np.uint8).reshape(-1))
        return t[2:2 + a.nbytes]
    with pytest.raises(capi.MoeError):
        if what == "experts":
            a = HostLayer(rng, d, mid, E, k)
            m.set_experts_q4cp(0, capi.wview(off(a.gate_up), capi.Q4CP, E * 2 * mid, d), capi.wview(off(a.down), capi.Q4CP, E * d, mid))
        elif what == "shared":
            sh = [off(S.make_gg(rng, 12, r, c)) for r, c in ((mid, d), (mid, d), (d, mid))]
            m.set_shared(0, capi.wview(sh[0], 0, mid, d), capi.wview(sh[1], 0, mid, d), capi.wview(sh[2], 0, d, mid),
                         capi.wview(dev["shsg"], capi.F32, 1, d), 12)
        else:
            a = HostLayer(rng, d, mid, E, k, fmt="q4k")
            m.set_experts_gguf(0, off(a.gate), off(a.up), off(a.down), 12, 12)
    for x, y in zip(xs, before):
        assert (m.forward(0, x).cpu().numpy() == y).all()
    m.close()
