"""moe_forward is enqueue-only with fixed scratch addresses: it can be captured into a HIP graph
(the reference captures its decode step, src/gpu/parts/40_model.inc:8011-8016).  The graph is
replayed several times with eager calls and synchronisations in between; every replay must
reproduce the eager result bit for bit (same kernels, same order)."""
import numpy as np
import pytest

from helpers import HostLayer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,T", [("q4cp", 1), ("q4cp", 7), ("q4cp", 20), ("q4cp", 48), ("q4k", 1), ("q4k", 9)])
def test_forward_under_graph_capture(oracle, fmt, T):
    import torch
    rng = np.random.default_rng(5 + T)
    d, mid, E, k = 1024, 256, 16, 4
    hl = HostLayer(rng, d, mid, E, k, fmt=fmt)
    m, dev = hl.to_gpu(max_tokens=64)
    xs = [torch.from_numpy(rng.standard_normal((T, d), dtype=np.float32)).cuda() for _ in range(3)]
    x = torch.empty((T, d), dtype=torch.float32, device="cuda")
    y = torch.empty((T, d), dtype=torch.float32, device="cuda")
    eager = []
    for xi in xs:  # eager results (also the warm-up that one-time kernel attributes need)
        x.copy_(xi)
        m.forward(0, x, y)
        eager.append(y.clone())
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    x.copy_(xs[0])
    with torch.cuda.graph(g):
        m.forward(0, x, y)
    for rep in range(3):
        for i, xi in enumerate(xs):
            x.copy_(xi)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager[i]), (rep, i)
            # eager work between replays
            y.zero_()
            m.forward(0, xs[(i + 1) % 3], y)
            torch.cuda.synchronize()
            assert torch.equal(y, eager[(i + 1) % 3])
    m.close()


@pytest.mark.parametrize("variant,T", [("table", 1), ("table", 4), ("table", 9), ("table", 48), ("dense", 1), ("dense", 6),
                                       ("dense", 48), ("ggmix", 3), ("ggmix", 48)])
def test_other_paths_under_graph_capture(oracle, variant, T):
    """The same for the paths that the configurations above do not reach: a table codebook (look-up decode kernels up
    to 5 tokens, plain f32 kernels beyond, table GEMM), a densely stored shared expert (extra launches behind the
    routed experts' kernels; the general GEMM on the side stream), a GGUF layer in mixed block types."""
    import torch
    from gfx1151_engine_amd import synth as S
    rng = np.random.default_rng(50 + T)
    d, mid, E, k = 1024, 256, 16, 4
    if variant == "table":
        hl = HostLayer(rng, d, mid, E, k, codebook=S.UNIVERSAL_CODEBOOK, scale_std=0.05)
    elif variant == "dense":
        hl = HostLayer(rng, d, mid, E, k, shared_dense="q8g32")
    else:
        hl = HostLayer(rng, d, mid, E, k, fmt="q4k", gg_types=(13, 8, 12))
    m, dev = hl.to_gpu(max_tokens=64)
    xs = [torch.from_numpy(rng.standard_normal((T, d), dtype=np.float32)).cuda() for _ in range(2)]
    x = torch.empty((T, d), dtype=torch.float32, device="cuda")
    y = torch.empty((T, d), dtype=torch.float32, device="cuda")
    eager = []
    for xi in xs:
        x.copy_(xi)
        m.forward(0, x, y)
        eager.append(y.clone())
    torch.cuda.synchronize()
    want, _, _ = oracle.moe_layer(hl.oracle_layer(), xs[0].cpu().numpy())
    assert np.abs(eager[0].cpu().numpy() - want).max() <= 2e-3 * np.abs(want).max()
    g = torch.cuda.CUDAGraph()
    x.copy_(xs[0])
    with torch.cuda.graph(g):
        m.forward(0, x, y)
    for rep in range(2):
        for i, xi in enumerate(xs):
            x.copy_(xi)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, eager[i]), (rep, i)
            y.zero_()
            m.forward(0, xs[1 - i], y)
            torch.cuda.synchronize()
            assert torch.equal(y, eager[1 - i])
    m.close()


def test_listed_tokens_under_graph_capture(oracle):
    """A batch whose router lists tokens: none, a few and all of them from replay to replay of one graph (the list, its
    count and its tickets are the call's own)."""
    import torch
    rng = np.random.default_rng(9)
    d, mid, E, k, T = 512, 256, 64, 4, 300
    hl = HostLayer(rng, d, mid, E, k)
    m, dev = hl.to_gpu(max_tokens=T)
    base = rng.standard_normal((T, d), dtype=np.float32)
    few = base.copy()
    few[::37] *= 400.0
    xs = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (base, few, base * np.float32(400.0))]
    x, y = torch.empty_like(xs[0]), torch.empty_like(xs[0])
    eager = []
    for xi in xs:
        x.copy_(xi)
        m.forward(0, x, y)
        eager.append((y.clone(), m.last_routing(T)[0]))
        io = oracle.router(hl.oracle_layer().router, xi.cpu().numpy(), k)[1]
        assert (eager[-1][1].cpu().numpy()[:, :k] == io[:, :k]).all()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        m.forward(0, x, y)
    for rep in range(3):
        for i in (0, 2, 1, 2, 0):
            x.copy_(xs[i])
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y.nan_to_num(), eager[i][0].nan_to_num()), (rep, i)
            assert torch.equal(m.last_routing(T)[0], eager[i][1])
            m.forward(0, xs[(i + 1) % 3], y)
            torch.cuda.synchronize()
            assert torch.equal(y.nan_to_num(), eager[(i + 1) % 3][0].nan_to_num())
    m.close()


def launches(m, x, y):
    """Nodes of a captured call."""
    import ctypes as C
    import torch
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        m.forward(0, x, y)
    n = C.c_size_t(0)
    assert C.CDLL("libamdhip64.so").hipGraphGetNodes(C.c_void_p(g.raw_cuda_graph()), None, C.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("E", [64, 62, 520])
@pytest.mark.parametrize("variant,ranked", [("q4cp", 3), ("table", 2), ("q4k", 4), ("ggmix", 4), ("i4r", 4)])
def test_up_to_how_many_tokens_the_gate_up_launch_selects(variant, ranked, E):
    """Router, gate/up and down launch, and the selection as a fourth from one token more on (rotated experts: two launches more).  Rows that cannot
    be ranked by logit -- more than 512 experts, or a number that is no multiple of four -- leave the launch earlier: with table codebooks
    at one token, else at three."""
    import torch
    from gfx1151_engine_amd import synth as S
    d, mid, k = 2048, 256, 4
    hl = HostLayer(np.random.default_rng(E), d, mid, E, k, fmt={"table": "q4cp", "ggmix": "q4k"}.get(variant, variant),
                   codebook=S.UNIVERSAL_CODEBOOK if variant == "table" else None, gg_types=(13, 8, 8) if variant == "ggmix" else (12, 12, 12))
    m, dev = hl.to_gpu(max_tokens=8)
    most = ranked if E == 64 else 0 if variant == "table" else 2
    count = {}
    for T in {max(most, 1), most + 1}:
        x = torch.randn((T, d), device="cuda")
        y = torch.empty_like(x)
        m.forward(0, x, y)
        count[T] = launches(m, x, y)
    m.close()
    least = 5 if variant == "i4r" else 3
    assert count == ({most: least, most + 1: least + 1} if most else {1: least + 1})
