"""The grouped GEMMs' dequantisation of codes that are read as f16 denormals (q4cp: with a power of two per expert): experts that
have it and experts that do not, in one layer, on the few-pair and the 128-pair kernels, against the oracle; what the form
does to the weights; and Q4_K experts, whose arithmetic has no such form, at the same scales.  Reference: src/gpu/parts/27_kernels_moe_lut.inc:16-29, 26_kernels_moe_gguf.inc:81-485."""
import numpy as np
import pytest

from helpers import HostLayer, max_abs_rel

pytestmark = pytest.mark.gpu
TOL_LAYER = 2e-3  # f16 MFMA operands and f16 intermediates, as in the other whole-layer tests of batches


def i4r_scales(blob, rows, cols):
    return blob[rows * cols // 2:].view(np.float16).reshape(rows, cols // 128)


def q4k_blocks(rows):
    return rows.reshape(-1, 144)


def change(hl, what):
    """Expert 1 (of its gate/up and down tensors) is changed; the others stay as they are."""
    d, mid, E = hl.d, hl.mid, hl.E
    if hl.fmt == "i4r":
        planes = [(i4r_scales(hl.gate_up, E * 2 * mid, d), 2 * mid), (i4r_scales(hl.down, E * d, mid), d)]
        for s, n in planes:
            if what == "wide":    # rows far below the expert's largest: no power of two for this expert
                s[n + 3:n + 9] *= np.float16(2.0 ** -9)
            elif what == "zero":
                s[n:2 * n] = 0
            elif what == "edge":  # a largest scale above the form's limit
                s[n, 0] = np.float16(0.12494)
    else:
        for w, rows, cols in ((hl.gate, mid, d), (hl.up, mid, d), (hl.down, d, mid)):
            b = q4k_blocks(w)
            n = rows * (cols // 256)
            dd = b[:, 0:4].copy().view(np.float16)
            if what == "wide":
                dd[n + 3 * (cols // 256):n + 6 * (cols // 256)] *= np.float16(2.0 ** -9)
            elif what == "zero":
                dd[n:2 * n] = 0
            elif what == "edge":  # super-blocks with a large d or dmin and no sub-scales at all
                dd[n], dd[n + 5] = (8.0, 0.0), (0.01, 4.0)
                b[n, 4:16] = 0
                b[n + 5, 4:16] = 0
            b[:, 0:4] = dd.view(np.uint8)


@pytest.mark.parametrize("T", [64, 150, 700])
@pytest.mark.parametrize("what", ["plain", "wide", "zero", "edge"])
@pytest.mark.parametrize("fmt", ["i4r", "q4k"])
def test_experts_with_and_without_a_power_of_two(oracle, fmt, what, T):
    import torch
    from gfx1151_engine_amd import capi
    rng = np.random.default_rng(T + len(what))
    hl = HostLayer(rng, 768, 512, 8, 2, fmt=fmt)
    change(hl, what)
    m, dev = hl.to_gpu(max_tokens=T)
    x = rng.standard_normal((T, 768), dtype=np.float32)
    yo, io, _ = oracle.moe_layer(hl.oracle_layer(), x)
    y = m.forward(0, torch.from_numpy(x).cuda())
    assert max_abs_rel(y.cpu().numpy(), yo) <= TOL_LAYER
    assert m.last_path() == capi.PATH_BATCH
    m.set_option(capi.OPT_STREAM_GEMM, 0)
    y = m.forward(0, torch.from_numpy(x).cuda())
    assert max_abs_rel(y.cpu().numpy(), yo) <= TOL_LAYER
    m.close()


def run_both_kernels(hl, x, *options):
    import torch
    from gfx1151_engine_amd import capi
    m, dev = hl.to_gpu(max_tokens=len(x))
    ys = []
    for o, v in options:
        m.set_option(o, v)
    for on in (1, 0):
        m.set_option(capi.OPT_STREAM_GEMM, on)
        ys.append(m.forward(0, torch.from_numpy(x).cuda()).cpu().numpy())
        assert m.last_path() == capi.PATH_BATCH
    m.close()
    return ys


@pytest.mark.parametrize("fused", [1, 0])
@pytest.mark.parametrize("T", [40, 88, 152, 700])
def test_rotated_experts_have_the_same_weights_in_either_form(T, fused):
    """Every expert with one scale above the form's limit, in a group whose weights are all zero, which keeps it on the plain form;
    and with that scale below it: the same results bit for bit, whatever the other groups' scales."""
    from gfx1151_engine_amd import capi
    d, mid, E = 768, 512, 16
    x = np.random.default_rng(T).standard_normal((T, d), dtype=np.float32)
    got = []
    for s0 in (0.0624, 0.0625, 0.5):
        hl = HostLayer(np.random.default_rng(5), d, mid, E, 4, fmt="i4r", bias=np.linspace(0, 0.5, E, dtype=np.float32))
        for w, n, cols in ((hl.gate_up, 2 * mid, d), (hl.down, d, mid)):
            codes = w[:E * n * cols // 2].reshape(E, n, cols // 128, 64)
            sc = i4r_scales(w, E * n, cols).reshape(E, n, cols // 128)
            sc[1, 8:40] *= np.float16(2.0 ** -6)   # rows and groups far below the expert's largest
            sc[2:, :, 1] *= np.float16(2.0 ** -8)
            sc[3, 9:20] = np.float16(2.0 ** -23)
            codes[:, 5, 0] = 0x88
            sc[:, 5, 0] = np.float16(s0)
        got += run_both_kernels(hl, x, (capi.OPT_V2_FUSED_MIDDLE, fused))
    assert np.isfinite(got[0]).all() and np.abs(got[0]).max() > 0
    for i in (2, 3, 4, 5):
        assert (got[i] == got[i & 1]).all()


def q4cp_scales(blob, rows, cols):
    return blob[64 + rows * cols // 2:].view(np.float16).reshape(rows, -1)


# slope * largest scale as a mantissa in [0.5, 1): with 1.5 * 5461 / 8192 it rounds to 1 as an f16 (the power of two has to leave
# that out, or the slope is infinite in the kernels), with 5459 / 8192 just not
@pytest.mark.parametrize("T", [40, 88, 152, 700])
@pytest.mark.parametrize("slope", [5461 / 8192, 5460 / 8192, 5459 / 8192, 1.0])
def test_slopes_that_round_up_to_a_power_of_two(oracle, slope, T):
    rng = np.random.default_rng(T)
    d, mid, E = 512, 640, 16
    cb = (np.arange(16) - 8).astype(np.float32) * np.float32(slope)
    assert all(cb[n] == np.float32(n * (float(cb[1]) - float(cb[0])) + float(cb[0])) for n in range(16))
    hl = HostLayer(rng, d, mid, E, 4, codebook=cb, bias=np.linspace(0, 0.5, E, dtype=np.float32))
    top = np.float16(1.5 * 2.0 ** -6)
    for w, n, cols in ((hl.gate_up, E * 2 * mid, d), (hl.down, E * d, mid), (hl.shared[0], mid, d), (hl.shared[1], mid, d), (hl.shared[2], d, mid)):
        sc = q4cp_scales(w, n, cols)[:, :cols // 32]
        sc[:] = np.minimum(sc, top)
        sc[3::7, 1] = top
    x = rng.standard_normal((T, d), dtype=np.float32)
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    for y in run_both_kernels(hl, x):
        assert np.isfinite(y).all() and max_abs_rel(y, yo) <= TOL_LAYER


@pytest.mark.parametrize("T", [40, 88, 152, 700])
@pytest.mark.parametrize("below", [5, 6, 7])
def test_rows_far_below_an_experts_largest_scale(oracle, below, T):
    """Rows whose largest scale lies 2^-5 below the expert's are the last that the scaled form takes; an expert with rows of 2^-6 has the
    plain form's weights bit for bit, those of a layer whose every expert has another row, of zeros, further below."""
    d, mid, E = 512, 640, 16
    x = np.random.default_rng(T).standard_normal((T, d), dtype=np.float32)
    got = []
    for zeros in (below, 9):
        hl = HostLayer(np.random.default_rng(9), d, mid, E, 4, shared=False, bias=np.linspace(0, 0.5, E, dtype=np.float32))
        for w, n, cols in ((hl.gate_up, 2 * mid, d), (hl.down, d, mid)):
            codes = w[64:64 + E * n * cols // 2].reshape(E, n, cols // 2)
            sc = q4cp_scales(w, E * n, cols)[:, :cols // 32].reshape(E, n, cols // 32)
            sc[:] = np.minimum(sc, np.float16(0.03))
            sc[:, :, 0] = np.float16(0.03)
            sc[:, 10:60] *= np.float16(2.0 ** -below)
            codes[:, 5] = 0x88
            sc[:, 5] = np.float16(0.03 * 2.0 ** -zeros)
        got.append(run_both_kernels(hl, x))
    yo, _, _ = oracle.moe_layer(hl.oracle_layer(), x)
    for y in got[0]:
        assert max_abs_rel(y, yo) <= TOL_LAYER
    if below > 5:
        assert (got[0][0] == got[1][0]).all() and (got[0][1] == got[1][1]).all()
