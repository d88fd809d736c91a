"""The grouped GEMMs' scaled dequantisation (codes read as f16 denormals, a power of two per expert) of rotated experts: experts
that have such a power and experts that do not, in one layer, on the few-pair and the 128-pair kernels, against the oracle; and
Q4_K experts, whose arithmetic has no such form, at the same scales.  Reference: src/gpu/parts/27_kernels_moe_lut.inc:16-29, 26_kernels_moe_gguf.inc:81-485."""
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
            elif what == "edge":  # a largest scale that ends just under a power of two
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
