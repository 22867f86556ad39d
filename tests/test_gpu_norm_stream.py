"""The persistent norm kernel (rms_adaln_stream), bit-exact against the oracle,
just above the row counts from which prefer_row_kernel leaves rows to it: every
chunk count per lane with and without a residual, tables of one row, in runs and
in random order, and rows of two sequences. Each case looks at its launch (a block per
row has 256 threads, this grid more), so one that the dispatch
moves to another kernel fails."""
import numpy as np
import pytest
import torch

import gpu_adapter as gpu
from graph_nodes import kernels as launched
from helpers import bf16_randn, from_np, to_np
from lynnreal_omni_amd import kernels
from oracle import reference as ref

pytestmark = pytest.mark.gpu

# (batch, tokens, hidden): the least rows that stream there with several table rows.
PLAIN = [(1, 2561, 8), (1, 2561, 512), (2, 1301, 520), (1, 2561, 1024), (1, 4097, 1032), (1, 4097, 2048),
         (2, 2051, 2056), (1, 4097, 3072), (1, 4097, 3080), (1, 4097, 4096), (1, 4097, 4104), (2, 2050, 5120),
         (1, 4097, 5632), (1, 4097, 6144)]
RESIDUAL = [(1, 2049, 8), (2, 1025, 512), (1, 2049, 520), (1, 3073, 1032), (2, 1601, 1544), (1, 3073, 2040),
            (1, 8193, 2048), (2, 4099, 2056), (1, 8193, 3072)]
BIG = 0x6A80   # bf16 2^86: rows modulated by it have |y| far above 2^80


def _inputs(batch, t, d, layout):
    g = torch.Generator().manual_seed(batch * t + d)
    rows = 1 if layout == "one row" else 5
    x, u = bf16_randn((batch, t, d), g, outliers=0.01), bf16_randn((batch, t, d), g)
    w = (1 + 0.05 * torch.randn(d, generator=g)).bfloat16()
    table = bf16_randn((rows, 6 * d), g, scale=0.1)
    idx = torch.randint(0, rows, (t,), generator=g)
    if layout == "runs":
        idx = idx.sort().values
    return [to_np(v) for v in (x, u, w, table)] + [idx.numpy()]


def _assert_streams(x, u, w, table, idx, residual):
    """One kernel on a persistent grid."""
    x, u, table, idx = (from_np(a, gpu.DEV) for a in (x, u, table, idx))
    norm = gpu._norm(w, 1e-6)
    if residual:
        nodes = launched(lambda: kernels.residual_rms_quant(x, u, norm, table, idx))
    else:
        nodes = launched(lambda: kernels._rms_adaln_quant_int8(x, norm, table, idx, 0, 1))
    assert len(nodes) == 1 and nodes[0][1] > 256, nodes


@pytest.mark.parametrize("layout", ["one row", "runs", "random"])
@pytest.mark.parametrize("batch,t,d", PLAIN)
def test_streamed_norm(batch, t, d, layout):
    x, u, w, table, idx = _inputs(batch, t, d, layout)
    y = gpu.rms_adaln(x, w, table, idx, 3, 4, 1e-6)
    assert np.array_equal(y, ref.rms_adaln(x, w, table, idx, 3, 4, 1e-6))
    q, s = gpu.rms_adaln_quant(x, w, table, idx, 0, 1, 1e-6)
    rq, rs = ref.rms_adaln_quant(x, w, table, idx, 0, 1, 1e-6)
    assert np.array_equal(q, rq) and np.array_equal(s, rs)
    _assert_streams(x, u, w, table, idx, False)


@pytest.mark.parametrize("t,d,layout", [(4097, 6152, "runs"), (4097, 7168, "runs"), (4097, 8192, "runs"),
                                        (768, 3080, "one row"), (768, 5120, "one row")])
def test_streamed_norm_without_quantization(t, d, layout):
    """Widths and counts that only the bf16 output streams."""
    x, u, w, table, idx = _inputs(1, t, d, layout)
    y = gpu.rms_adaln(x, w, table, idx, 0, 1, 1e-6)
    assert np.array_equal(y, ref.rms_adaln(x, w, table, idx, 0, 1, 1e-6))


@pytest.mark.parametrize("batch,t,d,layout", [(*shape, layout) for shape in RESIDUAL
                                              for layout in ("one row", "runs", "random")]
                         + [(1, 1024, 8, "one row"), (2, 512, 1528, "one row")])
def test_streamed_residual_norm(batch, t, d, layout):
    x, u, w, table, idx = _inputs(batch, t, d, layout)
    r, q, s = gpu.residual_rms_quant(x, u, w, table, idx, 1e-6)
    rr, rq, rs = ref.residual_rms_quant(x, u, w, table, idx, 1e-6)
    assert np.array_equal(r, rr) and np.array_equal(q, rq) and np.array_equal(s, rs)
    _assert_streams(x, u, w, table, idx, True)


def test_residual_slices_switch_quotients_at_a_boundary():
    """Slices of rows that span two runs of table rows, one of which takes the
    corrected quotient (absmax of 2^80 and more)."""
    x, u, w, table, idx = _inputs(1, 8193, 3072, "runs")
    for row in (1, 3):
        table[row, 4 * 3072:5 * 3072] = BIG
    r, q, s = gpu.residual_rms_quant(x, u, w, table, idx, 1e-6)
    rr, rq, rs = ref.residual_rms_quant(x, u, w, table, idx, 1e-6)
    huge = np.isin(idx, (1, 3))
    assert (rs[huge] > 2.0 ** 80 / 127).all() and (rs[~huge] < 2.0 ** 80 / 127).all()
    assert np.array_equal(r, rr) and np.array_equal(q, rq) and np.array_equal(s, rs)
    _assert_streams(x, u, w, table, idx, True)
