"""Every element of the fused norm's outputs over many rows of the widths past
5120 (the Flash model's 5376 among them) against its 64-bit value: an element
that a few lanes lose now and then shows only over whole outputs."""
import types

import pytest
import torch

from lynnreal_omni_amd import kernels as k

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden", [(12605, 5376), (6001, 6144), (4099, 7000), (3001, 8192), (12605, 5120),
                                         (333, 5384), (2, 5376)])
def test_whole_bf16_output(rows, hidden):
    """Bound: bf16 roundings (half an ulp, at most 2^-8 of the value) of norm,
    1 + scale and product, each of the product t's size, and of the sum y, with
    a tenth for their products and fp32 noise. A lost element is off by |y|."""
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    x = torch.randn(1, rows, hidden, device="cuda", generator=g).bfloat16()
    norm = types.SimpleNamespace(weight=(1 + 0.05 * torch.randn(hidden, device="cuda", generator=g)).bfloat16(),
                                 eps=1e-6)
    table = (0.1 * torch.randn(6, 6 * hidden, device="cuda", generator=g)).bfloat16()
    indices = torch.arange(rows, device="cuda") * 6 // rows
    slots = table.double().view(6, 6, hidden)[indices]
    n = x[0].double() * torch.rsqrt(x[0].double().square().mean(-1, keepdim=True) + 1e-6) * norm.weight.double()
    want = n * (1 + slots[:, 1]) + slots[:, 0]
    bound = 1.1 * 2 ** -8 * (3 * (want - slots[:, 0]).abs() + want.abs()) + 1e-5
    for fill in (0.0, 3.0):
        torch.empty(rows * hidden, device="cuda", dtype=torch.bfloat16).fill_(fill)   # what a lost store leaves
        got = k._rms_adaln(x, norm, table, indices, 0, 1)[0].double()
        bad = ((got - want).abs() > bound).sum().item()
        assert bad == 0, f"{bad} elements off"


@pytest.mark.parametrize("rows,hidden", [(12605, 5376), (4099, 6144), (2049, 5632), (700, 5376), (3, 6000), (2500, 8192)])
def test_quantizing_norms_equal_their_two_steps(rows, hidden):
    """rms_adaln_quant equals quantize_rows of rms_adaln, and residual_rms_quant
    equals gated_residual followed by it, bit for bit, at every row."""
    g = torch.Generator(device="cuda").manual_seed(rows * 3 + hidden)
    x = torch.randn(1, rows, hidden, device="cuda", generator=g).bfloat16()
    u = torch.randn(1, rows, hidden, device="cuda", generator=g).bfloat16()
    norm = types.SimpleNamespace(weight=(1 + 0.05 * torch.randn(hidden, device="cuda", generator=g)).bfloat16(),
                                 eps=1e-6)
    table = (0.1 * torch.randn(3, 6 * hidden, device="cuda", generator=g)).bfloat16()
    for indices in (torch.arange(rows, device="cuda") * 3 // rows,
                    torch.randint(0, 3, (rows,), device="cuda", generator=g)):
        q, s = k._rms_adaln_quant_int8(x, norm, table, indices, 0, 1)
        q0, s0 = k.quantize_rows(k._rms_adaln(x, norm, table, indices, 0, 1)[0])
        assert torch.equal(q, q0) and torch.equal(s, s0)
        r, q, s = k.residual_rms_quant(x, u, norm, table, indices)
        r0 = k._gated_residual(x, u, table, indices, 2)
        q0, s0 = k._rms_adaln_quant_int8(r0, norm, table, indices, 3, 4)
        assert torch.equal(r, r0) and torch.equal(q, q0) and torch.equal(s, s0)


@pytest.mark.parametrize("table_rows", [1, 3])
@pytest.mark.parametrize("hidden", [8, 2040, 2048, 2056, 4096, 4104, 6144, 6152, 8184, 8192])
def test_row_kernel_edges(hidden, table_rows):
    """One row per block at the edges of its chunk counts, two sequences (rows
    past the first index by row modulo the sequence), against the oracle."""
    import gpu_adapter as gpu
    from helpers import bf16_randn, to_np
    from oracle import reference as ref

    g = torch.Generator().manual_seed(hidden + table_rows)
    x, u = (to_np(bf16_randn((2, 3, hidden), g, outliers=0.01)) for _ in range(2))
    w = to_np((1 + 0.05 * torch.randn(hidden, generator=g)).bfloat16())
    table = to_np(bf16_randn((table_rows, 6 * hidden), g, scale=0.1))
    idx = torch.randint(0, table_rows, (3,), generator=g).numpy()
    args = (x, w, table, idx)
    assert (gpu.rms_adaln(*args, 0, 1, 1e-6) == ref.rms_adaln(*args, 0, 1, 1e-6)).all()
    for got, want in ((gpu.rms_adaln_quant(*args, 3, 4, 1e-6), ref.rms_adaln_quant(*args, 3, 4, 1e-6)),
                      (gpu.residual_rms_quant(x, u, w, table, idx, 1e-6),
                       ref.residual_rms_quant(x, u, w, table, idx, 1e-6))):
        assert all((a == b).all() for a, b in zip(got, want))
