"""More rows than one launch's blocks can have (2^24 of 256 threads): the last
rows' values, and the first ones', which a grid counted modulo 2^32 threads would
run in their place."""
import types

import pytest
import torch

from lynnreal_omni_amd import kernels

pytestmark = pytest.mark.gpu

ROWS = (1 << 24) + 5


def _rows(width, dtype):
    """[ROWS, width] whose first element is the row's number modulo 97 plus 1, the rest half of it."""
    head = (torch.arange(ROWS, device="cuda") % 97 + 1).to(dtype)
    x = (head * 0.5).unsqueeze(1).repeat(1, width)
    x[:, 0] = head
    return x


def _check(q, s, absmax):
    assert torch.equal(s.reshape(-1), absmax.float() / torch.tensor(127.0, device="cuda"))
    assert bool((q[:, 0] == 127).all())
    assert q.shape[1] == 1 or bool(((q[:, 1:] == 63) | (q[:, 1:] == 64)).all())


@pytest.mark.parametrize("width,dtype", [(1, torch.bfloat16), (3, torch.float32), (2, torch.float16)])
def test_quantizer(width, dtype):
    x = _rows(width, dtype)
    q, s = kernels.quantize_rows(x)
    _check(q, s, x[:, 0])


def test_norms_with_a_block_per_row():
    """One column: the normalized row is x / sqrt(x^2 + eps), exactly 1 in bf16.
    Sequences of three rows, one of which lies across each launch's edge, take three
    different shifts."""
    sequence = 3
    x = _rows(1, torch.bfloat16)[:ROWS // sequence * sequence].reshape(-1, sequence, 1)
    rows = x.shape[0] * sequence
    norm = types.SimpleNamespace(weight=torch.ones(1, device="cuda", dtype=torch.bfloat16), eps=1e-6)
    table = torch.zeros(sequence, 6, device="cuda", dtype=torch.bfloat16)
    table[:, 0] = table[:, 3] = torch.tensor([1.0, 3.0, 7.0])
    indices = torch.arange(sequence, device="cuda")
    want = (table[:, 0] + 1).repeat(rows // sequence)
    assert torch.equal(kernels._rms_adaln(x, norm, table, indices, 0, 1).reshape(-1), want)
    q, s = kernels._rms_adaln_quant_int8(x, norm, table, indices, 0, 1)
    _check(q, s, want)
    r, q, s = kernels.residual_rms_quant(x, torch.zeros_like(x), norm, table, indices)
    assert torch.equal(r, x)
    _check(q, s, want)
