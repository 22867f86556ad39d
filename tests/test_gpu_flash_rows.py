"""Row gather and restore at the widths where a thread's number of 16-byte chunks
changes: below one chunk per thread, at each multiple of 256 chunks and one chunk
past it, and past the widest row held in registers."""
import numpy as np
import pytest
import torch

from helpers import bf16_randn, to_np
from lynnreal_omni_amd import flash
from oracle import reference as ref

pytestmark = pytest.mark.gpu

CHUNKS = [1, 3, 63, 64, 256, 257, 511, 512, 513, 768, 769, 1024, 1025]


@pytest.mark.parametrize("chunks", CHUNKS)
@pytest.mark.parametrize("outer", [1, 3])
def test_gather_chunk_edges(chunks, outer):
    g = torch.Generator().manual_seed(chunks)
    src = torch.randint(-128, 128, (outer, 41, 16 * chunks), dtype=torch.int8, generator=g)
    index = torch.cat([torch.randperm(41, generator=g)[:17], torch.tensor([40, 0, 0])])
    out = flash.gather_rows(src.cuda(), index.cuda(), 1)
    assert torch.equal(out.cpu(), src.index_select(1, index))


@pytest.mark.parametrize("chunks", CHUNKS)
@pytest.mark.parametrize("batch", [1, 2])
def test_restore_chunk_edges(chunks, batch):
    rows, compressed, width = 43, 11, 8 * chunks
    g = torch.Generator().manual_seed(chunks)
    full = bf16_randn((batch, rows, width), g)
    cur, inp = (bf16_randn((batch, compressed, width), g) for _ in range(2))
    inverse = torch.randint(0, compressed, (rows,), generator=g)
    out = flash.restore(full.cuda(), cur.cuda(), inp.cuda(), inverse.cuda(), 0.75)
    want = ref.flash_restore(to_np(full), to_np(cur), to_np(inp), inverse.numpy(), 0.75)
    assert np.array_equal(to_np(out.cpu()), want)
