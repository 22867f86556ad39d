"""GPU parity of the mid-size GEMM tiles (8 waves, rings of any depth) and of
the automatic choice between tiles and K splits.

Every tile and split computes the same exact int32 sums and the same epilogue
arithmetic, so each must equal the generic kernel (int32 dot products, any
shape) bit for bit: at one k-step, at k-steps around each ring's depth, one row
or column past a tile and one short of it, and through every epilogue.
"""
import pytest
import torch

from helpers import bf16_randn
from lynnreal_omni_amd import _lib, int8_gemm

pytestmark = pytest.mark.gpu

TILES = [(224, 256), (160, 256), (128, 256), (256, 128), (192, 128), (128, 192), (96, 128)]


def _case(m, n, k, epilogue, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randint(-127, 128, (m, k), dtype=torch.int8, generator=g).cuda()
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, generator=g).cuda()
    rs = (torch.rand(m, generator=g) * 1e-2 + 1e-3).cuda()
    cs = (torch.rand(n, generator=g) * 4e-3 + 1e-3).cuda()
    b = (0.02 * torch.randn(n, generator=g)).bfloat16().cuda()
    kw = {}
    if epilogue == "gelu":
        kw = {"activation": "gelu_tanh"}
    elif epilogue == "gated":
        kw = {"residual": bf16_randn((1, m, n), g).cuda(),
              "table": (0.1 * torch.randn(3, 6 * n, generator=g)).bfloat16().cuda(),
              "indices": torch.randint(0, 3, (m,), generator=g).cuda(), "gate_slot": 2}
    return (a, w.t(), rs, cs, b), kw


@pytest.mark.parametrize("tile", TILES, ids=str)
@pytest.mark.parametrize("k", [128, 256, 384, 512, 640, 1408])
def test_tile_edges_int32(tile, k):
    """Rows and columns one past and one short of whole tiles, k-steps from one
    to past the deepest ring."""
    rows, cols = tile
    for m, n in ((rows + 1, cols + 8), (2 * rows - 1, cols - 4), (1, 2 * cols + 12)):
        (a, w, *_), _ = _case(m, n, k, "raw", m + n + k)
        want = int8_gemm.int8_matmul_int32(a, w, tile="generic")
        assert torch.equal(int8_gemm.int8_matmul_int32(a, w, tile=tile), want), (m, n)


@pytest.mark.parametrize("tile", TILES, ids=str)
@pytest.mark.parametrize("epilogue", ["bf16", "gelu", "gated"])
def test_tile_epilogues(tile, epilogue):
    """Staged (N % 8 == 0) and direct (N % 4, odd N) stores, K slices, and K off
    the k-step (which has no kernel of its own tile)."""
    rows, cols = tile
    for m, n, k in ((rows + 37, cols + 40, 512), (rows - 3, cols + 12, 384), (70, cols + 5, 256),
                    (rows + 1, cols + 16, 400)):
        args, kw = _case(m, n, k, epilogue, m + n + k)
        want = int8_gemm.int8_matmul(*args, tile="generic", **kw)
        assert torch.equal(int8_gemm.int8_matmul(*args, tile=tile, **kw), want), (m, n, k)
        if k % 128 == 0 and n % 4 == 0:
            assert torch.equal(int8_gemm.int8_matmul(*args, tile=tile, splits=2, **kw), want), (m, n, k)


@pytest.mark.parametrize("epilogue", ["bf16", "gelu", "gated"])
@pytest.mark.parametrize("m,n,k", [
    (1, 640, 2048), (33, 1056, 4096), (65, 264, 7168), (129, 2056, 1024), (257, 1036, 1152), (511, 772, 640),
    (900, 520, 512), (1500, 1288, 256), (97, 1001, 1040), (300, 510, 976)])
def test_automatic_choice(m, n, k, epilogue):
    """The automatic tile and split against the generic kernel, off-tile sizes
    and K off the k-step among them."""
    args, kw = _case(m, n, k, epilogue, m + n + k)
    assert torch.equal(int8_gemm.int8_matmul(*args, **kw), int8_gemm.int8_matmul(*args, tile="generic", **kw))


def test_automatic_split_under_capture():
    """Under capture an automatic split takes its slices from the graph's own
    memory: replays stay equal to the eager result while eager calls outgrow
    and replace the kept workspace on the same stream."""
    (a, w, rs, cs, b), _ = _case(32, 1024, 4096, "bf16", 3)
    assert _lib.load().lr_int8_gemm_workspace_size(32, 1024, 4096, 0, _lib.TILE_AUTO) > 0
    want = int8_gemm.int8_matmul(a, w, rs, cs, b, splits=1)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        int8_gemm.int8_matmul(a, w, rs, cs, b)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            got = int8_gemm.int8_matmul(a, w, rs, cs, b)
        big, kw = _case(256, 5120, 16384, "bf16", 4)
        for _ in range(3):
            int8_gemm.int8_matmul(*big, **kw)
            held = [torch.full((32, 1024), 7, dtype=torch.int32, device="cuda") for _ in range(8)]
            got.zero_()
            graph.replay()
            side.synchronize()
            assert torch.equal(got, want)
            assert all(bool((h == 7).all()) for h in held)
