"""Which kernel a named GEMM tile runs: its own grid of tiles, and for K off the
k-step the substitute that is documented where it has none."""
import pytest
import torch

from graph_nodes import kernels
from lynnreal_omni_amd import int8_gemm

pytestmark = pytest.mark.gpu

M, N = 513, 520      # a different number of tiles for every shape below


def _launched(tile, k):
    a = torch.zeros(M, k, dtype=torch.int8, device="cuda")
    w = torch.zeros(N, k, dtype=torch.int8, device="cuda")
    rs, cs = torch.ones(M, device="cuda"), torch.ones(N, device="cuda")
    int8_gemm.int8_matmul(a, w.t(), rs, cs, tile=tile)
    return kernels(lambda: int8_gemm.int8_matmul(a, w.t(), rs, cs, tile=tile))


def _tiles(rows, cols):
    return -(-M // rows) * -(-N // cols)


@pytest.mark.parametrize("tile", sorted(t for t in int8_gemm._TILES), ids=str)
def test_tile_runs_its_own_grid(tile):
    assert [blocks for blocks, _ in _launched(tile, 384)] == [_tiles(*tile)]
    own = (128, 128) if tile in int8_gemm._ALIGNED_ONLY else tile
    assert [blocks for blocks, _ in _launched(tile, 400)] == [_tiles(*own)]


def test_waves_of_the_tiles_with_two_kernels():
    """(256, 128) and (128, 256): 8 waves at K % 128 == 0, 4 otherwise."""
    for tile in ((256, 128), (128, 256)):
        assert [threads for _, threads in _launched(tile, 384) + _launched(tile, 400)] == [512, 256]
