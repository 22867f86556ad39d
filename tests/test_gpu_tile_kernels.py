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


@pytest.mark.parametrize("m,n,k,tile", [
    (1000, 3072, 256, (128, 128)), (2048, 1536, 512, (128, 128)), (8192, 512, 1024, (128, 128)),
    (4096, 2048, 256, (128, 128)), (7955, 192, 10112, (64, 128)), (1099, 1600, 7808, (64, 128)),
    (64, 1024, 2048, (64, 80)), (130, 20480, 5120, (128, 160)), (331, 5376, 7168, (64, 128))])
def test_automatic_choice_off_the_models_sizes(m, n, k, tile):
    """Shapes whose fastest tile (by 12-30% over the cost model's own constants for
    a block's projections) the automatic choice takes: one kernel, its tiles."""
    a = torch.zeros(m, k, dtype=torch.int8, device="cuda")
    w = torch.zeros(n, k, dtype=torch.int8, device="cuda")
    rs, cs = torch.ones(m, device="cuda"), torch.ones(n, device="cuda")
    int8_gemm.int8_matmul(a, w.t(), rs, cs)
    launched = kernels(lambda: int8_gemm.int8_matmul(a, w.t(), rs, cs))
    assert [blocks for blocks, _ in launched] == [-(-m // tile[0]) * -(-n // tile[1])]
