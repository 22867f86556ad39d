"""The automatic GEMM schedule on the CPU (lr_int8_gemm_workspace_size runs the
same choice as the launch): slices within their bounds, no split where there is
nothing to fill, the same answer on every call and in every thread."""
import random
import threading

from lynnreal_omni_amd import _lib

CAP = 22 << 20


def _size(m, n, k, splits=0):
    return _lib.load().lr_int8_gemm_workspace_size(m, n, k, splits, _lib.TILE_AUTO)


def test_automatic_slices_stay_within_bounds():
    rng = random.Random(3)
    for _ in range(600):
        m, n, k = rng.randint(1, 3000), 4 * rng.randint(1, 8000), 128 * rng.randint(1, 200)
        need = _size(m, n, k)
        assert 0 <= need <= CAP and need % (4 * m * n) == 0, (m, n, k)
        slices = need // (4 * m * n)
        assert slices != 1 and slices <= 8 and 4 * slices <= max(4, k // 128), (m, n, k, slices)
        assert _size(m, n + 2, k) == 0 and _size(m, n, k + 16) == 0   # N % 4, K % 128


def test_large_shapes_do_not_split_and_small_ones_do():
    for m, n, k in ((12288, 5120, 20480), (2048, 5120, 5120), (256, 5120, 5120), (3683, 5376, 14336)):
        assert _size(m, n, k) == 0
    for m, n, k in ((1, 5120, 5120), (32, 5376, 7168), (64, 5376, 14336), (256, 5120, 20480)):
        assert _size(m, n, k) > 0
    assert _size(32, 5376, 7168, 5) == 5 * 32 * 5376 * 4   # a forced split is kept


def test_choice_is_the_same_in_every_thread():
    shapes = [(m, 5376, k) for m in (1, 17, 32, 100, 256, 300) for k in (1024, 7168, 14336)] * 20
    want = [_size(*s) for s in shapes]
    got = {}

    def work(i):
        got[i] = [_size(*s) for s in (shapes if i % 2 else shapes[::-1])]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(got[i] == (want if i % 2 else want[::-1]) for i in range(4))


def test_light_shapes_do_not_split_where_a_split_costs():
    """Weights far below a block's projection, where the slices' second launch
    costs more than the shorter loops save (measured: 12-27% slower split)."""
    for m, n, k in ((64, 1024, 2048), (256, 512, 2048), (128, 2048, 2048), (4096, 256, 8192), (2048, 512, 8192),
                    (1000, 2048, 8192)):
        assert _size(m, n, k) == 0, (m, n, k)
