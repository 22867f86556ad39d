"""Problems whose launch would have 2^32 threads or more, of which the GPU runs only
the count modulo 2^32: refused before anything is launched (the pointers here
are never used)."""
import pytest

from lynnreal_omni_amd import _lib

P = 1 << 20          # aligned, not null
MAX = (1 << 24) - 1  # blocks of 256 threads


@pytest.mark.parametrize("name,args", [
    ("lr_gather_rows", (P, P, P, 1, 8, MAX + 1, 1024, None)),
    ("lr_gather_rows", (P, P, P, 1, 8, 256 * MAX + 1, 1, None)),
    ("lr_flash_restore", (P, P, P, P, P, 1, MAX, 8, 8, 1.0, None)),         # whole rows per XCD: MAX + 1 blocks
    ("lr_flash_restore", (P, P, P, P, P, 1, 256 * MAX + 1, 8, 1, 1.0, None)),
    ("lr_flash_nearest_anchor", (P, 8, P, 1 << 32, P, 8, P, None)),
    ("lr_swiglu_quant", (P, P, P, MAX + 1, 8, None)),
    ("lr_gelu_quant", (P, P, P, MAX + 1, 8, None)),
    ("lr_gelu_tanh", (P, P, 256 * MAX + 1, None)),
    ("lr_swiglu", (P, P, 256 * MAX + 1, 1, None)),
    ("lr_gated_residual", (P, P, P, P, P, 256 * MAX + 1, 1, 1, 1, 6, 2, None)),
    ("lr_int8_epilogue", (P, P, P, None, P, 256 * MAX + 1, 1, None)),
    ("lr_qk_norm_rope", None),
])
def test_refused(name, args):
    lib = _lib.load()
    if args is None:
        args = (P, P, P, P, None, None, P, P, 1, 4 * MAX + 1, 1, 32, 32, 32, 32, 32, 0, 1e-6, None)
    status = getattr(lib, name)(*args)
    message = lib.lr_last_error()
    assert status in (_lib.LR_EINVAL, _lib.LR_EUNSUPPORTED) and b"too" in message, (status, message)
