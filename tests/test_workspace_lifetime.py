"""The split-K workspace of int8_matmul is alive when its kernels are launched
(on the CPU, with the launch itself replaced): under capture, where nothing else
keeps it, and where another thread's larger call replaces the kept buffer in
between."""
import weakref

import pytest
import torch

from lynnreal_omni_amd import _lib, int8_gemm


@pytest.mark.parametrize("capturing", [True, False])
def test_workspace_is_held_until_the_launch(monkeypatch, capturing):
    m, n, k = 32, 1024, 4096
    a, b = torch.zeros(m, k, dtype=torch.int8), torch.zeros(n, k, dtype=torch.int8).t()
    need = int8_gemm._workspace_bytes(m, n, k, 0, _lib.TILE_AUTO)
    assert need > 0
    buffers, launched = [], []
    empty = torch.empty

    def recorded_empty(*args, **kw):
        t = empty(*args, **kw)
        buffers.append((weakref.ref(t), t.data_ptr(), t.numel()))
        return t

    def call(name, *args):
        _lib._workspaces.clear()      # what a larger call of another thread does to the kept buffer
        ref, pointer, size = buffers[-1]
        launched.append(ref() is not None and args[19] == pointer and args[20] == size >= need)

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    monkeypatch.setattr(torch, "empty", recorded_empty)
    monkeypatch.setattr(_lib, "_workspaces", {})
    monkeypatch.setattr(_lib, "stream", lambda t: 0)
    monkeypatch.setattr(_lib, "call", call)
    int8_gemm._launch(a, b, None, None, None, a, _lib.EPI_RAW_INT32, None)
    assert launched == [True]
