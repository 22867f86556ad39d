"""The kernels that a call launches, read from a captured graph."""
import ctypes

import torch


class _Dim3(ctypes.Structure):
    _fields_ = [(c, ctypes.c_uint32) for c in "xyz"]


class _KernelParams(ctypes.Structure):      # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def _hip():
    """The HIP runtime that this process has loaded."""
    with open("/proc/self/maps") as maps:
        path = next(line.split()[-1] for line in maps if "libamdhip64" in line)
    return ctypes.CDLL(path)


def kernels(call):
    """[(blocks, threads per block)] of the kernels that `call` launches on the
    current stream, in the order of the graph's nodes. `call` has run before."""
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    hip = _hip()
    handle = ctypes.c_void_p(graph.raw_cuda_graph())
    count = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(handle, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * count.value)()
    assert hip.hipGraphGetNodes(handle, nodes, ctypes.byref(count)) == 0
    found = []
    for node in nodes:
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value != 0:      # hipGraphNodeTypeKernel
            continue
        p = _KernelParams()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        found.append((p.grid.x * p.grid.y * p.grid.z, p.block.x * p.block.y * p.block.z))
    return found
