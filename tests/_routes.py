"""Which kernels a call enqueues: their names and workgroup sizes, read from the
nodes of a HIP graph that captures the call."""

from __future__ import annotations

import ctypes

import torch

_KERNEL_NODE = 0  # hipGraphNodeTypeKernel


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class _KernelNodeParams(ctypes.Structure):
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def _hip():
    lib = ctypes.CDLL("libamdhip64.so.7")
    lib.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    lib.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return lib


def kernels_of(call) -> list[tuple[str, int]]:
    """(mangled name, threads per workgroup) of every kernel that ``call``
    enqueues, in order. The call runs once before it is captured."""
    hip = _hip()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    side.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=side):
        call()
    raw = ctypes.c_void_p(graph.raw_cuda_graph())
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0 and kind.value == _KERNEL_NODE
        p = _KernelNodeParams()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        out.append((hip.hipKernelNameRefByPtr(p.func, None).decode(), p.block.x))
    return out
