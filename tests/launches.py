"""The kernels that a call launches: the call is captured into a HIP graph, whose nodes are read and which
is never run."""

import ctypes
import glob
import os

import torch


class _KernelNodeParams(ctypes.Structure):   # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint * 3), ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def launches(call, threads=False):
    """[(kernel name, number of workgroups), ...] of call(), which uses torch's current stream; with `threads` the
    threads of a workgroup behind them."""
    hip = ctypes.CDLL(glob.glob(os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so*"))[0])
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    hip.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    call()   # a first launch sets attributes of the kernel, outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    raw, count = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * max(count.value, 1))()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(count)) == 0
    found = []
    for node in nodes[:count.value]:
        kind, params = ctypes.c_int(-1), _KernelNodeParams()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        assert kind.value == 0, "a node that is no kernel"
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(params)) == 0
        name = hip.hipKernelNameRefByPtr(params.func, None)
        found.append(((name or b"").decode(), params.grid[0] * params.grid[1] * params.grid[2])
                     + ((params.block[0] * params.block[1] * params.block[2],) if threads else ()))
    return found
