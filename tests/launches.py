"""The kernel launches of a library call, read from a captured HIP graph
(nothing runs): a route or a launch shape can be checked without a clock."""
import ctypes
import re

import torch


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]


class _KernelNodeParams(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.POINTER(ctypes.c_void_p)), ("shared", ctypes.c_uint)]


class Launch:
    """One kernel node; `key` is (function, blocks, threads, dynamic LDS)."""

    def __init__(self, p, words):
        self.key = (p.func, p.grid.x, p.block.x, p.shared)
        self.blocks, self.threads, self.shared = p.grid.x, p.block.x, p.shared
        self.words = words  # first 32 bits of the parameters asked for


def _hip():
    with open("/proc/self/maps") as f:
        path = re.search(r"(/\S*libamdhip64\.so\S*)", f.read()).group(1)
    return ctypes.CDLL(path)


def _check(rc):
    if rc:
        raise RuntimeError(f"HIP error {rc}")


def launches(call, params=None):
    """The launches of call(stream), in capture order.  params[i]: indices of
    parameters of launch i whose first 32 bits to read."""
    hip = _hip()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph, n = ctypes.c_void_p(), ctypes.c_size_t()
    st = ctypes.c_void_p(stream.cuda_stream)
    _check(hip.hipStreamBeginCapture(st, 2))  # relaxed
    call(stream.cuda_stream)
    _check(hip.hipStreamEndCapture(st, ctypes.byref(graph)))
    _check(hip.hipGraphGetNodes(graph, None, ctypes.byref(n)))
    nodes = (ctypes.c_void_p * n.value)()
    _check(hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)))
    out = []
    for node in nodes:
        kind = ctypes.c_int()
        _check(hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)))
        if kind.value:  # not a kernel
            continue
        p = _KernelNodeParams()
        _check(hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)))
        want = (params or {}).get(len(out), ())
        out.append(Launch(p, [ctypes.cast(p.params[i], ctypes.POINTER(ctypes.c_uint32))[0] for i in want]))
    _check(hip.hipGraphDestroy(graph))
    return out
