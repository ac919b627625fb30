"""The kernel launches of a call, read from a captured graph (no kernel runs), for
GPU tests of which shape a dispatch chose."""
import ctypes

from hiprt import rt


class _KernelParams(ctypes.Structure):
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p),
                ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3),
                ("params", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


def launches(call, stream):
    """[(kernel, grid, block, dynamic LDS bytes)] of `call(stream)`, in the order of
    the graph's nodes; `stream` is a handle of tests/hiprt.py."""
    L, st, graph = rt(), ctypes.c_void_p(stream), ctypes.c_void_p()
    assert L.hipStreamBeginCapture(st, 2) == 0   # relaxed
    try:
        call(stream)
    finally:
        rc = L.hipStreamEndCapture(st, ctypes.byref(graph))
    assert rc == 0
    n = ctypes.c_size_t()
    assert L.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert L.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        p = _KernelParams()
        assert L.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        out.append((p.func, tuple(p.grid), tuple(p.block), p.lds))
    assert L.hipGraphDestroy(graph) == 0
    return out
