"""Launch shapes of a call, read from the kernel nodes of a captured graph that is never launched."""
import ctypes as C

import torch


class _KernelParams(C.Structure):
    _fields_ = [("block", C.c_uint * 3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", C.c_uint * 3),
                ("params", C.c_void_p), ("shared", C.c_uint)]


def _hip():
    for line in open("/proc/self/maps"):
        if "libamdhip64.so" in line:
            return C.CDLL(line.split()[-1])
    raise RuntimeError("libamdhip64.so is not loaded")


def kernel_launches(fn):
    """[(grid, block), ...] of the kernels that fn(stream) launches, in capture order."""
    s = torch.cuda.Stream()
    fn(s)
    s.synchronize()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g, stream=s):
        fn(s)
    hip, graph = _hip(), C.c_void_p(g.raw_cuda_graph())
    n = C.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    nodes = (C.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
    out = []
    for node in nodes:
        kind = C.c_int(-1)
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        if kind.value == 0:  # a kernel
            p = _KernelParams()
            assert hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)) == 0
            out.append((tuple(p.grid), tuple(p.block)))
    return out
