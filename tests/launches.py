"""The kernels that a call launches, from a capture of the call: no launch
runs, and nothing is timed."""
import ctypes as C
import functools
import re
import subprocess

import atg


class _Dim(C.Structure):
    _fields_ = [("x", C.c_uint32), ("y", C.c_uint32), ("z", C.c_uint32)]


class _KernelNode(C.Structure):
    _fields_ = [("block", _Dim), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", _Dim), ("params", C.c_void_p),
                ("shared", C.c_uint32)]


@functools.lru_cache(None)
def _names():
    """Address of each kernel's handle in the loaded library -> its name."""
    out = subprocess.run(["nm", "-D", "--defined-only", atg._lib.LIB_PATH], capture_output=True, text=True, check=True).stdout
    names = {}
    for line in out.splitlines():
        sym = line.split()[-1]
        m = re.match(r"_ZN3atg(\d+)", sym)
        if line.split()[-2] in "VDR" and m:
            n = int(m.group(1))
            names[C.addressof(C.c_char.in_dll(atg.lib(), sym))] = sym[m.end():m.end() + n]
    return names


def launches(torch, call):
    """[(kernel, blocks, threads, dynamic LDS)] that call(stream) enqueues."""
    L = atg.lib()
    stream = torch.cuda.Stream()
    graph = C.c_void_p()
    assert L.hipStreamBeginCapture(C.c_void_p(stream.cuda_stream), 1) == 0  # thread-local
    try:
        call(stream)
    finally:
        rc = L.hipStreamEndCapture(C.c_void_p(stream.cuda_stream), C.byref(graph))
    assert rc == 0 and graph.value
    count = C.c_size_t(0)
    assert L.hipGraphGetNodes(graph, None, C.byref(count)) == 0
    nodes = (C.c_void_p * max(count.value, 1))()
    assert L.hipGraphGetNodes(graph, nodes, C.byref(count)) == 0
    found = []
    for node in nodes[:count.value]:
        kind = C.c_int(-1)
        assert L.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        if kind.value == 0:
            p = _KernelNode()
            assert L.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)) == 0
            found.append((_names().get(p.func, "?"), p.grid.x, p.block.x, p.shared))
    assert L.hipGraphDestroy(graph) == 0
    return found


def kernels(torch, call):
    return [k[0] for k in launches(torch, call)]
