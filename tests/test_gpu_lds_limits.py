"""The dynamic LDS a kernel is allowed is state of the process: a call that
needs little must not lower it under another thread's launch, or under a
captured graph that holds a larger one."""
import ctypes as C
import subprocess

import numpy as np
import pytest

import atg

pytestmark = pytest.mark.gpu


class FuncAttributes(C.Structure):
    _fields_ = [("binaryVersion", C.c_int), ("cacheModeCA", C.c_int), ("constSizeBytes", C.c_size_t),
                ("localSizeBytes", C.c_size_t), ("maxDynamicSharedSizeBytes", C.c_int), ("maxThreadsPerBlock", C.c_int),
                ("numRegs", C.c_int), ("preferredShmemCarveout", C.c_int), ("ptxVersion", C.c_int),
                ("sharedSizeBytes", C.c_size_t)]


def limits(part):
    """Dynamic LDS limits of the library's kernels whose name holds `part`."""
    names = [l.split()[-1] for l in subprocess.run(["nm", "-D", atg._lib.LIB_PATH], capture_output=True, text=True,
                                                   check=True).stdout.splitlines() if " V _ZN3atg" in l and part in l]
    assert names
    L, out = atg.lib(), {}
    for name in names:
        a = FuncAttributes()
        assert L.hipFuncGetAttributes(C.byref(a), C.c_void_p(C.addressof(C.c_char.in_dll(L, name)))) == 0
        out[name] = a.maxDynamicSharedSizeBytes
    return out


def one_build(n):
    t = atg.Table(n)
    t.set_weights(atg.generate_weights("pareto", n, seed=1, param=1.1))
    t.build()
    t.sync()


def batch(n):
    b = atg.Batch(np.array([0, n], np.int64), section_size=1000, num_splits=-10)
    b.set_weights(atg.generate_weights("pareto", n, seed=1, param=1.1))
    b.build()
    b.sync()


def draws(torch, rows):
    t = atg.Table(20_000)
    t.set_weights(atg.generate_weights("pareto", 20_000, seed=1, param=1.1))
    t.build()
    t.rejection_build()
    hist = torch.zeros(20_000, dtype=torch.int32, device="cuda")
    t.sample(40_000, 3, section_rows=rows, hist=hist)
    t.rejection_sample_sectioned(40_000, 3, section_slots=rows, hist=hist)
    t.sync()


def test_smaller_calls_leave_the_limit(gpu):
    for part, call, sizes in (("build_small", one_build, (6300, 3500)), ("seg_small", batch, (12_000, 8000)),
                              ("sample_sectioned", lambda r: draws(gpu, r), (8192, 5000))):
        call(sizes[0])
        before = limits(part)
        call(sizes[1])
        after = limits(part)
        print(part, sorted(set(before.values())), sorted(set(after.values())))
        assert all(after[k] >= before[k] for k in before), (part, before, after)
