"""Single phases of a table whose last build was one launch, which leaves the
lists and splits but not what the partition's two passes hand each other."""
import numpy as np
import pytest

import atg
from test_gpu_build import assert_same_build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("phases", [("partition_place",), ("partition_place", "split", "pack"),
                                    ("sum", "partition_place", "split", "pack")])
@pytest.mark.parametrize("n,section", [(64, 64), (641, 0), (5000, 1700)])
def test_placement_alone(gpu, oracle, n, section, phases):
    w = atg.generate_weights("pareto", n, seed=23, param=1.1)
    ref = oracle.build(w, section_size=section, num_splits=81920)
    t = atg.Table(n, section_size=section, num_splits=81920)
    # Never built: a placement of nothing yet, then a build.
    t.set_weights(w)
    t.build_phase("partition_place")
    for _ in range(2):
        t.build()
        for _ in range(2):
            for ph in phases:
                t.build_phase(ph)
            t.sync()
            assert_same_build(t, ref, n)
    # Another partition's staging is not this build's.
    other = np.ascontiguousarray(w[::-1])
    t.build_phase("partition")
    t.set_weights(other)
    t.build()
    for ph in phases:
        t.build_phase(ph)
    t.sync()
    assert_same_build(t, oracle.build(other, section_size=section, num_splits=81920), n)


@pytest.mark.parametrize("dtype,layout", [("f64", "aos"), ("f32", "soa")])
@pytest.mark.parametrize("n,section,psa", [(641, 0, True), (1023, 2048, True), (5000, 1700, True), (5000, 0, False)])
def test_phases_write_what_they_should(gpu, oracle, dtype, layout, n, section, psa):
    """The phases after a one-launch build of other weights, and the last two
    over rows that were cleared."""
    torch = gpu
    w1, w2 = (atg.generate_weights(d, n, seed=5, param=1.1) for d in ("exponential", "pareto"))
    if dtype == "f32":
        w1, w2 = w1.astype(np.float32), w2.astype(np.float32)
    opts = dict(psa_plus=psa, section_size=section, num_splits=81920)
    dw = torch.from_numpy(w1).cuda()
    t = atg.Table(n, dtype=dtype, layout=layout, **opts)
    t.set_weights(dw)
    t.build()
    t.sync()
    dw.copy_(torch.from_numpy(w2))
    for ph in atg.Table.PHASES:
        t.build_phase(ph)
    t.sync()
    ref = oracle.build(w2.astype(np.float64), **opts)
    assert_same_build(t, ref, n)
    dw.copy_(torch.from_numpy(w1))
    t.build()
    t.sync()
    ref = oracle.build(w1.astype(np.float64), **opts)
    assert_same_build(t, ref, n)
    # The leftovers' rows, which the split and pack write, cleared.
    left = np.concatenate([ref["L_item"][:-1], ref["H_item"][:-1]])
    ptrs = t.device_table_ptr()

    class View:
        def __init__(self, ptr, shape, typestr):
            self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}
    at = torch.from_numpy(left.astype(np.int64)).cuda()
    rows = torch.as_tensor(View(ptrs[0], (n, 2) if layout == "aos" else (n,), "<f8"), device="cuda")
    rows[at] = -1.0
    t.build_phase("split")
    t.build_phase("pack")
    t.sync()
    assert_same_build(t, ref, n)
