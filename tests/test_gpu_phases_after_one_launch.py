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
