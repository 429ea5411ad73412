"""Replays of a captured batch build whose weights are rewritten in place
between replays: every replay builds all tables, small ones beside the phases
of the others, from the weights of that moment."""
import numpy as np
import pytest

import atg
from launches import kernels
from test_gpu_build import bits

pytestmark = pytest.mark.gpu

SMALL = [1, 2, 63, 64, 65, 129, 513, 1023, 1024, 1025, 2047, 2500]
TINY = [1, 2, 63, 64, 65, 127]  # one class: 1,920 of them pay beside other tables


def weights(sizes, seed, dtype):
    w = np.concatenate([atg.generate_weights(("pareto", "exponential", "unit_uniform")[(t + seed) % 3], n,
                                             seed=seed + t, param=1.1) for t, n in enumerate(sizes)])
    return w.astype(np.float32) if dtype == "f32" else w


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("sizes,kw,group_items,beside", [
    (SMALL * 20, {}, 0, False),                                         # small tables only
    (TINY * 520 + [9000, 40_000], {}, 0, True),                         # beside the phases
    (TINY * 1100 + [9000] * 3, {}, 200_000, True),                      # in two groups
    (SMALL * 4 + [9000, 9000], {}, 0, False),                           # too few: all through the phases
    ([700, 6_500, 13_000] * 160 + [40_000], {"section_size": 0, "num_splits": 81_920, "chains": 16}, 0, True),
])
def test_replays_build_the_weights_of_the_moment(gpu, oracle, dtype, sizes, kw, group_items, beside):
    torch = gpu
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    opts = dict({"section_size": 2048, "chains": 32, "num_splits": -38}, **kw)
    ws = [weights(sizes, seed, dtype) for seed in (1, 2, 3)]
    dw = torch.from_numpy(ws[0]).cuda()
    b = atg.Batch(offsets, dtype=dtype, group_items=group_items, **opts)
    b.set_weights(dw)
    names = kernels(torch, b.build)
    assert ("seg_small" in names and "seg_pack" in names) == beside
    b.use_graph(True)  # before any build: the rows hold nothing yet
    for w in ws:
        dw.copy_(torch.from_numpy(w))
        b.build()
        torch.zeros(1 << 20, device="cuda").add_(1.0)  # other work between the replays
        b.sync()
        rw, ra, W = b.tables()
        ow, oa, oW = oracle.build_batch(w, offsets, **opts)
        assert np.array_equal(bits(W), bits(oW))
        bad = np.nonzero((bits(rw) != bits(ow)) | (ra != oa))[0]
        assert bad.size == 0, (bad.size, bad[:5], np.searchsorted(offsets, bad[:5], side="right") - 1)
        # A build reads memory and meets barriers many times over: it takes
        # microseconds, and a table that was not built a clock tick (10 ns).
        lat = b.latencies_ns()
        assert (lat > 1e3).all() and (lat < 1e9).all()
