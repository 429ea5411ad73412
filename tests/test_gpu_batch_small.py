"""Batches whose small tables are built by a workgroup each, beside the phases
of the larger ones: the oracle's rows for every table, direct and replayed."""
import numpy as np
import pytest

import atg
from test_gpu_build import bits

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 63, 64, 65, 127, 128, 129, 511, 512, 513, 1023, 1024, 1025, 2047]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("sizes,kw,group_items", [
    (EDGES * 3, {}, 0),                                                  # small tables only, every class
    (EDGES * 2 + [2048, 4097, 30_000], {}, 0),                           # beside the phases
    (EDGES * 4 + [2048, 5000] * 3, {}, 20_000),                          # in groups
    ([40] * 300, {}, 0),                                                 # one class
    (EDGES, {"psa_plus": False}, 0),
    (EDGES * 2, {"chains": 1}, 0),
    (EDGES * 2 + [3000], {"split": "learned", "chains": 64}, 0),
    (EDGES * 2, {"section_size": 300, "num_splits": -11}, 0),            # several sections
    ([2049, 4095, 4096, 6143, 8190, 8192, 9000], {}, 0),                 # up to four long sections, past them the phases
    ([2500, 8000] * 3, {"psa_plus": False}, 0),                          # every item in the lists
    ([2500, 8000] * 3, {"chains": 64, "num_splits": -10}, 0),
    ([9, 10, 11, 99, 640, 1279, 1290, 5110, 5130, 8000, 10_230, 10_300, 14_000, 16_000],
     {"section_size": 0, "num_splits": 81_920, "chains": 16}, 0),             # eleven to sixteen sections; past them the phases
    ([700, 13_000, 6_500] * 5 + [40_000], {"section_size": 0, "num_splits": 81_920}, 40_000),
])
def test_small_tables_match_oracle(gpu, oracle, dtype, sizes, kw, group_items):
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    w = np.concatenate([atg.generate_weights(("pareto", "exponential", "unit_uniform")[t % 3], n, seed=50 + t, param=1.1)
                        for t, n in enumerate(sizes)])
    if dtype == "f32":
        w = w.astype(np.float32)
    opts = dict({"section_size": 2048, "chains": 32, "num_splits": -38}, **kw)
    b = atg.Batch(offsets, dtype=dtype, group_items=group_items, **opts)
    b.set_weights(w)
    opts.pop("split", None)
    ow, oa, oW = oracle.build_batch(w, offsets, **opts)
    torch = gpu
    for graph in (False, True):
        b.use_graph(graph)
        for _ in range(3):
            b.build()
            torch.zeros(1 << 20, device="cuda").add_(1.0)  # other work between the builds
            b.sync()
            rw, ra, W = b.tables()
            assert np.array_equal(bits(W), bits(oW))
            bad = np.nonzero((bits(rw) != bits(ow)) | (ra != oa))[0]
            assert bad.size == 0, (bad.size, bad[:5], np.searchsorted(offsets, bad[:5], side="right") - 1)
    lat = b.latencies_ns()
    assert (lat > 0).all() and (lat < 1e9).all()


def test_small_table_with_bad_weights(gpu):
    """One bad table among small ones: reported, its samples -1, the others whole."""
    torch = gpu
    sizes = [100] * 50
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    w = atg.generate_weights("exponential", int(offsets[-1]), seed=4)
    w[offsets[7] + 3] = np.nan
    b = atg.Batch(offsets)
    b.set_weights(w)
    b.build()
    with pytest.raises(atg.AtgError):
        b.sync()
    out = torch.zeros(50 * 8, dtype=torch.int32, device="cuda")
    b.sample(8, 1, out)
    got = out.cpu().numpy().reshape(50, 8)
    assert (got[7] == -1).all() and (np.delete(got, 7, 0) >= 0).all() and (got < 100).all()
