"""Counts per item of the samplers: the histogram a call adds to equals the
count of its own output, whether the counts go to device memory one by one or
through a block's LDS counters (few, many and clashing items; hot items)."""
import numpy as np
import pytest

import atg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["basic", "sectioned", "rejection", "rejection_sectioned"])
@pytest.mark.parametrize("n,dist,count", [
    (1, "unit_uniform", 20_000),         # one counter
    (4096, "pareto", 16_383),            # below the smallest call that counts in LDS
    (4096, "pareto", 16_384),            # a slot per item
    (4097, "unit_uniform", 50_001),      # two items share a slot
    (300_001, "heavy_mix", 1_000_003),   # hot items among many
    (100_003, "one_heavy", 3_000_000),   # one item draws nearly everything
])
def test_histogram_counts_the_output(gpu, kind, n, dist, count):
    torch = gpu
    w = atg.generate_weights(dist, n, seed=21, param={"pareto": 1.1, "heavy_mix": 0.9}.get(dist, 0.0))
    t = atg.Table(n)
    t.set_weights(w)
    out = torch.empty(count, dtype=torch.int32, device="cuda")
    hist = torch.ones(n, dtype=torch.int32, device="cuda")  # incremented, not overwritten
    if kind.startswith("rejection"):
        t.rejection_build()
        draw = t.rejection_sample if kind == "rejection" else t.rejection_sample_sectioned
    else:
        t.build()
        draw = lambda *a, **k: t.sample(*a, kind=kind, **k)  # noqa: E731
    cs = draw(count, 77, out=out, hist=hist, checksum=True)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(hist.cpu().numpy() - 1, np.bincount(got, minlength=n))
    assert cs == int(got.astype(np.int64).sum())
    # The histogram alone: the same counts on top.
    draw(count, 77, hist=hist)
    np.testing.assert_array_equal(hist.cpu().numpy() - 1, 2 * np.bincount(got, minlength=n))
