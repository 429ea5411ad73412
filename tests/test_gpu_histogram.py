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


@pytest.mark.parametrize("layout", ["aos", "soa"])
@pytest.mark.parametrize("n,rows,count", [
    (100_003, 4096, 12_500),       # n / 8 samples: the most that read their rows one by one
    (100_003, 4096, 12_501),       # staged sections
    (100_003, 64, 5_000),          # sections of a row count below a wave's lanes, a few samples each
    (1, 4096, 0), (9, 4096, 1),    # one section: no descent
    (1_000_003, 200, 125_000),     # 5,001 sections: their counts from a launch of their own
    (800_000, 200, 100_000),       # 4,000 sections: counts by the sampling waves
    (5_000_011, 4096, 33),         # at most 32 samples at every node of the descent
    (3_000_000, 8192, 375_000),    # rounds of four full wave loads and a rest
])
def test_sparse_sections_match_oracle(gpu, oracle, layout, n, rows, count):
    """Sectioned draws with few samples per row against the oracle's stream."""
    torch = gpu
    w = atg.generate_weights("pareto", n, seed=9, param=1.1)
    t = atg.Table(n, layout=layout)
    t.set_weights(w)
    t.build()
    tw, ta = t.table()
    out = torch.full((max(count, 1),), -7, dtype=torch.int32, device="cuda")
    hist = torch.zeros(n, dtype=torch.int32, device="cuda")
    t.sample(count, 31, section_rows=rows, out=out)
    exp = oracle.sample_sectioned(tw, ta, t.stats()["W_N"], rows, count, 31) if count else np.empty(0, np.int32)
    np.testing.assert_array_equal(out.cpu().numpy()[:count], exp)
    t.sample(count, 31, section_rows=rows, hist=hist)
    np.testing.assert_array_equal(hist.cpu().numpy(), np.bincount(exp, minlength=n))


@pytest.mark.parametrize("layout", ["aos", "soa"])
def test_longest_sections_with_counts(gpu, oracle, layout):
    """8,192 rows or slots and the block's counters: the most LDS of a draw."""
    torch = gpu
    n, count = 50_001, 60_000
    w = atg.generate_weights("pareto", n, seed=9, param=1.1)
    t = atg.Table(n, layout=layout)
    t.set_weights(w)
    t.build()
    tw, ta = t.table()
    out = torch.empty(count, dtype=torch.int32, device="cuda")
    hist = torch.zeros(n, dtype=torch.int32, device="cuda")
    t.sample(count, 31, section_rows=8192, out=out, hist=hist)
    exp = oracle.sample_sectioned(tw, ta, t.stats()["W_N"], 8192, count, 31)
    np.testing.assert_array_equal(out.cpu().numpy(), exp)
    np.testing.assert_array_equal(hist.cpu().numpy(), np.bincount(exp, minlength=n))
    t.rejection_build()
    W = t.rejection_weight_sum()
    _, A = oracle.rejection_build(w, W)
    hist.zero_()
    t.rejection_sample_sectioned(count, 32, section_slots=8192, out=out, hist=hist)
    exp = oracle.sample_rejection_sectioned(A, w, W, 8192, count, 32)
    np.testing.assert_array_equal(out.cpu().numpy(), exp)
    np.testing.assert_array_equal(hist.cpu().numpy(), np.bincount(exp, minlength=n))


@pytest.mark.parametrize("count", [1, 2047, 2048])
def test_few_staged_counts(gpu, count):
    """Staged draws below and at the fewest samples that count in LDS."""
    torch = gpu
    n = 1000
    t = atg.Table(n)
    t.set_weights(atg.generate_weights("pareto", n, seed=3, param=1.1))
    t.build()
    t.rejection_build()
    out = torch.empty(count, dtype=torch.int32, device="cuda")
    for draw in (lambda **k: t.sample(count, 5, **k), lambda **k: t.rejection_sample_sectioned(count, 5, **k)):
        hist = torch.zeros(n, dtype=torch.int32, device="cuda")
        draw(out=out, hist=hist)
        np.testing.assert_array_equal(hist.cpu().numpy(), np.bincount(out.cpu().numpy(), minlength=n))
