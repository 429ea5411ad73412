"""The partition pass of builds with more sections than the device holds at
once (rows written after the chains, whole sections or chain by chain) against
the oracle, bit for bit, at the edges of its chunks and chains."""
import numpy as np
import pytest

import atg
from test_gpu_build import assert_same_build, gpu_build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,layout", [("f64", "aos"), ("f32", "soa")])
@pytest.mark.parametrize("n,dist,chains,section", [
    (40_000, "pareto", 16, 1),                # a section per item or two
    (120_001, "exponential", 64, 7),          # more chains than items
    (400_003, "unit_uniform", 16, 33),        # partial chunks, nearly all rows from the chains
    (900_001, "pareto", 3, 64),               # sections of a chunk and one item
    (1_500_000, "heavy_mix", 16, 100),        # few rows from the chains: written chain by chain
    (2_000_003, "powerlaw2", 1, 200),         # one chain, several episodes of 64 steps
    (5_000_011, "unit_uniform", 16, 1000),    # the default section
    (5_000_000, "best_worst", 17, 1024),      # the longest short section
    (9_000_001, "exponential", 2, 2047),      # long chains in the long-section kernel
    (9_000_000, "pareto", 64, 2048),          # the longest section
])
def test_many_sections_match_oracle(gpu, oracle, dtype, layout, n, dist, chains, section):
    w = atg.generate_weights(dist, n, seed=17, param={"pareto": 1.1, "heavy_mix": 0.9}.get(dist, 0.0))
    if dtype == "f32":
        w = w.astype(np.float32)
    p = max(2, n // 40)
    t = gpu_build(w, dtype=dtype, layout=layout, chains=chains, section_size=section, num_splits=p)
    ref = oracle.build(w.astype(np.float64), chains=chains, section_size=section, num_splits=p)
    assert_same_build(t, ref, n)


def test_batch_with_many_sections_matches_single_tables(gpu, oracle):
    """More sections than fit at once in a batch: the same rows as the oracle."""
    sizes = [100_000, 1, 63, 64, 65, 2049, 4097, 300_001, 17] * 6
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    w = atg.generate_weights("pareto", int(offsets[-1]), seed=3, param=1.1)
    b = atg.Batch(offsets, section_size=64, chains=8, num_splits=-38)
    b.set_weights(w)
    b.build()
    b.sync()
    rw, ra, W = b.tables()
    ow, oa, oW = oracle.build_batch(w, offsets, chains=8, section_size=64, num_splits=-38)
    assert np.array_equal(W.view(np.uint64), oW.view(np.uint64))
    assert np.array_equal(rw.view(np.uint64), ow.view(np.uint64)) and np.array_equal(ra, oa)


@pytest.mark.parametrize("n,dist", [((1 << 24) + 5, "exponential"), ((1 << 24) - 5, "exponential")])
def test_long_sections_around_the_cached_rows(gpu, oracle, n, dist):
    """16-byte rows of sections of 2048 just past and just within what the rule
    takes for cached: whole sections after the chains, and rows by each step."""
    w = atg.generate_weights(dist, n, seed=17)
    t = gpu_build(w, chains=17, section_size=2048, num_splits=n // 64)
    assert_same_build(t, oracle.build(w, chains=17, section_size=2048, num_splits=n // 64), n)


def test_large_batch_with_many_long_sections(gpu, oracle):
    """A batch whose rows are written after the chains."""
    sizes = [3_000_000, 1, 2047, 2048, 2049, 64, 4_500_000, 100_001] * 3
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    assert offsets[-1] > 1 << 24
    w = atg.generate_weights("exponential", int(offsets[-1]), seed=3)
    b = atg.Batch(offsets, section_size=2048, chains=32, num_splits=-38)
    b.set_weights(w)
    b.build()
    b.sync()
    rw, ra, W = b.tables()
    ow, oa, oW = oracle.build_batch(w, offsets, chains=32, section_size=2048, num_splits=-38)
    assert np.array_equal(W.view(np.uint64), oW.view(np.uint64))
    assert np.array_equal(rw.view(np.uint64), ow.view(np.uint64)) and np.array_equal(ra, oa)
