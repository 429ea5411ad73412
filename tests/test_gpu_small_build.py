"""One-launch builds of small tables against the oracle, and against the same
handle built phase by phase: rows, lists, splits and state, bit for bit."""
import numpy as np
import pytest

import atg
from test_gpu_build import assert_same_build, bits, gpu_build

pytestmark = pytest.mark.gpu


def weights(n, dist, dtype="f64"):
    w = atg.generate_weights(dist, n, seed=23, param={"pareto": 1.1, "heavy_mix": 0.9}.get(dist, 0.0))
    return w.astype(np.float32) if dtype == "f32" else w


@pytest.mark.parametrize("dtype,layout", [("f64", "aos"), ("f32", "soa")])
@pytest.mark.parametrize("n,dist,psa,chains,section,p", [
    (1, "unit_uniform", True, 16, 0, 0),       # degenerate
    (2, "pareto", True, 16, 0, 0),
    (10, "pareto", False, 16, 0, 0),
    (63, "exponential", True, 64, 0, 0),
    (64, "exponential", True, 64, 64, 0),      # two sections, the second nearly empty
    (65, "unit_uniform", True, 1, 4096, 0),    # one section of a chunk and one item
    (641, "pareto", True, 16, 0, 0),           # eleven sections
    (1000, "one_heavy", True, 16, 0, 0),
    (1024, "best_worst", True, 17, 65, 0),     # sixteen sections, a wave each
    (1023, "pareto", True, 32, 2048, 27),      # one section, the longest short one
    (1024, "pareto", True, 32, 2048, 27),      # one section of the long kernel
    (2047, "heavy_mix", True, 16, 2048, 2),    # two long pack chains
    (5000, "exponential", False, 16, 0, 0),    # every item in the lists
    (5000, "powerlaw2", True, 3, 1700, 400),   # three long sections
    (6300, "pareto", True, 16, 0, 0),          # nearly all of the LDS
    (8192, "zipf_shuffled", True, 16, 0, 0),   # past it: the phases
])
def test_small_build_matches_oracle(gpu, oracle, dtype, layout, n, dist, psa, chains, section, p):
    w = weights(n, dist, dtype)
    p_req = p if p > 0 else 320 * gpu.cuda.get_device_properties(0).multi_processor_count
    t = gpu_build(w, dtype=dtype, layout=layout, psa_plus=psa, chains=chains, section_size=section, num_splits=p_req)
    ref = oracle.build(w.astype(np.float64), psa_plus=psa, chains=chains, section_size=section, num_splits=p_req)
    assert_same_build(t, ref, n)
    one = t.stats()
    # The last phases again over the lists it left, then all of them.
    for phases in (("split", "pack"), atg.Table.PHASES, ("pack",)):
        for ph in phases:
            t.build_phase(ph)
        t.sync()
        assert_same_build(t, ref, n)
    two = t.stats()
    assert {k: v for k, v in one.items() if k != "phase_ms"} == {k: v for k, v in two.items() if k != "phase_ms"}
    t.build()
    t.sync()
    assert_same_build(t, ref, n)


def test_small_build_rejects_bad_weights_and_recovers(gpu, oracle):
    n = 777
    t = atg.Table(n)
    for bad in (np.nan, -1.0, np.inf):
        w = weights(n, "pareto")
        w[500] = bad
        t.set_weights(w)
        t.build()
        with pytest.raises(atg.AtgError):
            t.sync()
    t.set_weights(np.zeros(n))
    t.build()
    with pytest.raises(atg.AtgError):
        t.sync()
    w = weights(n, "pareto")
    t.set_weights(w)
    t.build()
    t.sync()
    assert_same_build(t, oracle.build(w, num_splits=81920), n)


@pytest.mark.parametrize("split", ["bisect", "learned", "pary"])
@pytest.mark.parametrize("layout", ["aos", "soa"])
def test_small_noalloc_equals_table(gpu, layout, split):
    torch = gpu
    for n in (1, 500, 6000):
        w = torch.from_numpy(weights(n, "exponential")).cuda()
        t = atg.Table(n, layout=layout, split=split)
        t.set_weights(w)
        t.build()
        t.sync()
        tw, ta = t.table()
        rows = torch.zeros(2 * n if layout == "aos" else n, dtype=torch.float64, device="cuda")
        al = None if layout == "aos" else torch.zeros(n, dtype=torch.int32, device="cuda")
        W = torch.zeros(1, dtype=torch.float64, device="cuda")
        err = torch.full((1,), 9, dtype=torch.int32, device="cuda")
        atg.build_noalloc(w, rows, al, W, err, layout=layout, split=split)
        rw = rows.cpu().numpy()
        if layout == "aos":
            ra = rw.view(np.int32)[2::4]
            rw = rw[0::2]
        else:
            ra = al.cpu().numpy()
        assert np.array_equal(bits(rw), bits(tw)) and np.array_equal(ra, ta)
        assert W.item() == t.stats()["W"] and err.item() == 0


@pytest.mark.parametrize("n,section,dist,p", [
    (9_000, 0, "exponential", 0),              # the smallest default table built by the phases
    (20_000, 313, "pareto", 0),                # 64 sections: one whole block of 64
    (20_000, 312, "pareto", 500),              # 65
    (60_000, 29, "unit_uniform", 32_768),      # 2,069 sections: through the block tree
    (60_000, 30, "unit_uniform", 6_000),       # 2,001 sections: from the sections' sums
    (65_504, 32, "pareto", 0),                 # 2,048
    (400_000, 1000, "heavy_mix", 32_768),      # the most splits with four lanes each
    (400_000, 1000, "heavy_mix", 32_769),
    (50_000, 1000, "best_worst", 2),           # one split to find
    ((1 << 21) - 1, 2048, "pareto", 40_000),   # whole light lists
    (1 << 21, 2048, "pareto", 100_000),        # lean ones
    (1_000_000, 1000, "pareto", 30_700),       # windowed pack, 32 items a chain
    (1_000_000, 1000, "pareto", 31_000),       # staged
    ((1 << 22) - 1, 2048, "pareto", 40_000),   # windowed with whole light lists
    (1 << 22, 2048, "pareto", 40_000),         # with lean ones
    (4_300_000, 90, "unit_uniform", 2_000),    # lean: sections of few lights or none
    (4_300_000, 2048, "ascending", 9_001),     # lean: the lights in the first sections
    (4_300_000, 1024, "descending", 9_001),    # lean: in the last
    (4_300_000, 500, "heavy_mix", 5),          # lean: long chains over many sections
    (700_001, 2048, "exponential", 5_000),     # a last window block with one chain
    (300_000, 1000, "all_equal", 0),           # degenerate: filled by the split's launch
])
def test_mid_size_routes_match_oracle(gpu, oracle, n, section, dist, p):
    if dist == "all_equal":
        w = np.full(n, 2.5)
    elif dist in ("ascending", "descending"):
        w = np.sort(weights(n, "pareto"))[::1 if dist == "ascending" else -1].copy()
    else:
        w = weights(n, dist)
    p_req = p if p > 0 else 81920
    for layout in ("aos", "soa"):
        t = gpu_build(w, layout=layout, section_size=section, num_splits=p_req)
        ref = oracle.build(w, section_size=section, num_splits=p_req)
        assert_same_build(t, ref, n)
        t.build_phase("split")
        t.build_phase("pack")
        t.sync()
        assert_same_build(t, ref, n)


@pytest.mark.parametrize("n,section,dist,p,interleave", [
    (2_621_440, 2048, "pareto", 1 << 18, False),     # the fewest splits found in groups
    (2_621_440, 2048, "pareto", (1 << 18) - 1, False),
    (2_621_440, 2048, "exponential", 1 << 18, True),   # few splits left: found by bisection all the same
    (3_000_000, 40, "unit_uniform", 300_000, False),   # short chains leave heavies of less than the mean
    (3_000_000, 1000, "heavy_mix", 300_000, True),
    (2_700_000, 1000, "all_equal", 270_000, False),    # degenerate
])
def test_grouped_bisection_matches_oracle(gpu, oracle, n, section, dist, p, interleave):
    w = np.full(n, 2.5) if dist == "all_equal" else weights(n, dist)
    t = gpu_build(w, section_size=section, num_splits=p, interleave=interleave)
    ref = oracle.build(w, section_size=section, num_splits=p)
    assert_same_build(t, ref, n)
    assert t.stats()["monotone"] == -1 and t.stats()["learned_fallbacks"] == 0
    for phase in atg.Table.PHASES:
        t.build_phase(phase)
    t.sync()
    assert_same_build(t, ref, n)
