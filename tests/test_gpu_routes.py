"""Which kernels a call launches: explicit choices of the caller, and the
rules on sizes."""
import pytest

import atg
from launches import kernels, launches
from test_gpu_build import assert_same_build

pytestmark = pytest.mark.gpu


def build(torch, n, **kw):
    t = atg.Table(n, **kw)
    t.set_weights(atg.generate_weights("pareto", n, seed=3, param=1.1))
    return kernels(torch, t.build)


def noalloc(torch, n, **kw):
    w = torch.from_numpy(atg.generate_weights("pareto", n, seed=3, param=1.1)).cuda()
    rows = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
    atg.build_noalloc(w, rows)  # finds the scratch array, outside the capture
    return kernels(torch, lambda s: atg.build_noalloc(w, rows, stream=s, **kw))


@pytest.mark.parametrize("n", [11, 1000, 5000])
def test_small_tables_keep_explicit_methods(gpu, n):
    """The one-launch build stands for the default pack and the bisection; a
    pack or split method that the caller names is the one that runs."""
    assert build(gpu, n) == ["build_small"]
    assert noalloc(gpu, n) == ["build_small"]
    for pack, psa in (("basic", True), ("basic", False), ("no_weights", False)):
        ks = build(gpu, n, pack=pack, psa_plus=psa)
        assert "pack_basic" in ks and "build_small" not in ks
        ks = noalloc(gpu, n, pack=pack, psa_plus=psa)
        assert "pack_basic" in ks and "build_small" not in ks
    for split, kernel in (("learned", "split_learned"), ("pary", "split_pary")):
        assert kernel in build(gpu, n, split=split)
        assert kernel in noalloc(gpu, n, split=split)


def counted(torch, n, count, kind, rows=4096):
    t = atg.Table(n)
    t.set_weights(atg.generate_weights("pareto", n, seed=3, param=1.1))
    t.build()
    t.sync()
    hist = torch.zeros(n, dtype=torch.int32, device="cuda")
    t.sample(count, 1, kind=kind, section_rows=rows)  # grows the buffer of the sections' counts
    return launches(torch, lambda s: t.sample(count, 1, kind=kind, section_rows=rows, hist=hist, stream=s))


@pytest.mark.parametrize("count", [16_383, 16_384, 20_001, 65_536, 200_000, 1_000_000])
def test_basic_counts_of_few_samples_fill_the_card(gpu, count):
    """Few samples with counts are spread over blocks down to a sample a
    thread, up to 128 blocks."""
    (_, blocks, threads, _), = counted(gpu, 300_000, count, "basic")
    assert blocks * threads >= min(count - threads, 128 * 512)


@pytest.mark.parametrize("n,rows,count", [(3_000_000, 4096, 16_384), (3_000_000, 4096, 300_000),
                                          (3_000_000, 200, 20_000), (300_000, 4096, 16_384)])
def test_sparse_counts_have_a_wave_per_section(gpu, n, rows, count):
    """Draws that read their rows one by one find each section's samples by a
    wave: with counts there are as many waves as sections, or the card is full."""
    ks = counted(gpu, n, count, "sectioned", rows)
    name, blocks, threads, _ = ks[-1]
    assert name == "sample_sectioned_sparse"
    assert blocks * threads // 64 >= min((n + rows - 1) // rows, 8192)


@pytest.mark.parametrize("count,counters", [(2047, 0), (2048, 16_384)])
def test_staged_counts_of_few_samples(gpu, count, counters):
    """Staged sections hold LDS counters from 2,048 samples on."""
    n, hist = 1000, gpu.zeros(1000, dtype=gpu.int32, device="cuda")
    name, _, _, lds = counted(gpu, n, count, "sectioned")[-1]
    assert (name, lds) == ("sample_sectioned", 4096 * 16 + counters)
    t = atg.Table(n)
    t.set_weights(atg.generate_weights("pareto", n, seed=3, param=1.1))
    t.rejection_build()
    t.rejection_sample_sectioned(count, 1)  # reads the array's size back, outside the capture
    name, _, _, lds = launches(gpu, lambda s: t.rejection_sample_sectioned(count, 1, hist=hist, stream=s))[-1]
    assert (name, lds) == ("rej_sample_sectioned", 4096 * 16 + counters)


@pytest.mark.parametrize("n,p,pack", [(98_304 * 60, 98_304, "pack_windowed"), (98_305 * 64, 98_305, "pack_staged"),
                                      (147_456 * 75, 147_456, "pack_windowed")])
def test_pack_at_the_end_of_a_round(gpu, oracle, n, p, pack):
    """Where the windowed pack's waves just fit the card, have a few more than
    that, and again have enough: the pack that runs, and its rows."""
    w = atg.generate_weights("heavy_mix", n, seed=3, param=0.9)
    t = atg.Table(n, section_size=2048, num_splits=p)
    t.set_weights(w)
    assert pack in kernels(gpu, t.build)
    t.build()
    t.sync()
    assert_same_build(t, oracle.build(w, section_size=2048, num_splits=p), n)


@pytest.mark.parametrize("n,p,pack", [(100, 2, "pack_staged"), (2048, 10, "pack_staged"), (2049, 10, "pack_windowed")])
def test_pack_of_small_tables(gpu, oracle, n, p, pack):
    """Tables whose lists the staged pack holds at once, or nearly."""
    w = atg.generate_weights("unit_uniform", n, seed=3)
    for psa in (True, False):
        t = atg.Table(n, num_splits=p, split="learned", psa_plus=psa)
        t.set_weights(w)
        assert pack in kernels(gpu, t.build)
        t.build()
        t.sync()
        assert_same_build(t, oracle.build(w, num_splits=p, psa_plus=psa), n)


@pytest.mark.parametrize("layout,n,rows,count,sparse", [
    ("aos", 100_003, 4096, 12_500, True), ("aos", 100_003, 4096, 12_501, False),
    ("soa", 100_003, 4096, 12_500, True), ("soa", 100_003, 4096, 12_501, False),
    ("aos", 4_200_000, 4096, 525_000, True), ("soa", 4_200_000, 4096, 350_000, True),
    ("soa", 4_200_000, 4096, 350_001, False), ("soa", 4_200_000, 8192, 525_000, False),
    ("soa", 4_200_000, 4095, 525_000, True)])
def test_line_of_sparse_draws(gpu, oracle, layout, n, rows, count, sparse):
    """Few samples a row read the drawn rows, fewer where a row is in two pieces."""
    t = atg.Table(n, layout=layout)
    t.set_weights(atg.generate_weights("pareto", n, seed=3, param=1.1))
    t.build()
    tw, ta = t.table()
    out = gpu.empty(count, dtype=gpu.int32, device="cuda")
    t.sample(1, 4, section_rows=rows)  # grows the buffer of the sections' counts
    ks = kernels(gpu, lambda s: t.sample(count, 4, section_rows=rows, out=out, stream=s))
    assert (ks[-1] == "sample_sectioned_sparse") == sparse
    t.sample(count, 4, section_rows=rows, out=out)
    assert (out.cpu().numpy() == oracle.sample_sectioned(tw, ta, t.stats()["W_N"], rows, count, 4)).all()
