"""The host rules that choose kernels by size, compiled from the library's own
headers and asked on the CPU, also for sizes too large to allocate."""
import os
import subprocess

import pytest

import build_lib

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "atg_sample.h"
#include "atg_small.h"
using namespace atg;
int main(int argc, char** argv) {
    auto arg = [&](int k) { return atoll(argv[k]); };
    const char* what = argv[1];
    if (what[0] == 's') {  // small_class n G Ls p
        SmallClass c;
        if (small_class_of(arg(2), arg(3), arg(4), arg(5), c)) printf("%d %d %d\n", kSmallChunks[c.xu], c.waves, c.tier);
        else printf("none\n");
    }
    if (what[0] == 'b') printf("%d\n", (int)small_beside_ok(arg(2), (int)arg(3)));  // beside sections classes
    if (what[0] == 'l') printf("%d\n", (int)rows_later_ok(arg(2), arg(3), arg(4) != 0, arg(5), arg(6)));  // later sections resident aos n Ls
    if (what[0] == 'g') printf("%d\n", (int)batch_rows_later_ok(arg(2), arg(3), arg(4), arg(5)));  // group_later sections resident items Ls
    if (what[0] == 'w') printf("%d\n", (int)pack_windowed_ok(arg(2), arg(3), PACK_CHUNKED));  // windowed n p
    if (what[0] == 'r') printf("%u\n", rej_share((uint32_t)arg(2)));  // rej_share m
    return 0;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, exe = str(d / "rules.cpp"), str(d / "rules")
    with open(src, "w") as f:
        f.write(PROGRAM)
    r = subprocess.run([build_lib.HIPCC, "-O1", "-std=c++17", "-x", "hip", "--cuda-host-only",
                        f"--offload-arch={build_lib.ARCH}", "-I" + build_lib.CSRC, src, "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def ask(*args):
        return subprocess.run([exe] + [str(a) for a in args], capture_output=True, text=True, check=True,
                              timeout=10).stdout.strip()
    return ask


@pytest.mark.parametrize("n,G,Ls,p,want", [
    (1, 1, 1, 2, "2 1 0"),
    (1000, 11, 100, 100, "2 16 0"),
    (1600, 16, 100, 160, "2 16 0"),
    (1700, 17, 100, 170, "none"),              # a section more than a workgroup has waves
    (8192, 4, 2048, 200, "32 4 2"),
    (9000, 5, 2048, 200, "none"),              # a long section more
    (14_000, 15, 1000, 1400, "none"),          # past a CU's LDS
    ((1 << 30) + 1, (1 << 30) + 1, 1, 2, "none"),   # more sections than an int's powers of two
    ((1 << 31) - 17, (1 << 31) - 17, 1, 2, "none"),
])
def test_small_class(rule, n, G, Ls, p, want):
    assert rule("small_class", n, G, Ls, p) == want


@pytest.mark.parametrize("m,want", [(1, 64), (64, 64), (114, 64), (1024, 64), (1025, 65), (40_000, 2500),
                                    ((1 << 31) - 1, 1 << 27)])
def test_rejection_share(rule, m, want):
    """16 shares hold every sample, none of fewer than a wave's lanes."""
    assert rule("rej_share", m) == str(want) and 16 * want >= m


@pytest.mark.parametrize("sections,classes,want", [
    (47, 8, 0), (704, 1, 0), (1919, 1, 0), (1920, 1, 1), (3839, 4, 0), (3840, 4, 1), (22_595, 5, 1)])
def test_small_tables_beside_others(rule, sections, classes, want):
    assert rule("beside", sections, classes) == str(want)


@pytest.mark.parametrize("n,p,want", [
    (1_000_000, 30_700, 1), (1_000_000, 31_000, 0),
    (5_120_000, 80_000, 1), (98_304 * 64, 98_304, 1),
    (98_305 * 64, 98_305, 0), (7_040_000, 110_000, 0), (11_000_000, 110_000, 0),   # a second round of few waves
    (14_080_000, 110_000, 1), (147_455 * 128, 147_455, 0), (147_456 * 80, 147_456, 1),
    (16_000_000, 160_000, 1), (100_000_000, 1_000_000, 0), (100_000_000, 666_000, 1),
    (257 * 110_000, 110_000, 1),
    (100, 2, 0), (2048, 20, 0), (2049, 20, 1), (1000, 3, 1),                       # lists that are staged at once
])
def test_windowed_pack(rule, n, p, want):
    assert rule("windowed", n, p) == str(want)


@pytest.mark.parametrize("sections,resident,aos,n,Ls,want", [
    (2048, 2048, 1, 1 << 22, 2048, 0), (2048, 2048, 0, 1 << 22, 2048, 0),      # a wave each from the start
    (2442, 2048, 1, 5_000_000, 2048, 0), (8192, 2048, 1, 1 << 24, 2048, 0),    # long sections, rows in the cache
    (8193, 2048, 1, (1 << 24) + 1, 2048, 1), (48_829, 2048, 1, 100_000_000, 2048, 1),
    (2442, 2048, 0, 5_000_000, 2048, 1),                                       # split rows
    (10_001, 4096, 1, 10_000_019, 1000, 1), (5001, 4096, 1, 5_000_000, 1024, 1), (5001, 4096, 1, 5_000_000, 1025, 0),
])
def test_rows_later(rule, sections, resident, aos, n, Ls, want):
    assert rule("later", sections, resident, aos, n, Ls) == str(want)


@pytest.mark.parametrize("sections,resident,items,Ls,want", [
    (100_000, 2048, 100_000_000, 1000, 0), (100_000, 2048, 100_000_000, 2048, 1),
    (2048, 2048, 100_000_000, 2048, 0), (8192, 2048, 1 << 24, 2048, 0)])
def test_group_rows_later(rule, sections, resident, items, Ls, want):
    assert rule("group_later", sections, resident, items, Ls) == str(want)
