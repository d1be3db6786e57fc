"""The layout of a batch's launch (host code, compiled here with g++): the
clock and ledger waves of every member come first, and a cap on the resident
waves counts the LDS that the kernel has of its own."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "sw2d-efdc_amd" / "csrc"

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "sw2d_schedule.hpp"
using namespace sw2d;
int main(int argc, char **argv)
{
    if (!strcmp(argv[1], "lds")) {  // per_cu, per_block, own, cap
        printf("%zu\n", lds_pad(atol(argv[2]), atol(argv[3]), atol(argv[4]), atoi(argv[5])));
        return 0;
    }
    // order, then the block count of each member
    std::vector<int> counts, sids;
    for (int i = 2; i < argc; i++) { counts.push_back(atoi(argv[i])); sids.push_back(10 * (i - 2)); }
    std::vector<TileRef> tiles;
    order_tiles(counts, sids, atoi(argv[1]), tiles);
    for (const TileRef &t : tiles) printf("%d %d\n", t.sid, t.local);
    return 0;
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("schedule")
    (d / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", "-o", str(d / "main"),
                    str(d / "main.cpp")], check=True)
    return lambda *a: subprocess.run([str(d / "main"), *map(str, a)], check=True, text=True,
                                     capture_output=True).stdout


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("counts", [[3], [2, 2], [7, 3, 12], [40, 3, 3, 5, 90]])
def test_clock_and_ledger_waves_come_first(run, order, counts):
    tiles = [tuple(map(int, line.split())) for line in run(order, *counts).splitlines()]
    assert sorted(tiles) == [(10 * m, i) for m, c in enumerate(counts) for i in range(c)]
    first = tiles[: 2 * len(counts)]           # a clock wave and a ledger wave each
    assert {t[1] for t in first} == {0, 1}
    rest = tiles[2 * len(counts):]
    if order == 0:                             # then each member's blocks in a run
        assert rest == [(10 * m, i) for m, c in enumerate(counts) for i in range(2, c)]
    else:
        assert [t[1] for t in rest] == sorted(t[1] for t in rest)


CU, STEP = 160 << 10, 1280


@pytest.mark.parametrize("cap", range(1, 9))
@pytest.mark.parametrize("own", [0, 512, 2176, 2240, 10560, 24000])
def test_cap_counts_the_kernels_own_lds(run, cap, own):
    pad = int(run("lds", CU, CU, own, cap))
    fit = lambda nbytes: CU // (-(-nbytes // STEP) * STEP)
    # as many blocks a CU as the cap asks for, or the most below it that a whole
    # number of allocation steps leaves, or what the kernel's own LDS leaves
    most = max(fit(STEP * n) for n in range(1, 129) if fit(STEP * n) <= 4 * cap)
    assert fit(max(own + pad, 1)) == (min(most, fit(own)) if own else most)
    if cap in (1, 2, 3, 4, 8):
        assert most == 4 * cap
    assert int(run("lds", CU, 64 << 10, own, cap)) + own <= 64 << 10
    assert int(run("lds", CU, CU, own, 0)) == 0
