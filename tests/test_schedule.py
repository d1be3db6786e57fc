"""The order of the blocks of a batch's launch (host code, compiled here with
g++): the clock and ledger waves of every member come first."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "sw2d-efdc_amd" / "csrc"

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include "sw2d_schedule.hpp"
using namespace sw2d;
int main(int argc, char **argv)
{
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
