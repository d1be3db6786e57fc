"""sw2d_get_field of large grids (GPU): written by the device into pinned chunks
and moved on by two threads.  The values are those of sw2d_get_field_noalloc,
value for value, around the size from which it applies (2^20 cells) and with
a last chunk that is full, short and one cell."""
import threading

import numpy as np
import pytest

FIELD_NAMES = ("h", "um", "vn", "uu", "vv", "uua", "vva", "z", "hm", "hn", "uu1", "vv1")


def wet_case(pkg, cases, R, C, precision, seed=3):
    z = 0.2 * np.arange(R - 1, -1, -1.0)[:, None] + cases.fbm(R, C, 0.7, 2.0, seed)
    z[0, 0] = z[-1, -1] = -9999.0
    c = pkg.Case(z, np.zeros((R, C)), 10.0, dt=0.5, manning=0.03, precision=precision)
    c.set_rain(np.array([80.0, 20.0, 0.0]), 600.0)
    c.step(20)
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("R,C,precision", [(1023, 1025, "fp64"), (1024, 1024, "fp32"),
                                           (17, 61681, "fp64"), (1285, 2040, "mixed")])
def test_large_fields_equal_noalloc(pkg, cases, R, C, precision):
    c = wet_case(pkg, cases, R, C, precision)
    for _ in range(2):
        for n in FIELD_NAMES:
            assert np.array_equal(c.field(n), c.field_noalloc(n)), n
        c.step(7)
    assert c.field("h").max() > 0
    c.close()


@pytest.mark.gpu
def test_large_fields_of_two_handles_at_once(pkg, cases):
    cs = [wet_case(pkg, cases, 1100, 1201, "fp64", seed) for seed in (3, 4)]
    want = [c.field_noalloc("h").copy() for c in cs]
    got = [[], []]

    def read(i):
        for _ in range(5):
            got[i].append(cs[i].field("h").copy())

    ts = [threading.Thread(target=read, args=(i,)) for i in (0, 1)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for i in (0, 1):
        assert len(got[i]) == 5 and all(np.array_equal(g, want[i]) for g in got[i])
        cs[i].close()
