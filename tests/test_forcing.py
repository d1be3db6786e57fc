"""Forcing values are evaluated once an iteration, by the iteration before it
(or when a setter changed them): series that start, change and end while a
handle or a batch member runs, and point sources at the columns and rows where
tiles meet, equal the oracle value for value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def terrain(R, C, seed):
    rng = np.random.default_rng(seed)
    z = 0.05 * np.arange(R)[::-1, None] + 0.2 * rng.random((R, C))
    h0 = np.where(rng.random((R, C)) < 0.5, 0.3 * rng.random((R, C)), 0.0)
    return z, h0


def same(g, o):
    for f in ("h", "um", "vn"):
        assert np.array_equal(g.field(f), o.field(f)), f


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("adaptive", [False, True])
def test_series_changed_while_running(pkg, po, batch, adaptive):
    z, h0 = terrain(37, 130, 3)
    kw = dict(dt=0.5, manning=0.03, INT=0.1, LWL=0.05, EV_WL_min=0.1)
    gkw = dict(kw, adaptive=True, courant=0.4) if adaptive else kw
    o = po.Oracle(z, h0, 10.0, **kw)
    if adaptive:
        o.set_adaptive(0.4, 1.0)
    if batch:
        b = pkg.Batch(precision="fp64", pool_bytes=64 << 20)
        g = b.case(z, h0, 10.0, **gkw)
        b.attach(g)
        step = b.step
    else:
        g = pkg.Case(z, h0, 10.0, **gkw)
        step = g.step
    def both(n):
        step(n)
        o.step(n)
        same(g, o)
    both(3)
    for c in (g, o):
        c.set_rain(np.array([900.0, 100.0, 0.0]), 5.3)
    both(1)
    both(13)                       # past the end of the series
    for c in (g, o):
        c.set_rain(np.array([50.0, 500.0, 200.0, 10.0]), 11.1)
        c.set_evaporation(np.array([30.0, 60.0]))
    both(7)
    both(12)


@pytest.mark.parametrize("tile_rows", [1, 5])
def test_sources_where_tiles_meet(pkg, po, tile_rows):
    R, C, dx = 23, 180, 10.0
    z, h0 = terrain(R, C, 4)
    cols = np.array([1, 2, 55, 57, 58, 59, 60, 61, 115, 116, 118, 119, 174, 178, 179, 90])
    rows = np.array([0, 1, 4, 5, 6, 9, 10, 11, 14, 15, 16, 19, 20, 21, 22, 12])
    # the cell of a source at (x, y): row R - round(y / dx), column round(x / dx) + 1
    x, y = (cols - 1) * dx, (R - rows) * dx
    rng = np.random.default_rng(5)
    Q = rng.uniform(0.5, 20.0, (4, len(cols)))
    g = pkg.Case(z, h0, dx, dt=0.5, manning=0.03, tile_rows=tile_rows)
    o = po.Oracle(z, h0, dx, dt=0.5, manning=0.03)
    g.set_sources(x, y, Q, 4.7)
    o.set_sources(rows * C + cols, Q, 4.7)
    for n in (1, 2, 9):
        g.step(n)
        o.step(n)
        same(g, o)
    assert g.balance()["v_source"] > 0
