"""The per-wave results that an iteration combines: the CFL minimum (partial
minima in several words, combined when the next iteration starts) and the
volume ledger (one record a tile, 512 of them to a round of the reducing
wave), at tile counts around those of one word each and of one round."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,tile_rows", [((4, 20), 8), ((15, 58), 1), ((16, 58), 1), ((17, 59), 1),
                                             ((127, 200), 1), ((128, 200), 1), ((129, 200), 1),
                                             ((257, 250), 1)])
@pytest.mark.parametrize("adaptive", [False, True])
def test_ledger_and_step_match_oracle(pkg, po, shape, tile_rows, adaptive):
    rng = np.random.default_rng(shape[0])
    z = 0.05 * np.arange(shape[0])[::-1, None] + 0.1 * rng.random(shape)
    h0 = np.where(rng.random(shape) < 0.3, 0.5 * rng.random(shape), 0.0)
    kw = dict(adaptive=True, courant=0.3) if adaptive else {}
    g = pkg.Case(z, h0, 10.0, dt=0.5, manning=0.03, tile_rows=tile_rows, **kw)
    o = po.Oracle(z, h0, 10.0, dt=0.5, manning=0.03)
    if adaptive:
        o.set_adaptive(0.3, 1.0)
    for c in (g, o):
        c.set_rain(np.array([40.0, 10.0, 0.0]), 300.0)
    for n in (1, 2, 13):
        g.step(n)
        o.step(n)
        assert g.time == o.time
        assert np.array_equal(g.field("h"), o.field("h")), n
        b, ob = g.balance(), o.ledger()
        # sums of at most 65k terms in different orders: 65k * 2^-53 < 1e-11
        for k, ok in (("volume", "volume"), ("v_source", "v_src"), ("v_clip", "v_clip")):
            assert b[k] == pytest.approx(ob[ok], rel=1e-11), k
