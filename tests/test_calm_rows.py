"""Rows the fused kernel passes over: no face of the row (nor the next row's
north faces) carries flux and nothing is added or taken, so the row keeps its
depths.  Water bodies apart from each other in a dry basin give every meeting
of such rows with flowing ones, at tile borders too; FP64 equals the oracle
value for value, and the FP32 form's dry basin stays exactly dry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def basin(R, C, seed):
    rng = np.random.default_rng(seed)
    z = 5.0 + 0.3 * rng.random((R, C))
    z[R // 4, C // 3:C // 2] = -9999.0                  # inactive cells beside water
    h0 = np.zeros((R, C))
    for _ in range(4):                                  # ponds, some at an edge
        r, c = rng.integers(0, R), rng.integers(0, C)
        h0[max(0, r - 3):r + 3, max(0, c - 4):c + 4] = rng.random() + 0.2
    h0[R - 2, 1] = 5.0e-5                               # below the dry threshold: stays
    h0[R // 2, C // 2] = -1.0e-3                        # clipped to 0 in the first iteration
    h0[z == -9999.0] = 0.0
    return z, h0


@pytest.mark.parametrize("shape,tile_rows", [((2, 2), 1), ((9, 61), 2), ((40, 59), 1), ((64, 175), 7),
                                             ((64, 175), 64)])
@pytest.mark.parametrize("outlet", [False, True])
def test_still_rows_match_oracle(pkg, po, shape, tile_rows, outlet):
    z, h0 = basin(*shape, seed=shape[0] + tile_rows)
    g = pkg.Case(z, h0, 10.0, dt=0.5, manning=0.03, tile_rows=tile_rows)
    o = po.Oracle(z, h0, 10.0, dt=0.5, manning=0.03)
    for c in (g, o):
        if outlet:
            c.set_outlet(shape[0] - 1, 0)
            c.set_hydrograph(64)
    for n in (1, 2, 37):
        g.step(n)
        o.step(n)
        for f in ("h", "um", "vn"):
            assert np.array_equal(g.field(f), o.field(f)), (f, n)
    b, ob = g.balance(), o.ledger()
    assert b["volume"] == pytest.approx(ob["volume"], rel=1e-13)
    assert b["v_clip"] == pytest.approx(ob["v_clip"], rel=1e-13)
    if outlet:
        assert np.array_equal(g.hydrograph(64)[:, 1], o.hydrograph()[:len(g.hydrograph(64)), 1])


@pytest.mark.parametrize("precision", ["fp32", "mixed"])
def test_dry_cells_stay_dry(pkg, precision):
    z = np.full((70, 130), 2.0)
    h0 = np.zeros_like(z)
    h0[30:34, 60:64] = 1.0
    g = pkg.Case(z, h0, 10.0, dt=0.5, manning=0.03, precision=precision, tile_rows=5)
    g.step(3)                                           # water reaches at most 2 cells an iteration
    h = g.field("h")
    assert h[30:34, 60:64].max() > 0.5
    assert np.count_nonzero(h[:24]) == 0 and np.count_nonzero(h[41:]) == 0
    assert np.count_nonzero(h[:, :54]) == 0 and np.count_nonzero(h[:, 71:]) == 0
    assert g.balance()["volume"] == pytest.approx(16.0 * 100.0, rel=1e-6)
