"""Tiles at the edges of the grid and of their rows: grids lower than a tile and
its halo, a last tile of one row, one and two strips, tiles of 1 to 9 rows, the
outlet on every side beside a tile's border, films that dry while they flow
(fluxes taken out between the two depth updates) and that keep all fluxes, one
forcing for all depths and a wet and a dry one.  FP64 equals the oracle value
for value; the FP32 and mixed forms do not depend on the tile height."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3), (3, 58), (5, 59), (10, 117), (19, 64)]
OUTLETS = {"south": lambda R, C: (R - 1, C // 2), "north": lambda R, C: (0, C - 1),
           "west": lambda R, C: (R // 2, 0), "east": lambda R, C: (R // 2, C - 1)}


def film(R, C, seed):
    rng = np.random.default_rng(seed)
    z = 0.15 * np.arange(R, 0, -1.0)[:, None] + 0.05 * rng.random((R, C))
    h0 = np.maximum(0.02 * rng.random((R, C)) - 0.008, 0.0)   # patches of film
    h0[:, : C // 3] = 0.4 + 0.01 * rng.random((R, C // 3))    # and deep water
    if R > 4:
        z[R // 2, C // 2] = -9999.0
        h0[R // 2, C // 2] = 0.0
    return z, h0


def states(case, outlet, lake):
    """Fields before the rain starts, while films dry, and after."""
    case.set_rain(np.array([0.0, 0.0, 0.3, 0.0]), 9.7)
    if lake:
        case.set_evaporation(np.array([0.05, 0.02, 0.04, 0.0]))
    case.set_outlet(*outlet)
    out = []
    for n in (9, 22):
        case.step(n)
        out += [case.field(f).copy() for f in ("h", "um", "vn")]
    return out


FRACTIONS = dict(INT=0.1, INF=0.05, LWL=0.2, EV_WL_min=0.01)


@pytest.mark.parametrize("R,C", SHAPES)
@pytest.mark.parametrize("side", OUTLETS)
def test_fp64_equals_oracle_at_every_height(pkg, po, R, C, side):
    z, h0 = film(R, C, 17 * R + C)
    outlet = OUTLETS[side](R, C)
    for lake in (False, True):
        kw = dict(dt=0.4, manning=0.03, **(FRACTIONS if lake else {}))
        want = states(po.Oracle(z, h0, 10.0, **kw), outlet, lake)
        for H in (1, 2, 3, 9):
            g = pkg.Case(z, h0, 10.0, tile_rows=H, **kw)
            for i, (a, b) in enumerate(zip(states(g, outlet, lake), want)):
                assert np.array_equal(a, b), (i, H, lake)
            g.close()


@pytest.mark.parametrize("precision", ["fp32", "mixed"])
def test_reduced_forms_do_not_depend_on_the_height(pkg, precision):
    for R, C in SHAPES:
        z, h0 = film(R, C, 5 * R + C)
        got = []
        for H in (1, 2, 4, 9):
            g = pkg.Case(z, h0, 10.0, dt=0.4, manning=0.03, precision=precision, tile_rows=H, **FRACTIONS)
            got.append(states(g, OUTLETS["south"](R, C), True))
            g.close()
        for other in got[1:]:
            for a, b in zip(got[0], other):
                assert np.array_equal(a, b), (R, C)
