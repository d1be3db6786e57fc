"""A setter that finds no memory in its batch's pool leaves the member without
what it was to set: none of the arrays it gave back is read or written again,
the member steps on, and a later call that fits takes effect."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE, DX = (20, 70), 10.0
KW = dict(dt=0.5, manning=0.03, tile_rows=8)


def terrain():
    rng = np.random.default_rng(21)
    return 0.02 * np.arange(SHAPE[0])[::-1, None] + 0.05 * rng.random(SHAPE), np.full(SHAPE, 0.1)


def pair(pkg):
    """A member of a batch with a small pool, and the same grid alone."""
    z, h0 = terrain()
    batch = pkg.Batch(precision="fp64", pool_bytes=1 << 20)
    member, alone = batch.case(z, h0, DX, **KW), pkg.Case(z, h0, DX, **KW)
    batch.attach(member)
    return batch, member, alone


def step_both(batch, member, alone, n):
    batch.step(n)
    alone.step(n)
    for f in ("h", "um", "vn"):
        assert np.array_equal(member.field(f), alone.field(f)), f
    assert member.balance() == alone.balance()


def sources(n, nq):
    rng = np.random.default_rng(22)
    cells = rng.choice(SHAPE[0] * (SHAPE[1] - 1), n, replace=n > SHAPE[0] * (SHAPE[1] - 1))
    r, c = cells // (SHAPE[1] - 1), cells % (SHAPE[1] - 1)
    # the cell of a source at (x, y): row R - round(y / dx), column round(x / dx) + 1
    return c * DX, (SHAPE[0] - r) * DX, rng.uniform(0.1, 1.0, (nq, n)), 7.0


# the array that finds no room: the cells, their rates, the series
@pytest.mark.parametrize("n,nq", [(300000, 1), (20000, 1), (4, 100000)])
def test_sources(pkg, n, nq):
    batch, member, alone = pair(pkg)
    for c in (member, alone):
        c.set_sources(*sources(3, 4))
    step_both(batch, member, alone, 3)
    with pytest.raises(pkg.sw2d.Sw2dError, match="pool exhausted"):
        member.set_sources(*sources(n, nq))
    # seen on the host, before anything runs with the descriptors of now
    assert member.kernel_features()[0] & pkg.sw2d.FEAT_SOURCES == 0
    alone.set_sources(*sources(0, 0))
    step_both(batch, member, alone, 8)
    for c in (member, alone):
        c.set_sources(*sources(5, 3))
    step_both(batch, member, alone, 8)
