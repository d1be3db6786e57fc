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


def test_rain_and_evaporation(pkg):
    batch, member, alone = pair(pkg)
    for c in (member, alone):
        c.set_rain(np.array([400.0, 100.0, 300.0]), 4.3)
        c.set_evaporation(np.array([5.0, 9.0, 2.0]))
    step_both(batch, member, alone, 3)
    for setter, args in (("set_rain", (4.3,)), ("set_evaporation", ())):
        with pytest.raises(pkg.sw2d.Sw2dError, match="pool exhausted"):
            getattr(member, setter)(np.ones(300000), *args)
        # a series without values gives the rate 0 between the interval ends
        # (at one, where no step of 0.5 s comes, its formula divides 0 by 0)
        getattr(alone, setter)(np.zeros(0), *args)
        step_both(batch, member, alone, 8)
    for c in (member, alone):
        c.set_rain(np.array([200.0, 100.0, 50.0]), 9.0)
    step_both(batch, member, alone, 8)


def test_hydrograph(pkg):
    batch, member, alone = pair(pkg)
    for c in (member, alone):
        c.set_outlet(SHAPE[0] - 1, 30)
        c.set_hydrograph(40)
    step_both(batch, member, alone, 3)
    assert np.array_equal(member.hydrograph(), alone.hydrograph())
    with pytest.raises(pkg.sw2d.Sw2dError, match="pool exhausted"):
        member.set_hydrograph(100000)
    alone.set_hydrograph(0)
    step_both(batch, member, alone, 8)
    assert len(member.hydrograph()) == 0
    for c in (member, alone):
        c.set_hydrograph(40)
    step_both(batch, member, alone, 8)
    assert np.array_equal(member.hydrograph()[11:], alone.hydrograph()[11:])


# how many of the four arrays (4 bytes a record three times, then 8) find room
@pytest.mark.parametrize("rooms", [0, 2, 3])
def test_lake_records(pkg, rooms):
    batch, member, alone = pair(pkg)
    lake = np.zeros(SHAPE, np.int32)
    lake[8:12, 20:40] = 1
    for c in (member, alone):
        c.set_lake_bc(lake)
    step_both(batch, member, alone, 3)
    assert np.array_equal(member.lake_inflow(), alone.lake_inflow())
    many = (np.indices(SHAPE).sum(0) % 2).astype(np.int32)
    alone.set_lake_bc(many)
    assert alone.nbc > 1000
    # another member's hydrograph takes the rest of the pool
    z, h0 = terrain()
    filler = batch.case(z, h0, DX, **KW)
    used, _, cap = batch.memory()
    left = rooms * (-(-4 * alone.nbc // 256) * 256) + 512
    filler.set_hydrograph((cap - used - left) // 256 * 16)
    with pytest.raises(pkg.sw2d.Sw2dError, match="pool exhausted"):
        member.set_lake_bc(many)
    step_both(batch, member, alone, 8)
    assert len(member.lake_inflow()) == 0


def test_sources_without_a_series_give_nothing(pkg):
    """No rows in the table: the rates are 0 from the first step on, whatever
    lies behind it in the pool (here the rain series).  No step comes at the
    end of an interval, where the formula divides 0 by 0."""
    batch, member, alone = pair(pkg)
    x, y, _, _ = sources(100, 1)
    member.set_sources(x, y, np.zeros((0, 100)), 7.3)
    for c in (member, alone):
        c.set_rain(np.full(400, 30.0), 7.3)
    step_both(batch, member, alone, 8)
