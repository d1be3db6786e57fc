"""The forcing of an iteration is the same whether the iteration before it
evaluated it or a change of the descriptors did (a setter called again, another
member that joined or left), in every precision form: value for value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, SER = 0.5, 1799.3
# The series' interpolation divides by t - SER * k, which is one spacing of t
# here in the middle of the second iteration: a multiply-add that is fused in
# one place and not in another shows as a different value of the rate.
T_MID = np.nextafter(np.float64(SER) * 3, np.inf)
TIME0 = T_MID - 3 * DT


def case_of(make, kind):
    rng = np.random.default_rng(11)
    z = 0.02 * np.arange(20)[::-1, None] + 0.05 * rng.random((20, 70))
    h0 = np.full(z.shape, 0.3)
    c = make(z, h0, 10.0, dt=DT, manning=0.03, time0=TIME0, tile_rows=8)

    def forcing():
        if kind == "rain":
            c.set_rain(np.array([0.0, 0.0, 0.0, 0.0, 1e-6, 0.0]), SER)
        else:
            Q = np.zeros((6, 2))
            Q[4] = 1e-7, 2e-7
            c.set_sources(np.array([100.0, 400.0]), np.array([100.0, 60.0]), Q, SER)
    forcing()
    return c, forcing


@pytest.mark.parametrize("kind", ["rain", "sources"])
@pytest.mark.parametrize("precision", ["fp32", "mixed", "fp64"])
def test_results_do_not_depend_on_a_rebuild(pkg, precision, kind):
    assert TIME0 + DT + DT + DT == T_MID
    exact, _ = case_of(lambda *a, **k: pkg.Case(*a, precision=precision, **k), kind)
    exact.step(4)
    assert np.ptp(exact.field("h")) > 0 and exact.balance()["v_source"] > 0

    again, forcing = case_of(lambda *a, **k: pkg.Case(*a, precision=precision, **k), kind)
    again.step(1)
    forcing()
    again.step(3)

    batch = pkg.Batch(precision=precision, pool_bytes=64 << 20, tile_rows=8)
    member, _ = case_of(batch.case, kind)
    batch.attach(member)
    batch.step(1)
    other, _ = case_of(batch.case, kind)
    batch.attach(other)
    batch.step(3)

    for c in (again, member):
        assert c.time == exact.time
        for f in ("h", "um", "vn"):
            assert np.array_equal(c.field(f), exact.field(f)), f
        assert c.balance() == exact.balance()
