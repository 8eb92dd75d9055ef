"""FP64 near field alone: fewer particles than a leaf holds, so that the forces are the
pairs of one leaf, at the edges of its target tiles (16, 4 of them to an item) and source
groups (64; cut into items), against the direct sum in extended precision.

Bound: a sum of n terms in FP64, each within 8 roundings of its exact value: n + 8
roundings of 2^-53 of the sum of the terms' magnitudes; the points lie on a grid, so
their differences are exact.  The potential drops its own term m / eps afterwards, which
adds that term's size; the energy is half the sum of m times these."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


@pytest.mark.parametrize("n", [2, 15, 16, 17, 63, 64, 65, 66, 127, 129, 1000, 4103])
@pytest.mark.parametrize("eps", [0.0, 1e-3])
@pytest.mark.parametrize("masses", [False, True])
def test_one_leaf(vg, n, eps, masses):
    rng = np.random.default_rng(n)
    x = np.round(rng.random((n, 3)) * np.array([1.0, 0.6, 1.7]) * 2 ** 18) / 2 ** 18
    m = rng.uniform(0.5, 1.5, n) / n if masses else np.full(n, 1.0 / n)
    with vg.Gravity(n, 1500, 3, "f64", eps=eps, G=1.3) as g:
        g.upload(x, None, m if masses else None)
        a, u = g.accelerations(), g.energy()[1]
        assert np.array_equal(a, g.accelerations()) and g.counts()["cells"] == 1
    w = (n + 8) * 2.0 ** -53
    xl, pot, spot = x.astype(np.longdouble), 0.0, 0.0
    for i in range(n) if n < 2000 else rng.integers(0, n, 200):
        d = np.delete(xl, i, 0) - xl[i]
        mj = np.delete(m, i)
        r2 = (d * d).sum(1) + np.longdouble(eps) ** 2
        t = (1.3 * mj / (r2 * np.sqrt(r2)))[:, None] * d
        assert (abs(a[i] - t.sum(0)) <= w * abs(t).sum(0)).all()
        p = (mj / np.sqrt(r2)).sum()
        pot += m[i] * p
        spot += m[i] * (p + (m[i] / eps if eps else 0.0))
    if n < 2000:
        assert abs(abs(u) - 0.65 * pot) <= 2 * w * 0.65 * spot
