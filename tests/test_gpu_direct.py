"""Direct sum at the edges of its tiles (256 sources, slices of 4096 and more), with
and without potentials and masses, where the fast reciprocal root does not hold
(coincident points without softening, squares that overflow), against the formula
in extended precision.

Bound: a sum of n terms in FP64, each within 8 roundings of its exact value: n + 8
roundings of 2^-53 of the sum of the terms' magnitudes."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


def _reference(x, idx, m, G, eps):
    """Accelerations, potentials and the sums of magnitudes of both."""
    x = x.astype(np.longdouble)
    a, pot, sa, sp = (np.zeros((len(idx), 3)), np.zeros(len(idx)), np.zeros((len(idx), 3)), np.zeros(len(idx)))
    for k, i in enumerate(idx):
        j = np.arange(len(x)) != i
        d = x[j] - x[i]
        r2 = (d * d).sum(1) + np.longdouble(eps) ** 2
        f = G * m[j].astype(np.longdouble) / (r2 * np.sqrt(r2))
        t, p = f[:, None] * d, m[j] / np.sqrt(r2)
        a[k], pot[k], sa[k], sp[k] = t.sum(0), p.sum(), abs(t).sum(0), p.sum()
    return a, pot, sa, sp


@pytest.mark.parametrize("n", [2, 128, 129, 255, 256, 257, 1000, 4097, 9000])
@pytest.mark.parametrize("eps", [0.0, 1e-2])
@pytest.mark.parametrize("with_masses", [False, True])
def test_tile_edges(vg, n, eps, with_masses):
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 3)) * np.array([1.0, 1e-3, 30.0])
    m = rng.uniform(0.5, 2.0, n) / n if with_masses else np.full(n, 1.0 / n)
    idx = np.unique(np.r_[0, n - 1, rng.integers(0, n, 60)])
    with vg.Gravity(n, 16, 3, "f64", eps=eps, G=0.7) as g:
        g.upload(x, masses=m if with_masses else None)
        a, pot = g.direct(idx, potential=True)
        assert np.array_equal(a, g.direct(idx))
    ra, rp, sa, sp = _reference(x, idx, m, 0.7, eps)
    u = (n + 8) * 2.0 ** -53
    assert (abs(a - ra) <= u * sa).all() and (abs(pot - rp) <= u * sp).all()


def test_coincident_and_far(vg):
    """Without softening a source at the target's place gives NaN (0 / 0) and an infinite
    potential; one whose distance's square overflows pulls with 0."""
    n = 700
    rng = np.random.default_rng(1)
    x = rng.standard_normal((n, 3))
    x[5] = x[650]
    x[300, 0] = 1e200
    idx = np.arange(n)
    with vg.Gravity(n, 16, 3, "f64", eps=0.0) as g:
        g.upload(x)
        a, pot = g.direct(idx, potential=True)
    pair = np.isin(idx, (5, 650))
    assert np.isnan(a[pair]).all() and np.isposinf(pot[pair]).all()
    assert (a[300] == 0).all() and pot[300] == 0
    near = idx[~pair & (idx != 300)]
    keep = np.delete(np.arange(n), 300)
    ra, rp, sa, sp = _reference(x[keep], near - (near > 300), np.full(n - 1, 1.0 / n), 1.0, 0.0)
    u = (n + 8) * 2.0 ** -53
    assert (abs(a[near] - ra) <= u * sa).all() and (abs(pot[near] - rp) <= u * sp).all()


def test_direct_small_and_large_samples_in_one_context():
    """Samples whose buffers the context keeps, and one of more than a million targets that it does not."""
    import vipp_gravity as vg
    rng = np.random.default_rng(12)
    n = 3000
    with vg.Gravity(n, 64, 4, "f64", eps=1e-3) as g:
        g.upload(rng.random((n, 3)))
        ref, pot = g.direct(np.arange(n), potential=True)
        for k in (50, 1_100_000, 700):
            idx = rng.integers(0, n, k)
            a, b = g.direct(idx, potential=True)
            # the sources are cut into other slices: sums of 3000 terms in another order
            assert np.abs(a - ref[idx]).max() <= 1e-12 * np.abs(ref).max() and np.abs(b - pot[idx]).max() <= 1e-12 * pot.max()


@pytest.mark.parametrize("n", [43690, 43691, 90001])
def test_accelerations_through_the_staging_buffers(n):
    """FP32 results come in pieces of 2^17 values: one, one and one value, and three."""
    import vipp_gravity as vg
    x = np.random.default_rng(n).random((n, 3))
    a = {}
    for mode in ("f64", "f32"):
        with vg.Gravity(n, 64, 6, mode, eps=1e-2) as g:
            g.upload(x)
            a[mode] = g.accelerations()
            assert np.array_equal(a[mode], g.accelerations())
    assert np.abs(a["f32"] - a["f64"]).max() <= 1e-3 * np.abs(a["f64"]).max()


@pytest.mark.parametrize("potential", [False, True])
def test_coincident_pair_costs_its_tile_only(vg, potential):
    """256 targets, 2^18 sources in slices of 4096 (16 tiles): a sum that is not finite is formed again over
    its tile, at three times the cost of the fast form, one tile in 16 a slice.  Half the call again
    is room for the clock; a slice walked by one thread took three times the call."""
    n = 1 << 18
    x = np.random.default_rng(5).random((n, 3))
    idx = np.arange(256)
    best = []
    for pair in (False, True):
        if pair:
            x[n - 100] = x[7]
        with vg.Gravity(n, 64, 4, "f64", eps=0.0) as g:
            g.upload(x)
            g.direct(idx, potential=potential)
            t = []
            for _ in range(30):
                t0 = time.perf_counter()
                a = g.direct(idx, potential=potential)
                t.append(time.perf_counter() - t0)
            best.append(min(t))
            a = a[0] if potential else a
            assert np.isnan(a[7]).all() == pair and np.isfinite(np.delete(a, 7, 0)).all()
    assert best[1] <= 1.5 * best[0]
