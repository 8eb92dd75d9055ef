"""FP32 M2L on the matrix cores: every expansion order (row tiles 1 to 11, odd
ones split between wavefronts, last column groups of 1 to 4 products), few and
many parents (not multiples of the 64 of a block; offsets cut into parts), against the
FP64 path's local expansions of the same tree, cell by cell.

Bound: a coefficient is a sum of 189 K products, K = (p + 1)^2 <= 169, of FP32
operands (each off by 2^-24 of itself).  The products of one offset differ in
size by the expansion's decay, so a few dozen carry the sum: roundings of
2^-24 each add up to some 1e-6 of the cell's largest coefficient at worst, and
cancellation between offsets costs another factor of ten: 2e-5, the bound of
the FP32 path's other tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


@pytest.mark.parametrize("p", range(1, 13))
@pytest.mark.parametrize("n,s", [(1500, 4), (30011, 24)])
def test_f32_locals_match_f64(vg, p, n, s):
    rng = np.random.default_rng(p)
    k = n // 2
    x = np.concatenate([0.05 * rng.standard_normal((k, 3)), rng.standard_normal((n - k, 3)) * np.array([1.0, 0.5, 2.0])])
    L = {}
    for mode in ("f64", "f32"):
        with vg.Gravity(n, s, p, mode, eps=1e-3) as g:
            g.upload(x)
            g.accelerations(copy=False)
            L[mode] = g.expansions()[1]
    a, b = L["f64"], L["f32"]
    scale = np.abs(a).max(axis=(1, 2), keepdims=True) + 1e-300
    assert (np.abs(a - b) / scale).max() < 2e-5


# M2M and L2L on the matrix cores: 16 parents a tile on levels of few parents, two
# tiles where a level has hundreds (leaves of 11 points); same bound for both expansions.
@pytest.mark.parametrize("p", range(1, 13))
@pytest.mark.parametrize("n,s", [(700, 40), (30011, 4)])
def test_f32_expansions_match_f64(vg, p, n, s):
    rng = np.random.default_rng(100 + p)
    x = np.concatenate([0.05 * rng.standard_normal((n // 3, 3)), rng.random((n - n // 3, 3))])
    m = rng.uniform(0.5, 1.5, n) / n
    E = {}
    for mode in ("f64", "f32"):
        with vg.Gravity(n, s, p, mode, eps=1e-3) as g:
            g.upload(x, None, m)
            g.accelerations(copy=False)
            E[mode] = g.expansions()
    for a, b in zip(E["f64"][:2], E["f32"][:2]):
        scale = np.abs(a).max(axis=(1, 2), keepdims=True) + 1e-300
        assert (np.abs(a - b) / scale).max() < 2e-5


def test_fallback_order_changes(vg):
    """The closure's fallback order may change in a context: the operators' padding belongs to an order."""
    import closure
    rng = np.random.default_rng(4)
    x = rng.random((20000, 3))
    params = closure.init_params(1)

    def forces(orders):
        with vg.Gravity(len(x), 24, 4, "f32", eps=1e-3) as g:
            g.upload(x)
            for p in orders:
                g.set_closure(params, bound=0.0, p_fallback=p)
                a = g.accelerations()
        return a
    assert np.array_equal(forces([12, 8, 10]), forces([10]))
