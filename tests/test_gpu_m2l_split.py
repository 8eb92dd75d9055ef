"""Split M2L on the BF16 matrix cores: every expansion order (row tiles 1 to 11,
last k-steps half full or not, one or more targets per gathering load), few and
many parents (not multiples of the 64 of a block; offsets cut into parts), against
the FP64 path's local expansions of the same tree, cell by cell.

Bound: the split's two residuals are 2^-17 of their operand at most and the
dropped product 2^-18, 2^-16 of a product together.  A coefficient is a sum of
products of both signs; cancellation between offsets costs a factor of ten
against the cell's largest coefficient: 10 * 2^-16 < 2e-4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


@pytest.mark.parametrize("p", range(1, 13))
@pytest.mark.parametrize("n,s", [(1500, 4), (30011, 24)])
def test_split_locals_match_f64(vg, p, n, s):
    rng = np.random.default_rng(p)
    k = n // 2
    x = np.concatenate([0.05 * rng.standard_normal((k, 3)), rng.standard_normal((n - k, 3)) * np.array([1.0, 0.5, 2.0])])
    L = {}
    for mode in ("f64", "split"):
        with vg.Gravity(n, s, p, mode, eps=1e-3) as g:
            g.upload(x)
            g.accelerations(copy=False)
            L[mode] = g.expansions()[1]
    a, b = L["f64"], L["split"]
    scale = np.abs(a).max(axis=(1, 2), keepdims=True) + 1e-300
    assert (np.abs(a - b) / scale).max() < 2e-4
