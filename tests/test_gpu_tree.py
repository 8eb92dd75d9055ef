"""Octree at the edges of its kernels: particle counts around the leaf threshold,
around the 1024 (beyond 2^20 particles: 4096) sorted codes of a block and around the sort's
tiles (4096 codes; 64 tiles), leaves counted in
one block and in many, on a first and on a second build in one context.  Bit for bit the
oracle's tree and lists."""
import numpy as np
import pytest

from test_gpu_parity import assert_lists_equal, assert_tree_equal

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


def _points(n):
    """Half uniform, a quarter in a small cube, a quarter on a lattice with coincident points."""
    rng = np.random.default_rng(n)
    k = n // 4
    lattice = rng.integers(0, 32, (k, 3)) / 32
    return np.concatenate([rng.random((n - 2 * k, 3)), 0.3 + 1e-3 * rng.random((k, 3)), lattice])


# (threshold floor(sqrt(8) s): 2 at s = 1, 11 at 4, 181 at 64)
@pytest.mark.parametrize("n,s", [(1, 1), (11, 4), (12, 4), (181, 64), (182, 64), (1023, 4), (1024, 4), (1025, 4), (2047, 64), (4096, 4), (4097, 4),
                                 (5000, 4), (40000, 2), (64 * 4096, 64), (64 * 4096 + 1, 64), ((1 << 20) + 1025, 64)])
def test_tree_at_the_edges(vg, orc, n, s):
    x = _points(n)
    rt, rl = orc.tree_and_lists(x, s)
    with vg.Gravity(n, s, 2, "f64", eps=1e-3) as g:
        for _ in range(2):
            g.upload(x)
            assert_tree_equal(g.tree(), rt)
            assert_lists_equal(g.lists(), rl)


def test_first_tree_deeper_than_sixteen_levels(vg, orc):
    rng = np.random.default_rng(8)
    x = np.concatenate([rng.random((300, 3)), 0.7 + 1e-5 * rng.random((200, 3))])
    rt, rl = orc.tree_and_lists(x, 4)
    with vg.Gravity(len(x), 4, 2, "f64", eps=1e-3) as g:
        for _ in range(2):
            g.upload(x)
            assert_tree_equal(g.tree(), rt)
            assert_lists_equal(g.lists(), rl)


# The lists are enqueued before the tree's size is known where twice the last tree's cells
# are at most 2^18 (60,000 points: 114,000 cells), after it elsewhere (376,000 cells).
@pytest.mark.parametrize("n", [60000, 200000])
def test_lists_of_many_cells(vg, orc, n):
    rng = np.random.default_rng(n)
    with vg.Gravity(n, 1, 2, "f64", eps=1e-3) as g:
        for _ in range(3):
            x = rng.random((n, 3))
            rt, rl = orc.tree_and_lists(x, 1)
            g.upload(x)
            assert_tree_equal(g.tree(), rt)
            assert_lists_equal(g.lists(), rl)
