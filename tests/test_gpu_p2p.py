"""FP32 near field (matrix-core squared distances and the pass by differences).

The FP32 modes and the FP64 mode of one input share tree, lists and order, and
the points lie on a grid that FP32 positions relative to the root centre hold
exactly, so the modes differ by the rounding of FP32 sums and products alone.
Its bound: a source tile that is taken by the expansion
|x_j|^2 - 2 x_i x_j + |x_i|^2 lies at least R / 8 from the targets' box of
radius R, where the squared distance loses at most 2 (9/8 R)^2 / (R / 8)^2 ~ 160
roundings of 2^-24, 1e-5, and the pair force 1.5 times that; sums over pairs of
both signs of error stay below the single worst pair, and the FP32 expansions
add 1e-6: 5e-5 of the force in the 2-norm leaves a factor of 3."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BOUND = 5e-5


@pytest.fixture(scope="module")
def vg():
    import vipp_gravity
    return vipp_gravity


def _points(n, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "uniform":
        x = rng.random((n, 3)) * np.array([1.0, 0.6, 1.7])
    else:  # a dense core inside a sparse halo: leaves of a few points beside cells of thousands
        k = n // 2
        x = np.concatenate([0.01 * rng.standard_normal((k, 3)) + 0.3, np.clip(rng.standard_normal((n - k, 3)), -3.9, 3.9)])
    return np.round(x * 2 ** 18) / 2 ** 18


# leaf thresholds floor(sqrt(8) s) around the 16-target tiles, the 96 targets of
# one pass and beyond several passes; particle counts around the 64-source groups
@pytest.mark.parametrize("n,s,kind", [(3, 1, "uniform"), (700, 1, "core"), (1025, 6, "uniform"), (4100, 12, "core"), (9001, 34, "uniform"),
                                      (20011, 35, "core"), (30000, 130, "core"), (12000, 1500, "uniform")])
@pytest.mark.parametrize("eps,masses", [(0.0, False), (1e-3, True)])
def test_p2p_f32_against_f64_mode(vg, n, s, kind, eps, masses):
    x = _points(n, kind, n)
    m = np.random.default_rng(1).uniform(0.5, 1.5, n) / n if masses else None
    r = {}
    for mode in ("f64", "f32"):
        with vg.Gravity(n, s, 8, mode, eps=eps, G=1.3) as g:
            g.upload(x, None, m)
            r[mode] = g.accelerations(), g.energy()[1]
    a, b = r["f64"][0], r["f32"][0]
    assert np.linalg.norm(b - a) <= BOUND * np.linalg.norm(a)
    assert abs(r["f32"][1] - r["f64"][1]) <= 5e-6 * abs(r["f64"][1])


def test_p2p_f32_same_twice(vg):
    """Leaves whose sources are cut into many items: partial sums in a fixed order."""
    x = _points(40000, "core", 5)
    with vg.Gravity(len(x), 40, 4, "f32", eps=1e-3) as g:
        g.upload(x)
        a = g.accelerations()
        assert np.array_equal(a, g.accelerations())


def test_p2p_f32_beyond_the_range_of_squared_distances(vg):
    """A cluster at the root centre and 20 points at each of two corners 1e19
    away: those tiles' squared distances leave the range in which FP32 pairs
    still pull, and the cluster feels itself alone, as an FP64 direct sum over
    its own members gives it."""
    c = np.random.default_rng(3).uniform(-0.5, 0.5, (40, 3))
    far = np.full((20, 3), 6e18)
    x = np.concatenate([far, -far, c])
    with vg.Gravity(80, 16, 4, "f32", eps=1e-2, mass=1.0) as g:
        g.upload(x)
        a = g.accelerations()[40:]
    d = c[None] - c[:, None]
    w = ((d ** 2).sum(2) + 1e-4) ** -1.5
    ref = (w[..., None] * d).sum(1)
    assert np.isfinite(a).all()
    assert np.linalg.norm(a - ref) <= BOUND * np.linalg.norm(ref)


# floor(sqrt(8) s) = 181 and 4242: leaves put in order by a wavefront each, and by a block each after the tree's sizes are known
@pytest.mark.parametrize("s", [64, 1500])
@pytest.mark.parametrize("mode", ["f64", "f32", "split"])
def test_streams_equal_one_stream(vg, mode, s):
    """Per-phase timing keeps one stream: the same results bit for bit, evaluation after evaluation."""
    rng = np.random.default_rng(s)
    n, runs = 12000, []
    x = [rng.random((n, 3)) for _ in range(3)]
    for timing in (False, True):
        with vg.Gravity(n, s, 5, mode, eps=1e-3) as g:
            g.set_timing(timing)
            for y in x:
                g.upload(y)
                runs.append((g.accelerations(), g.energy()))
    for a, b in zip(runs[:3], runs[3:]):
        assert np.array_equal(a[0], b[0]) and a[1] == b[1]


# lengths times 2^l and masses times 2^k, as SI or cgs units have them, and G so that the
# accelerations keep their size: r^-3, m x and the sums leave the FP32 range unless taken
# in units of their own
@pytest.mark.parametrize("l,k", [(0, 0), (37, 110), (53, 100), (53, 0), (60, 40), (0, 100), (0, -60)])
@pytest.mark.parametrize("eps,masses", [(0.0, True), (1e-3, True), (1e-3, False)])
def test_p2p_f32_units(vg, l, k, eps, masses):
    n, s = 4100, 12
    x = _points(n, "core", n) * 2.0 ** l
    m = np.random.default_rng(1).uniform(0.5, 1.5, n) / n * 2.0 ** k if masses else None
    r = {}
    for mode in ("f64", "f32", "split"):
        with vg.Gravity(n, s, 8, mode, eps=eps * 2.0 ** l, G=1.3 * 2.0 ** (2 * l - k), mass=2.0 ** k / n) as g:
            g.upload(x, None, m)
            r[mode] = g.accelerations(), g.energy()[1]
    a = r["f64"][0]
    for mode in ("f32", "split"):
        b = r[mode][0]
        assert np.linalg.norm(b - a) <= BOUND * np.linalg.norm(a), mode  # false for NaN
        assert abs(r[mode][1] - r["f64"][1]) <= 5e-6 * abs(r["f64"][1]), mode


@pytest.mark.parametrize("k,eps,masses", [(88, 1e-3, True), (0, 1e-7, False)])
def test_p2p_f32_small_softening_in_a_wide_box(vg, k, eps, masses):
    """The pair of a particle with itself forms m / eps^3, which FP32 holds in the caller's
    units (2^106 and 2^70) and has to in those of a box 2^63 wide too."""
    n, s, l = 4100, 12, 60
    x = _points(n, "core", n) * 2.0 ** l
    m = np.random.default_rng(1).uniform(0.5, 1.5, n) / n * 2.0 ** k if masses else None
    a = {}
    for mode in ("f64", "f32", "split"):
        with vg.Gravity(n, s, 8, mode, eps=eps, G=1.3 * 2.0 ** (2 * l - k), mass=2.0 ** k / n) as g:
            g.upload(x, None, m)
            a[mode] = g.accelerations()
    for mode in ("f32", "split"):
        assert np.linalg.norm(a[mode] - a["f64"]) <= BOUND * np.linalg.norm(a["f64"]), mode  # false for NaN


def test_p2p_f32_softening_beyond_the_range(vg):
    """A softening whose square FP32 does not hold: the near field vanishes, and the potential is the far field's."""
    n = 2000
    x = _points(n, "uniform", 2)
    m = np.random.default_rng(2).uniform(0.5, 1.5, n) / n
    for s in (16, 1000):
        u = {}
        for mode in ("f64", "f32"):
            with vg.Gravity(n, s, 8, mode, eps=1e25) as g:
                g.upload(x, None, m)
                a, u[mode] = g.accelerations(), g.energy()[1]
                assert np.isfinite(a).all() and (s < 1000 or (abs(a) < 1e-38).all())
        assert abs(u["f32"] - u["f64"]) <= 5e-6 * abs(u["f64"])


@pytest.mark.parametrize("gap", [0.11, 0.13, 0.16, 0.25, 0.42, 0.45, 0.6])
def test_p2p_f32_single_pairs_of_a_large_leaf(vg, gap):
    """One heavy source near a leaf as large as an octant of the root (R = 0.85), all other
    masses negligible, so that each target's force is one pair's, on positions that
    FP32 holds exactly.  By differences a pair is within 16 roundings (r^2 3, the root's
    estimate 2, 3 x 3.5 for its cube, products 2.5); by the expansion, beyond R / 2,
    within 2 (3/2 R)^2 / (R / 2)^2 = 18 of r^2, 27 of the force, and 12 more: 40."""
    worst = 0.0
    for seed in range(25):
        rng = np.random.default_rng(seed)
        t = -1 + 0.98 * rng.random((96, 3))
        t[0], t[1] = -1, -0.02  # the leaf's corners
        c = np.array([gap - 0.015, *(-0.02 - 0.5 * rng.random(2))]) + 0.004 * (rng.random((32, 3)) - 0.5)
        x = np.round(np.concatenate([t, c, [[1.0, 1.0, 1.0]]]) * 2 ** 20) / 2 ** 20
        h = 96 + rng.integers(32)
        m = np.full(len(x), 2.0 ** -60)
        m[h] = 1
        with vg.Gravity(len(x), 40, 3, "f32", eps=0.0) as g:
            g.upload(x, None, m)
            a = g.accelerations()[:96]
            assert g.counts()["cells"] == 9
        d = x[h] - x[:96]
        ref = d / ((d * d).sum(1) ** 1.5)[:, None]
        worst = max(worst, (np.linalg.norm(a - ref, axis=1) / np.linalg.norm(ref, axis=1)).max())
    assert worst <= 40 * 2.0 ** -24


def test_p2p_memory_of_large_leaves(vg):
    """64 leaves of about 4096 particles with up to 27 x 4096 sources each, in FP64: partial sums of
    at most 12 rows of 2^18 entries (101 MB, 134 where buffers grow in powers of two) beside
    330 B a particle (173 MB for the same reason), and as much again for all else: 614 MB."""
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        f, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(total)) == 0
        return f.value

    n = 1 << 18
    x = np.random.default_rng(9).random((n, 3))
    with vg.Gravity(2000, 100, 4, "f64", eps=1e-3) as g:  # what the first context of a process takes
        g.upload(x[:2000])
        g.accelerations()
    before = free()
    with vg.Gravity(n, 5000, 4, "f64", eps=1e-3) as g:
        g.upload(x)
        g.accelerations()
        used = before - free()
        assert g.counts()["leaves"] == 64
    assert used <= 614e6


def test_p2p_items_in_pieces(vg):
    """64 leaves of about 8192 particles, whose 65,000 to 220,000 sources go to 12 items each, in
    pieces of 4096: accelerations against the direct sum, the two modes' energies against
    each other.  Level-2 cells that do not touch are far enough apart for p = 12 to truncate
    at 1e-5 of a force in the 2-norm; a piece left out or taken twice is 2 % of a leaf's
    sources or more."""
    n = 1 << 19
    rng = np.random.default_rng(10)
    x = rng.random((n, 3))
    m = rng.uniform(0.5, 1.5, n) / n
    idx = rng.choice(n, 2000, replace=False)
    u = {}
    for mode in ("f64", "f32"):
        with vg.Gravity(n, 5000, 12, mode, eps=1e-3) as g:
            g.upload(x, None, m)
            a, u[mode] = g.accelerations(), g.energy()[1]
            assert g.counts()["leaves"] == 64 and np.array_equal(a, g.accelerations())
            ref = g.direct(idx)
        assert np.linalg.norm(a[idx] - ref) <= 1e-4 * np.linalg.norm(ref), mode
    assert abs(u["f32"] - u["f64"]) <= 5e-6 * abs(u["f64"])


@pytest.mark.parametrize("mode", ["f64", "f32", "split"])
@pytest.mark.parametrize("n", [3, 17, 50, 700])
@pytest.mark.parametrize("masses", [False, True])
def test_potential_without_the_particle_itself(vg, mode, n, masses):
    """Softening far below the distances, m_i / eps far above the potential: the energy of one leaf
    against the sum over pairs.  Terms of one sign, each within 8 roundings, and their sums:
    n + 8 roundings of 2^-24 or 2^-53."""
    rng = np.random.default_rng(n)
    x = np.round(rng.random((n, 3)) * 2 ** 18) / 2 ** 18
    m = rng.uniform(0.5, 1.5, n) / n if masses else np.full(n, 1.0 / n)
    with vg.Gravity(n, 1500, 3, mode, eps=1e-5) as g:
        g.upload(x, None, m if masses else None)
        u = g.energy()[1]
    ref = np.longdouble(0)
    for i in range(n):
        d = (np.delete(x, i, 0) - x[i]).astype(np.longdouble)
        ref -= m[i] / 2 * (np.delete(m, i) / np.sqrt((d * d).sum(1) + np.longdouble(1e-5) ** 2)).sum()
    assert abs(u - ref) <= (n + 8) * 2.0 ** (-53 if mode == "f64" else -24) * abs(ref)
