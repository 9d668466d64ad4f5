"""Quadratic diagnostics over unordered pairs, split into (64 targets, source
range) items: at the edges of groups, tiles and ranges, for coupled and
independent wakes and single wake blocks, under both smoothing kernels, against
the oracle.  The sums are compared relative to the sums of their terms'
magnitudes, which bound what any order of adding them can lose."""
import numpy as np
import pytest

from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu

H, EN, ENF, KE, KEF = 9, 10, 11, 12, 13


def _wake(n, seed):
    rng = np.random.default_rng(seed)
    return W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=rng.normal(size=(n, 3)),
                            alpha=rng.normal(size=(n, 3)), radius=rng.uniform(0.1, 0.4, n), volume=np.ones(n))


def _scales(s):
    """Sums of magnitudes: |a_i||a_j|/(4 pi r^2) for the helicity, the same
    over r for the energies (with the self terms)."""
    d = np.linalg.norm(s.pos[:, None] - s.pos[None], axis=-1)
    a = np.linalg.norm(s.alpha, axis=1)
    sg = np.sqrt(0.5 * (s.radius[:, None] ** 2 + s.radius[None] ** 2))
    r = np.sqrt(d * d + sg * sg)
    aa = a[:, None] * a[None]
    return np.sum(aa * d / r ** 3) / (4 * np.pi), np.sum(aa / r) / (8 * np.pi)


# n eps for the order of the sums, and the kernels' own few roundings
def _check(d, ref, s):
    sh, sk = _scales(s)
    tol = 4 * (np.sqrt(s.n) + 8) * 2.0 ** -52
    assert abs(d[H] - ref[H]) <= tol * sh
    assert abs(d[KE] - ref[KE]) <= tol * sk and abs(d[KEF] - ref[KEF]) <= tol * sk


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 256, 257, 1000, 2311])
def test_one_system(oracle, n):
    s = _wake(n, n)
    with capi.Solver(s) as g:
        d = g.diagnose()[:15]
        again = g.diagnose()[:15]
    np.testing.assert_array_equal(d, again)
    _check(d, oracle.diagnose(s), s)


def test_independent_systems_and_wake_blocks(oracle):
    parts = [_wake(n, 70 + n) for n in (130, 1, 700, 64, 321)]
    s = W.concat(parts, coupled=False, nu=0.0, name="five")
    with capi.Solver(s) as g:
        d = g.diagnose().reshape(-1, 15)
    for k, p in enumerate(parts):
        _check(d[k], oracle.diagnose(p), p)
    c = W.concat(parts, coupled=True, nu=0.0, name="five")
    with capi.Solver(c) as g:
        tot = g.diagnose()[:15]
        blocks = [g.diagnose_wakes(a, b) for a in range(5) for b in range(a, 5)]
    _check(tot, oracle.diagnose(c), c)
    sh, sk = _scales(c)
    assert abs(sum(b[H] for b in blocks) - tot[H]) < 1e-13 * sh
    assert abs(sum(b[KE] for b in blocks) - tot[KE]) < 1e-13 * sk


def test_coincident_particles_are_not_finite():
    """0/0 in the reference's q; the energies stay finite."""
    s = _wake(100, 3)
    s.pos[40] = s.pos[7]
    for kernel in (capi.PW_KERNEL_GAUSSIAN, capi.PW_KERNEL_HIGHORDER):
        with capi.Solver(s) as g:
            g.set_kernel(kernel)
            d = g.diagnose()[:15]
        assert np.isnan(d[H]) and np.isfinite(d[KE]) and np.isfinite(d[KEF])
