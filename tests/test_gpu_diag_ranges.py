"""Quadratic diagnostics of systems whose items span source ranges of 128, 512
and 1,024 particles (several tiles an item, waves partly before and partly at
their targets, self terms only in the range that ends with the group), and
cross-wake blocks of as many, under both smoothing kernels, against the oracle.
The sums are compared relative to the sums of their terms' magnitudes."""
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
    """Bounds of the sums of magnitudes: |a_i||a_j| over 4 pi r^2 (helicity),
    over 8 pi r (energies) and 47 / (8 pi r^3) of them (the enstrophies of the
    high-order kernel), r^2 = d^2 + sigma^2."""
    a = np.linalg.norm(s.alpha, axis=1)
    sh = sk = se = 0.0
    for i in range(0, s.n, 256):
        d2 = sum((s.pos[i:i + 256, None, c] - s.pos[None, :, c]) ** 2 for c in range(3))
        r2 = d2 + 0.5 * (s.radius[i:i + 256, None] ** 2 + s.radius[None] ** 2)
        aa = a[i:i + 256, None] * a[None]
        sh += np.sum(aa / r2)
        sk += np.sum(aa / np.sqrt(r2))
        se += np.sum(aa / r2 ** 1.5)
    return sh / (4 * np.pi), sk / (8 * np.pi), 47 * se / (8 * np.pi)


def _check(d, ref, s, kernel, scales):
    sh, sk, se = scales
    tol = 4 * (np.sqrt(s.n) + 8) * 2.0 ** -52
    assert abs(d[H] - ref[H]) <= tol * sh
    assert abs(d[KE] - ref[KE]) <= tol * sk and abs(d[KEF] - ref[KEF]) <= tol * sk
    if kernel:
        assert abs(d[EN] - ref[EN]) <= tol * se and abs(d[ENF] - ref[ENF]) <= tol * se


@pytest.mark.parametrize("n", [6501, 13001, 18001])
@pytest.mark.parametrize("kernel", [0, 1])
def test_long_ranges(oracle, n, kernel):
    s = _wake(n, n)
    with oracle.smoothing(kernel):
        ref = oracle.diagnose(s)
    with capi.Solver(s) as g:
        g.set_kernel(kernel)
        d = g.diagnose()[:15]
        own = g.diagnose_wakes(0, 0)
    scales = _scales(s)
    _check(d, ref, s, kernel, scales)
    _check(own, ref, s, kernel, scales)


@pytest.mark.parametrize("kernel", [0, 1])
def test_blocks_of_two_wakes(oracle, kernel):
    parts = [_wake(5001, 5), _wake(8343, 6)]
    c = W.concat(parts, coupled=True, nu=0.0, name="two")
    with oracle.smoothing(kernel):
        ref = oracle.diagnose(c)
    with capi.Solver(c) as g:
        g.set_kernel(kernel)
        blocks = [g.diagnose_wakes(*p) for p in ((0, 0), (1, 1), (0, 1))]
    _check(np.sum(blocks, axis=0), ref, c, kernel, _scales(c))
