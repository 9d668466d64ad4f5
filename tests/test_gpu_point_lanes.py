"""Point velocities with the particles in the lanes: few and many particles per
lane, the block's waves sharing out the points or the range, with remainders on
both sides; against the oracle at the repository's FP64 bar, and the algebraic
kernel against its own FP64 sum."""
import numpy as np
import pytest

from conftest import normwise
from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu


def _wake(n):
    s = W.helix_wake(-(-n // 128) * 128)
    return W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=s.pos[:n].copy(), alpha=s.alpha[:n].copy(),
                            radius=s.radius[:n].copy(), volume=s.volume[:n].copy(), nu=0.0, coupled=True,
                            name="helix")


# (particles, points): one particle per lane; two, the waves sharing out the
# points (256 groups of points and fewer than 1,024 particles); four, the waves
# sharing out the range, whole and with a remainder, one range and several
@pytest.mark.parametrize("n,m", [(63, 17), (65, 1), (129, 64 * 256), (1023, 64 * 255 + 1), (1024, 64 * 255 + 1),
                                 (4097, 5003), (65600, 300)])
@pytest.mark.parametrize("highorder", [False, True])
def test_lane_edges(oracle, n, m, highorder):
    s = _wake(n)
    rng = np.random.default_rng(n + m)
    lo, hi = s.pos.min(0) - 0.1, s.pos.max(0) + 0.1
    pts = rng.uniform(lo, hi, size=(m, 3))
    pts[-1] = s.pos[-1]  # on a particle
    pick = np.unique(np.concatenate([np.arange(min(m, 70)), rng.integers(0, m, 40), [m - 1]]))
    with capi.Solver(s) as g:
        if highorder:
            g.set_kernel(capi.PW_KERNEL_HIGHORDER)
        u = g.velocity_at(pts)
        np.testing.assert_array_equal(g.velocity_at(pts), u)
    if highorder:
        d = pts[pick][:, None, :] - s.pos[None]
        r2 = (d * d).sum(-1)
        s2 = (s.radius * s.radius)[None]
        q = (r2 + 2.5 * s2) / (r2 + s2) ** 2.5 / (4.0 * np.pi)
        ref = (q[..., None] * np.cross(s.alpha[None], d)).sum(1)
    else:
        ref = oracle.velocity_at(s, pts[pick])
    assert normwise(u[pick], ref) < 1e-12
