"""Point velocities with the sources split over blocks: at the edges of the
64-point groups and 256-source tiles, with too few particles to hold a split's
partial sums, and through the entry point that allocates nothing; against the
oracle at the repository's FP64 bar."""
import numpy as np
import pytest

from conftest import normwise
from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(1, 1), (255, 64), (257, 63), (512, 65), (1000, 700), (8191, 1), (8193, 129)])
def test_split_edges(oracle, n, m):
    s = W.cored_ring(R=1.0, gamma=1.0, sigma=0.1, core=0.1, nst=-(-n // 5), ncs_ring=4)
    s = W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=s.pos[:n].copy(), alpha=s.alpha[:n].copy(),
                         radius=s.radius[:n].copy(), volume=s.volume[:n].copy(), nu=0.0, coupled=True, name="ring")
    rng = np.random.default_rng(n + m)
    pts = rng.uniform(-1.3, 1.3, size=(m, 3)) * np.array([1.0, 1.0, 0.3])
    pts[0] = s.pos[0]  # on a particle
    ref = oracle.velocity_at(s, pts)
    with capi.Solver(s) as g:
        u = g.velocity_at(pts)
        np.testing.assert_array_equal(g.velocity_at_noalloc(pts), u)
        np.testing.assert_array_equal(g.velocity_at(pts), u)  # the kept buffer
    assert normwise(u, ref) < 1e-12 or (n == 1 and not u.any() and not ref.any())
