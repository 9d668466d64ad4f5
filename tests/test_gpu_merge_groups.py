"""Merging in groups of flagged particles, each replayed by its own block, bit
for bit the sequential oracle: groups on either side of the linking distance, a
crowded cell that is linked whole, a wake that is one connected group, and
particles that travel further than the groups are kept apart (the replay starts
over as one)."""
import numpy as np
import pytest

from oracle import oracle as O
from pawan_amd import capi

pytestmark = pytest.mark.gpu

SIGMA = 0.1
H = 0.25 * SIGMA  # merge distance of two particles of this radius


def _compare(pos, alpha, radius, stepnum=100.0):
    n = len(pos)
    volume, active = np.linspace(1.0, 2.0, n), np.zeros(n)
    birth = np.linalg.norm(alpha, axis=1)
    w = O.WakeParticles(pos, alpha, radius, volume, birth, active)
    k_ref = O.wake_merge(w, stepnum)
    g = [np.ascontiguousarray(a).copy() for a in (pos, alpha, radius, volume, active)]
    k = capi.wake_merge(g[0], g[1], g[2], g[3], g[4], n, stepnum)
    print(f"n={n}: {k} merges, oracle {k_ref}", flush=True)
    assert k == k_ref
    np.testing.assert_array_equal(g[0], w.pos)
    np.testing.assert_array_equal(g[1], w.alpha)
    np.testing.assert_array_equal(g[3], w.volume)
    return k


@pytest.mark.parametrize("gap", [0.5, 1.0, 2.0, 4.0, 5.0, 6.2, 6.3, 9.0])
def test_clusters_at_a_distance(gap):
    """A line of clusters `gap` merge distances apart, 1-5 particles each,
    their indices interleaved."""
    rng = np.random.default_rng(int(10 * gap))
    m, per = 120, 5
    centre = np.zeros((m, 3))
    centre[:, 0] = gap * H * np.arange(m)
    pos = np.repeat(centre, per, axis=0) + rng.normal(scale=0.2 * H, size=(m * per, 3))
    order = rng.permutation(m * per)
    pos = pos[order]
    alpha = rng.normal(size=(m * per, 3))
    assert _compare(pos, alpha, np.full(m * per, SIGMA)) > m


@pytest.mark.parametrize("n", [40, 700])
def test_crowded_cell(n):
    """All flagged particles in one coarse cell (700: also more neighbours
    than the replay keeps in LDS would need at 27 cells of H)."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 3.0 * H, size=(n, 3))
    far = np.array([[1.0, 1.0, 1.0]]) + rng.normal(scale=0.3 * H, size=(20, 3))
    pos = np.concatenate([pos, far])[rng.permutation(n + 20)]
    _compare(pos, rng.normal(size=(n + 20, 3)), rng.uniform(0.6 * SIGMA, SIGMA, n + 20))


@pytest.mark.parametrize("hops", [2, 6, 40])
def test_travelling_particle(hops):
    """A weak particle dragged along a chain of strong ones of alternating
    direction, most of a merge distance per merge."""
    pos, alpha = [[0.0, 0.0, 0.0]], [[0.0, 1e-6, 0.0]]
    x = 0.0
    for k in range(hops):
        x += 0.9 * H
        pos.append([x, 0.0, 0.0])
        alpha.append([1.0 if k % 2 == 0 else -1.0, 0.0, 1e-3])
    rng = np.random.default_rng(hops)
    pos = np.concatenate([np.array(pos), 1.0 + rng.uniform(0.0, 20 * H, size=(200, 3))])
    alpha = np.concatenate([np.array(alpha), rng.normal(size=(200, 3))])
    _compare(pos, alpha, np.full(len(pos), SIGMA))
