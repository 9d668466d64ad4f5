"""The launch the library chooses when none is set: the split kernel (64
targets per block against a source range, a quarter of each tile per wave, the
items' slabs summed by the stage kernel) at the edges of its groups, tiles and
source ranges, for single and independent systems, and the scalar-fed kernels
just beyond the sizes it serves; against the oracle, under both smoothing
kernels."""
import contextlib

import numpy as np
import pytest

from conftest import normwise
from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu

# the repository's bars: FP64 parity, FP32C velocity and stretching
TOL = {"fp64": (1e-12, 1e-12), "fp32c": (1e-6, 1e-5)}


def _say(msg):
    print(msg, flush=True)


def _wake(n):
    """The first n particles of a viscous cored ring."""
    s = W.cored_ring(R=1.0, gamma=1.0, sigma=0.1, core=0.1, nst=-(-max(n, 40) // 5), ncs_ring=4)
    return W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=s.pos[:n].copy(), alpha=s.alpha[:n].copy(),
                            radius=s.radius[:n].copy(), volume=s.volume[:n].copy(), nu=1e-3, coupled=True,
                            name=f"ring_{n}")


@pytest.mark.parametrize("n", [2, 17, 63, 64, 65, 255, 256, 257, 1000, 3841])
@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
def test_split_edges(oracle, n, prec):
    s = _wake(n)
    ru, rw = oracle.solve(s)
    with capi.Solver(s) as g:
        u, w = g.solve(prec)
    eu, ew = normwise(u, ru), normwise(w, rw)
    _say(f"default launch N={n} {prec}: e_u={eu:.2e} e_w={ew:.2e}")
    assert eu < TOL[prec][0] and ew < TOL[prec][1]


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
def test_one_particle_moves_nothing(prec):
    with capi.Solver(_wake(1)) as g:
        u, w = g.solve(prec)
    assert not u.any() and not w.any()


@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
def test_split_independent_systems(oracle, prec):
    """Systems of 64-3,000 particles that start and end off the 64-target
    groups' and 256-source tiles' grid."""
    s = W.batched_rings(nwakes=12, nmin=64, nmax=3000, seed=9)
    with capi.Solver(s) as g:
        u, _ = g.solve(prec)
    for k in range(s.nw):
        a, b = int(s.off[k]), int(s.off[k + 1])
        ru, _ = oracle.solve(s.wake(k))
        assert normwise(u[a:b], ru) < TOL[prec][0], k


@pytest.mark.parametrize("n,prec,kernel", [(32768, "fp64", 0), (32769, "fp64", 0), (45057, "fp32c", 0),
                                           (65537, "fp64", 1)])
def test_around_the_sizes_where_the_launch_changes(oracle, n, prec, kernel):
    """Sampled targets, the last (ragged) group among them; the high-order
    case is past the item count at which the source ranges double."""
    s = W.helix_wake(128 * -(-n // 128))
    s = W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=s.pos[:n].copy(), alpha=s.alpha[:n].copy(),
                         radius=s.radius[:n].copy(), volume=s.volume[:n].copy(), nu=s.nu, coupled=True, name="helix")
    idx = np.unique(np.concatenate([np.linspace(0, n - 1, 60).astype(np.int64), np.arange(n - 4, n)]))
    with capi.Solver(s) as g:
        g.set_kernel(kernel)
        u, w = g.solve(prec)
        g.set_pair_config(prec, 2)  # the LDS-tiled kernels
        u2, w2 = g.solve(prec)
    if kernel == 0:
        ru, rw = oracle.rates_targets(s, idx)
        assert normwise(u[idx], ru) < TOL[prec][0] and normwise(w[idx], rw) < TOL[prec][1]
    assert normwise(u, u2) < TOL[prec][0] and normwise(w, w2) < TOL[prec][1]


def test_high_order_split_edges(oracle):
    for n in (65, 257, 1000):
        s = _wake(n)
        with contextlib.ExitStack() as st:
            g = st.enter_context(capi.Solver(s))
            g.set_kernel(capi.PW_KERNEL_HIGHORDER)
            ref = g.solve("fp64_ref")
            for prec in ("fp64", "fp32c"):
                u, w = g.solve(prec)
                g.set_pair_config(prec, 1, True)  # persistent: the LDS-tiled kernels
                u2, w2 = g.solve(prec)
                assert normwise(u, u2) < TOL[prec][0] and normwise(w, w2) < TOL[prec][1]
                assert normwise(u, ref[0]) < TOL[prec][0] and normwise(w, ref[1]) < TOL[prec][1]


@pytest.mark.parametrize("scheme", ["euler", "rk3", "rk4"])
@pytest.mark.parametrize("n", [65, 1000])
def test_steps_replayed_equal_eager(oracle, scheme, n):
    """Every stage form of the fused tail, eager and replayed (bit for bit),
    against the oracle's steps."""
    s = _wake(n)
    with capi.Solver(s) as ea, capi.Solver(s) as gr:
        gr.set_graph(True)
        for _ in range(3):
            ea.step(scheme, 2e-3, "fp64", 1)
            gr.step(scheme, 2e-3, "fp64", 1)
            np.testing.assert_array_equal(ea.state()[0], gr.state()[0])
            np.testing.assert_array_equal(ea.state()[1], gr.state()[1])
        pos, alpha = ea.state()
    end = oracle.step(s, scheme, 2e-3, 3)
    assert normwise(pos - s.pos, end.pos - s.pos) < 1e-11 and normwise(alpha, end.alpha) < 1e-12
