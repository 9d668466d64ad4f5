"""The default launch on both sides of every size at which it changes (the
split kernel up to 40,960 particles in FP64 and 65,536 in FP32C, then the
scalar-fed kernels over 64 source parts, over 32 from 196,608; the high-order
FP64 kernel split at every size), with ragged last groups, and the LDS-tiled
kernels, which no default launch of these sizes takes, on large wakes: sampled
targets, the last group among them, against the oracle."""
import os

import numpy as np
import pytest

from conftest import normwise
from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu

# the repository's bars: FP64 parity, FP32C velocity and stretching
TOL = {"fp64": (1e-12, 1e-12), "fp32c": (1e-6, 1e-5)}
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _helix(n):
    s = W.helix_wake(128 * -(-n // 128))
    return W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=s.pos[:n].copy(), alpha=s.alpha[:n].copy(),
                            radius=s.radius[:n].copy(), volume=s.volume[:n].copy(), nu=s.nu, coupled=True, name="helix")


def _targets(n):
    return np.unique(np.concatenate([np.linspace(0, n - 1, 60).astype(np.int64), np.arange(n - 4, n)]))


@pytest.mark.parametrize("prec,n", [("fp64", 40960), ("fp64", 40961), ("fp64", 196607), ("fp64", 196609),
                                    ("fp32c", 65536), ("fp32c", 65537), ("fp32c", 196607), ("fp32c", 196609)])
@pytest.mark.parametrize("kernel", [0, 1])
def test_default_launch(oracle, prec, n, kernel):
    s, idx = _helix(n), _targets(n)
    with oracle.smoothing(kernel):
        ru, rw = oracle.rates_targets(s, idx)
    with capi.Solver(s) as g:
        g.set_kernel(kernel)
        u, w = g.solve(prec)
    eu, ew = normwise(u[idx], ru), normwise(w[idx], rw)
    print(f"default launch N={n} {prec} kernel {kernel}: e_u={eu:.2e} e_w={ew:.2e}", flush=True)
    assert np.isfinite(u).all() and np.isfinite(w).all()
    assert eu < TOL[prec][0] and ew < TOL[prec][1]


@pytest.mark.parametrize("name,make", [("leapfrog_64k", W.leapfrog_64k), ("helix_1m", W.helix_wake)])
@pytest.mark.parametrize("prec", ["fp64", "fp32c"])
@pytest.mark.parametrize("parts,persistent", [(1, True), (2, False)])
def test_lds_tiled_on_large_wakes(name, make, prec, parts, persistent):
    ref = np.load(os.path.join(GOLDEN, f"{name}.npz"))
    with capi.Solver(make()) as g:
        g.set_pair_config(prec, parts, persistent)
        u, w = g.solve(prec)
    idx = ref["targets"]
    eu, ew = normwise(u[idx], ref["vel"]), normwise(w[idx], ref["retvor"])
    print(f"{name} {prec} LDS-tiled parts {parts} persistent {persistent}: e_u={eu:.2e} e_w={ew:.2e}", flush=True)
    assert eu < TOL[prec][0] and ew < TOL[prec][1]
