"""Scalar-fed kernels on coarse filaments, whose 64-particle chunks are wider
than the gaps between turns: sources that are clear of a wave's targets one by
one, in source ranges that start and end inside a chunk, with a ragged last
chunk and radii that vary along the wake; against the LDS-tiled FP64 kernel, FP32C held
to the LDS-tiled FP32C kernel's own error."""
import numpy as np
import pytest

from conftest import normwise
from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,parts", [(8257, 7), (40001, 3)])
@pytest.mark.parametrize("kernel", [0, 1])
def test_coarse_filaments(n, parts, kernel):
    s = W.helix_wake(128 * -(-n // 128))
    s = W.ParticleSystem(off=np.array([0, n], dtype=np.int64), pos=s.pos[:n].copy(), alpha=s.alpha[:n].copy(),
                         radius=s.radius[:n] * np.linspace(0.5, 1.5, n), volume=s.volume[:n].copy(), nu=1e-3,
                         coupled=True, name="helix")
    with capi.Solver(s) as g:
        g.set_kernel(kernel)
        g.set_pair_config("fp64", 2)
        ref = g.solve("fp64")
        g.set_pair_config("fp32c", 2)
        tiled = [normwise(a, r) for a, r in zip(g.solve("fp32c"), ref)]
        for persistent in (False, True):
            if kernel == 0:
                g.set_pair_config("fp64", parts, persistent, False, True)
                for a, r in zip(g.solve("fp64"), ref):
                    assert normwise(a, r) < 1e-12  # the repository's FP64 bar
            for waves8, two in ((False, False), (True, False), (False, True)):
                g.set_pair_config("fp32c", parts, persistent, waves8, True, two)
                for a, r, t in zip(g.solve("fp32c"), ref, tiled):
                    e = normwise(a, r)
                    print(f"N={n} kernel {kernel} waves8 {waves8} two {two}: {e:.2e}, tiled {t:.2e}", flush=True)
                    assert e < 1.2 * t + 2e-8  # FP32 rounding of the sums themselves
