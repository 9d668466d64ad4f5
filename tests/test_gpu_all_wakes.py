"""The rows of every wake in one transfer against wake-by-wake transfers: before
the particles are on the device, after a solve, and for one and many wakes."""
import numpy as np
import pytest

from pawan_amd import capi, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nwakes", [1, 7])
def test_all_wakes_match_each(nwakes):
    s = W.batched_rings(nwakes=nwakes, nmin=1, nmax=900, seed=3)
    with capi.Solver(s) as g:
        def each(get):
            parts = [get(w) for w in range(s.nw)]
            return [np.concatenate([p[k] for p in parts]) for k in (0, 1)]

        for solved in (False, True):
            if solved:
                g.step("rk3", 1e-3, "fp64", 1)
            for all_rows, get in ((g.state(), g.wake_state), (g.rates(), g.wake_rates)):
                for a, b in zip(all_rows, each(get)):
                    np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(g.state()[0].shape, (s.n, 3))
