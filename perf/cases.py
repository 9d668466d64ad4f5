"""Performance cases of the solver: what programs built on it spend their time in.

A case is a plain dict.  ``listed()`` names the fixed ones, ``draw(rng)`` gives
another one of the same ranges, ``prepare(case, seed)`` makes what a program has
in hand before the call (host arrays, a solver, a point set), ``run(state)`` is
one pass through the public entry points of ``pawan_amd.capi``, ``work(case)``
the bytes and operations that pass cannot do without, and ``exact(case, seed)``
the same results in 64 bits by plain torch, where that takes seconds.

The kinds:

  steps    a small or medium wake advanced by a host program that owns the
           state (load, a few RK steps on the device, read back): latency and
           launches count
  solve    one right-hand side of a wake, velocities and vorticity rates read
           back: direct sums in FP64 and FP32C, coupled wakes or independent
           ones, the Gaussian or the high-order kernel, with the default launch
           or one a program has tuned before
  tree     one right-hand side of the tree path, with the analytic expansion or
           the network
  diagnose the conserved quantities written at every output time
  points   the velocity at a set of points (inflow planes, probes)
  relax    particle management of one wake: split, then merge
  grad     loss and gradient of the far-field network on a batch of samples

Results of the single-precision paths (FP32C, tree) are handed on as float32
arrays, those of the FP64 paths as float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from pawan_amd import capi, workloads as W

FLOP_PER_PAIR = 88     # of one ordered (target, source) pair: velocity, stretching, diffusion
FLOP_PER_POINT = 45    # velocity alone
FLOP_PER_DIAG = 70     # helicity and the two energies of an unordered pair
STATE_BYTES, RATE_BYTES = 64, 48   # a particle's record, its rates
DTS = {"ring": 0.005, "leapfrog": 0.002, "batched": 0.002, "helix": 1e-3}
# Direct sums beyond this many pairs take plain torch too long
EXACT_PAIRS = 7e10


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # the smallest program: one vortex ring, FP64, ten RK4 steps between
        # two looks at the state, replayed as a HIP graph
        dict(name="ring_rk4_fp64", kind="steps", wake="ring", nst=200, precision="fp64", kernel="gaussian",
             scheme="rk4", nsteps=10, graph=True),
        # two leapfrogging rings of odd size with viscosity under the algebraic
        # kernel, third-order steps
        dict(name="leapfrog_rk3_highorder", kind="steps", wake="leapfrog", nst=301, precision="fp64",
             kernel="highorder", scheme="rk3", nsteps=2, graph=False),
        # a batch of independent rings of very different sizes in one context
        dict(name="batched_fp64", kind="solve", wake="batched", nwakes=48, precision="fp64", kernel="gaussian",
             tuned=False),
        # a rotor wake in the default precision and the default launch
        dict(name="helix_fp64", kind="solve", wake="helix", n=147200, precision="fp64", kernel="gaussian",
             tuned=False),
        # the same with compensated single-precision sums, no tuning
        dict(name="helix_fp32c", kind="solve", wake="helix", n=200064, precision="fp32c", kernel="gaussian",
             tuned=False),
        # the headline workload: 1,048,576 particles, the launch its autotuner picks
        dict(name="helix_1m_fp32c", kind="solve", wake="helix", n=1048576, precision="fp32c", kernel="gaussian",
             tuned=True),
        # the headline workload on the tree path, both far fields
        dict(name="tree_1m_quadrupole", kind="tree", n=1048576, network=False, tol=0.0),
        dict(name="tree_network", kind="tree", n=300032, network=True, tol=5e-4),
        # conserved quantities of two leapfrogging rings
        dict(name="diagnose_leapfrog", kind="diagnose", wake="leapfrog", nst=1500, kernel="gaussian"),
        # a rotor disk's inflow: some hundred points in a large wake
        dict(name="points_in_wake", kind="points", wake="helix", n=262144, kernel="gaussian", m=1200),
        # a wake's particles split and merged between steps
        dict(name="relax_wake", kind="relax", n=98304),
        # one training batch
        dict(name="network_gradient", kind="grad", batch=4096),
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng) -> dict:
    kind = rng.choice(["steps", "steps", "solve", "solve", "solve", "tree", "tree", "diagnose", "points", "relax",
                       "grad"])
    kernel = rng.choice(["gaussian", "gaussian", "highorder"])
    if kind == "steps":
        wake = rng.choice(["ring", "leapfrog"])
        nst = int(_log(rng, 40, 4000)) if wake == "ring" else int(_log(rng, 20, 1500))
        return dict(kind=kind, wake=wake, nst=nst, precision=rng.choice(["fp64", "fp32c"]), kernel=kernel,
                    scheme=rng.choice(["euler", "rk3", "rk4"]), nsteps=rng.choice([1, 2, 5, 10]),
                    graph=rng.choice([False, True]))
    if kind == "solve":
        wake = rng.choice(["helix", "leapfrog", "batched"])
        precision = rng.choice(["fp64", "fp32c"])
        c = dict(kind=kind, wake=wake, precision=precision, kernel=kernel, tuned=False)
        if wake == "helix":
            c["n"] = 128 * int(_log(rng, 32, 1200 if precision == "fp64" else 2000))
            c["tuned"] = precision == "fp32c" and rng.random() < 0.4
        elif wake == "leapfrog":
            c["nst"] = int(_log(rng, 200, 8000))
        else:
            c["nwakes"] = int(_log(rng, 4, 200))
        return c
    if kind == "tree":
        return dict(kind=kind, n=128 * int(_log(rng, 160, 8000)), network=rng.choice([False, True]),
                    tol=rng.choice([0.0, 2e-4, 1e-3]))
    if kind == "diagnose":
        return dict(kind=kind, wake="leapfrog", nst=int(_log(rng, 60, 4000)), kernel=kernel)
    if kind == "points":
        return dict(kind=kind, wake="helix", n=128 * int(_log(rng, 64, 4096)), kernel=kernel,
                    m=int(_log(rng, 1, 20000)))
    if kind == "relax":
        return dict(kind=kind, n=128 * int(_log(rng, 64, 1600)))
    return dict(kind="grad", batch=int(_log(rng, 64, 32768)))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _disturbed(s: W.ParticleSystem, seed: int) -> W.ParticleSystem:
    """The generator's wake with every particle moved by up to 2% of its
    smoothing radius and its strength scaled by up to 2%: a wake in motion."""
    n = s.n
    move = np.stack([W.uniform(seed, 31 + k, n, -0.02, 0.02) for k in range(3)], axis=-1)
    s.pos = np.ascontiguousarray(s.pos + s.radius[:, None] * move)
    s.alpha = np.ascontiguousarray(s.alpha * (1.0 + W.uniform(seed, 34, n, -0.02, 0.02))[:, None])
    return s


def _system(case: dict, seed: int) -> W.ParticleSystem:
    wake = case["wake"]
    if wake == "helix":
        return W.helix_wake(case["n"], seed=seed)
    if wake == "batched":  # the rings of one batch, in another state
        return _disturbed(W.batched_rings(case["nwakes"]), seed)
    if wake == "leapfrog":
        return _disturbed(W.leapfrog_64k(case["nst"]), seed)
    s = W.cored_ring(R=1.0, gamma=1.0, sigma=0.1, core=0.1, nst=case["nst"], ncs_ring=4)
    return _disturbed(s, seed)


def _solver(case: dict, s: W.ParticleSystem) -> capi.Solver:
    g = capi.Solver(s)
    if case.get("kernel") == "highorder":
        g.set_kernel(capi.PW_KERNEL_HIGHORDER)
    return g


def _weights(seed: int) -> np.ndarray:
    """Network parameters (W1 b1 W2 b2 W3 b3 W4 b4, input-major) of the scale
    training leaves them at: +-1/sqrt(fan-in), a weak output layer."""
    out, stream = [], 50
    for fan, units, scale in ((16, 128, 1.0), (128, 128, 1.0), (128, 128, 1.0), (128, 12, 0.3)):
        lim = scale / math.sqrt(fan)
        out.append(W.uniform(seed, stream, fan * units, -lim, lim))
        out.append(W.uniform(seed, stream + 1, units, -lim, lim))
        stream += 2
    return np.concatenate(out).astype(np.float32)


def _relax_arrays(case: dict, seed: int):
    """A helical wake in which one particle in 200 has turned (it merges with
    its neighbours) and one in 100 has doubled its strength (it splits)."""
    n = case["n"]
    s = W.helix_wake(n, seed=seed)
    pos, alpha = s.pos.copy(), s.alpha.copy()
    turn = W.uniform(seed, 41, n) < 0.005
    t = alpha[turn]
    alpha[turn] = np.stack([-t[:, 1], t[:, 0], t[:, 2]], axis=1)
    birth = np.linalg.norm(alpha, axis=1)
    birth[W.uniform(seed, 42, n) < 0.01] *= 0.4
    # strengths in the units of a rotor's circulation, so that the split's
    # floor on the birth strength is met
    alpha *= 20.0
    birth *= 20.0
    maxn = n + n // 8
    rows = []
    for a, cols in ((pos, 3), (alpha, 3), (s.radius, 0), (s.volume, 0), (birth, 0), (np.zeros(n), 0)):
        b = np.zeros((maxn, 3) if cols else maxn)
        b[:n] = a
        rows.append(b)
    return rows, maxn


def _points(case: dict, seed: int) -> np.ndarray:
    m = case["m"]
    r, psi = 1.2 * np.sqrt(W.uniform(seed, 43, m)), W.uniform(seed, 44, m, 0.0, 2.0 * math.pi)
    return np.ascontiguousarray(np.stack([r * np.cos(psi), r * np.sin(psi),
                                          W.uniform(seed, 45, m, -0.45, 0.05)], axis=-1))


def _samples(case: dict, seed: int):
    n = case["batch"]
    X = np.stack([W.uniform(seed, 60 + k, n, -1.0, 1.0) for k in range(16)], axis=-1).astype(np.float32)
    Y = np.stack([W.uniform(seed, 80 + k, n, -0.5, 0.5) for k in range(12)], axis=-1).astype(np.float32)
    return X, Y


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    st = dict(case=case, kind=kind)
    if kind == "relax":
        st["rows"], st["maxn"] = _relax_arrays(case, seed)
    elif kind == "grad":
        st["X"], st["Y"] = _samples(case, seed)
        st["g"] = capi.Solver(W.thin_ring(1.0, 1.0, 0.1, 64))
        st["g"].ff_set_weights(_weights(seed))
    elif kind == "tree":
        st["g"] = capi.Solver(W.helix_wake(case["n"], seed=seed))
        st["g"].ff_set_params(0.5, case["tol"], use_mlp=case["network"])
        if case["network"]:
            st["g"].ff_set_weights(_weights(seed))
    else:
        s = _system(case, seed)
        st["g"] = _solver(case, s)
        if kind == "steps":
            st["wakes"] = [(s.pos[a:b].copy(), s.alpha[a:b].copy()) for a, b in zip(s.off[:-1], s.off[1:])]
            st["g"].set_graph(case["graph"])
        elif kind == "points":
            st["points"] = _points(case, seed)
        elif case.get("tuned"):
            # what the autotuner picks for large wakes, kept by the program
            st["g"].set_pair_config(case["precision"], 32, True, True, True)
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _kept(arrays, single: bool):
    return tuple(a.astype(np.float32) for a in arrays) if single else tuple(arrays)


def run(st: dict):
    case, kind = st["case"], st["kind"]
    if kind == "steps":
        g = st["g"]
        for w, (pos, alpha) in enumerate(st["wakes"]):
            g.set_wake_state(w, pos, alpha)
        g.step(case["scheme"], DTS[case["wake"]], case["precision"], case["nsteps"])
        return _kept(g.state(), case["precision"] == "fp32c")
    if kind == "solve":
        return _kept(st["g"].solve(case["precision"]), case["precision"] == "fp32c")
    if kind == "tree":
        return _kept(st["g"].solve("learned"), True)
    if kind == "diagnose":
        return st["g"].diagnose()
    if kind == "points":
        return st["g"].velocity_at(st["points"])
    if kind == "relax":
        pos, alpha, radius, volume, birth, active = (a.copy() for a in st["rows"])
        n, splits = capi.wake_split(pos, alpha, radius, volume, birth, active, case["n"], 60.0, st["maxn"])
        merges = capi.wake_merge(pos, alpha, radius, volume, active, n, 60.0)
        return {"n": n, "splits": splits, "merges": merges, "pos": pos, "alpha": alpha, "radius": radius,
                "volume": volume, "birth": birth, "active": active}
    grad, loss = st["g"].ff_mlp_grad(st["X"], st["Y"])
    return {"grad": grad, "loss": np.float32(loss)}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _sizes(case: dict) -> list[int]:
    """Particles of each system that interacts with itself."""
    wake = case["wake"]
    if wake == "helix":
        return [case["n"]]
    if wake == "leapfrog":
        return [16 * case["nst"]]
    if wake == "ring":
        return [5 * case["nst"]]
    return np.diff(W.batched_rings(case["nwakes"]).off).tolist()


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "relax":
        # ten doubles of a particle read, and written
        return {"bytes": 160.0 * case["n"], "flops": 40.0 * case["n"]}
    if kind == "grad":
        # forward, and two products of the same size backward
        return {"bytes": 112.0 * case["batch"] + 8.0 * 36748, "flops": 3.0 * 72704 * case["batch"]}
    if kind == "tree":
        n = case["n"]
        # near pairs and far nodes of a target at the opening angle 0.5, from
        # the lists of the 1M wake (wakes of fewer particles have shorter ones)
        near, far = min(28000, n // 8), min(1700, n // 150)
        flops = n * (FLOP_PER_PAIR * near + (160 if case["network"] else 380) * far)
        if case["network"]:
            flops += 72704.0 * (n / 150) * far
        return {"bytes": float(n * (STATE_BYTES + RATE_BYTES)), "flops": float(flops)}
    if kind == "points":
        n, m = case["n"], case["m"]
        return {"bytes": float(STATE_BYTES * n + 48 * m), "flops": float(FLOP_PER_POINT) * n * m}
    sizes = _sizes(case)
    n, pairs = sum(sizes), float(sum(k * (k - 1) for k in sizes))
    if kind == "diagnose":
        return {"bytes": float(STATE_BYTES * n + 120), "flops": FLOP_PER_DIAG * 0.5 * pairs}
    if kind == "steps":
        rhs = case["nsteps"] * {"euler": 1, "rk3": 3, "rk4": 4}[case["scheme"]]
        return {"bytes": float(2 * 48 * n), "flops": FLOP_PER_PAIR * pairs * rhs}
    return {"bytes": float((STATE_BYTES + RATE_BYTES) * n), "flops": FLOP_PER_PAIR * pairs}


# ---------------------------------------------------------------------------
# The same in 64 bits, plain torch
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gauss(s: torch.Tensor):
    """(4 pi sigma^3 q, sigma^5 F, sigma^3 Z) of the Gaussian kernel at
    s = rho^2 / sigma^2; below s = 1 by the series of positive terms
    sum s^k / (2k + 5)!!, which has no cancellation at small s."""
    K = (2.0 * math.pi) ** -1.5
    e = torch.exp(-0.5 * s)
    small = s < 1.0
    ss = torch.where(small, s, torch.zeros_like(s))
    B, term, k = torch.zeros_like(s), torch.full_like(s, 1.0 / 15.0), 0
    while k < 22:
        B += term
        k += 1
        term = term * ss / (2 * k + 5)
    sb = torch.where(small, torch.ones_like(s), s)
    rb = sb.sqrt()
    q_far = (torch.erf(rb * math.sqrt(0.5)) / rb - 4.0 * math.pi * K * e) / sb
    q = torch.where(small, 4.0 * math.pi * K * e * (1.0 / 3.0 + ss * B), q_far)
    F = torch.where(small, -3.0 * K * e * B, (K * e - 3.0 * q_far / (4.0 * math.pi)) / sb)
    return q, F, K * e


def _kernel(r2: torch.Tensor, sig2: torch.Tensor, highorder: bool, need_f: bool = True):
    """q, F and Z of the pairs (r2 = inf: no pair)."""
    if highorder:
        b = (r2 + sig2).rsqrt()
        b2 = b * b
        b5 = b2 * b2 * b
        q = (0.25 / math.pi) * (r2 + 2.5 * sig2) * b5
        skip = torch.isinf(r2)
        q.masked_fill_(skip, 0.0)
        if not need_f:
            return q, None, None
        F = (-0.375 / math.pi) * (2.0 * r2 + 7.0 * sig2) * (b5 * b2)
        F.masked_fill_(skip, 0.0)
        Z = (13.125 / math.pi) * sig2 ** 3 * (b5 * b2 * b2)
        return q, F, Z
    ir = r2.rsqrt()
    q = (0.25 / math.pi) * ir * ir * ir
    F = -3.0 * q * ir * ir if need_f else None
    Z = torch.zeros_like(r2) if need_f else None
    near = torch.nonzero(r2 < 100.0 * sig2, as_tuple=True)
    if near[0].numel():
        sg = sig2[near] if sig2.shape == r2.shape else sig2.expand_as(r2)[near]
        gq, gF, gZ = _gauss(r2[near] / sg)
        s3 = sg * sg.sqrt()
        q[near] = gq / (4.0 * math.pi * s3)
        if need_f:
            F[near] = gF / (s3 * sg)
            Z[near] = gZ / s3
    return q, F, Z


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


def _rates(x, a, s2, vol, nu: float, highorder: bool, block: int = 1 << 24):
    """u and d(alpha)/dt of one interacting system (tensors on one device)."""
    n = x.shape[0]
    u, w = torch.empty_like(x), torch.empty_like(a)
    src, al = x.T.contiguous(), a.T.contiguous()
    step = max(1, block // n)
    for t0 in range(0, n, step):
        t1 = min(n, t0 + step)
        d = [src[k, t0:t1, None] - src[k, None, :] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        i = torch.arange(t1 - t0, device=x.device)
        r2[i, t0 + i] = math.inf
        sig2 = 0.5 * (s2[t0:t1, None] + s2[None, :])
        q, F, Z = _kernel(r2, sig2, highorder)
        at = al[:, t0:t1]
        # v = a_s x d, h = a_t . v
        v = [al[1] * d[2] - al[2] * d[1], al[2] * d[0] - al[0] * d[2], al[0] * d[1] - al[1] * d[0]]
        h = at[0, :, None] * v[0] + at[1, :, None] * v[1] + at[2, :, None] * v[2]
        for k in range(3):
            u[t0:t1, k] = (q * v[k]).sum(1)
        g = F * h
        # a_t x a_s pair by pair: the sum of q a_s would cancel against a_t
        cx = [at[1, :, None] * al[2] - at[2, :, None] * al[1], at[2, :, None] * al[0] - at[0, :, None] * al[2],
              at[0, :, None] * al[1] - at[1, :, None] * al[0]]
        for k in range(3):
            w[t0:t1, k] = (q * cx[k] + g * d[k]).sum(1)
        if nu:
            c = (2.0 * nu) * Z / sig2
            c[i, t0 + i] = 0.0
            S, V = c @ a, c @ vol
            w[t0:t1] += vol[t0:t1, None] * S - V[:, None] * a[t0:t1]
        del d, r2, q, F, Z, v, h, g, cx
    return u, w


def _far_rates(x, a, s2, vol, nu: float, block: int = 1 << 25):
    """The same for the Gaussian kernel and many particles: sums over the
    sources as matrix products (their cancellation, about 1e-12, is far
    below single precision)."""
    n = x.shape[0]
    c0 = x.mean(0)
    x = x - c0
    m = torch.linalg.cross(a, x)           # a_s x x_s
    A6 = torch.cat([a, m], 1)
    X4 = torch.cat([torch.ones_like(x[:, :1]), x], 1)
    u, w = torch.empty_like(x), torch.empty_like(a)
    src = x.T.contiguous()
    H = torch.cat([a, -m], 1).T.contiguous()
    step = max(1, block // n)
    for t0 in range(0, n, step):
        t1 = min(n, t0 + step)
        xt, at = x[t0:t1], a[t0:t1]
        d = src[0, t0:t1, None] - src[0, None, :]
        r2 = d * d
        for k in (1, 2):
            torch.sub(src[k, t0:t1, None], src[k, None, :], out=d)
            r2.addcmul_(d, d)
        i = torch.arange(t1 - t0, device=x.device)
        r2[i, t0 + i] = math.inf
        sig2 = 0.5 * (s2[t0:t1, None] + s2[None, :])
        q, F, Z = _kernel(r2, sig2, False)
        S6 = q @ A6
        S, M = S6[:, :3], S6[:, 3:]
        u[t0:t1] = torch.linalg.cross(S, xt) - M
        h = torch.cat([torch.linalg.cross(xt, at), at], 1) @ H
        g4 = (F * h) @ X4
        w[t0:t1] = torch.linalg.cross(at, S) + g4[:, :1] * xt - g4[:, 1:]
        if nu:
            c = (2.0 * nu) * Z / sig2
            c[i, t0 + i] = 0.0
            w[t0:t1] += vol[t0:t1, None] * (c @ a) - (c @ vol)[:, None] * at
    return u, w


def _tensors(s: W.ParticleSystem):
    dev = _device()
    return [torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in (s.pos, s.alpha, s.radius ** 2, s.volume)]


def _system_rates(s: W.ParticleSystem, x, a, s2, vol, highorder: bool, large: bool):
    parts = [(0, s.n)] if s.coupled else list(zip(s.off[:-1].tolist(), s.off[1:].tolist()))
    us, ws = [], []
    for p, e in parts:
        sl = slice(p, e)
        if large and not highorder and s.coupled:
            u, w = _far_rates(x[sl], a[sl], s2[sl], vol[sl], s.nu)
        else:
            u, w = _rates(x[sl], a[sl], s2[sl], vol[sl], s.nu, highorder)
        us.append(u)
        ws.append(w)
    return torch.cat(us), torch.cat(ws)


def _advance(f, x, a, scheme: str, dt: float):
    k1 = f(x, a)
    if scheme == "euler":
        return x + dt * k1[0], a + dt * k1[1]
    k2 = f(x + 0.5 * dt * k1[0], a + 0.5 * dt * k1[1])
    if scheme == "rk3":
        k3 = f(x - dt * k1[0] + 2.0 * dt * k2[0], a - dt * k1[1] + 2.0 * dt * k2[1])
        return tuple(y + dt / 6.0 * (p + 4.0 * q + r) for y, p, q, r in zip((x, a), k1, k2, k3))
    k3 = f(x + 0.5 * dt * k2[0], a + 0.5 * dt * k2[1])
    k4 = f(x + dt * k3[0], a + dt * k3[1])
    return tuple(y + dt / 6.0 * (p + 2.0 * q + 2.0 * r + t) for y, p, q, r, t in zip((x, a), k1, k2, k3, k4))


def _diagnosis(s: W.ParticleSystem, highorder: bool) -> torch.Tensor:
    x, a, s2, vol = _tensors(s)
    n = s.n
    out = torch.zeros(15 * s.nw if not s.coupled else 15 * max(1, s.nw), dtype=torch.float64, device=x.device)
    r = torch.linalg.cross(x, a)
    out[0:3] = a.sum(0)
    out[3:6] = 0.5 * r.sum(0)
    out[6:9] = torch.linalg.cross(x, r).sum(0) / 3.0
    pi = math.pi
    H = KE = KF = EN = EF = torch.zeros((), dtype=torch.float64, device=x.device)
    src, al = x.T.contiguous(), a.T.contiguous()
    step = max(1, (1 << 24) // n)
    for t0 in range(0, n, step):
        t1 = min(n, t0 + step)
        d = [src[k, None, :] - src[k, t0:t1, None] for k in range(3)]
        at = al[:, t0:t1, None]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        i = torch.arange(t1 - t0, device=x.device)
        off = torch.ones_like(r2)
        off[i, t0 + i] = 0.0
        sig2 = 0.5 * (s2[t0:t1, None] + s2[None, :])
        rq = r2.clone()
        rq[i, t0 + i] = math.inf
        q, _, _ = _kernel(rq, sig2, highorder, need_f=False)
        c = [at[1] * al[2] - at[2] * al[1], at[2] * al[0] - at[0] * al[2], at[0] * al[1] - at[1] * al[0]]
        H = H + (q * (d[0] * c[0] + d[1] * c[1] + d[2] * c[2])).sum()
        aa = at[0] * al[0] + at[1] * al[1] + at[2] * al[2]
        p1 = d[0] * at[0] + d[1] * at[1] + d[2] * at[2]
        p2 = d[0] * al[0] + d[1] * al[1] + d[2] * al[2]
        b = r2 + sig2
        b15 = b * b.sqrt()
        KE = KE + (off * ((r2 + 2.0 * sig2) * aa + p1 * p2) / b15).sum() / (16.0 * pi)
        KF = KF + (off * (r2 + 1.5 * sig2) * aa / b15).sum() / (8.0 * pi)
        if highorder:
            b35 = b15 * b * b
            f1 = (2.0 * r2 * r2 + 7.0 * sig2 * r2 + 20.0 * sig2 * sig2) / (8.0 * pi * b35)
            f2 = -(6.0 * r2 * r2 + 27.0 * sig2 * r2 + 21.0 * sig2 * sig2) / (8.0 * pi * b35 * b)
            EN = EN + (off * (f1 * aa + f2 * p1 * p2)).sum()
            EF = EF + (off * (15.0 / (8.0 * pi)) * sig2 * sig2 / b35 * aa).sum()
    sg, a2 = s2.sqrt(), (a * a).sum(1)
    KE = KE + (a2 / sg).sum() / (8.0 * pi)
    KF = KF + 3.0 * (a2 / sg).sum() / (16.0 * pi)
    if highorder:
        EN = EN + 2.5 / pi * (a2 / sg ** 3).sum()
        EF = EF + 1.875 / pi * (a2 / sg ** 3).sum()
    out[9], out[10], out[11], out[12], out[13] = H, EN, EF, KE, KF
    # the centroid of the last wake with any in-plane extent
    for w in range(s.nw):
        sl = slice(int(s.off[w]), int(s.off[w + 1]))
        oy, rr = a[sl].norm(dim=1), x[sl, 0] ** 2 + x[sl, 1] ** 2
        if float((oy * rr).sum()) != 0.0:
            out[14] = (oy * x[sl, 2] * rr).sum() / (oy * rr).sum()
    return out


def _point_velocity(s: W.ParticleSystem, pts: np.ndarray, highorder: bool) -> torch.Tensor:
    x, a, s2, _ = _tensors(s)
    p = torch.from_numpy(pts).to(x.device).T.contiguous()
    src, al = x.T.contiguous(), a.T.contiguous()
    out = torch.empty((pts.shape[0], 3), dtype=torch.float64, device=x.device)
    step = max(1, (1 << 24) // s.n)
    for t0 in range(0, pts.shape[0], step):
        d = [p[k, t0:t0 + step, None] - src[k, None, :] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        q, _, _ = _kernel(r2, s2[None, :].expand_as(r2), highorder, need_f=False)
        out[t0:t0 + step, 0] = (q * (al[1] * d[2] - al[2] * d[1])).sum(1)
        out[t0:t0 + step, 1] = (q * (al[2] * d[0] - al[0] * d[2])).sum(1)
        out[t0:t0 + step, 2] = (q * (al[0] * d[1] - al[1] * d[0])).sum(1)
    return out


def _network_gradient(case: dict, seed: int) -> dict:
    X, Y = _samples(case, seed)
    p = torch.from_numpy(_weights(seed)).double().requires_grad_(True)
    o, layers = 0, []
    for fan, units in ((16, 128), (128, 128), (128, 128), (128, 12)):
        layers.append((p[o:o + fan * units].view(fan, units), p[o + fan * units:o + fan * units + units]))
        o += fan * units + units
    h = torch.from_numpy(X).double()
    for i, (w, b) in enumerate(layers):
        h = h @ w + b
        if i < 3:
            z = math.sqrt(2.0 / math.pi) * (h + 0.044715 * h ** 3)
            h = h * torch.sigmoid(2.0 * z)
    loss = ((h - torch.from_numpy(Y).double()) ** 2).sum() / X.shape[0]
    loss.backward()
    return {"grad": p.grad, "loss": float(loss.detach())}


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "relax":
        return None
    if kind == "grad":
        return _network_gradient(case, seed)
    if kind == "tree":
        # the tree path's own error is far above any rounding: the direct sum,
        # for the analytic expansion (made-up weights approximate nothing)
        n = case["n"]
        if case["network"] or float(n) * n > EXACT_PAIRS:
            return None
        s = W.helix_wake(n, seed=seed)
        x, a, s2, vol = _tensors(s)
        return tuple(v.cpu() for v in _far_rates(x, a, s2, vol, s.nu))
    highorder = case["kernel"] == "highorder"
    s = _system(case, seed)
    if kind == "points":
        return _point_velocity(s, _points(case, seed), highorder).cpu()
    if kind == "diagnose":
        return _diagnosis(s, highorder).cpu()
    pairs = float(s.ordered_pairs())
    x, a, s2, vol = _tensors(s)
    if kind == "steps":
        f = lambda p, q: _system_rates(s, p, q, s2, vol, highorder, False)  # noqa: E731
        rhs = case["nsteps"] * {"euler": 1, "rk3": 3, "rk4": 4}[case["scheme"]]
        if rhs * pairs > 0.5 * EXACT_PAIRS:
            return None
        for _ in range(case["nsteps"]):
            x, a = _advance(f, x, a, case["scheme"], DTS[case["wake"]])
        return x.cpu(), a.cpu()
    single = case["precision"] == "fp32c"
    if pairs > (EXACT_PAIRS if single and not highorder and s.coupled else 0.5 * EXACT_PAIRS):
        return None
    u, w = _system_rates(s, x, a, s2, vol, highorder, single)
    return u.cpu(), w.cpu()
