"""The branch-free FP64 Gaussian core (pw_core64.h): G(s) = exp(-s/2) B(s)
from 64 degree-10 pieces on 0 <= s <= 90, and exp(-s/2) beside it.  The tables
compiled into the header are read from the source, compared with a fresh fit,
and evaluated step by step as the kernel does (each fused multiply-add rounded
once) against the series in 60-digit arithmetic: at the edges and centres of
the pieces, near s = 0 and over the whole range."""
import os
import re
import sys
from fractions import Fraction

import mpmath as mp
import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pawan_amd", "csrc")
sys.path.insert(0, CSRC)
import fit_core_table64 as F  # noqa: E402


def _source():
    return open(os.path.join(CSRC, "pw_core64.h")).read()


def _numbers(text):
    return [float.fromhex(v) for v in re.findall(r"-?0x[0-9a-f.]+p[+-]?\d+", text)]


def _tables():
    src = _source()
    exp = _numbers(re.search(r"kCore64Exp\[12\] = \{(.*?)\};", src, re.S).group(1))
    body = re.search(r"kCore64Table\[kCore64Pieces\]\[kCore64Row\] = \{(.*?)\n\};", src, re.S).group(1)
    rows = [_numbers(r) for r in re.findall(r"\{([^}]*)\}", body)]
    assert len(exp) == F.EXP_DEG + 1 and len(rows) == F.PIECES and all(len(r) == F.DEG + 2 for r in rows)
    return exp, rows


def test_tables_match_the_fit():
    exp, rows = _tables()
    assert exp == F.exp_coefficients()
    assert rows == F.table()


def test_core_against_its_series_in_high_precision():
    exp, rows = _tables()
    fma = lambda a, b, c: float(Fraction(a) * Fraction(b) + Fraction(c))  # noqa: E731
    w = 45.0 / 32.0
    edges = [k * w + d for k in range(F.PIECES + 1) for d in (-1e-9, 0.0, 1e-9)]
    centres = [(k + 0.5) * w for k in range(F.PIECES)]
    rng = np.random.default_rng(5)
    s_all = edges + centres + list(10.0 ** rng.uniform(-14, 0, 100)) + list(rng.uniform(0.0, 90.0, 800)) + [0.0, 90.0]
    worst_g = worst_e = 0.0
    for s in s_all:
        s = float(min(max(s, 0.0), 90.0))
        k = min(max(int(s * (32.0 / 45.0)), 0), F.PIECES - 1)
        t = fma(-w, k + 0.5, s)
        g = rows[k][F.DEG]
        for j in range(F.DEG - 1, -1, -1):
            g = fma(g, t, rows[k][j])
        x, p = -0.5 * t, exp[F.EXP_DEG]
        for j in range(F.EXP_DEG - 1, -1, -1):
            p = fma(p, x, exp[j])
        e = rows[k][F.DEG + 1] * p
        ref_g, ref_e = F.core_g(s), mp.exp(-mp.mpf(s) / 2)
        worst_g = max(worst_g, abs(float((g - ref_g) / ref_g)))
        worst_e = max(worst_e, abs(float((e - ref_e) / ref_e)))
    # a Horner step rounds once and its successors damp it (|c1 t / c0| < 0.5
    # on a piece): about two roundings of 2^-53 each for G, one more for e
    # (the product with the row's rounded exp(-s_c/2))
    assert worst_g < 3 * 2.0 ** -53 and worst_e < 4 * 2.0 ** -53, (worst_g, worst_e)
