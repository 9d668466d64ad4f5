"""Table and exponential of the FP64 Gaussian core (pw_core64.h): the function
    G(s) = exp(-s/2) B(s),  B(s) = sum_k s^k / (2k+5)!!,  s = rho^2/sigma^2,
on 0 <= s <= 90, from which the FP64 kernels form
    q sigma^3 = K (exp(-s/2)/3 + s G),   F sigma^5 = -3 K G,   K = (2 pi)^-3/2
(the incomplete-gamma series of erf, A&S 6.5.29, with exp(-s/2) factored:
every term positive, so q and F lose no digits as rho -> 0).

The range is cut into 64 pieces of width 45/32 (64 x 45/32 = 90, and every
piece's centre s_c = (k + 1/2) 45/32, is exact in FP64).  A row is
(c0 .. c10, exp(-s_c/2)): G as a degree-10 polynomial in t = s - s_c, and
exp(-s/2) = exp(-s_c/2) p(-t/2) with p a degree-11 fit of exp on
|x| <= 45/128.  Both fits interpolate at Chebyshev nodes in 60-digit
arithmetic and are rounded to FP64 last.

    python pawan_amd/csrc/fit_core_table64.py    (prints both tables)
"""
import mpmath as mp

PIECES = 64
DEG = 10
EXP_DEG = 11
WIDTH_NUM, WIDTH_DEN = 45, 32
mp.mp.dps = 60


def core_g(s):
    """G(s) by its series (positive terms) in the current precision."""
    s = mp.mpf(s)
    acc, term, k = mp.mpf(0), mp.mpf(1) / 15, 0
    while term > acc * mp.mpf(10) ** -55 or k < 4:
        acc += term
        term = term * s / (2 * k + 7)
        k += 1
    return mp.exp(-s / 2) * acc


def _fit(f, half, deg):
    """Monomial coefficients of the interpolant of f at the Chebyshev nodes of
    |t| <= half."""
    n = deg + 1
    nodes = [half * mp.cos(mp.pi * (2 * i + 1) / (2 * n)) for i in range(n)]
    vals = [f(t) for t in nodes]
    c = []
    for j in range(n):
        v = sum(vals[i] * mp.cos(mp.pi * j * (2 * i + 1) / (2 * n)) for i in range(n)) * 2 / n
        c.append(v / 2 if j == 0 else v)
    # Chebyshev to monomial in x = t / half
    tm, tp = [mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]
    out = [mp.mpf(0)] * n
    for j in range(n):
        poly = tm if j == 0 else tp
        for m, v in enumerate(poly):
            out[m] += c[j] * v
        if j >= 1:
            nx = [mp.mpf(0)] + [2 * v for v in tp]
            for m, v in enumerate(tm):
                nx[m] -= v
            tm, tp = tp, nx
    return [float(v / half ** m) for m, v in enumerate(out)]


def table() -> list[list[float]]:
    w = mp.mpf(WIDTH_NUM) / WIDTH_DEN
    rows = []
    for k in range(PIECES):
        sc = (k + mp.mpf(1) / 2) * w
        rows.append(_fit(lambda t: core_g(sc + t), w / 2, DEG) + [float(mp.exp(-sc / 2))])
    return rows


def exp_coefficients() -> list[float]:
    """p(x) ~ exp(x) on |x| <= 45/128."""
    return _fit(mp.exp, mp.mpf(WIDTH_NUM) / (4 * WIDTH_DEN), EXP_DEG)


if __name__ == "__main__":
    print("exp:", ", ".join(v.hex() for v in exp_coefficients()))
    for r in table():
        print("    {" + ", ".join(v.hex() for v in r) + "},")
