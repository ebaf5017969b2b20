"""Generate rys_table.inc: piecewise polynomial fits of Rys roots and weights.

The n-point Rys rule for the weight exp(-T x) / (2 sqrt(x)) on x = t^2 in [0, 1]
has moments mu_k = F_k(T) (Boys function).  For each n = 1..NMAX the exact nodes
x_i(T) and weights w_i(T) are computed in 50-digit arithmetic (Golub-Welsch from
the Hankel moment matrix), then fitted per interval [T_k, T_k + h_k) of T by a
polynomial of degree D(n) in the local variable s = 2 (T - T_k)/h_k - 1 (truncated
Chebyshev series of the exact values, converted to monomials in the same arithmetic).
The functions flatten as T grows, so the intervals widen with it: they are those of
T + T0(n) that share an exponent and the leading B(n) bits of the mantissa, which the
device reads from the number's bits.  FITS holds (T0, B, D), chosen so that every fit
is good to 1e-15 relative.
Above T_max(n) the large-T limit is used: x_i = s_i^2 / T, w_i = W_i / sqrt(T)
with s_i, W_i the positive nodes / weights of the 2n-point Gauss-Hermite rule
(the truncation of the weight at t = 1 is below 1e-16 relative there).

Output layout (double): for n, interval k: [x_0..x_{n-1} coeffs (D+1 each),
w_0..w_{n-1} coeffs (D+1 each), 2 unused], coefficient 0 = constant term.  The two
unused words make the interval stride an odd multiple of 16 bytes (n <= 3), so the
intervals start in all LDS banks.

    python iqcp_amd/csrc/gen_rys_table.py          # writes rys_table.inc next to this file
"""
from __future__ import annotations

import multiprocessing
import sys
from pathlib import Path

import mpmath as mp
import numpy as np

NMAX = 7
H = 2.0           # step of the search for T_max
FITS = {1: (8, 4, 9), 2: (8, 4, 9), 3: (4, 3, 11), 4: (8, 4, 11), 5: (8, 4, 11), 6: (8, 4, 11), 7: (8, 4, 11)}
NODES = 24        # Chebyshev sample nodes per interval
PAD = 2           # unused words per interval
mp.mp.dps = 50


def boys_mp(m, T):
    T = mp.mpf(T)
    if T == 0:
        return mp.mpf(1) / (2 * m + 1)
    return mp.gammainc(m + mp.mpf("0.5"), 0, T) / (2 * T ** (m + mp.mpf("0.5")))


def rys_exact(n, T):
    """Exact (50-digit) Rys nodes x_i = t_i^2 and weights, ascending nodes."""
    mom = [boys_mp(k, T) for k in range(2 * n + 1)]
    M = mp.matrix(n + 1, n + 1)
    for i in range(n + 1):
        for j in range(n + 1):
            M[i, j] = mom[i + j]
    R = mp.cholesky(M).T  # upper: M = R^T R
    alpha = []
    beta = []
    for k in range(n):
        a = R[k, k + 1] / R[k, k] - (R[k - 1, k] / R[k - 1, k - 1] if k > 0 else 0)
        alpha.append(a)
        if k < n - 1:
            beta.append(R[k + 1, k + 1] / R[k, k])
    J = mp.matrix(n, n)
    for k in range(n):
        J[k, k] = alpha[k]
        if k < n - 1:
            J[k, k + 1] = beta[k]
            J[k + 1, k] = beta[k]
    E, Q = mp.eigsy(J)
    order = sorted(range(n), key=lambda i: E[i])
    x = [E[i] for i in order]
    w = [mom[0] * Q[0, i] ** 2 for i in order]
    return x, w


def hermite_half(n):
    """Positive nodes squared and weights of the 2n-point Gauss-Hermite rule."""
    s, W = np.polynomial.hermite.hermgauss(2 * n)
    # refine in mpmath via Newton on H_{2n}
    xs, ws = [], []
    for si, wi in zip(s, W):
        if si <= 0:
            continue
        x = mp.mpf(si)
        for _ in range(8):
            h = mp.hermite(2 * n, x)
            dh = 4 * n * mp.hermite(2 * n - 1, x)
            x = x - h / dh
        w = (2 ** (2 * n - 1) * mp.factorial(2 * n) * mp.sqrt(mp.pi)) / ((2 * n) ** 2 * mp.hermite(2 * n - 1, x) ** 2)
        xs.append(x * x)
        ws.append(w)
    order = sorted(range(n), key=lambda i: xs[i])
    return [xs[i] for i in order], [ws[i] for i in order]


def tmax_for(n):
    """Smallest multiple of H where the large-T limit is accurate to < 2e-16 relative."""
    hx, hw = hermite_half(n)
    T = 10.0
    while True:
        x, w = rys_exact(n, T)
        err = max(max(abs((hx[i] / T - x[i]) / x[i]) for i in range(n)),
                  max(abs((hw[i] / mp.sqrt(T) - w[i]) / w[i]) for i in range(n)))
        if err < 2e-16:
            return T
        T += H


def intervals(n, tmax):
    """(T_k, h_k) of the fits, up to the one that holds tmax."""
    T0, bits, _ = FITS[n]
    out = []
    lo = float(T0)
    while lo <= tmax + T0:
        h = 2.0 ** (int(np.floor(np.log2(lo))) - bits)
        out.append((lo - T0, h))
        lo += h
    return out


def fit_interval(job):
    n, T0, h = job
    mp.mp.dps = 50
    deg = FITS[n][2]
    th = [mp.pi * (k + mp.mpf(1) / 2) / NODES for k in range(NODES)]
    vals = []
    for t in th:
        x, w = rys_exact(n, T0 + (mp.cos(t) + 1) * h / 2)
        vals.append(list(x) + list(w))
    cheb = [[mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]]  # Chebyshev polynomials in monomials
    while len(cheb) <= deg:
        p = [mp.mpf(0)] + [2 * v for v in cheb[-1]]
        for q, v in enumerate(cheb[-2]):
            p[q] -= v
        cheb.append(p)
    out = []
    for i in range(2 * n):
        m = [mp.mpf(0)] * (deg + 1)
        for j in range(deg + 1):
            c = (1 if j == 0 else 2) * sum(vals[k][i] * mp.cos(j * th[k]) for k in range(NODES)) / NODES
            for q, v in enumerate(cheb[j]):
                m[q] += c * v
        out += [float(v) for v in m]
    return out + [0.0] * PAD


def main():
    out = Path(__file__).with_name("rys_table.inc")
    tmax = {}
    jobs = []
    offsets = []
    nint = {}
    herm = {}
    total = 0
    for n in range(1, NMAX + 1):
        tmax[n] = tmax_for(n)
        iv = intervals(n, tmax[n])
        nint[n] = len(iv)
        offsets.append(total)
        jobs += [(n, t, h) for t, h in iv]
        total += len(iv) * (2 * n * (FITS[n][2] + 1) + PAD)
        herm[n] = hermite_half(n)
        print(f"n={n} tmax={tmax[n]} intervals={nint[n]}", file=sys.stderr)
    with multiprocessing.Pool() as pool:
        flat = np.concatenate(pool.map(fit_interval, jobs, chunksize=1))
    ns = range(1, NMAX + 1)

    def table(ctype, name, values):
        return f"constexpr {ctype} {name}[QCG_RYS_NMAX + 1] = {{0, " + ", ".join(str(v) for v in values) + "};"

    lines = ["// Generated by gen_rys_table.py: piecewise fits of Rys nodes/weights (see generator docstring).",
             f"#define QCG_RYS_NMAX {NMAX}",
             f"#define QCG_RYS_PAD {PAD}",
             table("int", "qcg_rys_deg", [FITS[n][2] for n in ns]),
             table("int", "qcg_rys_log2t0", [int(np.log2(FITS[n][0])) for n in ns]),
             table("int", "qcg_rys_bits", [FITS[n][1] for n in ns]),
             table("int", "qcg_rys_nint", [nint[n] for n in ns]),
             table("int", "qcg_rys_off", offsets),
             table("double", "qcg_rys_tmax", [tmax[n] for n in ns])]
    hx = []
    hw = []
    for n in range(1, NMAX + 1):
        hx += [mp.nstr(v, 25) for v in herm[n][0]]
        hw += [mp.nstr(v, 25) for v in herm[n][1]]
    lines.append("// large-T limit: x_i = qcg_rys_hx[tri(n)+i] / T, w_i = qcg_rys_hw[tri(n)+i] / sqrt(T); tri(n) = n(n-1)/2")
    lines.append("constexpr double qcg_rys_hx[] = {" + ", ".join(hx) + "};")
    lines.append("constexpr double qcg_rys_hw[] = {" + ", ".join(hw) + "};")
    lines.append(f"constexpr double qcg_rys_coef[{len(flat)}] = {{")
    for i in range(0, len(flat), 4):
        lines.append("  " + ", ".join(f"{v:.17e}" for v in flat[i:i + 4]) + ",")
    lines.append("};")
    out.write_text("\n".join(lines) + "\n")
    print("wrote", out, len(flat), "coefficients", file=sys.stderr)


if __name__ == "__main__":
    main()
