"""Rys quadrature tables: roots and weights as piecewise polynomials of T.

The n-point rule integrates t^2-polynomials of degree < 2n exactly,

  int_0^1 p(t^2) exp(-T t^2) dt = sum_i w_i(T) p(u_i(T)),

(Dupuis, Rys & King, J. Chem. Phys. 65, 111 (1976)); u_i are the zeros of the
degree-n polynomial orthogonal on [0, 1] for the weight exp(-T t^2) dt in t^2.
``roots_weights`` builds the rule with the discretised Stieltjes procedure
(Gautschi) over a Gauss-Legendre grid in extended precision; ``table`` turns
u_i(T) and w_i(T) into one polynomial of degree NCOEF - 1 per interval of width
WIDTH on [0, TMAX): Chebyshev interpolation in extended precision, re-expanded
in powers of the local variable x in [-1, 1] and rounded to FP64.  For
T >= TMAX the upper limit of the integral is infinite to FP64 precision (the
part beyond t = 1 is below 1e-16 of the smallest moment an n = 5 rule uses), so
u_i = h_i / T and w_i = W_i / sqrt(T) from the half-range Gauss-Hermite rule.
"""

from __future__ import annotations

import functools
import math

import numpy as np

LD = np.longdouble
WIDTH = 0.25
TMAX = 64.0
NROW = int(TMAX / WIDTH)
NCOEF = 8
NMAX = 5


def nroots(L: int) -> int:
    """Points that integrate the t^2-polynomial of total angular momentum L."""
    return L // 2 + 1


def _gauss_legendre(n):
    """Nodes and weights on [0, 1] in extended precision."""
    x = np.polynomial.legendre.leggauss(n)[0].astype(LD)
    for _ in range(3):
        p0, p1 = np.ones_like(x), x.copy()
        for k in range(2, n + 1):
            p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
        dp = n * (x * p1 - p0) / (x * x - 1)
        x = x - p1 / dp
    p0, p1 = np.ones_like(x), x.copy()
    for k in range(2, n + 1):
        p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
    dp = n * (x * p1 - p0) / (x * x - 1)
    return (x + 1) / 2, 1 / ((1 - x * x) * dp * dp)


def _stieltjes(x, w, n):
    """Recursion coefficients and norms of the monic polynomials orthogonal for
    the discrete measure w (last axis) at x, batched over the leading axis."""
    p0 = np.zeros_like(w)
    p1 = np.ones_like(w)
    alpha, beta, norm = [], [], []
    prev = None
    for k in range(n):
        nk = (w * p1 * p1).sum(-1)
        ak = (w * x * p1 * p1).sum(-1) / nk
        bk = np.zeros_like(nk) if prev is None else nk / prev
        alpha.append(ak)
        beta.append(bk)
        norm.append(nk)
        p0, p1 = p1, (x - ak[..., None]) * p1 - bk[..., None] * p0
        prev = nk
    return alpha, beta, norm


def _rule(alpha, beta, norm):
    """Roots and weights (batch, n) from the recursion coefficients."""
    n = len(alpha)
    m = alpha[0].shape[0]
    Jm = np.zeros((m, n, n))
    for k in range(n):
        Jm[:, k, k] = alpha[k].astype(np.float64)
        if k:
            Jm[:, k, k - 1] = Jm[:, k - 1, k] = np.sqrt(beta[k].astype(np.float64))
    u = np.linalg.eigvalsh(Jm).astype(LD)

    def values(u):
        q0, q1 = np.zeros_like(u), np.ones_like(u)
        d0, d1 = np.zeros_like(u), np.zeros_like(u)
        for k in range(n):
            a, b = alpha[k][:, None], beta[k][:, None]
            q0, q1, d0, d1 = q1, (u - a) * q1 - b * q0, d1, q1 + (u - a) * d1 - b * d0
        return q0, q1, d1                      # p_{n-1}, p_n, p_n'

    for _ in range(3):
        _, pn, dn = values(u)
        u = u - pn / dn
    pm, _, dn = values(u)
    return u, norm[-1][:, None] / (dn * pm)


def roots_weights(n, T):
    """u (len(T), n) ascending and w (len(T), n) for an array of T >= 0."""
    T = np.asarray(T, dtype=LD)
    t, g = _gauss_legendre(64)
    x = t * t
    return _rule(*_stieltjes(x, g * np.exp(-T[:, None] * x), n))


@functools.lru_cache(None)
def asymptotic(n):
    """h_i, W_i with u_i = h_i / T and w_i = W_i / sqrt(T) for T >= TMAX: the
    positive half of the 2n-point Gauss-Hermite rule (h_i the squared nodes),
    from int_0^inf exp(-T t^2) p(t^2) dt."""
    h = np.sort(np.polynomial.hermite.hermgauss(2 * n)[0])[n:].astype(LD)

    def herm(x):
        p0, p1 = np.ones_like(x), 2 * x
        for k in range(1, 2 * n):
            p0, p1 = p1, 2 * x * p1 - 2 * k * p0
        return p0, p1                          # H_{2n-1}, H_{2n}

    for _ in range(3):
        a, b = herm(h)
        h = h - b / (4 * n * a)
    a, _ = herm(h)
    w = LD(2) ** (2 * n - 1) * math.factorial(2 * n) * np.sqrt(LD(math.pi) + LD(1.2246467991473532e-16)) / ((2 * n) ** 2 * a * a)
    return h * h, w


@functools.lru_cache(None)
def table(n):
    """(NROW, 2n, NCOEF) FP64: per interval the polynomials of u_0..u_{n-1},
    then w_0..w_{n-1}, coefficients ascending in x = (T - centre) * 2 / WIDTH."""
    m = NCOEF
    th = (np.arange(m, dtype=LD) + LD(0.5)) * (LD(math.pi) + LD(1.2246467991473532e-16)) / m
    node = np.cos(th)
    centre = (np.arange(NROW, dtype=LD) + LD(0.5)) * LD(WIDTH)
    T = centre[:, None] + node[None, :] * LD(WIDTH) / 2
    u, w = roots_weights(n, T.ravel())
    f = np.concatenate([u, w], axis=1).reshape(NROW, m, 2 * n)
    cheb = np.stack([(2 if k else 1) / LD(m) * (f * np.cos(k * th)[None, :, None]).sum(1) for k in range(m)], axis=2)
    poly = np.zeros_like(cheb)
    t0, t1 = np.zeros(m, LD), np.zeros(m, LD)
    t0[0], t1[1] = 1, 1
    for k in range(m):
        tk = t0 if k == 0 else t1
        if k > 1:
            tk = 2 * np.concatenate([[LD(0)], t1[:-1]]) - t0
            t0, t1 = t1, tk
        poly += cheb[..., k:k + 1] * tk
    return poly.astype(np.float64)


def evaluate(n, T):
    """The kernels' evaluation of the rule in FP64 (NumPy)."""
    T = np.asarray(T, dtype=np.float64)
    k = np.minimum((T * (1.0 / WIDTH)).astype(np.int64), NROW - 1)
    x = T * (2.0 / WIDTH) - (2.0 * k + 1.0)
    c = table(n)[k]
    s = c[..., NCOEF - 1]
    for j in range(NCOEF - 2, -1, -1):
        s = s * x[:, None] + c[..., j]
    h, W = [v.astype(np.float64) for v in asymptotic(n)]
    big = T >= TMAX
    s[big, :n] = h / T[big, None]
    s[big, n:] = W / np.sqrt(T[big, None])
    return s[:, :n], s[:, n:]


def header_text(n):
    """C++ text of the table of the n-point rule (device constants)."""
    t = table(n)
    h, W = [v.astype(np.float64) for v in asymptotic(n)]
    o = ["// Generated by vlxmi.gen.rys: %d-point Rys rule, [row][u_0..u_%d, w_0..w_%d][coefficient], intervals of %g on [0, %g)."
         % (n, n - 1, n - 1, WIDTH, TMAX),
         "#pragma once",
         "namespace vlxmi {",
         "__device__ const double rys_table_%d[%d * %d * %d] __attribute__((aligned(64))) = {" % (n, NROW, 2 * n, NCOEF)]
    for row in t:
        for f in row:
            o.append(", ".join(float(v).hex() for v in f) + ",")
    o += ["};",
          "__device__ constexpr double rys_large_%d[%d] = {%s};" % (n, 2 * n, ", ".join(float(v).hex() for v in list(h) + list(W))),
          "}  // namespace vlxmi", ""]
    return "\n".join(o)
