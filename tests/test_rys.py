"""Rys quadrature: the tables against moments of the weight function, and the
generated one-dimensional integrals (values and gradient sums), evaluated in
Python, against the oracle for every class."""

import math

import numpy as np
import pytest

import oracle
from vlxmi.gen import emit, rys
from vlxmi.gen.osdag import tri
from vlxmi.gen.rysdag import RysPoint

CLASSES = [(la, lb, lc, ld) for la in range(3) for lb in range(3) for lc in range(3) for ld in range(3)]
IDS = ["".join("spd"[x] for x in c) for c in CLASSES]


@pytest.mark.parametrize("n", range(1, rys.NMAX + 1))
def test_table_moments(n):
    """sum_i w_i u_i^m = F_m(T), m < 2n, at interval ends, centres, both sides
    of the table's end and far above it.  Roots and weights carry a relative
    error of a few 1e-16 (weights: of F_0), the m-th power m times that; the
    rule at T >= 64 leaves out less than 1e-16."""
    T = np.array([0.0, 1e-12, 0.1, 0.125, np.nextafter(0.25, 0), 0.25, 7.3, 31.999, 40.0, np.nextafter(64.0, 0), 64.0,
                  64.1, 100.0, 5e3, 1e6])
    u, w = rys.evaluate(n, T)
    for k, t in enumerate(T):
        F = oracle.boys(2 * n - 1, t)
        for m in range(2 * n):
            assert abs(np.sum(w[k] * u[k] ** m) - F[m]) <= 4e-15 * (m + 1) * F[m] + 1e-17 * F[0], (t, m)


def _setup(cls, seed, extra=0):
    rng = np.random.default_rng(seed + sum(v * 3 ** i for i, v in enumerate(cls)))
    A, B, C, D = rng.uniform(-2, 2, (4, 3))
    a, b, c, d = np.exp(rng.uniform(math.log(0.1), math.log(20), 4))
    z, e = a + b, c + d
    S4, P, Q = z + e, (a * A + b * B) / z, (c * C + d * D) / e
    PQ, rho = Q - P, z * e / S4
    env = {"double": float, "h1": 0.5 / z, "h2": 0.5 / e, "h4": 0.5 / S4, "rz": e / S4, "re": z / S4,
           "two_ai": 2 * a, "two_aj": 2 * b, "two_ak": 2 * c}
    for i, x in enumerate("xyz"):
        env.update({"gPA_" + x: b / z * (B[i] - A[i]), "gQC_" + x: d / e * (D[i] - C[i]), "WP_" + x: e / S4 * PQ[i],
                    "WQ_" + x: -z / S4 * PQ[i], "gAB_" + x: A[i] - B[i], "gCD_" + x: C[i] - D[i]})
    n = rys.nroots(sum(cls) + extra)
    u, w = rys.evaluate(n, np.array([rho * PQ @ PQ]))
    return env, u[0], w[0] * math.sqrt(4 * rho / math.pi), (a, A, b, B, c, C, d, D)


def _run(lines, env, u, w):
    code = "\n".join(x.replace("const double ", "").replace("double ", "").rstrip(";") for x in lines)
    for ru, rw in zip(u, w):
        env.update(ru=ru, rw=rw)
        exec(code, env)


@pytest.mark.parametrize("cls", CLASSES, ids=IDS)
def test_points_match_oracle(cls):
    """Bar: that of the recursion's own check (test_generator)."""
    env, u, w, geo = _setup(cls, 3)
    pt, shape = RysPoint(), [(l + 1) * (l + 2) // 2 for l in cls]
    env["X"] = np.zeros(shape)
    for k in np.ndindex(*shape):
        pt.lines.append("X[%d,%d,%d,%d] += %s;" % (k + (pt.component(*[tri(cls[i])[k[i]] for i in range(4)]),)))
    _run(pt.lines, env, u, w)
    ref = oracle.eri_block(*cls, *geo)
    assert np.abs(env["X"] - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("cls", [c for c in CLASSES if sum(c) in (0, 1, 3, 4, 6, 8)],
                         ids=lambda c: "".join("spd"[x] for x in c))
def test_gradient_terms_match_oracle(cls):
    """The weighted sums over components of the A-, B- and C-centre derivatives."""
    env, u, w, geo = _setup(cls, 11, extra=1)
    shape = [(l + 1) * (l + 2) // 2 for l in cls]
    W = np.random.default_rng(5).normal(size=shape)
    pt, comps = RysPoint(), []
    for k in np.ndindex(*shape):
        name = "W%d_%d_%d_%d" % k
        env[name] = W[k]
        comps.append((name,) + tuple(tri(cls[i])[k[i]] for i in range(4)))
    pt.gradient_terms(comps, [(0, "two_ai", 0), (1, "two_aj", 3), (2, "two_ak", 6)], "gacc")
    env["gacc"] = np.zeros(9)
    _run(pt.lines, env, u, w)
    for centre in range(3):
        for g in range(3):
            d = oracle.eri_deriv_block(centre, *cls, *geo)[g]
            assert abs(env["gacc"][3 * centre + g] - np.sum(W * d)) <= 1e-11 * np.sum(np.abs(W * d)) + 1e-14, (centre, g)


@pytest.mark.parametrize("nab,nc,nd,maxx", [(1, 1, 1, 9), (18, 6, 6, 54), (36, 6, 6, 18), (6, 3, 6, 36), (9, 6, 3, 72), (3, 3, 1, 1)])
def test_passes_cover_every_ket_pair_once(nab, nc, nd, maxx):
    groups = emit.rys_groups(nab, nc, nd, maxx)
    flat = [p for g in groups for p in g]
    assert sorted(flat) == [(i, j) for i in range(nc) for j in range(nd)]
    assert len({len(g) for g in groups}) == 1
    assert len(groups[0]) * nab <= max(maxx, nab)
