"""Straight-line code of one Rys quadrature point.

(ab|cd) = sum_i w_i Ix(u_i) Iy(u_i) Iz(u_i): each direction needs only the
one-dimensional integrals I(i, j, k, l), i <= la, ..., so a point's values are
few however large the class, where the Head-Gordon-Pople recursion of
``osdag`` holds a table of three-dimensional intermediates.

One-dimensional recursion (Rys, Dupuis & King, J. Comput. Chem. 4, 154 (1983)),
with u = t^2 and the prefactors of ``osdag`` (PQ = Q - P):
  G(n+1, 0) = (PA + u WP) G(n, 0) + n B10 G(n-1, 0)
  G(n, m+1) = (QC + u WQ) G(n, m) + m B01 G(n, m-1) + n B00 G(n-1, m)
  B10 = (1 - u rho/zeta) / (2 zeta), B01 = (1 - u rho/eta) / (2 eta), B00 = u / (2 (zeta + eta))
and the horizontal recursions of eri.py:177-235 applied per direction:
  I(i, j+1, ..) = I(i+1, j, ..) + AB I(i, j, ..),  I(.., k, l+1) = I(.., k+1, l) + CD I(.., k, l).
G(0, 0) is 1 for x and y and the weight times the prefactor for z.

Expected in scope: ``ru`` (u_i), ``rw`` (w_i Lambda), gPA_*, gQC_*, WP_*, WQ_*,
gAB_*, gCD_*, h1, h2, h4, rz, re as in ``emit.quartet_prologue``.
"""

from __future__ import annotations

AX = "xyz"


class RysPoint:
    """Emits the one-dimensional integrals of one quadrature point on demand."""

    def __init__(self, prefix="g", ty="double"):
        self.prefix = prefix
        self.ty = ty
        self.lines = []
        self.memo = {}
        self.nflop = 0

    def _new(self, key, expr, flops=0):
        name = "%s%d" % (self.prefix, len(self.memo))
        self.memo[key] = name
        self.lines.append("const %s %s = %s;" % (self.ty, name, expr))
        self.nflop += flops
        return name

    def _coef(self, name):
        """C_x.., D_x.., B10, B01, B00 of this point and their small multiples."""
        key = ("coef",) + name
        if key in self.memo:
            return self.memo[key]
        kind, arg = name
        if kind == "C":
            return self._new(key, "gPA_%s + ru * WP_%s" % (arg, arg), 2)
        if kind == "D":
            return self._new(key, "gQC_%s + ru * WQ_%s" % (arg, arg), 2)
        if arg == 1:
            expr = {"B10": "h1 - ru * (h1 * rz)", "B01": "h2 - ru * (h2 * re)", "B00": "ru * h4"}[kind]
            return self._new(key, expr, 2)
        return self._new(key, "%d.0 * %s" % (arg, self._coef((kind, 1))), 1)

    @staticmethod
    def _mul(c, v):
        return c if v is None else "%s * %s" % (c, v)

    # values are names, or None for the constant 1 (x and y at order zero)
    def G(self, g, n, m):
        key = ("G", g, n, m)
        if key in self.memo:
            return self.memo[key]
        if n == 0 and m == 0:
            self.memo[key] = "rw" if g == 2 else None
            return self.memo[key]
        if m > 0:
            t = [self._mul(self._coef(("D", AX[g])), self.G(g, n, m - 1))]
            if m > 1:
                t.append(self._mul(self._coef(("B01", m - 1)), self.G(g, n, m - 2)))
            if n > 0:
                t.append(self._mul(self._coef(("B00", n)), self.G(g, n - 1, m - 1)))
        else:
            t = [self._mul(self._coef(("C", AX[g])), self.G(g, n - 1, 0))]
            if n > 1:
                t.append(self._mul(self._coef(("B10", n - 1)), self.G(g, n - 2, 0)))
        if len(t) == 1 and "*" not in t[0]:
            self.memo[key] = t[0]
            return t[0]
        return self._new(key, " + ".join(t), 2 * len(t) - 1)

    def _shift(self, key, up, fac, low):
        one = "%s(1)" % self.ty
        return self._new(key, "%s + %s" % (one if up is None else up, self._mul(fac, low)), 2)

    def W(self, g, n, k, l):
        """(n | k l) by the ket horizontal recursion."""
        key = ("W", g, n, k, l)
        if key not in self.memo:
            if l == 0:
                self.memo[key] = self.G(g, n, k)
            else:
                self._shift(key, self.W(g, n, k + 1, l - 1), "gCD_" + AX[g], self.W(g, n, k, l - 1))
        return self.memo[key]

    def I(self, g, i, j, k, l):
        """(i j | k l) by the bra horizontal recursion."""
        key = ("I", g, i, j, k, l)
        if key not in self.memo:
            if j == 0:
                self.memo[key] = self.W(g, i, k, l)
            else:
                self._shift(key, self.I(g, i + 1, j - 1, k, l), "gAB_" + AX[g], self.I(g, i, j - 1, k, l))
        return self.memo[key]

    def component(self, a, b, c, d):
        """Expression Ix Iy Iz of one component quartet."""
        f = [self.I(g, a[g], b[g], c[g], d[g]) for g in range(3)]
        f = [x for x in f if x is not None]
        return " * ".join(f) if f else "%s(1)" % self.ty

    # ---------------------------------------------------------------- gradients
    def dI(self, g, t, pos, two_exp):
        """Derivative of I(g, *t) with respect to the centre of index ``pos``:
        2 alpha I(.. r+1 ..) - r I(.. r-1 ..)."""
        key = ("dI", g, t, pos)
        if key in self.memo:
            return self.memo[key]
        up, dn = list(t), list(t)
        up[pos] += 1
        e = self._mul(two_exp, self.I(g, *up))
        if t[pos]:
            dn[pos] -= 1
            low = self.I(g, *dn)
            low = "%s(1)" % self.ty if low is None else low
            e += " - " + (low if t[pos] == 1 else "%d.0 * %s" % (t[pos], low))
        return self._new(key, e, 1 + 2 * (t[pos] > 0))

    def gradient_terms(self, weighted, cents, acc):
        """Lines adding this point's share of sum_q W_q d(Ix Iy Iz)_q to the
        accumulators: the weights and the two other directions are summed per
        one-dimensional index first (V), so a component costs five operations
        whatever the number of centres.  ``weighted``: [(W name, a, b, c, d)];
        ``cents``: [(index position, 2 x exponent, first accumulator)]."""
        V = [{}, {}, {}]

        def put(g, t, expr):
            if t in V[g]:
                self.lines.append("%s += %s;" % (V[g][t], expr))
            else:
                V[g][t] = "%sV%d_%d" % (self.prefix, g, len(V[g]))
                self.lines.append("%s %s = %s;" % (self.ty, V[g][t], expr))

        for n, (w, a, b, c, d) in enumerate(weighted):
            t = [(a[g], b[g], c[g], d[g]) for g in range(3)]
            x, y, z = [self.I(g, *t[g]) for g in range(3)]
            wz = self._new(("wz", n), self._mul(w, z))
            wx = w if x is None else self._new(("wx", n), self._mul(w, x))
            put(0, t[0], self._mul(wz, y))
            put(1, t[1], self._mul(wz, x))
            put(2, t[2], self._mul(wx, y))
        for g in range(3):
            for t, v in V[g].items():
                for pos, two, first in cents:
                    self.lines.append("%s[%d] += %s * %s;" % (acc, first + g, self.dI(g, t, pos, two), v))
