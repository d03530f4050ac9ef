"""GPU parity: HIP kernels (through the C ABI) vs the FP64 CPU oracle on the
same reference-layout inputs.

Tolerance (stated by the task for the plain FP64 path): 1e-11 max-abs on every
J and K element.  The oracle applies the reference's per-component screening.
"""

import numpy as np
import pytest

import _util as U
import oracle
from vlxmi import configs
from vlxmi import pairs as P

TOL = 1e-11

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def dev():
    from vlxmi.runtime import Device
    return Device()


@pytest.fixture(scope="module")
def small8(dev):
    from vlxmi.fock import FockEngine
    mol, D = configs.make_small8()
    eng = FockEngine(mol, dev=dev)
    return mol, D, eng


def test_boys_device(dev):
    _say("case: device Boys function vs oracle, L=0..8")
    rng = np.random.default_rng(7)
    T = np.concatenate([rng.uniform(0, 45, 4000), [0.0, 1e-12, 0.025, 39.999, 40.0, 40.001, 120.0, 1e4]])
    for L in range(9):
        F = dev.boys_eval(T, L)
        ref = np.array([oracle.boys(L, t) for t in T])
        rel = np.max(np.abs(F - ref) / np.abs(ref))
        assert rel < 1e-14, (L, rel)
        if L <= 4:
            # the polynomial rows in LDS that the light-class kernels use
            Fc = dev.boys_eval(T, L, coarse=True)
            relc = np.max(np.abs(Fc - ref) / np.abs(ref))
            assert relc < 1e-14, (L, "coarse", relc)


def test_schwarz_device(small8):
    _say("case: small8 GPU Schwarz vs oracle")
    mol, D, eng = small8
    for pc, ps in eng.fl.pairsets.items():
        ta, tb = eng.fl.prims[ps.la], eng.fl.prims[ps.lb]
        Qo = oracle.schwarz(ps.la, ps.lb, ta.info, tb.info, ps.I, ps.J, ps.S)
        rel = np.max(np.abs(Qo - ps.Q) / np.maximum(np.abs(Qo), 1e-300))
        assert rel < 1e-12, (pc, rel)


def test_j_per_class_small8(small8):
    mol, D, eng = small8
    Dc_np = U.cart_density(mol, D)
    Dc = eng.cart_density(D)
    kets = eng.prepare_kets(Dc)
    for ab, cd in P.j_classes():
        if ab not in eng.jl or cd not in eng.jl:
            continue
        _say("case: small8 J class %s%s" % (ab, cd))
        g = eng.run_J(Dc, kets=kets, classes=[(ab, cd)])[ab].cpu().numpy()
        r = U.oracle_matJ(eng.fl, Dc_np, "component", classes=[(ab, cd)])[ab]
        assert np.max(np.abs(g - r)) <= TOL, (ab, cd, np.max(np.abs(g - r)))


def test_k_per_class_small8(small8):
    mol, D, eng = small8
    Dc_np = U.cart_density(mol, D)
    Dc = eng.cart_density(D)
    for cls in P.k_classes():
        a, b, c, d = cls
        if a + c not in eng.ik or a + b not in eng.kc or c + d not in eng.kc:
            continue
        _say("case: small8 K class %s" % cls)
        g = eng.run_K(Dc, classes=[cls])[a + c].cpu().numpy()
        r = U.oracle_matK(eng.fl, Dc_np, "component", classes=[cls])[a + c]
        assert np.max(np.abs(g - r)) <= TOL, (cls, np.max(np.abs(g - r)))


def test_fock_small8(small8):
    _say("case: small8 AO J/K + energies vs oracle and 4-index brute force")
    mol, D, eng = small8
    J, K = eng.build(D)
    J, K = J.cpu().numpy(), K.cpu().numpy()
    Dc = U.cart_density(mol, D)
    Jr, Kr = U.oracle_fock(eng.fl, Dc, "component")
    assert np.max(np.abs(J - Jr)) <= TOL
    assert np.max(np.abs(K - Kr)) <= TOL
    eri = oracle.ao_eri_tensor(mol)
    Jb, Kb = oracle.jk_from_tensor(eri, Dc)
    # the screened build differs from the unscreened tensor only by screened terms
    assert np.max(np.abs(J - Jb)) < 1e-9
    assert np.max(np.abs(K - Kb)) < 1e-9
    EJ, EK = eng.energies(D, eng.dev.tensor(J), eng.dev.tensor(K))
    assert abs(EJ - 0.5 * np.sum(D * Jr)) < 1e-9 and EJ > 0 and EK > 0


def test_k_density_order_contract(small8):
    """Exchange classes listed in k_dorder.json read D_jl as D[l][j]: with a
    non-symmetric density they give the oracle's K for D^T, the other classes
    the oracle's K for D (the engines symmetrise the density, so both agree
    there; this pins what a caller passing a non-symmetric D gets)."""
    from vlxmi.gen import build as B
    mol, D, eng = small8
    Dc = U.cart_density(mol, D)
    rng = np.random.default_rng(5)
    A = rng.normal(size=Dc.shape) * 1e-3
    Dn = Dc + (A - A.T)
    Dt = eng.dev.tensor(np.ascontiguousarray(Dn))
    lj = B.load_layouts(B.DORDER_TABLE)
    kinds = set()
    mx = float(np.abs(Dn).max())
    for cls in ("spss", "spsp", "sppp", "pppp", "pspp"):
        a, b, c, d = cls
        _say("case: small8 K class %s, non-symmetric density (%s)" % (cls, "D[l][j]" if cls in lj else "D[j][l]"))
        g = eng.run_K(Dt, classes=[cls], maxD={b + d: mx})[a + c].cpu().numpy()
        read, other = (Dn.T, Dn) if cls in lj else (Dn, Dn.T)
        r = U.oracle_matK(eng.fl, np.ascontiguousarray(read), "component", classes=[cls], max_D=mx)[a + c]
        r2 = U.oracle_matK(eng.fl, np.ascontiguousarray(other), "component", classes=[cls], max_D=mx)[a + c]
        assert np.max(np.abs(g - r)) <= TOL, (cls, np.max(np.abs(g - r)))
        assert np.max(np.abs(g - r2)) > 1e3 * TOL, cls          # the read order is observable
        kinds.add(cls in lj)
    assert kinds == {True, False}
