"""A term that the screen |Q Q D| > threshold does not pass adds nothing, whatever
its value: a NaN compares false, and an infinity passes only against a finite
threshold.  Classes of every digestion (recursion with and without the unmasked
body, Rys quadrature)."""

import numpy as np
import pytest

from test_gpu_tiles import _chain

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from vlxmi.runtime import Device
    return Device()


@pytest.fixture(scope="module")
def eng(dev):
    from vlxmi.fock import FockEngine
    mol, D = _chain(9)
    e = FockEngine(mol, dev=dev)
    return e, e.cart_density(D)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("ab,cd", [("ss", "ss"), ("sp", "sp"), ("pp", "pp"), ("sp", "dd"), ("pd", "pd")])
def test_nan_density_is_screened_out_of_j(eng, ab, cd, precision):
    """One NaN among the ket's densities against the same list with a zero there:
    the same terms in the same order."""
    print("case: J (%s|%s) %s, a NaN density" % (ab, cd, precision), flush=True)
    e, Dc = eng
    e.precision, e.mixed_policy = precision, "all"
    try:
        out = []
        for x in (float("nan"), 0.0):
            kets = e.prepare_kets(Dc)
            kets[cd]["mat_D"][3] = x
            out.append(e.run_J(Dc, kets=kets, classes=[(ab, cd)])[ab].cpu().numpy())
    finally:
        e.precision, e.mixed_policy = "fp64", "measured"
    assert np.isfinite(out[0]).all()
    assert np.abs(out[0] - out[1]).max() <= 1e-14 * np.abs(out[1]).max()


@pytest.mark.parametrize("ab,cd", [("ss", "sp"), ("sp", "ss"), ("pp", "ss"), ("sp", "dd"), ("pd", "ss")])
def test_infinite_density_against_a_zero_bound(eng, ab, cd):
    """A bra entry with a zero Schwarz factor has an infinite threshold: nothing
    passes it, not even an infinite density."""
    print("case: J (%s|%s), an infinite density" % (ab, cd), flush=True)
    e, Dc = eng
    kets = e.prepare_kets(Dc)
    kets[cd]["mat_D"][2] = float("inf")
    Q = e.jl[ab]["mat_Q"]
    old = Q[1].clone()
    try:
        Q[1] = 0.0
        J = e.run_J(Dc, kets=kets, classes=[(ab, cd)])[ab].cpu().numpy()
    finally:
        Q[1] = old
    assert J[1] == 0.0
    assert not np.isfinite(J).all()                       # the others see it


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cls,pc", [("ssps", "ps"), ("spss", "ss"), ("sppp", "pp"), ("pppd", "pd"), ("sdpd", "pd")])
def test_nan_schwarz_factor_is_screened_out_of_k(eng, cls, pc, precision):
    """One NaN among the ket list's Schwarz factors against a zero there."""
    print("case: K %s %s, a NaN Schwarz factor" % (cls, precision), flush=True)
    e, Dc = eng
    assert pc == cls[2:] != cls[:2]
    e.precision, e.mixed_policy = precision, "all"
    Q = e.kc[pc]["Q"]
    old, maxD, out = Q[1].clone(), e.max_D(Dc), []
    try:
        for x in (float("nan"), 0.0):
            Q[1] = x
            out.append(e.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]].cpu().numpy())
    finally:
        Q[1] = old
        e.precision, e.mixed_policy = "fp64", "measured"
    assert np.isfinite(out[0]).all()
    assert np.abs(out[0] - out[1]).max() <= 1e-14 * np.abs(out[1]).max()
