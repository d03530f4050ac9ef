"""Density-dependent inputs: the ket order of the Coulomb lists and the density
maxima against the plain torch operations, at the edges of the kernels' blocks
(256) and of the list length that is ordered without a device sort (4096)."""

import numpy as np
import pytest

from vlxmi import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from vlxmi.runtime import Device
    return Device()


@pytest.mark.parametrize("nblk,nab", [(1, 1), (2, 36), (255, 3), (256, 9), (257, 6), (4096, 1), (4097, 3), (6001, 1)])
def test_ket_order_equals_stable_sort(dev, nblk, nab):
    from vlxmi.runtime import KET_RANK_MAX, KetClass, check, lib
    print("case: %d blocks of %d" % (nblk, nab), flush=True)
    t, n = dev.torch, 40
    rng = np.random.default_rng(nblk + nab)
    ent = nblk * nab
    D = dev.tensor(rng.normal(size=(n, n)))
    j = dict(ao_first=dev.tensor(rng.integers(0, n, ent)), ao_second=dev.tensor(rng.integers(0, n, ent)),
             keep=dev.tensor(rng.random(ent) < 0.8), mat_Q=dev.tensor(np.round(rng.random(ent), 2)),      # ties on purpose
             pair_data=dev.tensor(rng.normal(size=ent)), first=dev.tensor(np.arange(ent, dtype=np.uint32)),
             second=dev.tensor(rng.integers(0, 99, ent).astype(np.uint32)))
    D = t.round(D, decimals=1)
    cls = (KetClass * 1)()
    for k, v in j.items():
        setattr(cls[0], k, v.data_ptr())
    cls[0].nblk, cls[0].nab = nblk, nab
    mD = D[j["ao_first"], j["ao_second"]] * j["keep"].to(t.float64)
    beta = (j["mat_Q"] * mD).abs().view(-1, nab).amax(dim=1)
    order = t.sort(beta, descending=True, stable=True).indices
    if nblk > KET_RANK_MAX:
        cls[0].order = order.data_ptr()
    f64 = t.full((4, ent), float("nan"), dtype=t.float64, device=dev.device)
    ints = t.full((2, ent), -1, dtype=t.int32, device=dev.device)
    b = t.empty(nblk, dtype=t.float64, device=dev.device)
    st = dev.stream_ptr()
    check(lib().vlxmi_ket_bounds(cls, 1, D.data_ptr(), n, f64[0].data_ptr(), b.data_ptr(), st))
    check(lib().vlxmi_ket_order(cls, 1, b.data_ptr(), f64[0].data_ptr(), ints[0].data_ptr(), ints[1].data_ptr(),
                                f64[1].data_ptr(), f64[2].data_ptr(), f64[3].data_ptr(), st))
    e = (order[:, None] * nab + t.arange(nab, device=dev.device)[None, :]).reshape(-1)
    assert t.equal(f64[0], mD) and t.equal(b, beta)
    for got, ref in ((ints[0], j["first"]), (ints[1], j["second"]), (f64[1], j["pair_data"]), (f64[2], j["mat_Q"]), (f64[3], mD)):
        assert t.equal(got, ref[e])
    if nblk > KET_RANK_MAX:
        cls[0].order = None
        assert lib().vlxmi_ket_order(cls, 1, b.data_ptr(), f64[0].data_ptr(), ints[0].data_ptr(), ints[1].data_ptr(),
                                     f64[1].data_ptr(), f64[2].data_ptr(), f64[3].data_ptr(), st) == -3


def test_nan_bound_leads(dev):
    """A block with a NaN entry keeps NaN as its bound and leads its list, as in
    a device sort."""
    from vlxmi.runtime import KetClass, check, lib
    t = dev.torch
    D = dev.tensor(np.array([[1.0, np.nan], [2.0, 3.0]]))
    ao = dev.tensor(np.array([0, 0, 0, 1]))
    cls = (KetClass * 1)()
    keep, Q = t.ones(4, dtype=t.bool, device=dev.device), t.ones(4, dtype=t.float64, device=dev.device)
    second, idx = dev.tensor(np.array([0, 0, 1, 1])), dev.tensor(np.arange(4, dtype=np.uint32))
    for k, v in dict(ao_first=ao, ao_second=second, keep=keep, mat_Q=Q, pair_data=Q, first=idx, second=idx).items():
        setattr(cls[0], k, v.data_ptr())
    cls[0].nblk, cls[0].nab = 2, 2
    f64, b = t.empty((4, 4), dtype=t.float64, device=dev.device), t.empty(2, dtype=t.float64, device=dev.device)
    ints = t.empty((2, 4), dtype=t.int32, device=dev.device)
    st = dev.stream_ptr()
    check(lib().vlxmi_ket_bounds(cls, 1, D.data_ptr(), 2, f64[0].data_ptr(), b.data_ptr(), st))
    check(lib().vlxmi_ket_order(cls, 1, b.data_ptr(), f64[0].data_ptr(), ints[0].data_ptr(), ints[1].data_ptr(),
                                f64[1].data_ptr(), f64[2].data_ptr(), f64[3].data_ptr(), st))
    assert b[0].item() == 1.0 and t.isnan(b[1]).item()
    assert ints[0].tolist() == [2, 3, 0, 1]


def test_density_maxima_and_checks(dev):
    """The maxima equal FockEngine.max_D of the symmetrised density, which is
    exactly symmetric; densities that were refused still are."""
    from vlxmi.fock import FockEngine
    from vlxmi.pairs import DensityError
    mol, D = configs.make_lattice4()
    eng = FockEngine(mol, dev=dev)
    Dc, maxD = eng._density(D)
    T = eng.T.cpu().numpy()
    ref = T.T @ D @ T
    assert np.abs(Dc.cpu().numpy() - ref).max() <= 1e-14 * np.abs(ref).max() and dev.torch.equal(Dc, Dc.t())
    assert maxD == eng.max_D(Dc)
    bad = D.copy()
    bad[3, 5] += 1e-6
    for X in (bad, D * np.nan, D * 1e4, np.where(D == D.max(), np.inf, D)):
        with pytest.raises(DensityError):
            eng.build(X)
    with pytest.raises(ValueError):
        eng.build(D[None])
