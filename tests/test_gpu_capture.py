"""Ket-split Coulomb launches in HIP graphs: without a workspace large enough
they run unsplit, with one they keep it whatever else the stream runs later."""

import pytest

from test_gpu_tiles import _chain

pytestmark = pytest.mark.gpu

CLASSES = [("ss", "ss"), ("pd", "pd"), ("dd", "sd")]


@pytest.fixture(scope="module")
def dev():
    from vlxmi.runtime import Device
    return Device()


def _engine(dev, n):
    from vlxmi.fock import FockEngine
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    Dc = eng.cart_density(D)
    return eng, Dc, eng.prepare_kets(Dc)


def _run(eng, Dc, kets):
    return [eng.run_J(Dc, kets=kets, classes=[c])[c[0]] for c in CLASSES]


def _close(a, b):
    """Sums of the same terms in another order, at most 1e4 of them."""
    for x, y in zip(a, b):
        assert (x - y).abs().max() <= 1e-12 * max(1.0, float(y.abs().max()))


@pytest.mark.parametrize("warm", [False, True])
def test_coulomb_split_in_a_graph(dev, warm):
    from vlxmi.runtime import check, lib
    print("case: Coulomb launches in a graph, workspace %s" % ("grown before" if warm else "absent"), flush=True)
    t = dev.torch
    eng, Dc, kets = _engine(dev, 17)
    for ab, cd in CLASSES[1:]:
        a, c = eng.jl[ab], eng.jl[cd]
        assert eng._ket_split(a["nblk"], c["nblk"], a["nab"] * c["nab"]) > 1
    ref = [x.clone() for x in _run(eng, Dc, kets)]
    t.cuda.synchronize()
    check(lib().vlxmi_release_workspaces())
    s = t.cuda.Stream(device=dev.device)
    if warm:
        with t.cuda.stream(s):
            _run(eng, Dc, kets)
        t.cuda.synchronize()
    g = t.cuda.CUDAGraph()
    with t.cuda.graph(g, stream=s):
        out = _run(eng, Dc, kets)
    big, bDc, bkets = _engine(dev, 33)
    with t.cuda.stream(s):
        bref = [x.clone() for x in _run(big, bDc, bkets)]
    for _ in range(3):
        g.replay()
        t.cuda.synchronize()
        _close(out, ref)
        for x in out:
            x.fill_(-1.0)
        with t.cuda.stream(s):                         # grows the stream's buffer and writes it
            _close(_run(big, bDc, bkets), bref)
            big.run_K(bDc, classes=["pppp"])
        t.cuda.synchronize()
    _close(_run(eng, Dc, kets), ref)
    del g
    check(lib().vlxmi_release_workspaces())
