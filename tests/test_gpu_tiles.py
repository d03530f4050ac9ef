"""J, K and their gradients at the edges of the kernels' lane tiles.

A tile of few bra blocks (J) or partners (K) shares its lanes out among several
ket records, in powers of two up to the staged records, and a tile that would
be at most three quarters full is followed by a narrower one: the counts below
sit on both sides of every step of that rule, with one s, p and d primitive per
atom so that every class has exactly that many primitives of each type."""

import numpy as np
import pytest

import _util as U

pytestmark = pytest.mark.gpu


def _chain(n):
    """n atoms on a slightly bent line, one primitive of each type per atom,
    close enough that no pair is screened out."""
    from vlxmi.basis import Molecule, Shell
    rng = np.random.default_rng(40 + n)
    coords = np.stack([0.21 * np.arange(n), 0.3 * np.sin(np.arange(n)), 0.1 * rng.normal(size=n)], axis=1)
    shells = []
    for a in range(n):
        for l in range(3):
            shells.append(Shell(a, l, coords[a], [rng.uniform(0.3, 1.5)], [1.0], spherical=False))
    mol = Molecule(coords, shells, name="chain%d" % n)
    C = rng.normal(0.0, 0.2, size=(mol.nbf, max(1, mol.nbf // 4)))
    return mol, C @ C.T


@pytest.fixture(scope="module")
def dev():
    from vlxmi.runtime import Device
    return Device()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9])
def test_tiles_against_oracle(dev, n):
    """Every class with n primitives of each type against the CPU oracle (the
    parity suite's bar)."""
    from vlxmi.fock import FockEngine
    print("case: chain of %d atoms" % n, flush=True)
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    J, K = [x.cpu().numpy() for x in eng.build(D)]
    Dc = U.cart_density(mol, D)
    Jr, Kr = U.oracle_fock(eng.fl, Dc, "component")
    T = mol.cart2sph()
    assert np.abs(J - T @ Jr @ T.T).max() <= 1e-11 * max(1.0, np.abs(Jr).max())
    assert np.abs(K - T @ Kr @ T.T).max() <= 1e-11 * max(1.0, np.abs(Kr).max())


@pytest.mark.parametrize("n", [12, 13, 16, 17, 24, 25, 32, 33, 48, 49, 64, 65])
def test_tiles_sum_rule(dev, n):
    """Lists of n partners against the same molecule's kernels run one (I,K)
    block / one bra block at a time (a tile of one block each): sums of the
    same terms in another order, at most 1e4 of them."""
    from vlxmi.fock import FockEngine
    print("case: chain of %d atoms, sliced" % n, flush=True)
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    Dc = eng.cart_density(D)
    kets, maxD = eng.prepare_kets(Dc), eng.max_D(Dc)
    for ab, cd in (("ss", "sp"), ("sd", "pp"), ("pd", "sd"), ("dd", "ss")):
        whole = eng.run_J(Dc, kets=kets, classes=[(ab, cd)])[ab].cpu().numpy()
        nab = eng.jl[ab]["nab"]
        for b in (0, eng.jl[ab]["nblk"] - 1, eng.jl[ab]["nblk"] // 2):
            one = eng.run_J(Dc, kets=kets, classes=[(ab, cd)], bra_blocks={ab: [b]})[ab].cpu().numpy()
            assert np.abs(one - whole[b * nab:(b + 1) * nab]).max() <= 1e-12 * max(1.0, np.abs(whole).max())
    # K: the sum over the partners of an (I,K) block is symmetric in which side's
    # list is walked by lanes: (ab|cd) with I, K exchanged is the class (cd|ab)
    for cls, other in (("ssss", "ssss"), ("spsd", "sdsp"), ("pppp", "pppp"), ("dsdp", "dpds")):
        ac = cls[0] + cls[2]
        x = eng.run_K(Dc, classes=[cls], maxD=maxD)[ac].cpu().numpy()
        y = eng.run_K(Dc, classes=[other], maxD=maxD)[ac].cpu().numpy()
        na = {"s": 1, "p": 3, "d": 6}[cls[0]]
        ik = eng.ik[ac]
        I, Kk = ik["I"].cpu().numpy(), ik["K"].cpu().numpy()
        d = np.nonzero(I == Kk)[0]                        # diagonal blocks: both orders are in the list
        xs, ys = x.reshape(-1, na, na)[d], y.reshape(-1, na, na)[d]
        assert np.abs(xs - ys.transpose(0, 2, 1)).max() <= 1e-12 * max(1.0, np.abs(x).max())


@pytest.mark.parametrize("n", [1, 3, 5])
def test_gradient_tiles_against_oracle(dev, n):
    """The per-block gradient rows of every class, lists of a few blocks,
    against the oracle's derivative routines (the gradient suite's bar)."""
    from vlxmi.fock import FockEngine
    from vlxmi.grad import GradientEngine
    print("case: chain of %d atoms, gradient" % n, flush=True)
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    ge = GradientEngine(eng)
    Dc, Dn = eng.cart_density(D), U.cart_density(mol, D)
    for got, ref in ((ge.run_J(Dc), U.oracle_gradJ(eng.fl, Dn)), (ge.run_K(Dc), U.oracle_gradK(eng.fl, Dn))):
        scale = max(1.0, max(np.abs(v).max() for v in ref.values() if v.size))
        for k in ref:
            if ref[k].size:
                assert np.abs(got[k].cpu().numpy() - ref[k]).max() <= 1e-11 * scale, k


def test_exchange_split_under_capture(dev):
    """An exchange launch over few blocks splits its partners among wavefronts
    (partial sums in the library's workspace); while a stream is captured it
    stays unsplit, and the graph gives the same sums on every replay."""
    from vlxmi.fock import FockEngine
    print("case: exchange launches in a graph", flush=True)
    t = dev.torch
    mol, D = _chain(12)
    eng = FockEngine(mol, dev=dev)
    Dc = eng.cart_density(D)
    maxD = eng.max_D(Dc)
    for cls in ("ssss", "dpds", "pddd"):
        ref = eng.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]].clone()
        s = t.cuda.Stream(device=dev.device)
        s.wait_stream(t.cuda.current_stream(dev.device))
        g = t.cuda.CUDAGraph()
        with t.cuda.stream(s):
            eng.run_K(Dc, classes=[cls], maxD=maxD)
        t.cuda.synchronize()
        with t.cuda.graph(g):
            out = eng.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]]
        for _ in range(3):
            g.replay()
            t.cuda.synchronize()
            assert (out - ref).abs().max() <= 1e-12 * max(1.0, float(ref.abs().max()))
            eng.run_K(Dc, classes=[cls], maxD=maxD)


def test_exchange_split_two_threads_one_stream(dev):
    """Two threads launch split exchange classes of different sizes on one
    stream: each gets the sums it gets alone, bit for bit (a launch and its
    reduction hold the stream's workspace together)."""
    import threading
    from vlxmi.fock import FockEngine
    print("case: two threads, one stream", flush=True)
    t = dev.torch
    work = []
    for n in (9, 17):
        mol, D = _chain(n)
        eng = FockEngine(mol, dev=dev)
        Dc = eng.cart_density(D)
        work.append((eng, Dc, eng.max_D(Dc)))
    classes = ("ssss", "dpds", "pddd", "sdpd")

    def run(w):
        eng, Dc, maxD = w
        return [eng.run_K(Dc, classes=[c], maxD=maxD)[c[0] + c[2]].clone() for c in classes]

    alone = [run(w) for w in work]
    t.cuda.synchronize()
    got = [[], []]

    def loop(i):
        for _ in range(6):
            got[i].append(run(work[i]))

    ts = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
    for x in ts:
        x.start()
    for x in ts:
        x.join(60)
    assert not any(x.is_alive() for x in ts)
    t.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 6
        assert all(t.equal(a, b) for r in got[i] for a, b in zip(r, alone[i]))
