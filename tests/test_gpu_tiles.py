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
    """J of lists of n blocks against the same kernels on one bra block at a time
    (a tile of one block): sums of the same terms in another order, at most 1e4
    of them.  K of diagonal (I,I) blocks from both ends of the quartet."""
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
    for cls, other in (("spsd", "sdsp"), ("pppp", "pppp"), ("dsdp", "dpds")):
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


@pytest.mark.parametrize("n", [13, 17, 25, 33])
@pytest.mark.parametrize("cls", ["ssss", "ssps", "sppp", "pppp", "sdpd", "pddd"])
def test_exchange_tiles_against_oracle(dev, cls, n):
    """Partner counts on both sides of the narrowing step, with the launch split
    where it splits: sampled (I,K) blocks of the whole launch against the oracle."""
    from vlxmi.fock import FockEngine
    from vlxmi.pairs import NCART, LVAL
    print("case: chain of %d atoms, K %s" % (n, cls), flush=True)
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    Dc = eng.cart_density(D)
    ac = cls[0] + cls[2]
    got = eng.run_K(Dc, classes=[cls])[ac].cpu().numpy()
    nblk = eng.fl.iklists[ac].nblk
    sel = np.unique([0, 1, nblk // 3, nblk // 2, nblk - 2, nblk - 1]).astype(np.uint32)
    ref = U.oracle_matK(eng.fl, U.cart_density(mol, D), "component", ik_blocks=sel, classes=[cls])[ac]
    nac = NCART[LVAL[cls[0]]] * NCART[LVAL[cls[2]]]
    e = (sel[:, None].astype(np.int64) * nac + np.arange(nac)).ravel()
    assert np.abs(ref[e]).max() > 0
    assert np.abs(got[e] - ref[e]).max() <= 1e-11 * max(1.0, np.abs(ref[e]).max())


def _mixed_run(eng, thr32, run):
    """(FP64 result, mixed result, FP64 and FP32 quartets of the latter)."""
    ref = run().cpu().numpy()
    eng.precision, eng.mixed_policy, eng.fp32_threshold = "mixed", "all", thr32
    eng.reset_counts()
    got = run().cpu().numpy()
    counts = eng.quartet_counts()
    eng.precision = "fp64"
    return ref, got, counts


# an FP32 recursion's result carries at most some 64 roundings of the bound its
# quartet was let through by (below the threshold)
FP32_QUARTET = 64 * 2.0 ** -24


@pytest.mark.parametrize("n", [5, 13, 17, 25, 33])
def test_mixed_tiles_coulomb(dev, n):
    """Packed bra tiles that change from FP64 to FP32 within a ket tile: every
    quartet above the screen is evaluated once, none above the FP32 bound in
    FP32, and the sums differ by what FP32 leaves out."""
    from vlxmi import flops
    from vlxmi.fock import FockEngine
    print("case: chain of %d atoms, mixed J" % n, flush=True)
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    Dc, Dn = eng.cart_density(D), U.cart_density(mol, D)
    kets = eng.prepare_kets(Dc)
    for ab, cd in (("pp", "sp"), ("pp", "pp"), ("pd", "ss"), ("pd", "dd")):
        bra, ket = eng.fl.jlists[ab], eng.fl.jlists[cd]
        beta = np.abs(ket.mat_Q * ket.mat_D(Dn)).reshape(ket.nblk, -1).max(axis=1)
        thr32 = float(np.median(np.outer(bra.qmax_blk, beta)))
        ref, got, (n64, n32) = _mixed_run(eng, thr32, lambda: eng.run_J(Dc, kets=kets, classes=[(ab, cd)])[ab])
        assert n64 + n32 == flops.count_j(eng.fl, Dn, ab, cd) and n32 > 0, (ab, cd)
        thr, eng.fl.thr = eng.fl.thr, thr32
        assert n64 >= flops.count_j(eng.fl, Dn, ab, cd)
        eng.fl.thr = thr
        assert 0 < np.abs(got - ref).max() <= FP32_QUARTET * 2 * ket.count * thr32, (ab, cd)


@pytest.mark.parametrize("n", [5, 13, 17, 25, 33])
def test_mixed_tiles_exchange(dev, n):
    """As test_mixed_tiles_coulomb for packed partner tiles."""
    from vlxmi.fock import FockEngine
    print("case: chain of %d atoms, mixed K" % n, flush=True)
    mol, D = _chain(n)
    eng = FockEngine(mol, dev=dev)
    Dc = eng.cart_density(D)
    maxD = eng.max_D(Dc)
    for cls in ("ssps", "ppps", "sppp", "ppdp", "pddd"):
        A, C = eng.fl.kcsr[cls[:2]], eng.fl.kcsr[cls[2:]]
        mx = maxD[cls[1] + cls[3]]
        thr32 = float(A.blk_max.max() * np.median(C.blk_max) * mx)      # every tile changes half-way
        ref, got, (n64, n32) = _mixed_run(eng, thr32, lambda: eng.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]])
        assert n64 + n32 == eng.count_k_quartets(cls, mx), cls
        assert n32 > 0 or n < 8, cls                     # up to 8 records are one step of 8 lane groups
        thr, eng.thr = eng.thr, thr32
        assert n64 >= eng.count_k_quartets(cls, mx)
        eng.thr = thr
        terms = A.Q.size // eng.fl.prims[0].count * (C.Q.size // eng.fl.prims[0].count)
        assert np.abs(got - ref).max() <= FP32_QUARTET * terms * thr32, cls


@pytest.fixture(scope="module")
def split():
    """The number of chunks an exchange launch of an engine takes, by the rule in
    the launcher's source."""
    import re
    from vlxmi.gen import build
    src = build.sources()

    def chunks(eng, cls):
        m = re.search(r"tiles = \((\w)_prim_count \+ \d+\) / (\d+), want = \((\d+)u", src["k_%s.hip" % cls])
        nblk = eng.ik[cls[0] + cls[2]]["nblk"]
        tiles = -(-eng.prim_count["spd".index(m.group(1))] // int(m.group(2)))
        return min(tiles, -(-int(m.group(3)) // nblk), 16)
    return chunks


def test_exchange_split_under_capture(dev, split):
    """An exchange launch over few blocks splits its partners among wavefronts
    (partial sums in the library's workspace); while a stream is captured it
    stays unsplit, and the graph gives the same sums on every replay."""
    from vlxmi.fock import FockEngine
    print("case: exchange launches in a graph", flush=True)
    t = dev.torch
    mol, D = _chain(17)
    eng = FockEngine(mol, dev=dev)
    Dc = eng.cart_density(D)
    maxD = eng.max_D(Dc)
    for cls in ("ssss", "dpds", "pddd"):
        assert split(eng, cls) > 1
        ref = eng.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]].clone()
        s = t.cuda.Stream(device=dev.device)
        s.wait_stream(t.cuda.current_stream(dev.device))
        g = t.cuda.CUDAGraph()
        with t.cuda.stream(s):
            eng.run_K(Dc, classes=[cls], maxD=maxD)          # the capturing stream has a workspace
        t.cuda.synchronize()
        with t.cuda.graph(g, stream=s):
            out = eng.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]]
        for _ in range(3):
            g.replay()
            t.cuda.synchronize()
            assert (out - ref).abs().max() <= 1e-12 * max(1.0, float(ref.abs().max()))
            assert t.equal(eng.run_K(Dc, classes=[cls], maxD=maxD)[cls[0] + cls[2]], ref)


def test_exchange_split_two_threads_one_stream(dev, split):
    """Two threads launch split exchange classes of different sizes on one
    stream: each gets the sums it gets alone, bit for bit (a launch and its
    reduction hold the stream's workspace together; every launch of both threads
    uses it)."""
    import threading
    from vlxmi.fock import FockEngine
    print("case: two threads, one stream", flush=True)
    t = dev.torch
    work = []
    classes = ("ssss", "dpds", "pddd", "sdpd")
    for n in (17, 31):
        mol, D = _chain(n)
        eng = FockEngine(mol, dev=dev)
        assert all(split(eng, c) > 1 for c in classes)
        Dc = eng.cart_density(D)
        work.append((eng, Dc, eng.max_D(Dc)))

    def run(w):
        eng, Dc, maxD = w
        return [eng.run_K(Dc, classes=[c], maxD=maxD)[c[0] + c[2]].clone() for c in classes]

    alone = [run(w) for w in work]
    t.cuda.synchronize()
    got = [[], []]

    def loop(i):
        for _ in range(20):
            got[i].append(run(work[i]))

    ts = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
    for x in ts:
        x.start()
    for x in ts:
        x.join(60)
    assert not any(x.is_alive() for x in ts)
    t.cuda.synchronize()
    for i in range(2):
        assert len(got[i]) == 20
        assert all(t.equal(a, b) for r in got[i] for a, b in zip(r, alone[i]))
