"""What FockEngine.prepare_kets hands to its kernels, which read the density
through a raw pointer: any real matrix of the engine's device that holds the
density in its leading part, in the layout and type the kernels read."""

import types

import numpy as np
import pytest
import torch

import _util  # noqa: F401  (puts the package on sys.path)
from vlxmi import fock

N = 5


@pytest.fixture()
def eng(monkeypatch):
    """An engine of N AOs without lists; the library is not reached."""
    e = fock.FockEngine.__new__(fock.FockEngine)
    e.torch, e.naos, e.T = torch, N, torch.eye(N, dtype=torch.float64)
    e.dev = types.SimpleNamespace(device=torch.device("cpu"), stream_ptr=lambda: 0)
    e.jl = {}
    monkeypatch.setattr(fock, "lib", lambda: None)
    return e


def test_converted_to_contiguous_doubles(eng):
    D = torch.from_numpy(np.random.default_rng(1).normal(size=(N + 2, N + 3)))
    for X in (D, D.float(), D.half(), D.t()[:N, :N], D[:N, :N], (D * 9).int(), D[::2, ::1].repeat(2, 1)):
        out = eng._kernel_density(X)
        assert out.dtype == torch.float64 and out.is_contiguous() and out.shape == (N, N)
        assert torch.equal(out, X[:N, :N].double())
    own = torch.zeros((N, N), dtype=torch.float64)
    assert eng._kernel_density(own).data_ptr() == own.data_ptr()          # no copy of a density that fits


@pytest.mark.parametrize("bad", [torch.zeros(N, N - 1), torch.zeros(N - 1, N), torch.zeros(N * N), torch.zeros(1, N, N),
                                 torch.zeros(N, N, dtype=torch.complex128), torch.zeros(N, N, device="meta")],
                         ids=["narrow", "short", "flat", "batched", "complex", "device"])
def test_refused(eng, bad):
    with pytest.raises(ValueError):
        eng.prepare_kets(bad)


def test_lists_are_the_ones_in_place(eng):
    """A list put in the place of another is the one the next call reads."""
    def one(n):
        j = {f: torch.zeros(n) for f in ("ao_first", "ao_second", "keep", "mat_Q", "pair_data", "first", "second")}
        return dict(j, nblk=n, nab=1, count=n)
    eng.jl = {"ss": one(3), "sp": one(2)}
    for n in (3, 7):
        eng.jl["ss"] = one(n)
        cls, entries, blocks = eng._ket_classes()
        assert (entries, blocks) == (n + 2, n + 2)
        assert cls[0].mat_Q == eng.jl["ss"]["mat_Q"].data_ptr() and cls[0].nblk == n
        assert cls[1].pair_data == eng.jl["sp"]["pair_data"].data_ptr() and cls[1].entry_offset == n
