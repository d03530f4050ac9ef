"""The one-centre exchange-gradient kernels that include/vlxmi_device_kernels.h
declares for direct launches: _A (columns 0..2) and _C (columns 3..5) together
give the class kernel's rows."""

import ctypes as C

import numpy as np
import pytest

from test_gpu_tiles import _chain

pytestmark = pytest.mark.gpu

TYPES = {"double*": "Pd", "const uint32_t*": "PKj", "const double*": "PKd", "uint32_t": "j", "double": "d"}
CTYPES = {"Pd": C.c_void_p, "PKj": C.c_void_p, "PKd": C.c_void_p, "j": C.c_uint32, "d": C.c_double}


class Dim3(C.Structure):
    _fields_ = [(n, C.c_uint32) for n in "xyz"]


def _types(cls):
    """Itanium codes of the kernel's parameters."""
    from vlxmi.gen import emit, emit_grad
    out = []
    for p in emit._strip_restrict(emit_grad.kg_signature(cls)):
        t = " ".join(p.split()[:-1])
        out.append(TYPES[t if "*" in t else t.replace("const ", "")])
    return out


def _mangled(name, types):
    seen, out = [], "_Z%d%s" % (len(name), name)
    for t in types:
        if t in seen:
            k = seen.index(t)
            out += "S_" if k == 0 else "S%s_" % "0123456789"[k - 1]
            continue
        if len(t) == 1:
            out += t
            continue
        if t.startswith("PK"):
            seen.append(t[1:])
        seen.append(t)
        out += t
    return out


class Direct:
    """Stands for the library in GradientEngine: launches the kernels of a class
    launcher directly, with the launcher's arguments."""

    def __init__(self, lib, suffixes):
        self.lib, self.suffixes = lib, suffixes
        self.hip = lib.hipLaunchKernel            # of the HIP runtime the library itself is bound to
        self.hip.argtypes = [C.c_void_p, Dim3, Dim3, C.POINTER(C.c_void_p), C.c_size_t, C.c_void_p]

    def __getattr__(self, launcher):
        name = launcher.replace("vlxmi_launch_", "")
        cls = name[-4:].lower()
        types = _types(cls)

        def launch(*args):
            assert len(args) == len(types) + 1
            count, nac = args[3], [1, 3, 6]["spd".index(cls[0])] * [1, 3, 6]["spd".index(cls[2])]
            assert count % nac == 0
            vals = [CTYPES[t](a) for t, a in zip(types, args)]
            ptrs = (C.c_void_p * len(vals))(*[C.addressof(v) for v in vals])
            for s in self.suffixes:
                f = C.addressof(C.c_char.in_dll(self.lib, _mangled(name + s, types)))
                rc = self.hip(f, Dim3(count // nac, 1, 1), Dim3(64, 1, 1), ptrs, 0, args[-1])
                if rc:
                    return rc
            return 0
        return launch


def test_one_centre_kernels_add_up(monkeypatch):
    from vlxmi import grad
    from vlxmi.fock import FockEngine
    from vlxmi.gen import build
    from vlxmi.runtime import Device, lib
    classes = sorted(build.load_grad_passes()["centres"])
    assert len(classes) == 32
    mol, D = _chain(5)
    eng = FockEngine(mol, dev=Device())
    ge = grad.GradientEngine(eng)
    Dc = eng.cart_density(D)
    maxD = eng.max_D(Dc)
    for cls in classes:
        print("case: %s" % cls, flush=True)
        ac, rows = cls[0] + cls[2], {}
        for s in (None, ("_A",), ("_C",), ("",)):
            with monkeypatch.context() as m:
                if s is not None:
                    direct = Direct(lib(), s)
                    m.setattr(grad, "lib", lambda: direct)
                rows[s] = ge.run_K(Dc, classes=[cls], maxD=maxD)[ac].cpu().numpy().reshape(-1, 6)
        ref, scale = rows[None], max(1.0, np.abs(rows[None]).max())
        assert np.abs(ref).max() > 0
        assert np.abs(rows[("",)] - ref).max() <= 1e-12 * scale, cls
        assert np.abs(rows[("_A",)][:, :3] - ref[:, :3]).max() <= 1e-12 * scale and not rows[("_A",)][:, 3:].any(), cls
        assert np.abs(rows[("_C",)][:, 3:] - ref[:, 3:]).max() <= 1e-12 * scale and not rows[("_C",)][:, :3].any(), cls
