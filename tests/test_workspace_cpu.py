"""The ket-split workspaces (csrc/vlxmi_workspace.cpp) against a model of the few
HIP calls they make: what is allocated, freed and synchronised, also around
stream captures and when memory runs out."""

import ctypes as C
import os
import subprocess

import pytest

from _util import PKG

OK, ERR_ARG, OOM, SYNC_FAILED, UNSUPPORTED = 0, -1, 2, 719, 900

HIP = r"""
#include <cstddef>
#include <cstdio>
#include <set>
#include <string>
typedef void* hipStream_t;
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorLaunchFailure = 719,
                  hipErrorStreamCaptureUnsupported = 900, hipErrorStreamCaptureInvalidated = 901 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal = 0, hipStreamCaptureModeThreadLocal = 1, hipStreamCaptureModeRelaxed = 2 };
extern "C" hipError_t hipGetDevice(int*);
extern "C" hipError_t hipMalloc(void**, size_t);
extern "C" hipError_t hipFree(void*);
extern "C" hipError_t hipStreamSynchronize(hipStream_t);
extern "C" hipError_t hipDeviceSynchronize(void);
extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus*);
extern "C" hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*);
extern "C" hipError_t hipGetLastError(void);
"""

MODEL = r"""
#include "%s"
static std::string g_log;              // calls in order
static hipStream_t g_capture = nullptr;
static bool g_broken = false;          // an unsafe call reached a capture
static size_t g_room = (size_t)-1, g_used = 0;
static bool g_sync_fails = false;
static hipError_t g_last = hipSuccess;
static hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
static char g_mem[1 << 16];
static size_t g_next = 0;
static std::map<void*, size_t> g_live;
static hipError_t fail(hipError_t e) { g_last = e; return e; }
static bool unsafe() { if (g_capture && g_mode != hipStreamCaptureModeRelaxed) g_broken = true; return g_broken; }
extern "C" hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
extern "C" hipError_t hipMalloc(void** p, size_t n)
{
    if (unsafe()) return fail(hipErrorStreamCaptureUnsupported);
    if (g_used + n > g_room) return fail(hipErrorOutOfMemory);
    *p = g_mem + g_next++;
    g_live[*p] = n;
    g_used += n;
    g_log += "m";
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p)
{
    unsafe();
    if (!g_live.count(p)) { g_log += "!"; return hipSuccess; }
    g_used -= g_live[p];
    g_live.erase(p);
    g_log += "f";
    return hipSuccess;
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t s)
{
    if (s == g_capture) { g_broken = true; return fail(hipErrorStreamCaptureUnsupported); }
    g_log += "s";
    return g_sync_fails ? fail(hipErrorLaunchFailure) : hipSuccess;
}
extern "C" hipError_t hipDeviceSynchronize(void) { g_log += "d"; return hipSuccess; }
extern "C" hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c)
{
    *c = g_capture && s == g_capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
extern "C" hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) { std::swap(*m, g_mode); return hipSuccess; }
extern "C" hipError_t hipGetLastError(void) { hipError_t e = g_last; g_last = hipSuccess; return e; }
extern "C" void model_capture(void* s) { g_capture = s; }
extern "C" void model_room(size_t n) { g_room = n; }
extern "C" void model_sync_fails(int on) { g_sync_fails = on; }
extern "C" int model_broken(void) { return g_broken; }
extern "C" int model_mode(void) { return g_mode; }
extern "C" int model_last(void) { return g_last; }
extern "C" int model_live(void* p) { return g_live.count(p); }
extern "C" size_t model_used(void) { return g_used; }
extern "C" const char* model_log(void) { static std::string out; out = g_log; g_log.clear(); return out.c_str(); }
"""

S1, S2 = 0x1000, 0x2000
UNIT = 1 << 18                # the smallest buffer, in doubles


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    d = tmp_path_factory.mktemp("workspace")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    csrc = os.path.join(PKG, "csrc")
    (d / "model.cpp").write_text(MODEL % os.path.join(csrc, "vlxmi_workspace.cpp"))
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", str(d), "-I", csrc, str(d / "model.cpp"),
                    "-o", str(d / "model.so")], check=True)
    return str(d / "model.so")


@pytest.fixture()
def ws(so, tmp_path):
    """A fresh copy of the library (its state is static)."""
    p = tmp_path / "model.so"
    p.write_bytes(open(so, "rb").read())
    L = C.CDLL(str(p))
    L.model_log.restype = C.c_char_p
    for f in ("vlxmi_ket_workspace", "vlxmi_try_workspace"):
        getattr(L, f).argtypes = [C.c_size_t, C.c_void_p, C.POINTER(C.c_void_p)]
    L.model_capture.argtypes = L.model_live.argtypes = [C.c_void_p]
    L.model_room.argtypes, L.model_used.restype = [C.c_size_t], C.c_size_t
    return L


def _take(L, n, stream=S1, exchange=False):
    p = C.c_void_p()
    rc = (L.vlxmi_try_workspace if exchange else L.vlxmi_ket_workspace)(int(n * UNIT), stream, C.byref(p))
    return rc, p.value


def test_grows_after_a_synchronisation_and_is_kept(ws):
    rc, a = _take(ws, 100)
    assert (rc, ws.model_log()) == (OK, b"m")
    assert _take(ws, 100) == (OK, a) and _take(ws, 1) == (OK, a) and ws.model_log() == b""
    assert _take(ws, 100, S2)[1] != a and ws.model_log() == b"m"
    rc, b = _take(ws, 1000)
    assert rc == OK and b != a and not ws.model_live(a) and ws.model_log() == b"msf"
    assert ws.vlxmi_release_workspaces() == OK and ws.model_log() == b"dff" and ws.model_used() == 0


def test_exchange_growth_leaves_the_coulomb_buffer(ws):
    a = _take(ws, 100)[1]
    b = _take(ws, 10, exchange=True)[1]
    assert a != b and _take(ws, 5000, exchange=True)[0] == OK
    assert ws.model_live(a) and not ws.model_live(b) and _take(ws, 100)[1] == a


def test_capture_allocates_nothing_and_goes_on(ws):
    """Without memory of its own size a captured Coulomb launch is told so, an
    exchange launch always; the capture stays whole."""
    ws.model_capture(S1)
    assert _take(ws, 100) == (UNSUPPORTED, None) and _take(ws, 100, exchange=True) == (ERR_ARG, None)
    ws.model_capture(None)
    _take(ws, 100), _take(ws, 100, exchange=True)
    ws.model_log()
    ws.model_capture(S1)
    assert _take(ws, 101 * 2)[0] == UNSUPPORTED and _take(ws, 10, exchange=True)[0] == ERR_ARG
    assert ws.model_log() == b"" and not ws.model_broken() and ws.model_last() == 0


def test_a_graphs_buffer_outlives_growth(ws):
    """The address in a graph stays good until the workspaces are released; the
    buffers set aside are together smaller than the current one."""
    kept, n = [], 100
    for _ in range(6):
        assert _take(ws, n)[0] == OK
        ws.model_capture(S1)
        rc, p = _take(ws, n)
        ws.model_capture(None)
        assert rc == OK
        kept.append((p, n))
        n = int(n * 1.3)
    rc, last = _take(ws, 100 * n)
    assert rc == OK and all(ws.model_live(p) for p, _ in kept)
    assert ws.model_used() < 2 * 8 * UNIT * 125 * n
    _take(ws, 200 * n)                                     # not a graph's: freed
    assert not ws.model_live(last) and all(ws.model_live(p) for p, _ in kept)
    assert ws.vlxmi_release_workspaces() == OK and ws.model_used() == 0


@pytest.mark.parametrize("exchange", [False, True])
def test_another_threads_capture_is_left_alone(ws, exchange):
    ws.model_capture(S2)
    assert _take(ws, 100, exchange=exchange)[0] == OK and _take(ws, 1000, exchange=exchange)[0] == OK
    assert not ws.model_broken() and ws.model_mode() == 0


def test_out_of_memory(ws):
    """An exchange launch keeps its old buffer and leaves no error behind; a
    Coulomb launch gives its old buffer up for the new one."""
    a, b = _take(ws, 80)[1], _take(ws, 80, exchange=True)[1]
    ws.model_room(8 * UNIT * 250)
    assert _take(ws, 120, exchange=True)[0] == OOM and ws.model_live(b) and ws.model_last() == 0
    assert _take(ws, 80, exchange=True) == (OK, b)
    ws.model_log()
    rc, c = _take(ws, 110)
    assert rc == OK and not ws.model_live(a) and ws.model_log() == b"sfm" and ws.model_last() == 0
    assert ws.model_used() == 8 * UNIT * (100 + 137.5)
    assert _take(ws, 1000)[0] == OOM
    ws.model_room(1 << 40)
    assert _take(ws, 1000)[0] == OK


def test_failed_synchronisation_leaks_nothing(ws):
    a = _take(ws, 80)[1]
    used = ws.model_used()
    ws.model_sync_fails(1)
    assert _take(ws, 800)[0] == SYNC_FAILED and ws.model_live(a) and ws.model_used() == used
    ws.model_sync_fails(0)
    assert _take(ws, 80) == (OK, a)


def test_first_buffer_holds_what_small_molecules_ask_for(ws):
    """One allocation for all requests up to 2 MiB; only what was asked for when
    no more is to be had."""
    for n in (1, 50, 3000, 1 << 18):
        assert _take(ws, n / UNIT, exchange=True)[0] == OK
    assert ws.model_log() == b"m" and ws.model_used() == 1 << 21
    ws.model_room((1 << 21) + 8000)
    assert _take(ws, 1000 / UNIT, S2)[0] == OK and ws.model_used() == (1 << 21) + 8000
    assert ws.model_last() == 0
