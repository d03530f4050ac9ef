// Device memory for the partial sums of ket-split launches, kept per (device,
// stream): launches on one stream run in order, so they can share a buffer;
// another stream gets its own.  Host code only.
//
// Coulomb and exchange launches have buffers of their own.  A Coulomb launch
// recorded into a graph keeps its buffer's address, so a buffer that was handed
// out during a capture is never freed by growth: it is retired (freed by
// vlxmi_release_workspaces, or never), and its successor has at least twice its
// size, so what a stream's retired buffers hold stays below its current one.
// Exchange launches record none.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <map>
#include <mutex>
#include <new>
#include <tuple>
#include <vector>

#include "vlxmi_status.h"

namespace {
struct Workspace {
    double* p = nullptr;
    size_t n = 0;
    bool in_graph = false;
    std::vector<double*> retired;
};
std::recursive_mutex g_ws_mutex;   // a launcher's hold spans its own workspace call
std::map<std::tuple<int, void*, bool>, Workspace> g_ws;   // (device, stream, exchange) -> buffer

enum class Capture { no, yes, unknown };

Capture capturing(hipStream_t stream)
{
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &s) != hipSuccess) {
        (void)hipGetLastError();
        return Capture::unknown;
    }
    return s == hipStreamCaptureStatusNone ? Capture::no : Capture::yes;
}

// While one is alive this thread's allocations leave other threads' captures
// alone (relaxed mode): a launch that was not split allocated nothing.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    bool swapped = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    ~RelaxedCapture()
    {
        if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
};

// A new buffer holds at least 2 MiB, as much as any exchange launch asks for (its
// chunks times blocks are fewer than 4096, at most 36 sums each): growing class
// by class, each time with a synchronisation, an allocation and a free, lengthened
// the first build on a stream.
constexpr size_t MIN_DOUBLES = (size_t)1 << 18;

// A buffer of n doubles, with room to spare if it is to be had (``spare``).
hipError_t allocate(size_t n, size_t spare, double** p, size_t* got)
{
    hipError_t e = hipSuccess;
    for (size_t want : {spare, n}) {
        e = hipMalloc((void**)p, want * sizeof(double));
        if (e == hipSuccess) {
            *got = want;
            break;
        }
        if (want != n) (void)hipGetLastError();
    }
    return e;
}

// Grows w to n doubles; the old buffer stays as it was on failure, unless
// ``need`` and only its memory makes room for the new one.
hipError_t grow(Workspace& w, size_t n, hipStream_t stream, bool need)
{
    RelaxedCapture relaxed;
    if (w.in_graph) w.retired.reserve(w.retired.size() + 1);
    size_t spare = n + n / 4, least = n, got = 0;
    if (spare < MIN_DOUBLES) spare = MIN_DOUBLES;
    if (w.in_graph) {
        if (spare < 2 * w.n) spare = 2 * w.n;
        least = spare;
    }
    double* p = nullptr;
    hipError_t e = allocate(least, spare, &p, &got);
    if (e != hipSuccess && (!need || !w.p || w.in_graph)) return e;
    if (w.p && w.in_graph) {
        w.retired.push_back(w.p);
    } else if (w.p) {
        // the stream's earlier launches may still use it
        hipError_t se = hipStreamSynchronize(stream);
        if (se != hipSuccess) {
            if (p) (void)hipFree(p);
            return se;
        }
        (void)hipFree(w.p);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            w.p = nullptr;
            w.n = 0;
            e = allocate(least, spare, &p, &got);
            if (e != hipSuccess) return e;
        }
    }
    w.p = p;
    w.n = got;
    w.in_graph = false;
    return hipSuccess;
}

int take(size_t ndoubles, void* stream, bool exchange, double** out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    const Capture c = capturing((hipStream_t)stream);
    if (exchange && c != Capture::no) return VLXMI_ERR_ARG;
    try {
        std::lock_guard<std::recursive_mutex> lock(g_ws_mutex);
        Workspace& w = g_ws[std::make_tuple(dev, stream, exchange)];
        if (w.n < ndoubles) {
            if (c == Capture::yes) return (int)hipErrorStreamCaptureUnsupported;
            e = grow(w, ndoubles, (hipStream_t)stream, !exchange);
            if (e != hipSuccess) return (int)e;
        }
        if (c == Capture::yes) w.in_graph = true;
        *out = w.p;
    } catch (const std::bad_alloc&) {
        return (int)hipErrorOutOfMemory;
    }
    return VLXMI_OK;
}
}  // namespace

// A device buffer of at least ndoubles doubles for Coulomb launches on (current
// device, stream), grown on demand and kept until vlxmi_release_workspaces().
// While the stream is being captured nothing is allocated: a buffer that is
// large enough is the capture's from then on, else the call returns
// hipErrorStreamCaptureUnsupported and the capture goes on.
extern "C" int vlxmi_ket_workspace(size_t ndoubles, void* stream, double** out)
{
    if (!out) return VLXMI_ERR_ARG;
    return take(ndoubles, stream, false, out);
}

// The exchange launches' buffer, for launches that can do without: an error,
// with the old buffer kept and no HIP error left behind, while the stream is
// being captured or when the memory is not to be had.
extern "C" int vlxmi_try_workspace(size_t ndoubles, void* stream, double** out)
{
    const int rc = take(ndoubles, stream, true, out);
    if (rc > 0) (void)hipGetLastError();
    return rc;
}

// See vlxmi::WorkspaceHold.
extern "C" void vlxmi_workspace_hold(int on)
{
    if (on)
        g_ws_mutex.lock();
    else
        g_ws_mutex.unlock();
}

// Frees every workspace, those of graphs included (after a device
// synchronization).
extern "C" int vlxmi_release_workspaces(void)
{
    std::lock_guard<std::recursive_mutex> lock(g_ws_mutex);
    if (!g_ws.empty()) {
        hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) return (int)e;
    }
    for (auto& kv : g_ws) {
        if (kv.second.p) (void)hipFree(kv.second.p);
        for (double* p : kv.second.retired) (void)hipFree(p);
    }
    g_ws.clear();
    return VLXMI_OK;
}
