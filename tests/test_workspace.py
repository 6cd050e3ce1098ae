"""The operators' scratch blocks (csrc/workspace.cpp) and the split of a batch that has
no room for them (in_parts), on the host: the file itself compiled against a stand-in
for the HIP calls it makes, which counts what the device holds and can be full."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
GIB = 1 << 30

SOURCE = r"""
#include "ct_recon_extensions_amd/csrc/workspace.cpp"

#include <map>
#include <vector>

namespace {
std::map<void*, size_t> g_live;       // blocks the "device" holds
size_t g_bytes = 0, g_room = ~size_t{0};
uintptr_t g_next = 1 << 20;
bool g_busy = false;                  // events have not passed
int g_events = 0, g_waits = 0;
}  // namespace

extern "C" {
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)(uintptr_t)++g_events; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { --g_events; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return g_busy ? hipErrorNotReady : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { ++g_waits; return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t)
{
    if (g_bytes + n > g_room) return hipErrorOutOfMemory;
    *p = (void*)g_next;
    g_next += (n + 0xfff) & ~size_t{0xfff};
    g_live[*p] = n;
    g_bytes += n;
    return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t)
{
    auto it = g_live.find(p);
    if (it == g_live.end()) return hipErrorInvalidValue;
    g_bytes -= it->second;
    g_live.erase(it);
    return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { return hipSuccess; }
hipError_t hipFree(void* p) { return hipFreeAsync(p, nullptr); }
}

namespace ctr {
void set_error(const std::string&) {}
}

extern "C" {
void* take(size_t n, size_t stream)
{
    void* p = nullptr;
    return ctr::ws_alloc(&p, n, (hipStream_t)stream) == hipSuccess ? p : nullptr;
}
int give(void* p, size_t stream) { return ctr::ws_free(p, (hipStream_t)stream); }
size_t held() { return g_bytes; }
int blocks() { return (int)g_live.size(); }
int events() { return g_events; }
void room(size_t n) { g_room = n; }
void busy(int b) { g_busy = b != 0; }
int release() { return ctr_release_workspace(); }

// in_parts over n slices of `bytes`: a part allocates its scratch and, where that
// fails, is done slice by slice.  log: (first, count) of each call that did its work.
int parts(int n, size_t bytes, int* log, int* nlog, int* rc)
{
    *nlog = 0;
    const auto part = [&](int b, int count) -> int {
        void* p = nullptr;
        const int e = ctr::ws_part(&p, count * bytes, nullptr);
        if (e) return e;
        log[2 * *nlog] = b;
        log[2 * *nlog + 1] = count;
        ++*nlog;
        CTR_HIP(ctr::ws_free(p, nullptr));
        return 0;
    };
    *rc = ctr::in_parts(n, bytes, part, [&](int b, int count) {
        return ctr::one_by_one(b, count, [&](int i) { return part(i, 1); });
    });
    return 0;
}
}
"""


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    d = tmp_path_factory.mktemp("ws")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    (d / "ws.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-Wl,-Bsymbolic",
                    "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}", f"-I{ROOT}/ct_recon_extensions_amd/csrc",
                    f"-I{rocm}/include", str(d / "ws.cpp"), "-o", str(d / "ws.so")], check=True)
    return d / "ws.so"


@pytest.fixture
def ws(built, tmp_path):
    shutil.copy(built, tmp_path / "ws.so")  # a copy has state of its own
    lib = C.CDLL(str(tmp_path / "ws.so"))
    lib.take.restype, lib.take.argtypes = C.c_void_p, [C.c_size_t, C.c_size_t]
    lib.give.argtypes = [C.c_void_p, C.c_size_t]
    lib.held.restype = C.c_size_t
    lib.room.argtypes = [C.c_size_t]
    return lib


def test_kept_bytes_and_blocks_are_bounded(ws):
    got = [ws.take(200 << 20, 1) for _ in range(10)]
    assert all(got) and ws.blocks() == 10
    for p in got:
        assert ws.give(p, 1) == 0
    assert 0 < ws.held() <= GIB
    assert ws.release() == 0 and ws.held() == 0 and ws.events() == 0
    got = [ws.take(1 << 16, 1) for _ in range(100)]
    for p in got:
        ws.give(p, 1)
    assert ws.blocks() <= 64
    # one block larger than all that may be kept is not kept
    p = ws.take(3 * GIB, 1)
    ws.give(p, 1)
    assert ws.held() <= GIB


def test_release_gives_everything_back(ws):
    p = ws.take(512 << 20, 1)
    ws.give(p, 1)
    assert ws.held() >= 512 << 20
    q = ws.take(1 << 20, 1)  # a block in use stays
    assert ws.release() == 0
    assert ws.held() == 1 << 20
    ws.give(q, 1)
    assert ws.release() == 0 and ws.held() == 0 and ws.events() == 0


def test_blocks_are_shared_between_streams_only_when_done(ws):
    p = ws.take(1 << 20, 1)
    ws.give(p, 1)
    ws.busy(1)
    assert ws.take(1 << 20, 2) != p
    assert ws.take(1 << 20, 1) == p
    ws.give(p, 1)
    ws.busy(0)
    assert ws.take(1 << 20, 2) == p


def test_kept_blocks_make_room(ws):
    ws.room(GIB)
    p = ws.take(700 << 20, 1)
    ws.give(p, 1)
    # too small for the next call, and no room beside it
    assert ws.take(900 << 20, 2) is not None
    assert ws.blocks() == 1


@pytest.mark.parametrize("n", [1, 16, 18, 40])
def test_batches_without_room_go_slice_by_slice(ws, n):
    log, nlog, rc = (C.c_int * 200)(), C.c_int(), C.c_int()

    def run(room):
        ws.release()
        ws.room(room)
        ws.parts(n, C.c_size_t(100 << 20), log, C.byref(nlog), C.byref(rc))
        calls = [(log[2 * i], log[2 * i + 1]) for i in range(nlog.value)]
        return rc.value, calls

    code, calls = run(1 << 40)
    assert code == 0 and calls == [(b, min(16, n - b)) for b in range(0, n, 16)]
    code, calls = run(150 << 20)  # one slice at a time fits
    assert code == 0 and calls == [(b, 1) for b in range(n)]
    code, calls = run(50 << 20)  # nothing does
    assert code != 0 and calls == []
