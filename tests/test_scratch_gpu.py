"""A call whose scratch the device has no room for gives the bits that it gives with
room.  The room is taken away by a hipMallocAsync of our own, which a child process puts
before the runtime's and which refuses blocks above a limit."""
import os
import subprocess
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu
ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))

SHIM = r"""
#include <cstddef>
#include <dlfcn.h>
static size_t g_limit = ~size_t{0};
static int g_refused = 0;
extern "C" {
void limit(size_t n) { g_limit = n; }
int refused() { return g_refused; }
int hipMallocAsync(void** p, size_t n, void* stream)
{
    using F = int (*)(void**, size_t, void*);
    static F real = (F)dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMallocAsync");
    if (n <= g_limit) return real(p, n, stream);
    ++g_refused;
    return 2;  // hipErrorOutOfMemory
}
}
"""

CHILD = r"""
import ctypes as C, math, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
shim.limit.argtypes = [C.c_size_t]
sys.path.insert(0, sys.argv[2])
import torch
import ct_recon_extensions_amd as F
from ct_recon_extensions_amd import _lib
_lib.load()
torch.manual_seed(3)
na, ns, side = 240, 96, 70
kw = dict(img_shape=[side, side], img_space=[0.7, 0.7], proj_shape=[na, ns], channel_space=1.3,
          orbit=math.pi / na)
fan = dict(kw, orbit=2 * math.pi / na, dso=595.0, dsd=1085.6)
ops = {
    "fan": lambda n: F.fan_backprojection_2d(sino[:n], **fan),
    "par": lambda n: F.parallel_backprojection_2d(sino[:n], **kw),
    "fp": lambda n: F.parallel_projection_2d(img[:n], **kw),
    "dd": lambda n: F.parallel_projection_2d(img[:n], method="disdriven", **kw),
    "ddg": lambda n: F.parallel_projection_2d_grad(sino[:n], method="disdriven", **kw),
}
sino = torch.randn((35, na, ns), device="cuda")
img = torch.randn((35, side, side), device="cuda")
for name, op in ops.items():
    for n in (2, 3, 5, 8, 9, 11, 17, 18, 35):
        shim.limit(1 << 40)
        want = op(n)
        torch.cuda.synchronize()
        _lib.call("ctr_release_workspace")
        shim.limit(65536)  # one slice's scratch, not two's
        before = shim.refused()
        got = op(n)
        torch.cuda.synchronize()
        assert shim.refused() > before, (name, n)
        assert torch.equal(got, want), (name, n)
        _lib.call("ctr_release_workspace")
print("same bits")
"""


def test_results_do_not_depend_on_free_memory(tmp_path):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    (tmp_path / "shim.cpp").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    so = str(tmp_path / "shim.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(tmp_path / "shim.cpp"), "-o", so, "-ldl"],
                   check=True)
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), so, ROOT], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "same bits" in r.stdout, r.stdout + r.stderr[-2000:]


def test_release_workspace_gives_memory_back_to_the_device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import math

    import ct_recon_extensions_amd as F
    kw = dict(img_shape=[16, 16], img_space=[0.7, 0.7], proj_shape=[1440, 5888], channel_space=1.3,
              orbit=2 * math.pi / 1440, dso=595.0, dsd=1085.6)
    x = torch.zeros((8, 1440, 5888), device="cuda")
    scratch = x.numel() * 4
    F.fan_backprojection_2d(x[:1], **kw)  # tables
    F.release_workspace()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    y = F.fan_backprojection_2d(x, **kw)
    torch.cuda.synchronize()
    kept = torch.cuda.mem_get_info()[0]
    assert before - kept >= scratch
    F.release_workspace(y.device)
    assert torch.cuda.mem_get_info()[0] - kept >= scratch


def test_calls_beside_another_threads_capture():
    """Operators that take scratch (kept blocks of other streams, new ones) while
    another thread captures a graph neither fail nor invalidate the capture."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ctypes as C
    import math
    import threading

    import ct_recon_extensions_amd as F
    from ct_recon_extensions_amd import _lib
    from ct_recon_extensions_amd.geometry import FanBackprojection2DParam, device_tables
    x = torch.randn((1, 90, 96), device="cuda")
    kw = dict(img_shape=[64, 64], img_space=[0.7, 0.7], proj_shape=[90, 96], channel_space=1.3,
              orbit=math.pi / 90)  # one slice: the captured call itself takes no scratch
    streams = [torch.cuda.Stream() for _ in range(3)]
    sinos = [torch.randn((n, 240, ns), device="cuda") for n, ns in ((4, 96), (16, 960), (3, 2000))]
    outs = [torch.empty((len(s), 64, 64), device="cuda") for s in sinos]

    def bp(k, stream):  # no allocation but the operator's own
        n, na, ns = sinos[k].shape
        p = FanBackprojection2DParam(ns, na, 1.3, 2 * math.pi / na, 0.0, 0.0, 64, 64, 0.7, 0.7,
                                     0.0, 0.0, 595.0, 1085.6)
        tabs = device_tables("fan", p, x.device)
        _lib.call("ctr_fan_bp", C.byref(p.ctr()), 0, C.c_void_p(sinos[k].data_ptr()),
                  C.c_void_p(outs[k].data_ptr()), n, *(C.c_void_p(t.data_ptr()) for t in tabs),
                  p.scale, C.c_void_p(stream.cuda_stream))

    want = F.parallel_backprojection_2d(x, **kw) * 2
    for k in range(2):  # kept blocks, last used on two streams; the third size has none
        bp(k, streams[0])
        bp(k, streams[1])
    bp(2, streams[0])
    torch.cuda.synchronize()
    F.release_workspace()
    for k in range(2):
        bp(k, streams[0])
    images = [o.clone() for o in outs]
    torch.cuda.synchronize()
    go, done, errors = threading.Event(), threading.Event(), []

    def work():
        go.wait(60)
        try:
            for k in (0, 1, 2, 0, 1):
                bp(k, streams[2])
        except Exception as e:  # noqa: BLE001
            errors.append(e)
        done.set()

    t = threading.Thread(target=work)
    t.start()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = F.parallel_backprojection_2d(x, **kw)
        go.set()
        assert done.wait(60)
        z = y * 2
    t.join()
    assert not errors
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, want)
    assert all(torch.equal(a, b) for a, b in zip(images, outs))
