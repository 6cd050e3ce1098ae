"""The run-polynomial BP kernels (bp_stream.hpp) at the sizes where they can go
wrong, against the oracle: every group size and its remainders (16, 8, 4, 2, 1
slices), fewer views than waves and view counts that split unevenly, images
smaller than a tile and with partial tiles, tiles that reach past the detector,
both run orders and the geometries that stay on the engine kernel, spans of one
and of two DMA rows.  Tolerance: the suite's 1e-5 relative L2 (positions are
within a few 1e-6 channel, i.e. a few 1e-6 on N(0, 1) sinograms)."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import randn, rel_l2

pytestmark = pytest.mark.gpu
TOL32 = 1e-5


@pytest.fixture(scope="module")
def F():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ct_recon_extensions_amd as F
    from ct_recon_extensions_amd import _lib
    _lib.load()
    return F


def kwargs(g, fan):
    kw = dict(img_shape=[g["ny"], g["nx"]], img_space=[g["dy"], g["dx"]],
              proj_shape=[g["na"], g["ns"]], channel_space=g["ds"],
              img_offset=[g["offset_y"], g["offset_x"]], channel_offset=g["offset_s"],
              orbit_start=g["orbit_start"], orbit=g["orbit"])
    return dict(kw, dso=g["dso"], dsd=g["dsd"]) if fan else kw


def geom(n, na, ns, dx, ds, fan=True, offset_s=0.25, ny=None):
    g = dict(nx=n, ny=ny or n, na=na, ns=ns, dx=dx, dy=dx, ds=ds, offset_x=0.3, offset_y=-0.7,
             offset_s=offset_s, orbit_start=0.1, orbit=(2 if fan else 1) * math.pi / na)
    return dict(g, dso=595.0, dsd=1085.6) if fan else g


# (geometry, slices)
FAN = [
    (geom(64, 90, 96, 0.7, 1.3), 1), (geom(64, 90, 96, 0.7, 1.3), 2),
    (geom(64, 90, 96, 0.7, 1.3), 3), (geom(50, 45, 80, 0.7, 1.3, ny=37), 5),
    (geom(50, 45, 80, 0.7, 1.3, ny=37), 9), (geom(33, 61, 70, 0.7, 1.3), 10),
    (geom(33, 61, 70, 0.7, 1.3), 18),
    (geom(40, 5, 64, 0.7, 1.3), 1), (geom(40, 7, 64, 0.7, 1.3), 8),    # fewer views than waves
    (geom(7, 33, 40, 0.7, 1.3), 4), (geom(17, 130, 40, 0.7, 1.3), 16),  # partial tiles
    (geom(96, 60, 40, 0.7, 1.3), 1), (geom(96, 60, 40, 0.7, 1.3), 4),   # truncated detector
    (geom(96, 60, 41, 0.7, 1.3, offset_s=11.0), 8),
    (geom(96, 60, 40, 0.7, 1.3), 2), (geom(96, 60, 40, 0.7, 1.3), 16),
    (geom(48, 70, 120, 1.6, 1.3), 1), (geom(48, 70, 120, 1.6, 1.3), 6),  # long runs
    (geom(32, 50, 64, 5.0, 2.0), 2),                                     # engine kernel
    (geom(64, 40, 400, 0.7, 0.35), 1), (geom(64, 40, 400, 0.7, 0.35), 4),  # two DMA rows a span
    (geom(64, 40, 400, 0.7, 0.35), 16),
    (geom(20, 1537, 48, 0.7, 1.3), 2),  # more views than the waves hold
    (geom(20, 1100, 48, 0.7, 1.3), 16), (geom(20, 1536, 48, 0.7, 1.3), 8),
]


@pytest.mark.parametrize("case", range(len(FAN)))
def test_fan_bp_stream_matches_oracle(F, case):
    g, n = FAN[case]
    og = O.geom(**g)
    t = O.fan_prep(og)
    proj = randn(900 + case, (n, g["na"], g["ns"]))
    out = F.fan_backprojection_2d(torch.from_numpy(proj).cuda(), **kwargs(g, True)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.fan_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 2, 4, 7, 16, 17])
@pytest.mark.parametrize("ns,offset_s", [(60, 0.0), (23, 5.5)])
def test_par_bp_stream_matches_oracle(F, n, ns, offset_s):
    g = geom(45, 50, ns, 1.0, 1.0, fan=False, offset_s=offset_s, ny=38)
    og = O.geom(**g)
    t = O.par_prep(og)
    proj = randn(950 + n, (n, g["na"], ns))
    out = F.parallel_backprojection_2d(torch.from_numpy(proj).cuda(),
                                       **kwargs(g, False)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.par_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 2, 4])
@pytest.mark.parametrize("ns", [24, 25, 26, 27])
def test_last_channels_of_the_last_view(F, n, ns):
    """One tile, one view a wave, the last view's taps ending at channel ns - 1:
    a 16-byte load there reaches past the sinogram's end, and the channels
    before the end still count."""
    g = geom(16, 8, ns, 1.0, 1.0, fan=False)
    last = g["orbit_start"] + 7 * g["orbit"]
    reach = ((7.5 + abs(g["offset_x"])) * abs(math.cos(last))
             + (7.5 + abs(g["offset_y"])) * abs(math.sin(last)))
    g["offset_s"] = ns - 1.3 - reach - (ns - 1) / 2
    og = O.geom(**g)
    t = O.par_prep(og)
    proj = randn(980 + ns, (n, 8, ns))
    out = F.parallel_backprojection_2d(torch.from_numpy(proj).cuda(),
                                       **kwargs(g, False)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.par_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 2, 3, 8, 11, 17])
@pytest.mark.parametrize("ns", [80, 31])
def test_fpt_stream_matches_oracle_and_noalloc(F, n, ns):
    from ct_recon_extensions_amd import _lib
    from ct_recon_extensions_amd.geometry import ParallelProjection2DParam, device_tables
    g = geom(40, 50, ns, 1.0, 1.1, fan=False)
    og = O.geom(**g)
    t = O.fp_grad_prep(og)
    proj = randn(970 + n, (n, g["na"], ns))
    x = torch.from_numpy(proj).cuda()
    out = F.parallel_projection_2d_grad(x, **kwargs(g, False))
    for b in range(n):
        assert rel_l2(out[b].cpu().numpy(), O.fp_grad(og, proj[b], t)) < TOL32, b
    # the allocation-free entry point stages the same spans: the same bits
    p = ParallelProjection2DParam(ns, g["na"], g["ds"], g["orbit"], g["offset_s"],
                                  g["orbit_start"], 40, 40, 1.0, 1.0, g["offset_x"], g["offset_y"])
    w, pos, usex = device_tables("fp_grad", p, x.device)
    got = torch.empty_like(out)
    _lib.call("ctr_fp_t_noalloc", C.byref(p.ctr()), 0, C.c_void_p(x.data_ptr()),
              C.c_void_p(got.data_ptr()), n, C.c_void_p(w.data_ptr()), C.c_void_p(pos.data_ptr()),
              C.c_void_p(usex.data_ptr()), 40,
              C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert torch.equal(got, out)


def test_nonfinite_samples_stay_in_their_pixels(F):
    """inf and nan samples reach the pixels whose taps they are, as in the
    engine kernel (an explicit launch shape), and no others."""
    from ct_recon_extensions_amd import _lib
    from ct_recon_extensions_amd.geometry import FanBackprojection2DParam, device_tables
    g = geom(60, 37, 44, 0.7, 1.3)  # truncated: edge and inner tiles
    proj = randn(990, (4, g["na"], g["ns"]))
    proj[0, 3, 20], proj[1, 36, 43], proj[2, 0, 0] = np.inf, np.nan, -np.inf
    x = torch.from_numpy(proj).cuda()
    out = F.fan_backprojection_2d(x, **kwargs(g, True))
    p = FanBackprojection2DParam(g["ns"], g["na"], g["ds"], g["orbit"], g["offset_s"],
                                 g["orbit_start"], 60, 60, 0.7, 0.7, 0.3, -0.7, 595.0, 1085.6)
    tabs = device_tables("fan", p, x.device)
    ref = torch.empty_like(out)
    _lib.call("ctr_fan_bp_ex", C.byref(p.ctr()), 0, C.c_void_p(x.data_ptr()),
              C.c_void_p(ref.data_ptr()), 4, *(C.c_void_p(t.data_ptr()) for t in tabs), p.scale,
              C.byref(_lib.CtrFanBpLaunch(0, 6, 4)),
              C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert torch.equal(torch.isfinite(out), torch.isfinite(ref))
    assert not torch.isfinite(out[:3]).all() and torch.isfinite(out[3]).all()
    one = F.fan_backprojection_2d(x[1:2], **kwargs(g, True))
    assert torch.equal(torch.isfinite(one), torch.isfinite(ref[1:2]))


def test_workspace_is_given_back(F):
    from ct_recon_extensions_amd import _lib
    g = geom(64, 90, 96, 0.7, 1.3)
    x = torch.from_numpy(randn(999, (4, 90, 96))).cuda()
    a = F.fan_backprojection_2d(x, **kwargs(g, True))
    torch.cuda.synchronize()
    _lib.call("ctr_release_workspace")
    assert torch.equal(a, F.fan_backprojection_2d(x, **kwargs(g, True)))


# (nx, ny, views, channels, ds, slices, orbit_start): partial row segments and
# chunks, groups with views of both branches, rays that run along an image edge
# or cross a pixel corner exactly (odd sizes, no offsets), few views (one per
# workgroup), coarse detectors (256 staged columns, and beyond: the FP64-position
# kernel), detectors narrower and wider than the image
FP = [(33, 33, 40, 47, 1.0, 1, 0.0), (33, 33, 40, 47, 1.0, 5, 0.0), (32, 32, 40, 47, 1.0, 4, 0.0),
      (64, 48, 37, 80, 1.0, 2, 0.1), (48, 64, 37, 80, 1.0, 3, -0.7), (5, 3, 9, 12, 1.0, 1, 0.0),
      (3, 70, 22, 90, 0.8, 4, 0.3), (130, 130, 6, 150, 1.0, 1, 0.05), (130, 130, 6, 150, 1.0, 6, 0.05),
      (90, 90, 45, 70, 2.0, 1, 0.2), (90, 90, 45, 70, 2.0, 4, 0.2), (90, 90, 45, 30, 4.5, 2, 0.2),
      (200, 200, 50, 41, 1.0, 1, 0.0), (65, 65, 72, 200, 0.7071067811865476, 9, 0.0),
      (257, 255, 16, 257, 1.0, 1, 0.7853981633974483)]


@pytest.mark.parametrize("case", range(len(FP)))
@pytest.mark.parametrize("offset", [0.0, 0.3])
def test_fp_stream_matches_oracle(F, case, offset):
    nx, ny, na, ns, ds, n, start = FP[case]
    g = dict(nx=nx, ny=ny, na=na, ns=ns, dx=1.0, dy=1.0, ds=ds, offset_x=offset, offset_y=-offset,
             offset_s=offset, orbit_start=start, orbit=math.pi / na)
    og = O.geom(**g)
    t = O.fp_prep(og)
    img = randn(1000 + case, (n, ny, nx))
    out = F.parallel_projection_2d(torch.from_numpy(img).cuda(), **kwargs(g, False)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.fp(og, img[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 4])
def test_fp_nonfinite_pixels_stay_in_their_rays(F, n):
    g = geom(40, 30, 60, 1.0, 1.0, fan=False)
    img = randn(1100, (n, 40, 40))
    img[0, 0, 39], img[0, 20, 11], img[n - 1, 39, 0] = np.inf, np.nan, -np.inf
    og = O.geom(**g)
    t = O.fp_prep(og)
    out = F.parallel_projection_2d(torch.from_numpy(img).cuda(), **kwargs(g, False)).cpu().numpy()
    for b in range(n):
        np.testing.assert_array_equal(np.isfinite(out[b]), np.isfinite(O.fp(og, img[b], t)))


# distance-driven pair on interleaved planes, bitwise: group sizes 8 and 4 and
# their remainders, footprints of one, two and many cells (and channels), spans
# and footprints cut by the image's and the detector's ends
@pytest.mark.parametrize("n", [1, 4, 5, 9])
@pytest.mark.parametrize("ds,ns,na", [(1.0, 51, 24), (0.3, 60, 9), (4.5, 14, 16), (1.0, 9, 8)])
def test_dd_planes_match_oracle_bitwise(F, n, ds, ns, na):
    g = geom(35, na, ns, 1.0, ds, fan=False, offset_s=0.0)
    g.update(offset_x=0.0, offset_y=0.0, orbit_start=0.0)
    og = O.geom(**g)
    img, proj = randn(1200 + n, (n, 35, 35)), randn(1210 + n, (n, na, ns))
    kw = kwargs(g, False)
    fp = F.parallel_projection_2d(torch.from_numpy(img).cuda(), method="disdriven", **kw)
    gr = F.parallel_projection_2d_grad(torch.from_numpy(proj).cuda(), method="disdriven", **kw)
    t, tg = O.fp_dd_prep(og), O.fp_dd_grad_prep(og)
    for b in range(n):
        np.testing.assert_array_equal(fp[b].cpu().numpy(), O.fp_dd(og, img[b], t))
        np.testing.assert_array_equal(gr[b].cpu().numpy(), O.fp_dd_grad(og, proj[b], tg))


def test_workspace_across_streams_and_threads(F):
    """Calls that need scratch, from several streams and threads at once and
    with changing sizes, give the results of calls one after the other."""
    import threading
    cases = [(geom(40 + 8 * k, 30 + k, 60 + 10 * k, 1.0, 1.0, fan=False), 1 + k % 5)
             for k in range(6)]
    xs = [torch.from_numpy(randn(1300 + k, (n, g["ny"], g["nx"]))).cuda()
          for k, (g, n) in enumerate(cases)]
    want = [F.parallel_projection_2d(x, **kwargs(g, False)) for x, (g, _) in zip(xs, cases)]
    torch.cuda.synchronize()
    bad = []

    def work(seed):
        st = torch.cuda.Stream()
        rng = np.random.default_rng(seed)
        with torch.cuda.stream(st):
            got = [(k, F.parallel_projection_2d(xs[k], **kwargs(cases[k][0], False)))
                   for k in rng.integers(0, len(cases), 60)]
        st.synchronize()
        bad.extend(k for k, y in got if not torch.equal(y, want[k]))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_captured_call_replays(F):
    """A captured call takes its scratch from the graph: replays with new
    inputs, eager work on other sizes in between."""
    g = geom(48, 40, 70, 1.0, 1.0, fan=False)
    kw = kwargs(g, False)
    x = torch.from_numpy(randn(1400, (4, 48, 48))).cuda()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        F.parallel_projection_2d(x, **kw)
    torch.cuda.current_stream().wait_stream(st)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = F.parallel_projection_2d(x, **kw)
    for k in range(4):
        x.copy_(torch.from_numpy(randn(1401 + k, (4, 48, 48))))
        graph.replay()
        torch.cuda.synchronize()
        got = y.clone()
        assert torch.equal(got, F.parallel_projection_2d(x, **kw)), k
        F.parallel_projection_2d(x[:2], **kw)


FAN64 = [
    (geom(64, 90, 96, 0.7, 1.3), 1), (geom(50, 45, 80, 0.7, 1.3, ny=37), 2),
    (geom(33, 61, 70, 0.7, 1.3), 3), (geom(17, 129, 40, 0.7, 1.3), 4),  # rounds of 128 views
    (geom(7, 257, 40, 0.7, 1.3), 7), (geom(96, 60, 41, 0.7, 1.3, offset_s=11.0), 5),
    (geom(40, 1, 64, 0.7, 1.3), 2), (geom(40, 20, 2, 0.7, 300.0, offset_s=0.1), 2),
    (geom(32, 50, 64, 6.0, 2.0), 3),  # |u| above 0.1: the plain kernel
    # pixels exactly at the first and at the last channel of the first view
    (dict(geom(33, 8, 32, 1.0, 1.3, offset_s=-15.5), offset_x=0.0, orbit_start=0.0), 1),
    (dict(geom(33, 8, 32, 1.0, 1.3, offset_s=15.5), offset_x=0.0, orbit_start=0.0), 2),
]


@pytest.mark.parametrize("case", range(len(FAN64)))
def test_fan_bp_float64_matches_oracle(F, case):
    """Tile anchors in FP64: positions are the reference's to a few 1e-13 channel
    (the rounding of s, |s| < 1e3, and of its offset), so 1e-12 relative L2."""
    g, n = FAN64[case]
    og = O.geom(**g)
    t = O.fan_prep(og)
    proj = np.random.default_rng(1100 + case).standard_normal((n, g["na"], g["ns"]))
    out = F.fan_backprojection_2d(torch.from_numpy(proj).cuda(), **kwargs(g, True))
    assert out.dtype == torch.float64
    out = out.cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.fan_bp(og, proj[b], t)) < 1e-12, b


@pytest.mark.parametrize("ns", [2, 3, 8, 15, 16, 17, 31, 255, 256, 257, 513, 1025, 1706])
def test_ramp_float64_matches_oracle(F, ns):
    """Rows around a lane's 4 outputs, a block's 8 samples, the near field's 15 taps
    and a wave's 256 outputs, up to the longest; sums of at most 853 FP64 products,
    so 1e-12 relative L2."""
    g = O.geom(ns=ns, nrow=5, ds=0.9, dsd=1085.6, type=1)
    x = np.random.default_rng(1200 + ns).standard_normal((5, ns))
    out = F.ramp_filter(torch.from_numpy(x).cuda(), ns, 5, 0.9, 1085.6, "fan").cpu().numpy()
    assert rel_l2(out, O.ramp(g, x, O.ramp_prep(g))) < 1e-12


@pytest.mark.parametrize("op", ["fan", "fp", "dd", "dd_grad"])
def test_batches_whose_scratch_comes_in_parts(F, op):
    """18 slices of 64 MiB: the scratch of 16 at a time; the last two equal a call of
    their own, bit for bit."""
    torch.manual_seed(7)
    if op == "fan":
        g = geom(16, 1500, 11185, 0.7, 1.3)
        x = torch.randn((18, 1500, 11185), device="cuda")
        call = lambda x: F.fan_backprojection_2d(x, **kwargs(g, True))
    else:
        g = geom(4096 if op != "dd_grad" else 24, 4 if op != "dd_grad" else 1500,
                 64 if op != "dd_grad" else 11185, 1.0, 1.0, fan=False)
        kw = kwargs(g, False)
        size = (4096, 4096) if op != "dd_grad" else (1500, 11185)
        x = torch.randn((18, *size), device="cuda")
        if op == "dd_grad":
            call = lambda x: F.parallel_projection_2d_grad(x, method="disdriven", **kw)
        else:
            method = "disdriven" if op == "dd" else "raydriven"
            call = lambda x: F.parallel_projection_2d(x, method=method, **kw)
    out = call(x)
    assert torch.equal(out[16:], call(x[16:]))
    assert torch.equal(out[:16], call(x[:16]))
