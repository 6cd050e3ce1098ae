"""The stream BP kernels (bp_stream.hpp) with the view counts that take a call to them
(stream_pays) and on both sides of those counts, against the oracle: every group size
and its remainders, images smaller than a tile and with partial tiles, tiles that reach
past the detector, both run orders, spans of one and of two DMA rows.  Tolerance: the
suite's 1e-5 relative L2 (positions are within a few 1e-6 channel, i.e. a few 1e-6 on
N(0, 1) sinograms)."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import randn, rel_l2
from tests.test_stream_gpu import geom, kwargs

pytestmark = pytest.mark.gpu
TOL32 = 1e-5


@pytest.fixture(scope="module")
def F():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ct_recon_extensions_amd as F
    return F


SMALL = geom(64, 240, 96, 0.7, 1.3)
CUT = geom(96, 250, 41, 0.7, 1.3, offset_s=11.0)
# (geometry, slices)
FAN = [(SMALL, n) for n in (1, 2, 3, 4, 5, 8, 9, 10, 15, 16, 17, 18, 24)]
FAN += [(CUT, n) for n in (1, 2, 4, 8, 16)]
FAN += [(geom(64, na, 96, 0.7, 1.3), n)  # about the counts of views
        for na, n in ((55, 1), (56, 1), (143, 2), (144, 3), (175, 4), (176, 16), (239, 17))]
FAN += [(geom(50, 203, 80, 0.7, 1.3, ny=37), 5), (geom(33, 181, 70, 0.7, 1.3), 10),
        (geom(7, 199, 40, 0.7, 1.3), 4), (geom(17, 197, 40, 0.7, 1.3), 16),
        (geom(48, 190, 120, 1.6, 1.3), 1), (geom(48, 190, 120, 1.6, 1.3), 6),  # long runs
        (geom(64, 180, 400, 0.7, 0.35), 1), (geom(64, 180, 400, 0.7, 0.35), 4),
        (geom(64, 180, 400, 0.7, 0.35), 16), (geom(40, 1536, 100, 0.7, 0.6), 16)]


@pytest.mark.parametrize("case", range(len(FAN)))
def test_fan_bp_matches_oracle(F, case):
    g, n = FAN[case]
    og = O.geom(**g)
    t = O.fan_prep(og)
    proj = randn(1700 + case, (n, g["na"], g["ns"]))
    out = F.fan_backprojection_2d(torch.from_numpy(proj).cuda(), **kwargs(g, True)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.fan_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 2, 4, 7, 16, 17])
@pytest.mark.parametrize("ns,offset_s", [(60, 0.0), (23, 5.5)])
def test_par_bp_matches_oracle(F, n, ns, offset_s):
    g = geom(45, 240, ns, 1.0, 1.0, fan=False, offset_s=offset_s, ny=38)
    og = O.geom(**g)
    t = O.par_prep(og)
    proj = randn(1750 + n, (n, g["na"], ns))
    out = F.parallel_backprojection_2d(torch.from_numpy(proj).cuda(),
                                       **kwargs(g, False)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.par_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 2, 4])
@pytest.mark.parametrize("ns", [24, 25, 26, 27])
def test_last_channels_of_the_last_view(F, n, ns):
    """The last view's taps end at channel ns - 1 and all views are inside: a 16-byte load
    there reaches past the sinogram's end, and the channels before the end still count."""
    g = geom(16, 200, ns, 1.0, 1.0, fan=False)
    g.update(offset_x=0.0, offset_y=0.0, orbit_start=math.pi / 4 - 199 * g["orbit"])
    g["offset_s"] = ns - 1.3 - 7.5 * math.sqrt(2.0) - (ns - 1) / 2
    og = O.geom(**g)
    t = O.par_prep(og)
    proj = randn(1760 + ns, (n, 200, ns))
    proj[:, -1, -4:] *= 10.0
    out = F.parallel_backprojection_2d(torch.from_numpy(proj).cuda(),
                                       **kwargs(g, False)).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.par_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("n", [1, 2, 3, 8, 11, 16])
@pytest.mark.parametrize("ns", [80, 31])
def test_fpt_matches_oracle_and_noalloc(F, n, ns):
    from ct_recon_extensions_amd import _lib
    from ct_recon_extensions_amd.geometry import ParallelProjection2DParam, device_tables
    g = geom(40, 240, ns, 1.0, 1.1, fan=False)
    og = O.geom(**g)
    t = O.fp_grad_prep(og)
    proj = randn(1770 + n, (n, g["na"], ns))
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
    """inf and nan samples reach the pixels whose taps they are, as in the engine kernel
    (an explicit launch shape), and no others."""
    from ct_recon_extensions_amd import _lib
    from ct_recon_extensions_amd.geometry import FanBackprojection2DParam, device_tables
    g = geom(60, 201, 44, 0.7, 1.3)  # truncated: edge and inner tiles
    proj = randn(1790, (4, g["na"], g["ns"]))
    proj[0, 3, 20], proj[1, 200, 43], proj[2, 0, 0] = np.inf, np.nan, -np.inf
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
