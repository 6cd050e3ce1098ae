"""Backprojection at the edges of sinograms and detectors, against the oracle at the
suite's 1e-5 relative L2.  Where the first view's first tap is channel 0, its span
starts at channel -1, before the sinogram, four (or two) channels a lane, and the
channels from 0 on still count."""
import math

import pytest
import torch

from oracle import oracle as O
from tests.conftest import randn, rel_l2

pytestmark = pytest.mark.gpu
TOL32 = 1e-5


@pytest.mark.parametrize("n", [1, 2, 4])
@pytest.mark.parametrize("first", [0.3, 0.6, 0.95])
def test_first_channels_of_the_first_view(n, first):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ct_recon_extensions_amd as F
    # the tile reaches farthest in view 0, so all views are inside the detector
    ns, na, start = 48, 200, math.pi / 4
    reach = 7.5 * (math.cos(start) + math.sin(start))  # of the tile in view 0, both ways
    g = dict(nx=16, ny=16, na=na, ns=ns, dx=1.0, dy=1.0, ds=1.0, offset_x=0.0, offset_y=0.0,
             offset_s=first + reach - (ns - 1) / 2, orbit_start=start, orbit=math.pi / na)
    og = O.geom(**g)
    t = O.par_prep(og)
    proj = randn(1600 + n, (n, na, ns))
    proj[:, 0, :4] *= 10.0
    out = F.parallel_backprojection_2d(
        torch.from_numpy(proj).cuda(), img_shape=[16, 16], img_space=[1.0, 1.0],
        proj_shape=[na, ns], channel_space=1.0, channel_offset=g["offset_s"], orbit_start=start,
        orbit=g["orbit"]).cpu().numpy()
    for b in range(n):
        assert rel_l2(out[b], O.par_bp(og, proj[b], t)) < TOL32, b


@pytest.mark.parametrize("kind", ["ragged", "fan"])
def test_first_channels_of_the_first_fan_view(kind):
    """The same for a fan, alone and as a ragged problem's tile."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import numpy as np

    import ct_recon_extensions_amd as F
    from ct_recon_extensions_amd import ragged
    from ct_recon_extensions_amd.geometry import FanBackprojection2DAngleParam
    ns, na, n, dx, ds, dso, dsd = 64, 200, 16, 0.7, 1.3, 595.0, 1085.6
    # the first view is the one in which the tile reaches farthest, so all views are
    # inside the detector
    x = (np.arange(n) - (n - 1) / 2) * dx
    y = x[::-1, None]

    def first(b):
        r, d = x * np.cos(b) + y * np.sin(b), dso + x * np.sin(b) - y * np.cos(b)
        return (np.arctan2(r, d) * dsd / ds).min()

    start = min(2 * math.pi / na * np.arange(na), key=first)
    off = 0.6 - first(start) - (ns - 1) / 2
    angles = start + 2 * math.pi / na * np.arange(na)
    og = O.geom(nx=n, ny=n, na=na, ns=ns, dx=dx, dy=dx, ds=ds, offset_x=0.0, offset_y=0.0,
                offset_s=off, orbit_start=start, orbit=2 * math.pi / na, dso=dso, dsd=dsd)
    proj = randn(1650, (na, ns))
    proj[0, :4] *= 10.0
    want = O.fan_bp(og, proj, O.fan_prep(og))
    if kind == "fan":
        out = F.fan_backprojection_2d(
            torch.from_numpy(proj)[None].cuda(), img_shape=[n, n], img_space=[dx, dx],
            proj_shape=[na, ns], channel_space=ds, channel_offset=off, orbit_start=start,
            orbit=2 * math.pi / na, dso=dso, dsd=dsd)[0]
    else:
        p = FanBackprojection2DAngleParam(ns, na, ds, off, n, n, dx, dx, 0.0, 0.0, dso, dsd)
        plan = ragged.RaggedFanBackprojection2DAngle([p], [angles], autotune=False, tile=0,
                                                     vchunk=16)
        plan.projs[0].copy_(torch.from_numpy(proj))
        out = plan()[0]
    out = out.cpu().numpy()
    # (scales differ by a constant)
    assert rel_l2(out / np.linalg.norm(out), want / np.linalg.norm(want)) < TOL32


def test_ragged_sinogram_of_more_than_4_gib():
    """The stream tile reaches a sinogram through 31 bits of bytes; a longer one is the
    engine tile's.  2^28 channels, of which the image uses the middle 120."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import numpy as np

    from ct_recon_extensions_amd import ragged
    from ct_recon_extensions_amd.geometry import FanBackprojection2DAngleParam
    na, n, few, ns = 5, 40, 120, 1 << 28
    angles = 2 * math.pi / na * np.arange(na)
    og = O.geom(nx=n, ny=n, na=na, ns=few, dx=0.7, dy=0.7, ds=1.3, offset_x=0.0, offset_y=0.0,
                offset_s=0.0, orbit_start=0.0, orbit=2 * math.pi / na, dso=595.0, dsd=1085.6)
    proj = randn(1660, (na, few))
    want = O.fan_bp(og, proj, O.fan_prep(og))
    p = FanBackprojection2DAngleParam(ns, na, 1.3, 0.0, n, n, 0.7, 0.7, 0.0, 0.0, 595.0, 1085.6)
    plan = ragged.RaggedFanBackprojection2DAngle([p], [angles], autotune=False, tile=0, vchunk=16)
    a = (ns - few) // 2
    plan.projs[0][:, a:a + few] = torch.from_numpy(proj).cuda()
    out = plan()[0].cpu().numpy()
    assert rel_l2(out / np.linalg.norm(out), want / np.linalg.norm(want)) < TOL32


@pytest.mark.parametrize("n", [1, 2, 4])
def test_float64_integer_positions_read_one_channel(n):
    """A pixel whose position is a whole channel (the central rays of an odd detector)
    reads that channel only, as the reference's floor(s) and ceil(s) do: inf and nan
    next to it stay out of its sum."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import numpy as np

    import ct_recon_extensions_amd as F
    ns, na, side = 45, 12, 33
    g = dict(nx=side, ny=side, na=na, ns=ns, dx=0.7, dy=0.7, ds=1.3, offset_x=0.0, offset_y=0.0,
             offset_s=0.0, orbit_start=0.0, orbit=2 * math.pi / na, dso=595.0, dsd=1085.6)
    og = O.geom(**g)
    t = O.fan_prep(og)
    proj = np.random.default_rng(1670).standard_normal((n, na, ns))
    c = (ns - 1) // 2
    proj[0, 0, c + 1], proj[0, 3, c + 1], proj[0, 5, c - 1] = np.inf, np.nan, -np.inf
    out = F.fan_backprojection_2d(
        torch.from_numpy(proj).cuda(), img_shape=[side, side], img_space=[0.7, 0.7],
        proj_shape=[na, ns], channel_space=1.3, channel_offset=0.0, orbit_start=0.0,
        orbit=g["orbit"], dso=595.0, dsd=1085.6).cpu().numpy()
    assert np.isfinite(out[0, 16, 16])
    for b in range(n):
        want = O.fan_bp(og, proj[b], t)
        np.testing.assert_array_equal(np.isfinite(out[b]), np.isfinite(want))
        ok = np.isfinite(want)
        assert rel_l2(out[b][ok], want[ok]) < 1e-12, b


@pytest.mark.parametrize("fan", [True, False])
@pytest.mark.parametrize("ns,offset_s", [(40, 0.0), (41, 11.0), (40, 0.25)])
@pytest.mark.parametrize("n", [1, 4, 16])
def test_pair_is_adjoint_on_truncated_detectors(fan, ns, offset_s, n):
    """Forward (runs of pixels) and transpose (pixel by pixel) where many tiles reach
    past the detector.  1e-6 for rounding, and one pixel-view that lies within rounding
    of the detector's end may count in one only: 1 / (pixels sqrt(views)) of the norms."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ct_recon_extensions_amd as F
    side, na = 96, 180
    kw = dict(img_shape=[side, side], img_space=[0.7, 0.7], proj_shape=[na, ns], channel_space=1.3,
              img_offset=[0.3, -0.7], channel_offset=offset_s, orbit_start=0.1,
              orbit=(2 if fan else 1) * math.pi / na)
    if fan:
        kw.update(dso=595.0, dsd=1085.6)
        A, At = F.fan_backprojection_2d, F.fan_backprojection_2d_grad
    else:
        A, At = F.parallel_backprojection_2d, F.parallel_backprojection_2d_grad
    x = torch.from_numpy(randn(1680, (n, na, ns))).cuda()
    y = torch.from_numpy(randn(1681, (n, side, side))).cuda()
    ax, aty = A(x, **kw).double(), At(y, **kw).double()
    gap = abs((ax * y).sum() - (x * aty).sum()) / (ax.norm() * y.double().norm())
    assert gap < 1e-6 + 1.0 / (side * side * math.sqrt(na))
