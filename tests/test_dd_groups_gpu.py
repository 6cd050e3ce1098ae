"""Distance-driven pair and ray-driven FP where a batch's last slices join a padded group,
and where the gradient keeps the kernel without interleaved planes (few views, sinograms
of 2^31 elements and more): the distance-driven pair bitwise against the oracle, the
ray-driven FP's slices bitwise against calls of their own."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import randn
from tests.test_stream_gpu import geom, kwargs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ct_recon_extensions_amd as F
    return F


@pytest.mark.parametrize("n", [2, 9, 10, 12, 13, 17, 20])
@pytest.mark.parametrize("na", [7, 40, 41])
def test_dd_pair_bitwise(F, n, na):
    g = geom(35, na, 51, 1.0, 1.0, fan=False, offset_s=0.0)
    g.update(offset_x=0.0, offset_y=0.0, orbit_start=0.0)
    og = O.geom(**g)
    img, proj = randn(1800 + n, (n, 35, 35)), randn(1810 + n, (n, na, 51))
    kw = kwargs(g, False)
    fp = F.parallel_projection_2d(torch.from_numpy(img).cuda(), method="disdriven", **kw)
    gr = F.parallel_projection_2d_grad(torch.from_numpy(proj).cuda(), method="disdriven", **kw)
    t, tg = O.fp_dd_prep(og), O.fp_dd_grad_prep(og)
    for b in range(n):
        np.testing.assert_array_equal(fp[b].cpu().numpy(), O.fp_dd(og, img[b], t))
        np.testing.assert_array_equal(gr[b].cpu().numpy(), O.fp_dd_grad(og, proj[b], tg))


@pytest.mark.parametrize("side,na,n", [(32, 60, 5), (128, 90, 9), (70, 300, 17), (512, 6, 5)])
def test_fp_slice_has_its_bits_of_the_batch(F, side, na, n):
    """Padded into a group of four, alone, or in a call of its own."""
    kw = dict(img_shape=[side, side], img_space=[1.0, 1.0], proj_shape=[na, int(1.4 * side)],
              channel_space=1.0, orbit=math.pi / na)
    x = torch.from_numpy(randn(1820 + n, (n, side, side))).cuda()
    out = F.parallel_projection_2d(x, **kw)
    for b in (0, n - 2, n - 1):
        assert torch.equal(out[b], F.parallel_projection_2d(x[b:b + 1], **kw)[0]), b


def test_dd_gradient_of_a_sinogram_past_32_bits(F):
    """4.5e9 elements a slice, of which the image uses the middle 60 channels."""
    na, n, few, ns = 3, 24, 60, 1_500_000_000
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("36 GB of sinograms")
    g = geom(n, na, few, 1.0, 1.0, fan=False, offset_s=0.0)
    g.update(offset_x=0.0, offset_y=0.0, orbit_start=0.0)
    proj = randn(1830, (2, na, few))
    og = O.geom(**g)
    tg = O.fp_dd_grad_prep(og)
    x = torch.zeros((2, na, ns), device="cuda")
    a = (ns - few) // 2
    x[:, :, a:a + few] = torch.from_numpy(proj).cuda()
    out = F.parallel_projection_2d_grad(x, method="disdriven", **dict(kwargs(g, False),
                                                                      proj_shape=[na, ns]))
    del x
    torch.cuda.empty_cache()
    for b in range(2):  # positions near 7.5e8 are good to 1e-7 channel
        want = O.fp_dd_grad(og, proj[b], tg)
        assert np.linalg.norm(out[b].cpu().numpy() - want) < 1e-6 * np.linalg.norm(want)
