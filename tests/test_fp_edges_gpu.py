"""Ray-driven FP on sizes where rays stand exactly on the image's last column and
the staged width is a multiple of 64 columns (or one more, or one less): their
right tap, of weight 0, is a staged zero and not what the LDS held before (the
projection of a NaN image runs first).  Against the oracle, at the suite's 1e-5
relative L2."""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.conftest import randn, rel_l2

pytestmark = pytest.mark.gpu
TOL32 = 1e-5


@pytest.mark.parametrize("side,ns,ds", [(64, 64, 1.0), (63, 63, 1.0), (65, 65, 1.0), (128, 250, 1.0),
                                        (256, 378, 1.0), (256, 382, 1.0), (129, 253, 1.0),
                                        (195, 307, 1.0), (195, 311, 1.0), (128, 65, 2.0)])
def test_rays_on_the_last_column(side, ns, ds):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ct_recon_extensions_amd as F
    na = 90
    kw = dict(img_shape=[side, side], img_space=[1.0, 1.0], proj_shape=[na, ns], channel_space=ds,
              img_offset=[0.0, 0.0], channel_offset=0.0, orbit_start=0.0, orbit=math.pi / na)
    og = O.geom(nx=side, ny=side, na=na, ns=ns, dx=1.0, dy=1.0, ds=ds, offset_x=0.0, offset_y=0.0,
                offset_s=0.0, orbit_start=0.0, orbit=math.pi / na)
    img = randn(1500 + ns, (5, side, side))
    t = O.fp_prep(og)
    want = [O.fp(og, s, t) for s in img]
    for n in (1, 2, 4, 5):
        F.parallel_projection_2d(torch.full((n, side, side), float("nan"), device="cuda"), **kw)
        out = F.parallel_projection_2d(torch.from_numpy(img[:n]).cuda(), **kw).cpu().numpy()
        assert np.isfinite(out).all(), n
        for b in range(n):
            assert rel_l2(out[b], want[b]) < TOL32, (n, b)
