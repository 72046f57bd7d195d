"""The ramp filter by matrix instructions at its edges, against the FP64 oracle:
relative L2 1e-6 (the near taps are summed in FP64, the far ones, under 1 % of the
taps' weight, in FP32: about 1e-7).  Rows around multiples of 16 and 64 samples, one
wave to several passes, rows too long for it, view counts around multiples of 16, and
a row of NaN, which stays alone."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu,nview,B,ftype", [(1, 3, 1, 0), (15, 17, 1, 2), (17, 16, 2, 0), (64, 5, 3, 1), (65, 33, 1, 3),
                                              (255, 31, 1, 2), (257, 20, 1, 0), (736, 18, 2, 2), (790, 7, 1, 0),
                                              (1000, 7, 1, 2)])
def test_filter_edges(nu, nview, B, ftype):
    import oracle as orc
    from reconnet_amd.torch_ops import FanPlan

    geo = FanGeometry(nx=8, ny=8, dx=4.0, dy=4.0, nu=nu, nview=nview, da=0.5 / max(nu, 8), dsd=1085.6, dso=595.0,
                      off_a=0.25)
    y = np.random.default_rng(nu).uniform(0, 1, (B, nu, nview)).astype(np.float32)
    plan = FanPlan(geo)
    t = torch.from_numpy(y).cuda()
    out = plan.filter(t, ftype)
    ref = np.asarray(orc.ramp_filter(y.reshape(B, nu, nview, 1, 1), geo.oracle_geo(), filter_type=ftype))
    assert rel_l2(out.cpu().numpy(), ref.reshape(B, nu, nview)) <= 1e-6
    bad = t.clone()
    bad[0, :, 1] = float("nan")
    outb = plan.filter(bad, ftype)
    keep = [v for v in range(nview) if v != 1]
    assert torch.equal(outb[:, :, keep], out[:, :, keep]) and bool(outb[0, :, 1].isnan().all())
