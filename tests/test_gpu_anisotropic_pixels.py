"""Fan projectors and backprojections on pixels with dx != dy, uneven angles, a
detector offset of several bins and a mirrored detector, against the oracle
(relative L2 1e-5, the parity bar), one slice and a batch; the DD adjoint as the
transpose of the DD projector (2e-6, as its edge test)."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slices", [1, 5])
@pytest.mark.parametrize("dx,dy,s,off", [(4.0, 1.5, 1.0, 3.5), (1.2, 3.0, -0.8, -2.25)])
def test_anisotropic_pixels(dx, dy, s, off, slices):
    import oracle as orc
    from reconnet_amd.torch_ops import FanPlan

    nx, ny, nu, nview = 45, 52, 110, 37
    geo = FanGeometry(nx=nx, ny=ny, dx=dx, dy=dy, nu=nu, nview=nview, da=s * 2.5 / 1085.6, dsd=1085.6, dso=595.0,
                      off_a=off)
    rng = np.random.default_rng(nu)
    deg = np.sort(rng.uniform(0, 2 * np.pi, nview)).astype(np.float32)
    plan = FanPlan(geo, deg)
    x = rng.uniform(0, 1, (slices, nx, ny)).astype(np.float32)
    y = rng.uniform(0, 1, (slices, nu, nview)).astype(np.float32)
    tx, ty = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    og, xr, yr = geo.oracle_geo(), x.reshape(slices, nx, ny, 1, 1), y.reshape(slices, nu, nview, 1, 1)
    for out, ref in ((plan.forward(tx, "dd"), orc.dd_fan_fp(xr, deg, og, nu)),
                     (plan.forward(tx, "siddon"), orc.siddon_fan_fp(xr, deg, og, nu)),
                     (plan.backward(ty, "siddon"), orc.siddon_fan_bp(yr, deg, og, (nx, ny, 1))),
                     (plan.backward(ty, "dd"), orc.dd_fan_bp(yr, deg, og, (nx, ny, 1), type_projector=0)),
                     (plan.backward(ty, "dd_fbp"), orc.dd_fan_bp(yr, deg, og, (nx, ny, 1), type_projector=1))):
        assert rel_l2(out.cpu().numpy(), np.asarray(ref).reshape(out.shape)) <= 1e-5
    lhs = (plan.forward(tx, "dd").double() * ty.double()).sum()
    rhs = (tx.double() * plan.backward(ty, "dd_adjoint").double()).sum()
    assert float(abs(lhs - rhs) / abs(lhs)) <= 2e-6
