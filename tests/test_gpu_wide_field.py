"""Images that reach far out towards the source circle (fan angles of 40 to 60
degrees, where the polynomial arctangents leave their inner range and a tile's distance
from the source varies tenfold): the DD backprojections against the oracle (relative L2
1e-5, the parity bar), the Siddon one by tiles against the per-pixel gathers, a view at a
time and added in FP64 (1e-6 of the largest value: the same weights from the same FP32
ray table, which alone is 1.3e-5 from the oracle here), the DD adjoint as the transpose
of the DD projector (2e-6)."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry, fan_angles
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slices", [1, 4])
@pytest.mark.parametrize("n,d", [(64, 7.8), (300, 2.3)])
def test_wide_field(n, d, slices):
    import oracle as orc
    from reconnet_amd._lib import autotune, autotune_pin
    from reconnet_amd.torch_ops import FanPlan

    nu, nview = 400, 9
    geo = FanGeometry(nx=n, ny=n, dx=d, dy=d, nu=nu, nview=nview, da=2.0 / nu, dsd=1085.6, dso=595.0, off_a=0.25)
    rng = np.random.default_rng(n)
    deg = fan_angles(nview)
    plan = FanPlan(geo)
    x = rng.uniform(0, 1, (slices, n, n)).astype(np.float32)
    y = rng.uniform(0, 1, (slices, nu, nview)).astype(np.float32)
    tx, ty = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    og, yr = geo.oracle_geo(), y.reshape(slices, nu, nview, 1, 1)
    for out, ref in ((plan.backward(ty, "dd"), orc.dd_fan_bp(yr, deg, og, (n, n, 1), type_projector=0)),
                     (plan.backward(ty, "dd_fbp"), orc.dd_fan_bp(yr, deg, og, (n, n, 1), type_projector=1))):
        assert rel_l2(out.cpu().numpy(), np.asarray(ref).reshape(out.shape)) <= 1e-5
    batch = ty if slices >= 4 else ty.repeat(4, 1, 1)
    try:
        autotune(enable=True, reset=True)
        plan.backward(batch, "siddon")
        last = [len(ms) for k, (_, ms) in autotune().items() if k[0] == 2][0] - 1
        autotune_pin("siddon_bp", last)
        ref = torch.zeros((slices, n, n), dtype=torch.float64, device="cuda")
        for v in range(nview):
            one = torch.zeros_like(batch)
            one[:, :, v] = batch[:, :, v]
            ref += plan.backward(one, "siddon")[:slices]
    finally:
        autotune_pin("siddon_bp", None)
        autotune(enable=True, reset=True)
    assert float((plan.backward(ty, "siddon") - ref).abs().max() / ref.abs().max()) <= 1e-6
    ax = plan.forward(tx if slices >= 4 else tx.repeat(4, 1, 1), "dd")[:slices]
    lhs = (ax.double() * ty.double()).sum()
    rhs = (tx.double() * plan.backward(ty, "dd_adjoint").double()).sum()
    assert float(abs(lhs - rhs) / abs(lhs)) <= 2e-6
