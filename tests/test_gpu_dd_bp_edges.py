"""The distance-driven backprojection (iterative and FBP) by tiles, every launch
shape, against the oracle: relative L2 1e-5, the bar of the fan parity tests.
Sizes: images below a tile and a pixel over it, nx != ny, fewer views than waves and
more than 64 of one wave, windows wider than a staged chunk (fine bins), detectors
that miss most tiles, 1 to 33 slices, negative bin spacing; the last geometry's
pixels are too coarse for tiles and keep the per-pixel kernels."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry, fan_angles
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, pixel, nu, bin scale, nview, slices
    (5, 3, 3.0, 40, 1.0, 3, 1), (8, 9, 6.0, 33, 2.0, 7, 2), (33, 17, 4.0, 90, 1.0, 9, 3),
    (40, 64, 3.0, 700, 0.25, 30, 5), (64, 40, 2.0, 64, -1.2, 24, 9), (72, 72, 1.5, 150, 1.0, 600, 33),
    (6, 7, 40.0, 60, 10.0, 12, 2), (6, 7, 40.0, 60, 10.0, 12, 5),
]


@pytest.mark.parametrize("nx,ny,d,nu,s,nview,slices", CASES)
def test_dd_bp_shapes(nx, ny, d, nu, s, nview, slices):
    import oracle as orc
    from reconnet_amd._lib import autotune, autotune_pin
    from reconnet_amd.torch_ops import FanPlan

    geo = FanGeometry(nx=nx, ny=ny, dx=d, dy=d, nu=nu, nview=nview, da=s * 1.2 / 1085.6, dsd=1085.6, dso=595.0,
                      off_a=0.3)
    plan = FanPlan(geo)
    y = np.random.default_rng(nu + nview).uniform(0, 1, (slices, nu, nview)).astype(np.float32)
    t = torch.from_numpy(y).cuda()
    for kind, tp, ids in (("dd", 0, (5, 10)), ("dd_fbp", 1, (7, 11))):
        name = kind.replace("dd", "dd_bp") if kind == "dd" else kind
        name += "_q" if slices >= 4 else ""
        ref = orc.dd_fan_bp(y.reshape(slices, nu, nview, 1, 1), fan_angles(nview), geo.oracle_geo(), (nx, ny, 1),
                            type_projector=tp)
        ref = np.asarray(ref).reshape(slices, nx, ny)
        try:
            autotune(enable=True, reset=True)
            plan.backward(t, kind)
            n = [len(ms) for k, (_, ms) in autotune().items() if k[0] == ids[slices >= 4]][0]
            for c in range(n):
                autotune_pin(name, c)
                assert rel_l2(plan.backward(t, kind).cpu().numpy(), ref) <= 1e-5, (kind, c)
        finally:
            autotune_pin(name, None)
            autotune(enable=True, reset=True)
