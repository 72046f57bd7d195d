"""A NaN or an infinity in one sinogram bin stays with the pixels that meet the bin
(and, where zero-weight candidates are read, their direct neighbours): the fan
backprojections of one slice, of several and by every launch shape.  The pixels that
meet a bin are those with a non-zero backprojection of that bin alone."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry

pytestmark = pytest.mark.gpu

KINDS = {"siddon": ("siddon_bp", (2,)), "dd": (None, ()), "dd_fbp": (None, ()), "dd_adjoint": ("dd_adjoint", (4,))}


@pytest.mark.parametrize("slices", [1, 5, 20])
@pytest.mark.parametrize("kind", list(KINDS))
def test_nonfinite_bins_stay_local(kind, slices):
    from reconnet_amd._lib import autotune, autotune_pin
    from reconnet_amd.torch_ops import FanPlan

    nx, ny, nu, nview = 70, 52, 100, 40
    geo = FanGeometry(nx=nx, ny=ny, dx=3.0, dy=3.0, nu=nu, nview=nview, da=0.45 / nu, dsd=1085.6, dso=595.0, off_a=0.3)
    plan = FanPlan(geo)
    y = torch.from_numpy(np.random.default_rng(1).uniform(0.1, 1, (slices, nu, nview)).astype(np.float32)).cuda()
    name, ids = KINDS[kind]
    try:
        autotune(enable=True, reset=True)
        plan.backward(y, kind)
        n = [len(ms) for k, (_, ms) in autotune().items() if k[0] in ids]
        for c in range(n[0]) if n else [None]:
            if name:
                autotune_pin(name, c)
            for v, k, bad in ((0, 50, float("nan")), (7, 3, float("inf")), (23, 99, float("nan")), (31, 41, float("inf"))):
                one = torch.zeros_like(y)
                one[slices // 2, k, v] = 1.0
                hit = plan.backward(one, kind) != 0
                z = y.clone()
                z[slices // 2, k, v] = bad
                out = plan.backward(z, kind)
                near = torch.nn.functional.max_pool2d(hit.float()[None], 3, 1, 1)[0] > 0
                assert bool(torch.isfinite(out[~near]).all()), (kind, c, v, k)
                if kind in ("dd", "dd_fbp") and bad == float("inf"):
                    assert bool((out[hit] == bad).all()), (kind, c, v, k)
    finally:
        if name:
            autotune_pin(name, None)
        autotune(enable=True, reset=True)
