"""Batches of 4 and more slices (groups of 4 interleaved, last group padded)
against the same slices one at a time (one-slice layout), Siddon pair and DD
forward: 1e-6 of the largest value, the FP32 reordering of a ray's or pixel's sum
(the bar every launch shape is held to).  A slice of NaN and one of infinities
leave the others' bits unchanged.  Sizes: images below one 32 x 32 tile, a cell
over and nx != ny; bins beyond the image."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nu,nview,ns", [(5, 7, 30, 9, 4), (33, 31, 60, 12, 5), (32, 65, 90, 17, 7),
                                               (70, 40, 64, 31, 9), (96, 97, 200, 20, 33)])
def test_batch_equals_single_slices(nx, ny, nu, nview, ns):
    from reconnet_amd.torch_ops import FanPlan

    d = 260.0 / max(nx, ny)
    geo = FanGeometry(nx=nx, ny=ny, dx=d, dy=d, nu=nu, nview=nview, da=0.7 / nu, dsd=1085.6, dso=595.0, off_a=0.25)
    plan = FanPlan(geo)
    rng = np.random.default_rng(nx + ns)
    x = torch.from_numpy(rng.uniform(0, 1, (ns, nx, ny)).astype(np.float32)).cuda()
    y = torch.from_numpy(rng.uniform(0, 1, (ns, nu, nview)).astype(np.float32)).cuda()
    for src, run in ((x, lambda t: plan.forward(t, "siddon")), (y, lambda t: plan.backward(t, "siddon")),
                     (x, lambda t: plan.forward(t, "dd"))):
        out = run(src)
        for s in range(ns):
            one = run(src[s:s + 1].contiguous())[0]
            assert float((out[s] - one).abs().max() / one.abs().max()) <= 1e-6, s
        bad = src.clone()
        bad[1] = float("nan")
        bad[ns - 2] = float("inf")
        outb = run(bad)
        for s in range(ns):
            if s not in (1, ns - 2):
                assert torch.equal(outb[s], out[s]), s
