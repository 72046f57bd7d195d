"""The staged DD adjoint at its edges, as the transpose of the forward
projector: <A x, y> = <x, A' y> in FP64 sums for every slice (bar 2e-6, the
FP32 rounding of a line's footprint, about 1e-5 of a bin per term, averaged over
the >= 1e3 terms of either side), and one slice equal to the same slice in a
batch bit for bit (the view segments are summed in one order by every launch
shape).  Sizes: images smaller than a tile and a few pixels over it, fewer
views than segments, windows wider than a staged chunk (fine bins), detectors
that miss most tiles, 1 to 33 slices."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, pixel, nu, bin scale, nview, slices
    (5, 3, 9.0, 40, 1.0, 3, 1), (8, 9, 6.0, 33, 2.0, 7, 2), (33, 17, 4.0, 90, 1.0, 9, 3),
    (40, 64, 3.0, 700, 0.25, 30, 5), (64, 40, 2.0, 64, 1.2, 24, 9), (72, 72, 1.5, 150, 1.0, 41, 33),
]


@pytest.mark.parametrize("nx,ny,d,nu,s,nview,slices", CASES)
def test_transpose_and_batch(nx, ny, d, nu, s, nview, slices):
    from reconnet_amd._lib import autotune, autotune_pin
    from reconnet_amd.torch_ops import FanPlan

    geo = FanGeometry(nx=nx, ny=ny, dx=d, dy=d, nu=nu, nview=nview, da=s * 1.2 / 1085.6, dsd=1085.6, dso=595.0,
                      off_a=0.3)
    plan = FanPlan(geo)
    rng = np.random.default_rng(nu + nview)
    x = torch.from_numpy(rng.uniform(0, 1, (slices, nx, ny)).astype(np.float32)).cuda()
    y = torch.from_numpy(rng.uniform(0, 1, (slices, nu, nview)).astype(np.float32)).cuda()
    ax = plan.forward(x, "dd")
    try:
        autotune(enable=True, reset=True)
        plan.backward(y, "dd_adjoint")
        n = [len(ms) for k, (_, ms) in autotune().items() if k[0] == 4][0]
        outs = []
        for c in range(n):
            autotune_pin("dd_adjoint", c)
            outs.append(plan.backward(y, "dd_adjoint"))
            one = plan.backward(y[-1:].contiguous(), "dd_adjoint")
            assert torch.equal(one[0], outs[-1][-1])
    finally:
        autotune_pin("dd_adjoint", None)
        autotune(enable=True, reset=True)
    for c in range(1, n):
        assert torch.equal(outs[c], outs[0]), c
    lhs = (ax.double() * y.double()).sum((1, 2))
    rhs = (x.double() * outs[0].double()).sum((1, 2))
    assert float(((lhs - rhs).abs() / lhs.abs()).max()) <= 2e-6


def test_ragged_batch_of_ordinary_and_very_long_images_equals_single_slices():
    # a slice whose image reaches past the source's line in some view (870 mm of 1190:
    # FanK::dwide is 0) leaves the bits of the others as those of calls of their own
    from reconnet_amd.geometry import FanGeometry
    from reconnet_amd.ragged import RaggedFanBatch
    from reconnet_amd.torch_ops import FanPlan

    a, b = (FanGeometry(nx=nx, ny=ny, dx=1.0, dy=dy, nu=140, nview=33, da=da, dsd=1085.6, dso=595.0)
            for nx, ny, dy, da in ((48, 48, 1.0, 1.2 / 1085.6), (8, 64, 13.6, 0.0143)))
    geos = [a, b, a, a, b]
    rng = np.random.default_rng(8)
    ys = [torch.from_numpy(rng.uniform(0, 1, (g.nu, g.nview)).astype(np.float32)).cuda() for g in geos]
    out = RaggedFanBatch(geos).backward(torch.cat([y.reshape(-1) for y in ys]), "dd")
    for g, y, o in zip(geos, ys, out.split([g.nx * g.ny for g in geos])):
        one = FanPlan(g).backward(y[None].contiguous(), "dd_adjoint").reshape(-1)
        assert torch.equal(o, one), (g.nx, float((o - one).abs().max()))
