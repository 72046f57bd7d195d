"""The Siddon backprojection by tiles and of fewer than 4 slices, every launch shape,
against the per-pixel gathers that serve every geometry (the last shape of a batch of
4 and more slices, which the parity tests hold to the oracle), a few views at a time
and added in FP64: the same weights from the same ray table, so 1e-6 of the largest
value, the FP32 rounding of the sums.  And a ragged batch's Siddon and
DD adjoint against one-slice plan calls bit for bit (both sum the views in the same
fixed segments).  Sizes: images below a tile and a pixel over it, nx != ny, fewer views than
segments, more than 64 views of one wave, windows wider than a staged chunk, detectors
that miss most tiles, 1 to 33 slices, negative bin spacing; the last geometries'
pixels are too coarse for tiles."""

import numpy as np
import pytest
import torch

from reconnet_amd.geometry import FanGeometry

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, pixel, nu, bin scale, nview, slices
    (5, 3, 3.0, 40, 1.0, 3, 1), (8, 9, 6.0, 33, 2.0, 7, 2), (33, 17, 4.0, 90, 1.0, 9, 3), (40, 64, 3.0, 700, 0.25, 30, 5),
    (64, 40, 2.0, 64, -1.2, 24, 9), (72, 72, 1.5, 150, 1.0, 600, 33), (6, 7, 60.0, 60, 10.0, 12, 2),
    (6, 7, 60.0, 60, 10.0, 12, 5),
]


def _geo(nx, ny, d, nu, s, nview):
    return FanGeometry(nx=nx, ny=ny, dx=d, dy=d, nu=nu, nview=nview, da=s * 1.2 / 1085.6, dsd=1085.6, dso=595.0,
                       off_a=0.3)


@pytest.mark.parametrize("nx,ny,d,nu,s,nview,slices", CASES)
def test_siddon_bp_shapes(nx, ny, d, nu, s, nview, slices):
    from reconnet_amd._lib import autotune, autotune_pin
    from reconnet_amd.torch_ops import FanPlan

    geo = _geo(nx, ny, d, nu, s, nview)
    plan = FanPlan(geo)
    y = np.random.default_rng(nu + nview).uniform(0, 1, (slices, nu, nview)).astype(np.float32)
    t = torch.from_numpy(y).cuda()
    batch = t if slices >= 4 else t.repeat(4, 1, 1)

    def shapes(x):
        autotune(enable=True, reset=True)
        plan.backward(x, "siddon")
        return [len(ms) for k, (_, ms) in autotune().items() if k[0] == 2][0]

    outs = []
    try:
        n = shapes(batch)
        autotune_pin("siddon_bp", n - 1)
        ref = torch.zeros((slices, nx, ny), dtype=torch.float64, device="cuda")
        for v in range(0, nview, 3):
            few = torch.zeros_like(batch)
            few[:, :, v:v + 3] = batch[:, :, v:v + 3]
            ref += plan.backward(few, "siddon")[:slices]
        autotune_pin("siddon_bp", None)
        # (a batch's shapes end with the 10 gathers)
        for c in range(n - 10 if slices >= 4 else shapes(t)):
            autotune_pin("siddon_bp", c)
            outs.append(plan.backward(t, "siddon"))
            assert float((outs[-1] - ref).abs().max() / ref.abs().max()) <= 1e-6, c
            autotune_pin("siddon_bp", None)
    finally:
        autotune_pin("siddon_bp", None)
        autotune(enable=True, reset=True)
    if slices < 4:
        assert all(torch.equal(o, outs[0]) for o in outs)


def test_ragged_batch_equals_single_slices():
    from reconnet_amd.ragged import RaggedFanBatch
    from reconnet_amd.torch_ops import FanPlan

    geos = [_geo(*CASES[k][:6]) for k in (2, 2, 2, 2, 2, 5, 0, 6, 6, 4)]
    rb = RaggedFanBatch(geos)
    rng = np.random.default_rng(5)
    ys = [torch.from_numpy(rng.uniform(0, 1, (g.nu, g.nview)).astype(np.float32)).cuda() for g in geos]
    for kind, adj in (("siddon", "siddon"), ("dd", "dd_adjoint")):
        out = rb.backward(torch.cat([y.reshape(-1) for y in ys]), kind)
        off = 0
        for g, y in zip(geos, ys):
            n = g.nx * g.ny
            one = FanPlan(g).backward(y[None].contiguous(), adj)
            assert torch.equal(out[off:off + n], one.reshape(-1)), (kind, g.nx)
            off += n
