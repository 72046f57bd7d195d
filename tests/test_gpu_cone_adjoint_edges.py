"""The list-driven cone projectors against the FP64 oracle where their paths
change: up to 2, 3 and more rows per voxel, detector columns much finer than a
voxel (several list rounds), volumes taller than a workgroup's z block, fewer
views than a batch, detector rows that run against z, and a source close enough
that the row-sum tables take over (bar 1e-5 relative L2, the suite's parity bar)."""

import numpy as np
import pytest
import torch

import oracle as orc
from reconnet_amd.geometry import circular_cone_vectors
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

CASES = [  # nx, ny, nz, dz, nu, nv, du, dv, nview, dso, flip
    (9, 14, 20, 1.0, 20, 12, 2.0, 1.0, 5, 300.0, False),        # < 2 rows per voxel
    (17, 6, 11, 1.0, 30, 20, 1.3, 0.7, 33, 120.0, False),       # 2 to 3
    (8, 8, 10, 2.0, 24, 40, 1.3, 0.8, 17, 120.0, True),         # 3 to 7, rows against z
    (6, 7, 150, 0.5, 90, 30, 0.2, 1.0, 9, 120.0, False),        # fine columns, two z blocks
    (8, 8, 6, 4.0, 20, 60, 1.3, 0.5, 8, 90.0, False),           # more than 7: row sums
]


@pytest.mark.parametrize("nx,ny,nz,dz,nu,nv,du,dv,nview,dso,flip", CASES)
def test_cone_adjoint_paths(nx, ny, nz, dz, nu, nv, du, dv, nview, dso, flip):
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.torch_ops import ConePlan

    ctr, u, v, src = circular_cone_vectors(nview, dso, 200.0 + dso, th0=0.3)
    if flip:
        v = -v
    plan = ConePlan(nx, ny, nz, 1.0, 1.0, dz, nu, nv, du, dv, ctr, u, v, src, cx=0.3, cy=-0.2, cz=0.4, off_v=0.2)
    geo = dict(dx=1.0, dy=1.0, dz=dz, du=du, dv=dv, off_u=0.0, off_v=0.2, cx=0.3, cy=-0.2, cz=0.4)
    p = np.random.default_rng(nu + nv).uniform(0, 1, (1, nu, nview, nv, 1)).astype(np.float32)
    ref = orc.dd_cone_adj(p, ctr, u, v, src, geo, (nx, ny, nz))
    try:
        for c in range(3):
            autotune_pin("dd_cone_adj", c)
            assert rel_l2(plan.backward(torch.from_numpy(p).cuda(), "dd").cpu().numpy(), ref) <= 1e-5, c
    finally:
        autotune_pin("dd_cone_adj", None)


SIDDON = [  # nx, ny, nz, dz, nu, nv, du, dv, nview, dso, det (distance of the detector behind the axis), flip
    (9, 14, 20, 1.0, 20, 13, 2.0, 1.6, 5, 300.0, 200.0, False),     # < 2 rows, a level row
    (17, 6, 11, 1.0, 30, 20, 1.3, 0.8, 33, 120.0, 80.0, False),     # 2 to 3
    (8, 8, 10, 2.0, 24, 40, 1.3, 1.0, 17, 120.0, 80.0, True),       # 3 to 4, rows against z
    (8, 9, 12, 2.0, 24, 41, 1.3, 0.6, 7, 120.0, 80.0, False),       # 4 to 7, a level row
    (6, 7, 150, 0.5, 90, 30, 0.2, 1.0, 9, 120.0, 80.0, False),      # fine columns, two z blocks
    (16, 12, 9, 1.0, 40, 21, 0.6, 0.7, 11, 90.0, 3.0, False),       # the detector inside the volume
    (8, 8, 6, 4.0, 20, 60, 1.3, 0.5, 8, 90.0, 80.0, False),         # more than 7 rows: tested view by view
]


@pytest.mark.parametrize("nx,ny,nz,dz,nu,nv,du,dv,nview,dso,det,flip", SIDDON)
def test_siddon_cone_backprojection_paths(nx, ny, nz, dz, nu, nv, du, dv, nview, dso, det, flip):
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.torch_ops import ConePlan

    ctr, u, v, src = circular_cone_vectors(nview, dso, det + dso, th0=0.3)
    if flip:
        v = -v
    plan = ConePlan(nx, ny, nz, 1.0, 1.0, dz, nu, nv, du, dv, ctr, u, v, src, cx=0.3, cy=-0.2)
    geo = dict(dx=1.0, dy=1.0, dz=dz, du=du, dv=dv, off_u=0.0, off_v=0.0, cx=0.3, cy=-0.2, cz=0.0)
    p = np.random.default_rng(nu + nv).uniform(0, 1, (1, nu, nview, nv, 2)).astype(np.float32)
    ref = orc.siddon_cone_bp(p, ctr, u, v, src, geo, (nx, ny, nz))
    try:
        for c in range(3):
            autotune_pin("siddon_cone_bp", c)
            assert rel_l2(plan.backward(torch.from_numpy(p).cuda(), "siddon").cpu().numpy(), ref) <= 1e-5, c
    finally:
        autotune_pin("siddon_cone_bp", None)


def test_siddon_cone_backprojection_keeps_a_nan_in_its_rays():
    # a NaN detector cell reaches the voxels its ray meets (the forward
    # projection of each has the cell non-zero) and no others
    from reconnet_amd.torch_ops import ConePlan

    vecs = circular_cone_vectors(6, 120.0, 200.0, th0=0.3)
    plan = ConePlan(10, 10, 12, 1.0, 1.0, 1.0, 24, 18, 1.3, 1.0, *vecs)
    p = torch.rand((1, 24, 6, 18, 1), device="cuda")
    p[0, 11, 2, 7, 0] = float("nan")
    got = torch.isnan(plan.backward(p, "siddon"))
    q = torch.zeros_like(p)
    q[0, 11, 2, 7, 0] = 1.0
    assert torch.equal(got, plan.backward(q, "siddon") > 0)
    assert bool(got.any())


FORWARD = [  # nx, ny, nz, dz, nu, nv, du, dv, nview, dso, channels
    (9, 14, 40, 1.0, 20, 12, 1.0, 1.0, 5, 300.0, 1),       # z footprints under a voxel, inside the volume
    (9, 14, 40, 0.6, 20, 17, 1.0, 1.2, 5, 300.0, 2),       # one to two voxels; 32 rows a group
    (17, 6, 9, 0.3, 30, 70, 1.3, 1.4, 33, 120.0, 1),       # over two, and out of the volume; 16 rows a group
    (70, 67, 12, 1.0, 9, 33, 9.0, 1.0, 7, 200.0, 1),       # cells several voxels wide, two plane batches
    (8, 8, 10, 2.0, 300, 40, 0.1, 0.8, 3, 120.0, 1),       # columns much finer than a voxel
]


@pytest.mark.parametrize("nx,ny,nz,dz,nu,nv,du,dv,nview,dso,nc", FORWARD)
def test_cone_forward_paths(nx, ny, nz, dz, nu, nv, du, dv, nview, dso, nc):
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.torch_ops import ConePlan

    vecs = circular_cone_vectors(nview, dso, 200.0 + dso, th0=0.3)
    plan = ConePlan(nx, ny, nz, 1.0, 1.0, dz, nu, nv, du, dv, *vecs, cx=0.3, cy=-0.2, cz=0.4, off_v=0.2)
    geo = dict(dx=1.0, dy=1.0, dz=dz, du=du, dv=dv, off_u=0.0, off_v=0.2, cx=0.3, cy=-0.2, cz=0.4)
    x = np.random.default_rng(nu + nv).uniform(0, 1, (1, nx, ny, nz, nc)).astype(np.float32)
    ref = orc.dd_cone_fp(x, *vecs, geo, nu, nv)
    try:
        for c in range(2):
            autotune_pin("dd_cone_fp", c)
            assert rel_l2(plan.forward(torch.from_numpy(x).cuda(), "dd").cpu().numpy(), ref) <= 1e-5, c
    finally:
        autotune_pin("dd_cone_fp", None)


def test_cone_forward_keeps_a_nan_in_its_rays():
    # a NaN (or infinite) voxel reaches the rays that meet it or a cell next to it
    # (those of a volume of ones around it, 0 elsewhere) and no others, the corner
    # columns of the volume among the voxels
    from reconnet_amd.torch_ops import ConePlan

    n, nz = 21, 16
    vecs = circular_cone_vectors(7, 120.0, 200.0, th0=0.3)
    plan = ConePlan(n, n, nz, 1.0, 1.0, 1.0, 50, 18, 1.0, 1.0, *vecs)
    x = torch.rand((1, n, n, nz, 1), device="cuda")
    ref = plan.forward(x, "dd")
    for ix, iy in ((0, 0), (0, n - 1), (n - 1, 0), (10, 10)):
        for bad in (float("nan"), float("inf")):
            z = x.clone()
            z[0, ix, iy, 7, 0] = bad
            near = torch.zeros_like(x)
            near[0, max(ix - 1, 0):ix + 2, max(iy - 1, 0):iy + 2, 5:10] = 1.0
            met = plan.forward(near, "dd") > 0
            out = plan.forward(z, "dd")
            assert bool((~met).any()) and torch.equal(out[~met], ref[~met]), (ix, iy, bad)
            hit = torch.zeros_like(x)
            hit[0, ix, iy, 7, 0] = 1.0
            assert not bool(torch.isfinite(out[plan.forward(hit, "dd") > 0]).any())


@pytest.mark.parametrize("dist", [51.0, 56.0, 63.0, 95.0, 105.0, 120.0])
def test_cone_adjoint_at_exactly_seven_rows_per_voxel(dist):
    # the nearest plane, `dist` from the source, has 7 rows per voxel: the bound up to
    # which the adjoint takes row windows, in FP64 and not in FP32's reciprocal.  One view
    # along x, 8 planes of 1 mm, the detector 7 x dist behind the source, cells as high as
    # a voxel.
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.torch_ops import ConePlan

    nx, ny, nz, nu, nv = 8, 5, 6, 30, 60
    src = np.array([[-(dist + 3.5), 0.0, 0.0]], np.float32)
    ctr = np.array([[7.0 * dist - (dist + 3.5), 0.0, 0.0]], np.float32)
    u, v = np.array([[0.0, 1.0, 0.0]], np.float32), np.array([[0.0, 0.0, 1.0]], np.float32)
    plan = ConePlan(nx, ny, nz, 1.0, 1.0, 1.0, nu, nv, 2.0, 1.0, ctr, u, v, src)
    geo = dict(dx=1.0, dy=1.0, dz=1.0, du=2.0, dv=1.0, off_u=0.0, off_v=0.0, cx=0.0, cy=0.0, cz=0.0)
    p = np.random.default_rng(3).uniform(0, 1, (1, nu, 1, nv, 1)).astype(np.float32)
    ref = orc.dd_cone_adj(p, ctr, u, v, src, geo, (nx, ny, nz))
    try:
        for c in range(3):
            autotune_pin("dd_cone_adj", c)
            assert rel_l2(plan.backward(torch.from_numpy(p).cuda(), "dd").cpu().numpy(), ref) <= 1e-5, c
    finally:
        autotune_pin("dd_cone_adj", None)


@pytest.mark.parametrize("nx,nz,dz,nu,nv,du,dv,dso", [(10, 20, 1.0, 20, 12, 2.0, 1.0, 300.0),     # up to 2 rows per voxel
                                                      (17, 11, 1.0, 30, 20, 1.3, 0.7, 120.0),     # 2 to 3
                                                      (8, 10, 1.6, 24, 40, 1.3, 0.8, 120.0)])     # 3 to 7
def test_cone_adjoint_keeps_a_nan_in_its_rays(nx, nz, dz, nu, nv, du, dv, dso):
    # a NaN or infinite detector cell reaches the voxels that its footprint meets (those
    # of the cell's own backprojection) and no others, by every row-window shape
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.torch_ops import ConePlan

    plan = ConePlan(nx, nx, nz, 1.0, 1.0, dz, nu, nv, du, dv, *circular_cone_vectors(6, dso, 200.0 + dso, th0=0.3))
    p = torch.rand((1, nu, 6, nv, 1), device="cuda")
    try:
        for c in range(3):
            autotune_pin("dd_cone_adj", c)
            ref = plan.backward(p, "dd")
            for u, view, v, bad in ((nu // 2, 2, nv // 2, float("nan")), (nu // 2 - 1, 4, nv // 2 - 2, float("inf"))):
                z, q = p.clone(), torch.zeros_like(p)
                z[0, u, view, v, 0], q[0, u, view, v, 0] = bad, 1.0
                met, out = plan.backward(q, "dd") > 0, plan.backward(z, "dd")
                assert bool(met.any()) and not bool(torch.isfinite(out[met]).any()), (c, bad)
                assert torch.equal(out[~met], ref[~met]), (c, bad)
    finally:
        autotune_pin("dd_cone_adj", None)
