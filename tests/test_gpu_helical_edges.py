"""The helical backprojection against the oracle (relative L2 1e-5, the parity bar)
where its shortcuts can go wrong: rows and columns that fall off the detector on
either side (a short detector, offsets of several cells), voxels that no view sees
inside the taper, heights outside the scan, an odd and a single detector row, image
sizes below and over a wave's 8 x 8 columns, no taper at all (Q = 1)."""

import numpy as np
import pytest

from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,nu,nv,off_u,off_v,vol_z0,zrot,m_pi,Q", [
    (7, 9, 5, 40, 9, 0.25, 0.0, 8.0, 12.0, 1, 0.5), (17, 8, 9, 12, 4, -3.0, 2.5, -6.0, 10.0, 1, 0.6),
    (12, 13, 3, 50, 1, 0.25, 0.25, 9.0, 3.0, 1, 0.5), (9, 9, 17, 33, 24, 0.0, -6.0, 30.0, 12.0, 2, 0.4),
    (16, 16, 8, 48, 16, 0.3, -0.5, 10.0, -9.0, 1, 0.9), (10, 11, 6, 40, 12, 0.25, 0.0, 9.0, 11.0, 1, 1.0),
])
def test_helical_bp_edges(nx, ny, nz, nu, nv, off_u, off_v, vol_z0, zrot, m_pi, Q):
    import oracle as orc
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.recon import ReconNet

    npp, turns = 48, 3
    r = ReconNet()
    r.nx, r.ny, r.nz, r.dx, r.dy, r.dz = nx, ny, nz, 1.0, 1.0, 1.0
    r.du, r.dv, r.off_u, r.off_v, r.dsd, r.dso = 1.0, 1.0, off_u, off_v, 1000.0, 600.0
    prj = np.random.default_rng(nx + nv).uniform(0, 1, (1, nu, 2 * npp * turns, nv, 1)).astype(np.float32)
    g = dict(dx=1.0, dy=1.0, dz=1.0, du=1.0, dv=1.0, off_u=off_u, off_v=off_v, dsd=1000.0, dso=600.0)
    ref = orc.helical_bp(prj, g, (nx, ny, nz), npp, 0.1, vol_z0, zrot, m_pi=m_pi, Q=Q)
    try:
        for cand in range(3):
            autotune_pin("helical_bp", cand)
            out = r.cHelicalBP4d(prj, npp, 0.1, vol_z0, zrot, mPI=m_pi, Q=Q)
            assert rel_l2(out, ref) <= 1e-5 if np.abs(ref).max() > 0 else not out.any(), cand
    finally:
        autotune_pin("helical_bp", None)


@pytest.mark.parametrize("nv", [1, 4])
def test_helical_rows_on_the_detector_edge_without_a_taper(nv):
    # Q = 1: weight 1 up to and on the detector's edge (q = 1).  One voxel on the axis,
    # magnification 2 and dyadic heights: view 64 + d sees it at v = -nv d / 8 exactly, so
    # the views d = -4 and 4 on the edge, where the sample is half of the last row, and no
    # other voxel of the wave sees them inside it
    from reconnet_amd._lib import autotune_pin
    from reconnet_amd.recon import ReconNet

    npp, turns, zrot = 32, 3, 4.0 * nv
    r = ReconNet()
    r.nx, r.ny, r.nz, r.dx, r.dy, r.dz = 1, 1, 1, 1.0, 1.0, 64.0
    r.du, r.dv, r.off_u, r.off_v, r.dsd, r.dso = 1.0, 1.0, 0.25, 0.0, 1024.0, 512.0
    prj = np.random.default_rng(nv).uniform(0, 1, (1, 8, 2 * npp * turns, nv, 1)).astype(np.float32)
    ref = 0.0
    for d in range(-4, 5):
        rows = np.zeros(nv + 2)
        rows[1:-1] = 0.25 * prj[0, 3, 64 + d, :, 0] + 0.75 * prj[0, 4, 64 + d, :, 0]     # u = 0: column 3.75
        pv = -nv * d / 8 + (nv - 1) / 2 + 1
        k = int(np.floor(pv))
        ref += ((1 - pv + k) * rows[k] + (pv - k) * rows[k + 1]) / (1 + 1e-6)
    try:
        for cand in range(3):
            autotune_pin("helical_bp", cand)
            out = r.cHelicalBP4d(prj, npp, 0.0, zrot, zrot, mPI=1, Q=1.0)
            assert abs(float(out.ravel()[0]) - ref) <= 1e-5 * ref, cand
    finally:
        autotune_pin("helical_bp", None)


def test_helical_voxels_beyond_the_sources_circle():
    # where a view's u exceeds dso the row has no value: not a number, as the oracle's,
    # also when no voxel of the wave has one in that view
    import oracle as orc
    from reconnet_amd.recon import ReconNet

    npp, turns, zrot = 16, 3, 8.0
    r = ReconNet()
    r.nx, r.ny, r.nz, r.dx, r.dy, r.dz = 2, 1, 2, 1200.0, 1.0, 1.0
    r.du, r.dv, r.off_u, r.off_v, r.dsd, r.dso = 1.0, 1.0, 0.0, 0.0, 1024.0, 512.0
    prj = np.random.default_rng(1).uniform(0, 1, (1, 8, 2 * npp * turns, 4, 1)).astype(np.float32)
    g = dict(dx=1200.0, dy=1.0, dz=1.0, du=1.0, dv=1.0, off_u=0.0, off_v=0.0, dsd=1024.0, dso=512.0)
    ref = orc.helical_bp(prj, g, (2, 1, 2), npp, 0.0, zrot, zrot, m_pi=1, Q=0.5)
    assert np.isnan(ref).all()
    assert np.isnan(r.cHelicalBP4d(prj, npp, 0.0, zrot, zrot, mPI=1, Q=0.5)).all()
