"""The voxel-driven 3D gather on sinogram tables whose rays cross each other in z (slopes of any
order among growing means): it and the tile form give the oracle's image.  Tables of more runs
than the column kernel's LDS holds take the one-voxel kernel."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import assert_voxel_close, ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsino,nz,slope", [(60, 40, 16.0), (300, 24, 8.0), (1500, 9, 6.0)])
def test_crossing_rays(torch, ctx, nsino, nz, slope):
    log(f"case: gather of {nsino} sinograms of crossing rays")
    nx, dx, dz, nang, nr = 20, 4.0, 2.0, 5, 22
    rng = np.random.default_rng(nsino)
    mid = np.sort(rng.uniform(1.0, nz * dz - 1.0, nsino))
    half = rng.uniform(-slope, slope, nsino)
    za, zb = (mid - half).astype(np.float32), (mid + half).astype(np.float32)
    w = np.float32(2.0)
    p = hip.Plan(ctx, nx, nx, nz, dx, dz, nang, nr, nx * dx / 2, 300.0, z1=za, z2=zb, ring_width=w)
    za, zb = (((z - w / 2) + w / 2).astype(np.float32) for z in (za, zb))
    im = O.image_desc(nx, nx, nz, dx, dz)
    ang, r = O.sino_grid(nang, nr, nx * dx / 2)
    sino = rng.uniform(0.5, 1.5, p.subset_shape()).astype(np.float32)
    ref = O.backproject3d(im, sino, ang, r, 300.0, za, zb)
    sd = dev(torch, sino)
    # the oracle's float sums: its rounding over some hundreds of terms is within the forms' bar
    assert_voxel_close(host(p.backproject(sd, mode=hip.BP_TILE)), ref)
    for zlanes, zvox in ((1, 1), (1, 3), (2, 3)):
        p.set_tuning(gather_zlanes=zlanes, gather_zvox=zvox)
        assert_voxel_close(host(p.backproject(sd, mode=hip.BP_GATHER, precision=hip.PREC_KAHAN)),
                           ref)


@pytest.mark.parametrize("nx,ny,wide", [(14, 16, 2.0), (2, 54, 1.2), (3, 40, 0.9), (30, 9, 1.5)])
def test_beside_the_square(torch, ctx, nx, ny, wide):
    """Images that are not square: the reference clips LORs to a square of the image's width, and
    those that miss it still cross the rows beyond it; of images less tall, the rows end before."""
    log(f"case: backprojection of {nx} x {ny}, sinogram {wide} times as wide")
    nz, dx, dz, nang, nr, nsino = 14, 4.5, 2.0, 26, 91, 37
    rng = np.random.default_rng(nx)
    mid = np.sort(rng.uniform(1.0, nz * dz - 1.0, nsino))
    za, zb = (mid - 6.0).astype(np.float32), (mid + 6.0).astype(np.float32)
    w = np.float32(2.0)
    rfov = wide * nx * dx / 2
    p = hip.Plan(ctx, nx, ny, nz, dx, dz, nang, nr, rfov, 200.0, z1=za, z2=zb, ring_width=w)
    za, zb = (((z - w / 2) + w / 2).astype(np.float32) for z in (za, zb))
    im = O.image_desc(nx, ny, nz, dx, dz)
    ang, r = O.sino_grid(nang, nr, rfov)
    sino = rng.uniform(0.5, 1.5, p.subset_shape()).astype(np.float32)
    ref = O.backproject3d(im, sino, ang, r, 200.0, za, zb)
    sd = dev(torch, sino)
    for mode in (hip.BP_TILE, hip.BP_GATHER, hip.BP_SCATTER):
        assert_voxel_close(host(p.backproject(sd, mode=mode)), ref, rtol=2e-5)
    for zlanes, zvox in ((1, 1), (1, 3), (2, 3)):
        p.set_tuning(gather_zlanes=zlanes, gather_zvox=zvox)
        assert_voxel_close(host(p.backproject(sd, mode=hip.BP_GATHER, precision=hip.PREC_KAHAN)),
                           ref, rtol=2e-5)
    x = rng.uniform(0.5, 1.5, p.image_shape()).astype(np.float32)
    want = O.project3d(im, x, ang, r, 200.0, za, zb)
    c, s = np.cos(np.radians(ang))[:, None], np.sin(np.radians(ang))[:, None]
    meets = np.abs(r) < 0.999 * nx * dx / 2 * (np.abs(c) + np.abs(s))
    got = host(p.project(dev(torch, x)))
    off = int((got.view(np.int32) != want.view(np.int32))[:, meets].sum())
    assert off == 0
