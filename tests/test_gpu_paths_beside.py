"""The path forward projector on sinograms wider than the image (a zoomed image).  LORs beside the
image have lists that the reference walks along columns outside it, some of them back into rows of
the array: with compensated sums they are a ray per lane's, bit for bit.  LORs that meet the image
are the oracle's in the reference arithmetic."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def build(ctx, nx, nz, nang, nr, nsino, wide, dx=2.0, dz=2.0, rscanner=400.0):
    rng = np.random.default_rng(nx)
    L = nz * dz
    mid = np.sort(rng.uniform(1.0, L - 1.0, nsino))
    half = rng.uniform(-0.4 * L, 0.4 * L, nsino)
    za, zb = (mid - half).astype(np.float32), (mid + half).astype(np.float32)
    w = np.float32(2.0)
    rfov = wide * nx * dx / 2
    p = hip.Plan(ctx, nx, nx, nz, dx, dz, nang, nr, rfov, rscanner, z1=za, z2=zb, ring_width=w)
    za, zb = (((z - w / 2) + w / 2).astype(np.float32) for z in (za, zb))
    ang, r = O.sino_grid(nang, nr, rfov)
    return p, O.image_desc(nx, nx, nz, dx, dz), ang, r, za, zb, rng


# nx, nz, angles, bins, sinograms, the bins' half-width over the image's
@pytest.mark.parametrize("g", [(64, 17, 24, 60, 100, 1.1), (64, 17, 24, 60, 100, 1.42),
                               (64, 17, 24, 60, 100, 3.0), (32, 9, 36, 60, 70, 4.0)])
def test_meeting_the_image_vs_oracle(torch, ctx, g):
    log(f"case: path projector, sinogram wider than the image, {g}")
    p, im, ang, r, za, zb, rng = build(ctx, *g)
    img = rng.uniform(0.5, 1.5, p.image_shape()).astype(np.float32)
    ref = O.project3d(im, img, ang, r, 400.0, za, zb)
    c, s = np.cos(np.radians(ang))[:, None], np.sin(np.radians(ang))[:, None]
    meets = np.abs(r) < 0.999 * im.nx * im.dx / 2 * (np.abs(c) + np.abs(s))
    assert meets.any() and not meets.all()
    x = dev(torch, img)
    got = host(p.project(x))
    off = int((got.view(np.int32) != ref.view(np.int32))[:, meets].sum())
    assert off == 0
    meas = rng.poisson(3.0, ref.shape).astype(np.float32)
    ratio, _ = p.project_ratio(x, dev(torch, meas))
    ok = (meas != 0) & (ref != 0)
    want = np.where(ok, meas / np.where(ok, ref, 1), 0).astype(np.float32)
    off = int((host(ratio).view(np.int32) != want.view(np.int32))[:, meets].sum())
    assert off == 0


@pytest.mark.parametrize("precision", ["PREC_KAHAN", "PREC_F64_SETUP"])
def test_beside_the_image_equals_ray_per_lane(torch, ctx, precision):
    """A long enough projection takes the path in these precisions, its single angles a ray per
    lane: the same bins, bit for bit."""
    log(f"case: path against ray per lane beside the image, {precision}")
    nang, nr, nsino, nx = 36, 260, 130, 64
    p, *_, rng = build(ctx, nx, 15, nang, nr, nsino, 3.0)
    assert nsino * nang * nr * 2 * nx >= 1e8 > nsino * nr * 2 * nx
    x = dev(torch, rng.random(p.image_shape(), dtype=np.float32))
    prec = getattr(hip, precision)
    whole = host(p.project(x, precision=prec)).view(np.int32)
    off = 0
    for a in range(nang):
        one = host(p.project(x, subset=a, nsubsets=nang, precision=prec)).view(np.int32)
        off += int((one[:, 0] != whole[:, a]).sum())
    assert off == 0
