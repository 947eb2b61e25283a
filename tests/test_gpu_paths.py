"""The path forward projector at the sizes where its workgroups, batches and column walk
can go wrong: one sinogram, one more than a wavefront, several passes per wavefront;
paths shorter than a batch; rays that cross several slices per column (the step-by-step
form), that run along the slices, and that leave the image through its axial faces.
The projection is the oracle's, bit for bit, in the reference arithmetic; the
compensated sum stays within its error bound of the same terms summed in double."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# nx, ny, nz, dx, dz, angles, bins, sinograms, z range of the ends, slope range
GEOMS = {
    "one_sinogram": (5, 5, 3, 4.0, 3.0, 4, 7, 1, (3.0, 9.0), 0.0),
    "flat": (33, 40, 9, 2.0, 2.5, 5, 21, 63, (2.0, 22.0), 0.0),
    "wave_and_one": (40, 33, 17, 2.0, 2.0, 6, 24, 65, (2.0, 34.0), 12.0),
    "two_passes": (64, 64, 21, 2.0445, 2.027, 4, 33, 321, (2.0, 41.0), 20.0),
    "five_passes": (24, 24, 40, 3.0, 1.5, 3, 12, 1030, (1.0, 59.0), 30.0),
    "steep": (48, 48, 64, 4.0, 0.5, 6, 31, 130, (0.5, 31.0), 300.0),
    "leaving": (48, 48, 12, 2.0, 2.0, 6, 31, 200, (-20.0, 45.0), 60.0),
}


def build(ctx, name):
    nx, ny, nz, dx, dz, nang, nr, nsino, (z0, z1), slope = GEOMS[name]
    rng = np.random.default_rng(len(name))
    mid = np.sort(rng.uniform(z0, z1, nsino))
    half = 0.5 * rng.uniform(-slope, slope, nsino) if slope else np.zeros(nsino)
    za, zb = (mid - half).astype(np.float32), (mid + half).astype(np.float32)
    w = np.float32(2.0)
    rfov = 0.5 * min(nx, ny) * dx
    p = hip.Plan(ctx, nx, ny, nz, dx, dz, nang, nr, rfov, 300.0, z1=za, z2=zb, ring_width=w)
    # the plan's ends: z - w / 2 + w / 2, in float
    za, zb = (((z - w / 2) + w / 2).astype(np.float32) for z in (za, zb))
    im = O.image_desc(nx, ny, nz, dx, dz)
    ang, r = O.sino_grid(nang, nr, rfov)
    img = rng.random((nz, ny, nx), dtype=np.float32)
    return p, im, ang, r, za, zb, img


@pytest.mark.parametrize("name", sorted(GEOMS))
def test_path_projector_bitexact_vs_oracle(torch, ctx, name):
    log(f"case: path projector, {name}")
    p, im, ang, r, za, zb, img = build(ctx, name)
    ref = O.project3d(im, img, ang, r, 300.0, za, zb)
    x = dev(torch, img)
    got = host(p.project(x))
    assert np.array_equal(got.view(np.int32), ref.view(np.int32))
    meas = np.random.default_rng(1).poisson(3.0, ref.shape).astype(np.float32)
    ratio, lik = p.project_ratio(x, dev(torch, meas))
    ok = (meas != 0) & (ref != 0)
    want = np.where(ok, meas / np.where(ok, ref, 1), 0).astype(np.float32)
    assert np.array_equal(host(ratio).view(np.int32), want.view(np.int32))
    est = ref[ref != 0].astype(np.float64)
    term = meas[ref != 0] * np.log(est) - est
    # each term is rounded to float before it is summed in double
    assert abs(float(lik) - term.sum()) <= 4e-7 * np.abs(term).sum() + 1e-30


@pytest.mark.parametrize("name", sorted(GEOMS))
def test_path_projector_compensated_sums(torch, ctx, name):
    log(f"case: compensated path projector, {name}")
    p, im, ang, r, za, zb, img = build(ctx, name)
    got = host(p.project(dev(torch, img), precision=hip.PREC_KAHAN))
    rng = np.random.default_rng(2)
    for _ in range(40):
        s, a, q = rng.integers(len(za)), rng.integers(len(ang)), rng.integers(len(r))
        _, p1, p2 = O.lor_points(float(ang[a]), float(r[q]), 300.0)
        p1, p2 = np.float32(p1), np.float32(p2)
        v = (p2[0] - p1[0], p2[1] - p1[1], zb[s] - za[s])
        total = mag = 0.0
        for i, j, k, wt in O.siddon3d((p1[0], p1[1], za[s]), v, im):
            if 0 <= i < im.nx and 0 <= j < im.ny and 0 <= k < im.nz:
                t = float(np.float32(np.float32(wt) * img[k, j, i]))
                total, mag = total + t, mag + abs(t)
        # Kahan's bound, 2 eps + O(n eps^2) of the terms' magnitudes, eps = 2^-24
        assert abs(float(got[s, a, q]) - total) <= 3 * 2.0 ** -24 * mag


@pytest.mark.parametrize("precision", ["PREC_KAHAN", "PREC_F64_SETUP"])
def test_path_projector_equals_ray_per_lane(torch, ctx, precision):
    """A long enough projection of more than 112 sinograms takes the path in these precisions,
    its single angles a ray per lane: the same bins, bit for bit."""
    log(f"case: path against ray per lane, {precision}")
    rng = np.random.default_rng(5)
    nx, nz, nang, nr, nsino = 190, 21, 9, 240, 130
    mid = np.sort(rng.uniform(1.0, 41.0, nsino))
    half = rng.uniform(-15.0, 15.0, nsino)
    p = hip.Plan(ctx, nx, nx, nz, 2.0, 2.0, nang, nr, nx * 1.0, 300.0,
                 z1=(mid - half).astype(np.float32), z2=(mid + half).astype(np.float32),
                 ring_width=np.float32(2.0))
    assert nsino * nang * nr * 2 * nx >= 1e8 > nsino * nr * 2 * nx
    x = dev(torch, rng.random((nz, nx, nx), dtype=np.float32))
    prec = getattr(hip, precision)
    whole = host(p.project(x, precision=prec))
    for a in range(nang):
        one = host(p.project(x, subset=a, nsubsets=nang, precision=prec))
        assert np.array_equal(one.view(np.int32)[:, 0], whole.view(np.int32)[:, a])


def test_few_sinograms_equal_path_and_ray_per_lane(torch, ctx):
    """A projection of few sinograms of close bins takes a ray per lane, its single angles the
    path: the same bins, bit for bit."""
    log("case: path against ray per lane, reference arithmetic")
    rng = np.random.default_rng(6)
    nx, nz, nang, nr, nsino = 100, 15, 12, 120, 40
    mid = np.sort(rng.uniform(1.0, 29.0, nsino))
    half = rng.uniform(-10.0, 10.0, nsino)
    p = hip.Plan(ctx, nx, nx, nz, 2.0, 2.0, nang, nr, nx * 1.0, 300.0,
                 z1=(mid - half).astype(np.float32), z2=(mid + half).astype(np.float32),
                 ring_width=np.float32(2.0))
    assert nsino * nang * nr * 2 * nx >= 5e6 > nsino * nr * 2 * nx
    x = dev(torch, rng.random((nz, nx, nx), dtype=np.float32))
    whole = host(p.project(x))
    meas = dev(torch, rng.poisson(3.0, whole.shape).astype(np.float32))
    ratio, lik = p.project_ratio(x, meas)
    total = 0.0
    for a in range(nang):
        one = host(p.project(x, subset=a, nsubsets=nang))
        assert np.array_equal(one.view(np.int32)[:, 0], whole.view(np.int32)[:, a])
        part, l1 = p.project_ratio(x, meas, subset=a, nsubsets=nang)
        assert np.array_equal(host(part).view(np.int32)[:, 0], host(ratio).view(np.int32)[:, a])
        total += float(l1)
    # the same terms summed in double, in another order
    assert abs(float(lik) - total) <= 1e-9 * abs(total)
