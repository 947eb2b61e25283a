"""The tile backprojector at the sizes where its tiles, slabs, chunks and queue can go wrong:
images smaller than a tile and a row over one, one slab and one slice over it, one sinogram,
64 and one more of a run, more runs than lanes, steep rays, bins mostly zero or one alone.
A single bin's backprojection is the oracle's bit for bit (each voxel takes one term); dense
ones stay within the reference's own rounding; scatter, gather and tile forms are one sum.
The threshold of a sensitivity: images of one workgroup, of a few and of more than there are."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# nx, ny, nz, dx, dz, angles, bins, sinograms, z range of the ends, slope range, order
GEOMS = {
    "one_voxel": (1, 1, 1, 8.0, 4.0, 3, 5, 1, (1.0, 3.0), 0.0, "up"),
    "under_a_tile": (7, 5, 3, 4.0, 3.0, 4, 9, 3, (1.0, 8.0), 4.0, "up"),
    "a_row_over": (9, 17, 13, 3.0, 2.0, 5, 21, 64, (1.0, 25.0), 6.0, "up"),
    "a_slice_over": (16, 16, 14, 3.0, 2.0, 6, 20, 65, (1.0, 27.0), 6.0, "up"),
    "runs": (24, 24, 30, 3.0, 1.5, 4, 16, 150, (1.0, 44.0), 8.0, "down"),
    "long_run": (12, 12, 27, 4.0, 2.0, 3, 14, 300, (1.0, 53.0), 3.0, "up"),
    "steep": (33, 33, 40, 4.0, 0.5, 7, 31, 70, (0.5, 19.0), 200.0, "up"),
    "many_angles": (10, 10, 9, 2.0, 2.0, 60, 24, 20, (-4.0, 22.0), 12.0, "up"),
}


def build(ctx, name):
    nx, ny, nz, dx, dz, nang, nr, nsino, (z0, z1), slope, order = GEOMS[name]
    rng = np.random.default_rng(len(name))
    mid = np.sort(rng.uniform(z0, z1, nsino))
    if order == "down":  # every sinogram a run of its own
        mid = mid[::-1]
    half = 0.5 * rng.uniform(-slope, slope, nsino) if slope else np.zeros(nsino)
    za, zb = (mid - half).astype(np.float32), (mid + half).astype(np.float32)
    w = np.float32(2.0)
    rfov = 0.5 * min(nx, ny) * dx
    p = hip.Plan(ctx, nx, ny, nz, dx, dz, nang, nr, rfov, 300.0, z1=za, z2=zb, ring_width=w)
    za, zb = (((z - w / 2) + w / 2).astype(np.float32) for z in (za, zb))
    ang, r = O.sino_grid(nang, nr, rfov)
    return p, O.image_desc(nx, ny, nz, dx, dz), ang, r, za, zb, rng


@pytest.mark.parametrize("name", sorted(GEOMS))
def test_tile_backprojection(torch, ctx, name):
    log(f"case: tile backprojection, {name}")
    p, im, ang, r, za, zb, rng = build(ctx, name)
    shape = (len(za), len(ang), len(r))
    for _ in range(12):
        sino = np.zeros(shape, np.float32)
        sino[tuple(rng.integers(n) for n in shape)] = rng.uniform(0.5, 2.0)
        got = host(p.backproject(dev(torch, sino), mode=hip.BP_TILE))
        want = O.backproject3d(im, sino, ang, r, 300.0, za, zb)
        assert np.array_equal(got.view(np.int32).ravel(), want.view(np.int32).ravel())
    dr = (r[-1] - r[0]) / (len(r) - 1)
    # terms of a voxel: those of the bins within its half-diagonal, of every angle and sinogram
    terms = len(ang) * len(za) * (int(1.42 * max(im.dx, im.dy) / dr) + 2)
    for keep in (1.0, 0.05):
        sino = rng.random(shape, dtype=np.float32)
        sino[rng.random(shape) >= keep] = 0
        sd = dev(torch, sino)
        got = {m: host(p.backproject(sd, mode=m))
               for m in (hip.BP_TILE, hip.BP_GATHER, hip.BP_SCATTER)}
        want = O.backproject3d(im, sino, ang, r, 300.0, za, zb).reshape(got[hip.BP_TILE].shape)
        # the oracle's float sum of non-negative terms: terms * 2^-24 of the sum, twice for safety
        # of the second order
        assert np.all(np.abs(got[hip.BP_TILE] - want) <= 2 * terms * 2.0 ** -24 * want + 1e-30)
        for m in got:
            assert np.array_equal(got[m].view(np.int32), got[hip.BP_TILE].view(np.int32))


@pytest.mark.parametrize("n", [1, 255, 8192, 8193, 4096 * 512, 4096 * 512 + 1])
def test_threshold_of_many_workgroups(torch, ctx, n):
    log(f"case: threshold of {n} values")
    rng = np.random.default_rng(n % 1000)
    x = rng.uniform(1.0, 9.0, n).astype(np.float32)
    x[rng.random(n) < 0.2] = 0
    x[-1], x[n // 2] = 11.0, 0.25
    for first in (x[0], np.float32(0), np.float32(20.0), np.float32("nan")):
        y = x.copy()
        y[0] = first
        got, want = hip.mlem_threshold(ctx, dev(torch, y)), O.mlem_threshold(y)
        assert np.float32(got) == np.float32(want) or (np.isnan(got) and np.isnan(want))
