"""The 2D gather at the sizes where its patches, rounds and staged rays can go wrong: images
smaller than a patch and one voxel over one, fewer angles than a round's wavefronts and one
more, many bins per voxel (several stagings per angle, then the one-lane-per-voxel kernel).
Backprojections, fused updates and sensitivities are the oracle's, bit for bit, and a batch
of 2D jobs gives the single job's image."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# nx, dx, angles, bins
GEOMS = [(1, 8.0, 3, 9), (7, 4.0, 1, 11), (8, 4.0, 15, 13), (9, 4.0, 16, 40), (33, 2.0, 31, 30),
         (65, 2.0, 48, 130), (24, 5.0, 17, 170), (5, 26.0, 6, 344)]


def build(ctx, g):
    nx, dx, nang, nr = g
    rfov = nx * dx / 2
    p = hip.Plan.for_2d(ctx, nx, dx, nang, nr, rfov, 400.0)
    ang, r = O.sino_grid(nang, nr, rfov)
    return p, O.image_desc(nx, nx, 1, dx), ang, r, rfov


def same(a, b):
    a, b = np.ascontiguousarray(a).ravel(), np.ascontiguousarray(b).ravel()
    assert np.array_equal(a.view(np.int32), b.view(np.int32))


@pytest.mark.parametrize("g", GEOMS)
def test_gather2d_bitexact_vs_oracle(torch, ctx, g):
    log(f"case: 2D gather {g}")
    p, im, ang, r, rfov = build(ctx, g)
    rng = np.random.default_rng(3)
    sino = rng.random((1, g[2], g[3]), dtype=np.float32)
    sino[rng.random(sino.shape) < 0.3] = 0
    sd = dev(torch, sino)
    start = rng.random((1, g[0], g[0]), dtype=np.float32)
    out = p.backproject(sd, out=dev(torch, start), mode=hip.BP_GATHER)
    want = O.backproject2d(im, sino[0], ang, r, rfov, 400.0, img=start[0].copy())
    same(host(out), want)
    S = min(3, g[2])
    idx = O.subset_angles(g[2], S, S - 1)
    sens = p.sensitivity(mult=sd, subset=S - 1, nsubsets=S, mode=hip.BP_GATHER, force_positive=0)
    same(host(sens), O.backproject2d(im, sino[0][idx], ang[idx], r, rfov, 400.0))
    b = O.backproject2d(im, sino[0], ang, r, rfov, 400.0)
    ones = O.backproject2d(im, np.ones_like(sino[0]), ang, r, rfov, 400.0)
    same(host(p.sensitivity(mode=hip.BP_GATHER, force_positive=0)), ones)
    thr = float(np.median(ones))
    upd = p.backproject_update(sd, dev(torch, start), dev(torch, ones[None]), thr=thr, strict=1)
    same(host(upd), O.em_update(start[0].copy(), b, ones, thr, 1))


def test_gather2d_batch_equals_alone(torch, ctx):
    log("case: 2D jobs of every geometry in one batch")
    jobs = []
    batch = hip.Batch(ctx, max_jobs=len(GEOMS), max_sinograms=1)
    for k, g in enumerate(GEOMS):
        p, *_ = build(ctx, g)
        meas = torch.poisson(torch.full(p.subset_shape(), 5.0, device="cuda"))
        init = torch.ones(p.image_shape(), device="cuda")
        out = torch.empty_like(init)
        S = min(2, g[2])
        alone, _ = p.reconstruct(meas, init, 2, subsets=S, bp_mode=hip.BP_GATHER)
        jobs.append((alone, out, batch.submit(p, meas, init, out, 2, S)))
    batch.run()
    for alone, out, _ in jobs:
        a, b = host(alone), host(out)
        assert np.array_equal(np.isnan(a), np.isnan(b))
        same(np.nan_to_num(a), np.nan_to_num(b))
    batch.close()


@pytest.mark.parametrize("g", GEOMS)
def test_scatter2d_is_the_gather(torch, ctx, g):
    """The scatter form runs the patches where they fit: the oracle's sums, bit for bit."""
    log(f"case: 2D scatter form {g}")
    p, im, ang, r, rfov = build(ctx, g)
    rng = np.random.default_rng(4)
    sino = rng.random((1, g[2], g[3]), dtype=np.float32)
    sd = dev(torch, sino)
    same(host(p.backproject(sd, mode=hip.BP_SCATTER)),
         O.backproject2d(im, sino[0], ang, r, rfov, 400.0))
    same(host(p.sensitivity(mode=hip.BP_SCATTER, force_positive=0)),
         O.backproject2d(im, np.ones_like(sino[0]), ang, r, rfov, 400.0))
