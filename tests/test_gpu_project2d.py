"""The 2D forward projector at the sizes where its 64-ray workgroups and 16-step turns can go
wrong: rays shorter than a turn, one workgroup and a ray over, two rounds of 16 wavefronts,
8 wavefronts with many rounds, rays along the axes (one crossing chain has no end), along the
voxel faces and beside the image, images read through their transposed copy.  Projections and
ratios are the oracle's, bit for bit; the likelihood is the sum of its rounded terms."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

# nx, dx, angles, bins, the bins' half-width over the image's, subsets
GEOMS = [(1, 8.0, 4, 9, 1.0, 1), (5, 4.0, 8, 16, 1.0, 3), (16, 4.0, 4, 64, 1.0, 1),
         (17, 4.0, 5, 13, 1.5, 1), (128, 2.0, 4, 129, 1.0, 1), (130, 2.0, 12, 65, 1.0, 5),
         (64, 3.0, 180, 190, 1.2, 1), (300, 1.0, 8, 50, 1.0, 2), (363, 1.0, 4, 40, 1.0, 1)]


@pytest.mark.parametrize("g", GEOMS)
def test_project2d_bitexact_vs_oracle(torch, ctx, g):
    nx, dx, nang, nr, wide, S = g
    log(f"case: 2D projector {g}")
    rfov = nx * dx / 2 * wide
    p = hip.Plan.for_2d(ctx, nx, dx, nang, nr, rfov, 900.0)
    im = O.image_desc(nx, nx, 1, dx)
    ang, r = O.sino_grid(nang, nr, rfov)
    rng = np.random.default_rng(nx)
    img = rng.random((1, nx, nx), dtype=np.float32)
    x = dev(torch, img)
    ref = O.project2d(im, img[0], ang, r, rfov, 900.0).reshape(1, nang, nr)
    meas = rng.poisson(3.0, ref.shape).astype(np.float32)
    for s in range(S):
        part = np.ascontiguousarray(ref[:, O.subset_angles(nang, S, s)])
        y = np.ascontiguousarray(meas[:, O.subset_angles(nang, S, s)])
        got = host(p.project(x, subset=s, nsubsets=S))
        assert np.array_equal(got.view(np.int32), part.view(np.int32))
        ratio, lik = p.project_ratio(x, dev(torch, meas), subset=s, nsubsets=S)
        ok = (y != 0) & (part != 0)
        want = np.where(ok, y / np.where(ok, part, 1), 0).astype(np.float32)
        assert np.array_equal(host(ratio).view(np.int32), want.view(np.int32))
        est = part[part != 0].astype(np.float64)
        term = y[part != 0] * np.log(est) - est
        # each term is rounded to float before it is summed in double
        assert abs(float(lik) - term.sum()) <= 4e-7 * (np.abs(y[part != 0] * np.log(est)) + est).sum() + 1e-30
