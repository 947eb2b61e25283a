"""Backprojections on the mMR's LORs where a tile's candidate bins are the most: few angles (the
odd bins lie half an angular step from the even ones), voxels finer than the bins, wide images,
and plans whose own radial grid (rfov_mm), which the mMR's LORs do not use, is coarser than the
mMR's.  Every form is within the oracle's own rounding, and rfov_mm changes nothing."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

RINGS, ZFOV, SPAN, MRD = 4, 16.0, 3, 1
# form, nx, dx, nz, angles, rfov
CASES = [("mmr", 64, 4.2, 4, 36, 297.0), ("mmr", 128, 4.2, 4, 36, 800.0),
         ("mmr_subset", 128, 4.2, 4, 36, 800.0), ("mmr", 256, 2.0445, 2, 12, 297.0),
         ("mmr", 512, 1.0, 2, 12, 297.0)]


@pytest.mark.parametrize("case", CASES)
def test_mmr_backprojection_vs_oracle(torch, ctx, case):
    form, nx, dx, nz, nang, rfov = case
    log(f"case: mMR backprojection {case}")
    nr = 344
    p = hip.Plan.for_3d(ctx, nx, nx, nz, dx, ZFOV / nz, nang, nr, rfov, 328.0, RINGS, ZFOV, SPAN,
                        MRD)
    p.set_scanner(form)
    pts = (O.mmr_lor_table if form == "mmr" else O.mmr_subset_lor_table)(nang, nr)
    za, zb = O.ring_table(RINGS, ZFOV, SPAN, MRD)
    im = O.image_desc(nx, nx, nz, dx, ZFOV / nz)
    rng = np.random.default_rng(nang)
    sino = rng.uniform(0.5, 1.5, p.subset_shape()).astype(np.float32)
    want = O.backproject3d_pts(im, sino, pts, za, zb).astype(np.float64)
    # the oracle's float sum of at most `terms` positive terms: terms * 2^-24 of the sum; bins
    # are 0.8 mm apart at the least, a voxel 1.42 dx wide
    terms = nang * len(za) * (int(1.42 * dx / 0.8) + 2)
    for mode in (hip.BP_TILE, hip.BP_GATHER, hip.BP_SCATTER):
        got = host(p.backproject(dev(torch, sino), mode=mode)).reshape(want.shape)
        off = int((np.abs(got - want) > 2 * terms * 2.0 ** -24 * want).sum())
        assert off == 0, (mode, off)


@pytest.mark.parametrize("form", ["mmr", "mmr_subset"])
def test_mmr_images_do_not_depend_on_rfov(torch, ctx, form):
    """Subset sensitivities and an update of plans of three radial fields of view, bit for bit."""
    log(f"case: {form} plans of three rfov_mm")
    out = []
    for rfov in (297.0, 600.0, 800.0):
        p = hip.Plan.for_3d(ctx, 172, 172, 4, 3.0, 4.0, 252, 344, rfov, 328.0, RINGS, ZFOV, SPAN,
                            MRD)
        p.set_scanner(form)
        rng = np.random.default_rng(1)
        sino = dev(torch, rng.uniform(0.5, 1.5, p.subset_shape(1, 21)).astype(np.float32))
        sens = p.sensitivity(subset=1, nsubsets=21, mode=hip.BP_GATHER)
        x = p.backproject_update(sino, torch.ones_like(sens), sens, subset=1, nsubsets=21,
                                 mode=hip.BP_GATHER)
        out.append((host(sens).view(np.int32), host(x).view(np.int32)))
    for sens, x in out[1:]:
        assert int((sens != out[0][0]).sum()) == 0
        assert int((x != out[0][1]).sum()) == 0


@pytest.mark.parametrize("form", ["mmr", "mmr_subset"])
def test_mmr_on_a_plan_of_other_angles(torch, ctx, form):
    """The mMR's LORs have angles of their own, whatever the plan's are."""
    log(f"case: {form} on a plan of explicit angles")
    nx, nz, dx, nang, nr = 40, 4, 6.0, 20, 120
    rng = np.random.default_rng(9)
    z1, z2 = hip.ring_table(RINGS, ZFOV, SPAN, MRD)
    p = hip.Plan(ctx, nx, nx, nz, dx, ZFOV / nz, nang, nr, 297.0, 328.0, z1=z1, z2=z2,
                 ring_width=np.float32(ZFOV) / np.float32(RINGS), ang=rng.permutation(180)[:nang])
    p.set_scanner(form)
    pts = (O.mmr_lor_table if form == "mmr" else O.mmr_subset_lor_table)(nang, nr)
    za, zb = O.ring_table(RINGS, ZFOV, SPAN, MRD)
    sino = rng.uniform(0.5, 1.5, p.subset_shape()).astype(np.float32)
    im = O.image_desc(nx, nx, nz, dx, ZFOV / nz)
    want = O.backproject3d_pts(im, sino, pts, za, zb).astype(np.float64)
    terms = nang * len(za) * (int(1.42 * dx / 0.8) + 2)
    for mode, prec in ((hip.BP_TILE, hip.PREC_REFERENCE), (hip.BP_GATHER, hip.PREC_REFERENCE),
                       (hip.BP_SCATTER, hip.PREC_REFERENCE), (hip.BP_GATHER, hip.PREC_KAHAN)):
        got = host(p.backproject(dev(torch, sino), mode=mode, precision=prec)).reshape(want.shape)
        off = int((np.abs(got - want) > 2 * terms * 2.0 ** -24 * want).sum())
        assert off == 0, (mode, prec, off)
