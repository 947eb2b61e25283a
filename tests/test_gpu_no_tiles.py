"""3D backprojections in the reference arithmetic on plans that the tile backprojector refuses
(here: slabs whose sums exceed its LDS): the voxel-driven kernels and the atomics that such plans
run.  One bin's backprojection is the oracle's bit for bit; every voxel mapping gives the same
bits; stored, clamped and updated voxels are those of the separate passes; batched jobs equal the
job alone; and all stay within the float sum's rounding of the tile form of a plan that takes it."""
import numpy as np
import pytest

import _oracle as O
from apirl_amd import hip
from test_gpu_parity import assert_bitexact, assert_voxel_close, ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

NX, NZ, DX, DZ, NANG, NR, NSINO = 26, 140, 3.0, 1.0, 12, 30, 60


def build(ctx, tiles=False):
    rng = np.random.default_rng(3)
    mid = np.sort(rng.uniform(1.0, NZ * DZ - 1.0, NSINO))
    half = rng.uniform(-20.0, 20.0, NSINO)
    za, zb = (mid - half).astype(np.float32), (mid + half).astype(np.float32)
    p = hip.Plan(ctx, NX, NX, NZ, DX, DZ, NANG, NR, NX * DX / 2, 300.0, z1=za, z2=zb,
                 ring_width=np.float32(2.0))
    if not tiles:
        p.set_tuning(tile_zs=140)
        with pytest.raises(hip.ApirlError, match="64 KiB"):
            p.backproject(p.project(_ones(p)), mode=hip.BP_TILE)
    return p


def _ones(p):
    import torch
    return torch.ones(p.image_shape(), device="cuda")


def bins(torch, p, s=0, S=1, seed=5, low=0.0):
    rng = np.random.default_rng(seed)
    x = rng.uniform(low, 1.5, p.subset_shape(s, S)).astype(np.float32)
    x[rng.random(x.shape) < 0.3] = 0
    return dev(torch, x)


MAPPINGS = [dict(gather_zlanes=2)] + [dict(gather_zlanes=1, gather_zvox=v, gather_xcd=x)
                                      for v in (1, 2, 3, 4)
                                      for x in (hip.GATHER_XCD_ROUND_ROBIN, hip.GATHER_XCD_WEDGES)]


def test_voxel_mappings_and_single_bins(torch, ctx):
    log("case: voxel-driven kernels, every mapping")
    p = build(ctx)
    sino = bins(torch, p, 1, 3)
    start = dev(torch, np.random.default_rng(1).random(p.image_shape(), dtype=np.float32))
    got = []
    for m in MAPPINGS:
        p.set_tuning(**m)
        got.append(host(p.backproject(sino, out=start.clone(), subset=1, nsubsets=3,
                                      mode=hip.BP_GATHER)))
        assert_bitexact(got[-1], got[0])
    t = build(ctx, True)
    assert_voxel_close(got[0], host(t.backproject(sino, out=start.clone(), subset=1, nsubsets=3,
                                                  mode=hip.BP_TILE)))
    assert_voxel_close(got[0], host(p.backproject(sino, out=start.clone(), subset=1, nsubsets=3,
                                                  mode=hip.BP_SCATTER)))
    rng = np.random.default_rng(2)
    for m in (MAPPINGS[0], MAPPINGS[6]):
        p.set_tuning(**m)
        for _ in range(6):
            one = np.zeros(p.subset_shape(), np.float32)
            one[tuple(rng.integers(n) for n in one.shape)] = rng.uniform(0.5, 2.0)
            gather = host(p.backproject(dev(torch, one), mode=hip.BP_GATHER))
            assert_bitexact(gather, host(t.backproject(dev(torch, one), mode=hip.BP_TILE)))
            assert_bitexact(host(p.backproject(dev(torch, one), mode=hip.BP_SCATTER)), gather)


def test_single_bins_vs_oracle(torch, ctx):
    log("case: voxel-driven kernels, single bins")
    p = build(ctx)
    rng = np.random.default_rng(3)
    mid = np.sort(rng.uniform(1.0, NZ * DZ - 1.0, NSINO))
    half = rng.uniform(-20.0, 20.0, NSINO)
    w = np.float32(2.0)
    za, zb = ((z.astype(np.float32) - w / 2) + w / 2 for z in (mid - half, mid + half))
    im = O.image_desc(NX, NX, NZ, DX, DZ)
    ang, r = O.sino_grid(NANG, NR, NX * DX / 2)
    for _ in range(8):
        one = np.zeros(p.subset_shape(), np.float32)
        one[tuple(rng.integers(n) for n in one.shape)] = rng.uniform(0.5, 2.0)
        want = O.backproject3d(im, one, ang, r, 300.0, za.astype(np.float32), zb.astype(np.float32))
        assert_bitexact(host(p.backproject(dev(torch, one), mode=hip.BP_GATHER)), want)


@pytest.mark.parametrize("mapping", [MAPPINGS[0], MAPPINGS[6]])
def test_sensitivities(torch, ctx, mapping):
    """Stored over what the image held; clamped when asked for (a multiplicative sinogram of both
    signs gives negative sums)."""
    log(f"case: sensitivities without tiles, {mapping}")
    p = build(ctx)
    p.set_tuning(**mapping)
    mult = bins(torch, p, low=-1.0)
    junk = torch.full(p.image_shape(), 7.0, device="cuda")
    for m in (None, mult):
        b = host(p.backproject(torch.ones(p.subset_shape(), device="cuda") if m is None else m,
                               mode=hip.BP_GATHER))
        if m is not None:
            assert (b < 0).any() and (b > 0).any()
        for force in (0, 1):
            want = np.where(b < 0, np.float32(0), b) if force else b
            got = p.sensitivity(out=junk.clone(), mult=m, mode=hip.BP_GATHER, force_positive=force)
            assert_bitexact(host(got), want)
            got = p.sensitivity(out=junk.clone(), mult=m, mode=hip.BP_SCATTER, force_positive=force)
            if m is None:
                assert_voxel_close(host(got), want)
            else:  # sums of both signs: the float sums' rounding of their magnitudes
                mag = host(p.backproject(m.abs(), mode=hip.BP_GATHER))
                assert np.all(np.abs(host(got) - want) <= 1e-5 * mag)


@pytest.mark.parametrize("mapping", [MAPPINGS[0], MAPPINGS[6]])
@pytest.mark.parametrize("strict", [0, 1])
def test_fused_update(torch, ctx, mapping, strict):
    log(f"case: fused update without tiles, {mapping}, strict={strict}")
    p = build(ctx)
    p.set_tuning(**mapping)
    sino = bins(torch, p, 1, 3)
    sens = p.sensitivity(subset=1, nsubsets=3, mode=hip.BP_GATHER)
    thr = float(np.median(host(sens)[host(sens) > 0]))
    x0 = dev(torch, np.random.default_rng(4).uniform(0.5, 2.0, p.image_shape()).astype(np.float32))
    b = p.backproject(sino, subset=1, nsubsets=3, mode=hip.BP_GATHER)
    want = hip.em_update(ctx, x0.clone(), b, sens, thr, strict)
    got = p.backproject_update(sino, x0.clone(), sens, thr, strict, subset=1, nsubsets=3,
                               mode=hip.BP_GATHER)
    assert_bitexact(host(got), host(want), nan_ok=True)


def test_batch_equals_alone(torch, ctx):
    """OSEM and MLEM jobs (whose thresholds stay on the device)."""
    log("case: batched jobs without tiles")
    p = build(ctx)
    b = hip.Batch(ctx, max_jobs=4, max_sinograms=64)
    jobs = []
    for k, S in enumerate((1, 3, 1)):
        g = torch.Generator(device="cuda").manual_seed(k)
        meas = torch.poisson(torch.full(p.subset_shape(), 4.0, device="cuda"), generator=g)
        init, out = _ones(p), _ones(p)
        alone, _ = p.reconstruct(meas, init, 2, subsets=S, bp_mode=hip.BP_GATHER)
        b.submit(p, meas, init, out, 2, S)
        jobs.append((alone, out))
    b.run()
    for alone, out in jobs:
        assert_bitexact(host(out), host(alone), nan_ok=True)
    b.close()


def test_tile_form_vs_voxel_driven_at_full_size(torch, ctx):
    """256 x 256 x 81 from 12 of 252 angles: single bins (one term a voxel, which a compensated
    sum leaves as it is) bit for bit, dense ones within the forms' bar."""
    log("case: tile form against the voxel-driven gather, 256x256x81")
    p = hip.Plan.for_3d(ctx, 256, 256, 81, 2.0445, 2.027, 252, 344, 261.696, 400.0, 64, 164.187, 11,
                        60)
    S, s = 21, 3
    shape = p.subset_shape(s, S)
    rng = np.random.default_rng(11)
    for _ in range(6):
        one = np.zeros(shape, np.float32)
        one[tuple(rng.integers(n) for n in shape)] = rng.uniform(0.5, 3.0)
        x = dev(torch, one)
        assert_bitexact(host(p.backproject(x, subset=s, nsubsets=S, mode=hip.BP_TILE)),
                        host(p.backproject(x, subset=s, nsubsets=S, mode=hip.BP_GATHER,
                                           precision=hip.PREC_KAHAN)))
    x = bins(torch, p, s, S)
    assert_voxel_close(host(p.backproject(x, subset=s, nsubsets=S, mode=hip.BP_TILE)),
                       host(p.backproject(x, subset=s, nsubsets=S, mode=hip.BP_GATHER,
                                          precision=hip.PREC_KAHAN)))
