"""apirl_batch_job_bytes covers what a 3D job's submission takes from the device, the tile geometry
that its plan keeps from then on among it, or in its scratch where the plan keeps none; and a
serving loop over several plans stays within its budget, dropping geometry that idle plans keep
when a job needs the room."""
import numpy as np
import pytest

from apirl_amd import hip, serving
from test_gpu_parity import ctx, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu

MB = 1 << 20
# six buffers at most, each in whole 2 MiB pages, and an event
PAGES = 7 * 2 * MB


def plan(ctx, rscanner=400.0):
    return hip.Plan.for_3d(ctx, 128, 128, 20, 2.0, 2.0, 96, 128, 128.0, rscanner, 10, 40.0, 3, 5)


def free_bytes(torch):
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("subsets", [1, 6])
@pytest.mark.parametrize("cache_mb", [0, -1, 20])
def test_job_bytes_cover_the_submission(torch, ctx, subsets, cache_mb):
    log(f"case: job bytes, {subsets} subsets, tile_cache_mb {cache_mb}")
    p = plan(ctx)
    if cache_mb:
        p.set_tuning(tile_cache_mb=cache_mb)
    meas = torch.ones(p.subset_shape(), device="cuda")
    init = torch.ones(p.image_shape(), device="cuda")
    outs = [torch.empty_like(init) for _ in range(2)]
    b = hip.Batch(ctx, max_jobs=2, max_sinograms=256)
    before = free_bytes(torch)
    first = hip.Batch.job_bytes(p, subsets)
    b.submit(p, meas, init, outs[0], 1, subsets)
    middle = free_bytes(torch)
    second = hip.Batch.job_bytes(p, subsets)
    b.submit(p, meas, init, outs[1], 1, subsets)
    after = free_bytes(torch)
    b.run()
    b.close()
    assert before - middle <= first + PAGES
    assert middle - after <= second + PAGES
    assert second < first if cache_mb == 0 else second <= first


def test_serving_drops_idle_geometry(torch, ctx):
    """Three plans whose geometry does not fit the budget beside a job of another: every job is
    served, and equals the job alone."""
    log("case: serving with a budget of one job")
    plans = {f"p{k}": plan(ctx, 400.0 + 20 * k) for k in range(3)}
    jobs, want = [], []
    for k in range(6):
        p = plans[f"p{k % 3}"]
        g = torch.Generator(device="cuda").manual_seed(k)
        d = dict(meas=torch.poisson(torch.full(p.subset_shape(), 4.0, device="cuda"), generator=g),
                 init=torch.ones(p.image_shape(), device="cuda"), mult=None,
                 out=torch.empty(p.image_shape(), device="cuda"))
        jobs.append((dict(kind=f"p{k % 3}", iterations=1, subsets=4), d))
    need = max(hip.Batch.job_bytes(p, 4) for p in plans.values())
    low = [free_bytes(torch)]
    submit = hip.Batch.submit

    def watched(self, *a, **k):
        r = submit(self, *a, **k)
        low.append(free_bytes(torch))
        return r

    hip.Batch.submit = watched
    try:
        lat, _ = serving.serve(ctx, plans, jobs, 1000.0, torch, max_jobs=4, hbm_budget=need)
    finally:
        hip.Batch.submit = submit
    assert np.all(np.isfinite(lat))
    # the table and streams of the batch itself are not a job's
    assert low[0] - min(low) <= need + PAGES + 32 * MB
    for spec, d in jobs:
        p = plans[spec["kind"]]
        img, _ = p.reconstruct(d["meas"], d["init"], 1, subsets=4,
                               bp_mode=hip.Batch.backprojector(p))
        a, b = host(img), host(d["out"])
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(np.nan_to_num(a).view(np.int32), np.nan_to_num(b).view(np.int32))
    assert all(p.get_tuning()["tile_cache_mb"] == 16384 for p in plans.values())
