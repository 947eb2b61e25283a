"""Captured calls at the limits of what earlier calls have allocated: a subset larger than any
before, another form or precision than before, no call before at all.  What can run without an
allocation does, and every replay gives the eager result; the rest is refused with an error that
leaves the capture and the plan as they were.  A graph outlives the scratch it was captured over:
a later, larger call leaves it its own."""
import ctypes

import numpy as np
import pytest

from apirl_amd import hip
from test_gpu_parity import assert_voxel_close, ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu


class Captured:
    """A graph of calls on the context's stream, captured on a side stream."""

    def __init__(self, torch, c):
        self.torch, self.c = torch, c
        self.graph, self.side = torch.cuda.CUDAGraph(), torch.cuda.Stream()

    def __enter__(self):
        self.torch.cuda.synchronize()
        self.c.check(self.c.lib.apirl_ctx_set_stream(
            self.c.h, ctypes.c_void_p(self.side.cuda_stream)), "set_stream")
        self.inner = self.torch.cuda.graph(self.graph, stream=self.side)
        self.inner.__enter__()
        return self

    def __exit__(self, *e):
        self.inner.__exit__(*e)
        self.c.check(self.c.lib.apirl_ctx_set_stream(self.c.h, None), "set_stream")
        self.torch.cuda.synchronize()


def plan3(c):
    return hip.Plan.for_3d(c, 40, 40, 21, 3.0, 2.0, 30, 44, 60.0, 400.0, 11, 42.0, 3, 6)


def bins(torch, p, s, S, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.rand(p.subset_shape(s, S), device="cuda", generator=g)
    return x * (torch.rand(x.shape, device="cuda", generator=g) > 0.3)


def replays(torch, cap, x, img, eager, same):
    for k in range(3):
        x.copy_(torch.rand_like(x) * (torch.rand_like(x) > 0.3))
        img.zero_()
        torch.cuda.synchronize()
        cap.graph.replay()
        torch.cuda.synchronize()
        got, want = host(img), host(eager())
        if same:
            assert int((got.view(np.int32) != want.view(np.int32)).sum()) == 0, k
        else:
            assert_voxel_close(got, want)


def test_scatter_of_a_larger_subset(torch):
    """The scatter form needs no memory: captured for all angles after a call for a tenth."""
    log("case: captured scatter of a larger subset")
    c = hip.Context(0)
    p = plan3(c)
    p.backproject(bins(torch, p, 0, 10), subset=0, nsubsets=10, mode=hip.BP_SCATTER)
    x, img = bins(torch, p, 0, 1), torch.zeros(p.image_shape(), device="cuda")
    with Captured(torch, c) as cap:
        p.backproject(x, out=img, mode=hip.BP_SCATTER)
    replays(torch, cap, x, img, lambda: p.backproject(x, mode=hip.BP_SCATTER), False)


def test_scatter_sensitivity_of_a_larger_subset(torch):
    log("case: captured scatter sensitivity of a larger subset")
    c = hip.Context(0)
    p = plan3(c)
    p.sensitivity(subset=0, nsubsets=10, mode=hip.BP_SCATTER)
    mult, sens = bins(torch, p, 0, 1), torch.full(p.image_shape(), 7.0, device="cuda")
    with Captured(torch, c) as cap:
        p.sensitivity(mult=mult, out=sens, mode=hip.BP_SCATTER)
    replays(torch, cap, mult, sens, lambda: p.sensitivity(mult=mult, mode=hip.BP_SCATTER), False)


def test_scatter_divide_after_plain_calls(torch):
    """DivideAndBackproject keeps its atomics; a plain call before it runs the tiles."""
    log("case: captured scatter divide rule after a plain scatter")
    c = hip.Context(0)
    p = plan3(c)
    x, img = bins(torch, p, 1, 3), torch.zeros(p.image_shape(), device="cuda")
    est = torch.rand_like(x) + 0.5
    p.backproject(x, subset=1, nsubsets=3, mode=hip.BP_SCATTER)
    with Captured(torch, c) as cap:
        p.divide_backproject(x, est, out=img, subset=1, nsubsets=3, mode=hip.BP_SCATTER)
    replays(torch, cap, x, img,
            lambda: p.divide_backproject(x, est, subset=1, nsubsets=3, mode=hip.BP_SCATTER), False)


# few sinograms: the tile geometry is the larger part of the scratch; many: the axial records are
@pytest.mark.parametrize("first,then,rings,mrd", [("PREC_KAHAN", "PREC_REFERENCE", 8, 4),
                                                  ("PREC_REFERENCE", "PREC_KAHAN", 24, 20)])
def test_gather_after_another_precision(torch, first, then, rings, mrd):
    """A gather call makes room for a capture of any subset and precision of as many angles,
    also where a call of the other precision has left enough for itself."""
    log(f"case: captured gather, {first} then {then}")
    c = hip.Context(0)
    p = hip.Plan.for_3d(c, 256, 256, 40, 2.0, 2.0, 8, 344, 256.0, 400.0, rings, 80.0, 3, mrd)
    S = 3
    p.backproject(bins(torch, p, 0, 4), subset=0, nsubsets=4, mode=hip.BP_GATHER,
                  precision=getattr(hip, first))
    p.backproject(bins(torch, p, 0, S), subset=0, nsubsets=S, mode=hip.BP_GATHER,
                  precision=hip.PREC_REFERENCE)
    x, img = bins(torch, p, 1, S), torch.zeros(p.image_shape(), device="cuda")
    prec = getattr(hip, then)
    with Captured(torch, c) as cap:
        p.backproject(x, out=img, subset=1, nsubsets=S, mode=hip.BP_GATHER, precision=prec)
    replays(torch, cap, x, img, lambda: p.backproject(x, subset=1, nsubsets=S, mode=hip.BP_GATHER,
                                                      precision=prec), True)


@pytest.mark.parametrize("mode", ["BP_GATHER", "BP_TILE"])
def test_refused_capture_leaves_the_plan(torch, mode):
    """No call before: an error, the capture goes on, and the plan works afterwards."""
    log(f"case: capture on a fresh plan, {mode}")
    c = hip.Context(0)
    p = plan3(c)
    m = getattr(hip, mode)
    x, img = bins(torch, p, 0, 1), torch.ones(p.image_shape(), device="cuda")
    with Captured(torch, c) as cap:
        with pytest.raises(hip.ApirlError, match="scratch"):
            p.backproject(x, out=img, mode=m)
        img.mul_(3.0)
    cap.graph.replay()
    torch.cuda.synchronize()
    assert bool((img == 3.0).all())
    want = host(plan3(c).backproject(x, mode=m))
    assert np.array_equal(host(p.backproject(x, mode=m)).view(np.int32), want.view(np.int32))


@pytest.mark.parametrize("mode", ["BP_SCATTER", "BP_GATHER", "BP_TILE"])
def test_graph_outlives_its_scratch(torch, mode):
    """A larger call replaces the scratch, and a smaller tile_cache_mb the kept geometry, of a
    captured call; its replays read the ones they were captured over."""
    log(f"case: replays after the scratch has grown, {mode}")
    c = hip.Context(0)
    p = plan3(c)
    m = getattr(hip, mode)
    S = 10
    x, img = bins(torch, p, 1, S), torch.zeros(p.image_shape(), device="cuda")
    cap = Captured(torch, c)
    # the geometry kept on the capture's own stream
    c.check(c.lib.apirl_ctx_set_stream(c.h, ctypes.c_void_p(cap.side.cuda_stream)), "set_stream")
    torch.cuda.synchronize()
    p.backproject(x, out=img, subset=1, nsubsets=S, mode=m)
    with cap:
        p.backproject(x, out=img, subset=1, nsubsets=S, mode=m)
    p.backproject(bins(torch, p, 0, 1), mode=m)
    p.set_tuning(tile_cache_mb=-1)
    fill = [torch.full((1 << 20,), float("nan"), device="cuda") for _ in range(16)]
    replays(torch, cap, x, img, lambda: p.backproject(x, subset=1, nsubsets=S, mode=m), True)
    del fill


def test_ratio_after_another_precision(torch):
    """The likelihood's partials: a captured call of any precision finds room for them, and a
    graph keeps its own when a larger call takes more."""
    log("case: captured ratio, other precision, then a larger sinogram")
    c = hip.Context(0)
    p = hip.Plan.for_2d(c, 64, 4.0, 600, 200, 128.0, 400.0)
    x = torch.rand(p.image_shape(), device="cuda")
    meas = torch.poisson(torch.full(p.subset_shape(), 5.0, device="cuda"))
    ratio = torch.empty_like(meas)
    lik = torch.zeros(1, dtype=torch.float64, device="cuda")
    p.project_ratio(x, meas, precision=hip.PREC_KAHAN)

    def call(r, out):
        c.check(c.lib.apirl_project_ratio(p.h, x.data_ptr(), meas.data_ptr(), None, r.data_ptr(),
                                          out.data_ptr(), 0, 1, 0, hip.PREC_REFERENCE), "ratio")

    with Captured(torch, c) as cap:
        call(ratio, lik)
    big = hip.Plan.for_2d(c, 64, 4.0, 9000, 600, 128.0, 400.0)
    big.project_ratio(x, torch.ones(big.subset_shape(), device="cuda"))
    for _ in range(3):
        x.copy_(torch.rand_like(x))
        lik.zero_()
        torch.cuda.synchronize()
        cap.graph.replay()
        torch.cuda.synchronize()
        r2, l2 = torch.empty_like(meas), torch.zeros_like(lik)
        call(r2, l2)
        assert bool((ratio == r2).all()) and float(lik) == float(l2)
