"""Backprojections captured into a graph on a stream, and for a subset, that the plan has not
run before: the scratch of an earlier call holds what the capture needs, nothing is allocated,
and every replay, with the program's own work between them, gives the eager result."""
import ctypes

import numpy as np
import pytest

import _oracle as O  # noqa: F401
from apirl_amd import hip
from test_gpu_parity import ctx, dev, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("mode", ["BP_SCATTER", "BP_GATHER", "BP_TILE"])
def test_capture_on_another_stream_and_subset(torch, dims, mode):
    if dims == 2 and mode == "BP_TILE":
        pytest.skip("the tile form is 3D")
    log(f"case: captured backprojection, {dims}D {mode}")
    c = hip.Context(0)
    if dims == 2:
        p = hip.Plan.for_2d(c, 40, 3.0, 30, 44, 60.0, 400.0)
    else:
        p = hip.Plan.for_3d(c, 40, 40, 21, 3.0, 2.0, 30, 44, 60.0, 400.0, 11, 42.0, 3, 6)
    m = getattr(hip, mode)
    S = 3
    rng = np.random.default_rng(dims)
    full = [dev(torch, rng.random(p.subset_shape(s, S), dtype=np.float32)) for s in range(S)]
    p.backproject(full[0], subset=0, nsubsets=S, mode=m)  # the largest subset, another stream
    torch.cuda.synchronize()
    img = torch.zeros(p.image_shape(), dtype=torch.float32, device="cuda")
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    c.check(c.lib.apirl_ctx_set_stream(c.h, ctypes.c_void_p(side.cuda_stream)), "set_stream")
    with torch.cuda.graph(graph, stream=side):
        p.backproject(full[1], out=img, subset=1, nsubsets=S, mode=m)
    c.check(c.lib.apirl_ctx_set_stream(c.h, None), "set_stream")
    torch.cuda.synchronize()
    for k in range(3):
        full[1].copy_(torch.rand_like(full[1]) * (torch.rand_like(full[1]) > 0.3))
        img.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = host(p.backproject(full[1], subset=1, nsubsets=S, mode=m))
        assert np.array_equal(host(img).view(np.int32), want.view(np.int32)), k
