"""The first backprojection of a plan, which allocates its scratch and builds the tile geometry,
does not wait for the work already enqueued, as the later ones do not."""
import numpy as np
import pytest

from apirl_amd import hip
from test_gpu_parity import ctx, host, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["BP_SCATTER", "BP_GATHER", "BP_TILE"])
def test_first_backprojection_is_only_enqueued(torch, ctx, mode):
    log(f"case: first 3D backprojection behind busy work, {mode}")

    def plan():
        return hip.Plan.for_3d(ctx, 40, 40, 21, 3.0, 2.0, 30, 44, 60.0, 400.0, 11, 42.0, 3, 6)

    m = getattr(hip, mode)
    old, new = plan(), plan()
    sino = torch.rand(old.subset_shape(1, 3), device="cuda")
    want = host(old.backproject(sino, subset=1, nsubsets=3, mode=m))
    out = torch.zeros(new.image_shape(), device="cuda")
    busy = torch.cuda.Event()
    torch.cuda.synchronize()
    torch.cuda._sleep(1_000_000_000)  # some 0.4 s
    busy.record()
    new.backproject(sino, out=out, subset=1, nsubsets=3, mode=m)
    assert not busy.query()
    torch.cuda.synchronize()
    assert np.array_equal(host(out).view(np.int32), want.view(np.int32))
