"""apirl_project_ratio_noalloc up to its documented number of bins, however many of them share a
path: few sinograms of more than 2^19 (angle, radial bin) pairs."""
import numpy as np
import pytest
import ctypes

from apirl_amd import hip
from test_gpu_parity import ctx, log, torch  # noqa: F401

pytestmark = pytest.mark.gpu


def test_many_pairs_of_few_sinograms(torch, ctx):
    log("case: ratio without allocation, 2 sinograms of 540000 pairs")
    nang, nr = 45000, 12
    z1, z2 = np.float32([3.0, 5.0]), np.float32([5.0, 3.0])
    p = hip.Plan(ctx, 16, 16, 4, 1.0, 2.0, nang, nr, 8.0, 400.0, z1=z1, z2=z2,
                 ring_width=np.float32(2.0))
    assert nang * nr > 1 << 19
    x = torch.rand(p.image_shape(), device="cuda")
    meas = torch.poisson(torch.full(p.subset_shape(), 3.0, device="cuda"))
    want, lik = p.project_ratio(x, meas)
    got, out = torch.empty_like(want), torch.zeros(1, dtype=torch.float64, device="cuda")
    ctx.check(ctx.lib.apirl_project_ratio_noalloc(
        p.h, *(ctypes.c_void_p(t) for t in (x.data_ptr(), meas.data_ptr(), None, got.data_ptr(),
                                            out.data_ptr())), 0, 1, 0, hip.PREC_REFERENCE),
        "apirl_project_ratio_noalloc")
    torch.cuda.synchronize()
    assert bool((got == want).all())
    # the same terms summed in double, in another order
    assert abs(float(out) - float(lik)) <= 1e-9 * abs(float(lik))
