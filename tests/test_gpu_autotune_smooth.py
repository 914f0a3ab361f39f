"""The plan autotuner on lines of 96 and 160 points, whose kernel has one form:
no shape is timed twice, and results stay."""

import numpy as np
import pytest

from oracle import fft as F

from helpers import rel_l2, seeded_input

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n", [96, 160])
def test_lines_of_one_form(dev, n, real, fp64):
    import torch
    import dfft
    from torch.profiler import ProfilerActivity, profile
    rdt, cdt = (torch.float64, torch.complex128) if fp64 else (torch.float32, torch.complex64)
    x = seeded_input([40, n], real, n)
    a = torch.from_numpy(x).to(dev, rdt if real else cdt)
    b = torch.empty((40, n // 2 + 1 if real else n), dtype=cdt, device=dev)
    plan = dfft.Plan([a], [b], [1], [1, 1], [1, 1], global_in_extents=[40, n], global_out_extents=list(b.shape))
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        plan.autotune([a], [b])
        torch.cuda.synchronize()
    launches = sum(e.count for e in p.key_averages() if "fft_" in e.key)
    if fp64 or not real:
        # per direction 6 block sizes x lane order, block numbering and kind of access, each 4
        # launches, and 6 of them 3 times more
        assert 0 < launches <= 2 * (6 * 8 * 4 + 6 * 3 * 4)
    a.copy_(torch.from_numpy(x))
    dfft.execute(plan, [a], [b], dfft.Direction.forward)
    # a few rounding units per stage
    assert rel_l2(b.cpu().numpy(), F.fftn(a.cpu().numpy().astype(np.float64 if real else np.complex128), [1], real)) < \
        (4e-15 if fp64 else 2e-6)
    plan.destroy()
