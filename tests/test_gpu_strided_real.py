"""R2C and C2R passes across the lines (LayoutLeft views, the real axis not the
innermost one in storage) at their default launch shapes."""

import numpy as np
import pytest

from oracle import fft as F
from oracle import planner as PL
from oracle import plan_exec as PE

from helpers import device_full, gather_rel_l2, out_extents, run_gpu_plan, seeded_input

pytestmark = pytest.mark.gpu

# a few rounding units per stage, as in the tests of the lengths
TOL = {True: 4e-15, False: 2e-6}


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("gin,tin,tout", [
    ([9, 7, 64], [1, 1, 1], [1, 1, 1]),
    ([6, 10, 256], [2, 1, 1], [1, 2, 1]),
    ([6, 10, 512], [2, 1, 1], [1, 2, 1]),
    ([5, 6, 1024], [1, 1, 1], [1, 1, 1]),
    ([8, 4, 2048], [2, 1, 1], [1, 2, 1]),
    ([4, 6, 4096], [1, 1, 1], [1, 1, 1]),
    ([33, 40, 512], [1, 1, 1], [1, 1, 1]),
    ([33, 40, 1024], [1, 1, 1], [1, 1, 1]),
])
def test_left_views(dev, gin, tin, tout, fp64):
    axes = [0, 1, 2]
    x = seeded_input(gin, True, sum(gin)).astype(np.float64 if fp64 else np.float32)
    outs, backs, ins, plan = run_gpu_plan(dev, x, gin, axes, tin, tout, True, fp64, view_layout="left")
    plan.destroy()
    ref = PE.scatter(F.fftn(x.astype(np.float64), axes, True), out_extents(gin, axes, True), tout, PL.LAYOUT_RIGHT)
    assert gather_rel_l2(outs, ref) < TOL[fp64]
    assert gather_rel_l2(backs, ins) < TOL[fp64]


# Streamed stores of every other real of a row took two to three times as long
# as cached ones; runs of one shape differ by a few percent.
SLOWER = 1.3


@pytest.mark.parametrize("gin,fp64", [([256, 256, 256], True), ([256, 256, 256], False), ([512, 512, 64], True),
                                      ([1024, 1024, 64], True), ([384, 384, 384], True)])
def test_default_stores_are_no_slower_than_cached_ones(dev, gin, fp64):
    import torch
    import dfft
    rdt, cdt = (torch.float64, torch.complex128) if fp64 else (torch.float32, torch.complex64)
    a = device_full(gin, 0.0, rdt, dev, True)
    b = device_full(out_extents(gin, [0, 1, 2], True), 0.0, cdt, dev, True)
    plan = dfft.Plan([a], [b], [0, 1, 2], [1, 1, 1], [1, 1, 1], layout=dfft.LayoutLeft)

    def best():
        fwd = min(plan.execute_timed([a], [b], dfft.Direction.forward)[0] for _ in range(8))
        return fwd, min(plan.execute_timed([b], [a], dfft.Direction.backward)[2] for _ in range(8))

    default = best()
    plan.set_option("fwd.0.nt", 0)
    plan.set_option("bwd.2.nt", 0)
    cached = best()
    plan.destroy()
    assert default[0] < SLOWER * cached[0] and default[1] < SLOWER * cached[1], (default, cached)
