"""Compiled line kernels of the lengths with factors 7 up to 256 against the
oracle, lines along and across the rows, an odd line out."""

import numpy as np
import pytest

from oracle import fft as F

from helpers import gather_rel_l2, rel_l2, run_gpu_plan, seeded_input

pytestmark = pytest.mark.gpu

# an error of a few rounding units per stage: eps * sqrt(log2 n) with room for
# the twiddle products
TOL = {True: 4e-15, False: 2e-6}


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n", [7, 14, 21, 28, 35, 42, 49, 56, 63, 70, 84, 98, 105, 112, 126, 140, 147, 168, 175, 189, 196,
                               210, 224, 245, 252, 343])
def test_every_length(dev, n, real, fp64):
    for gin, axes in (([7, n], [1]), ([n, 37], [0])):
        x = seeded_input(gin, real, sum(gin))
        x = x if fp64 else x.astype(np.float32 if real else np.complex64)
        outs, backs, ins, plan = run_gpu_plan(dev, x, gin, axes, [1, 1], [1, 1], real, fp64)
        ref = F.fftn(x.astype(np.float64 if real else np.complex128), axes, real)
        assert rel_l2(outs[0], ref) < TOL[fp64], (gin, axes)
        assert gather_rel_l2(backs, ins) < TOL[fp64], (gin, axes)
        plan.destroy()
