"""Compiled line kernels of the lengths 2^a 3^b 5^c up to 1024: every length
against the oracle, lines along and across the rows, a line left over in the
last block and real lines with an odd one out; and their passes against the
per-element and power-of-two kernels, which serve the same lengths where the
line axis is split or real lines go one by one."""

import numpy as np
import pytest

from oracle import fft as F
from oracle import planner as PL
from oracle import plan_exec as PE

from helpers import gather_rel_l2, out_extents, rel_l2, run_gpu_plan, seeded_input

pytestmark = pytest.mark.gpu

# an error of a few rounding units per stage: eps * sqrt(log2 n) with room for
# the twiddle products
TOL = {True: 4e-15, False: 2e-6}


def _smooth(n):
    for r in (2, 3, 5):
        while n % r == 0:
            n //= r
    return n == 1


LENGTHS = [n for n in range(3, 1025) if _smooth(n) and n & (n - 1)]


def _input(gin, real, fp64):
    x = seeded_input(gin, real, sum(gin))
    return x if fp64 else x.astype(np.float32 if real else np.complex64)


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n", LENGTHS)
def test_every_length(dev, n, real, fp64):
    for gin, axes in (([7, n], [1]), ([n, 37], [0])):
        x = _input(gin, real, fp64)
        outs, backs, ins, plan = run_gpu_plan(dev, x, gin, axes, [1, 1], [1, 1], real, fp64)
        ref = F.fftn(x.astype(np.float64 if real else np.complex128), axes, real)
        assert rel_l2(outs[0], ref) < TOL[fp64], (gin, axes)
        assert gather_rel_l2(backs, ins) < TOL[fp64], (gin, axes)
        plan.destroy()


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n,m,p", [(12, 45, 2), (96, 18, 3), (160, 25, 4), (375, 10, 2), (300, 30, 4), (640, 6, 2)])
def test_ranks_and_layouts(dev, n, m, p, real, fp64):
    """Uneven blocks in both view layouts, there and back."""
    gin, axes, tin, tout = [m, n, 20], [0, 1, 2], [p, 1, 1], [1, p, 1]
    x = _input(gin, real, fp64)
    ref = F.fftn(x.astype(np.float64 if real else np.complex128), axes, real)
    for view in (None, "left"):
        outs, backs, ins, plan = run_gpu_plan(dev, x, gin, axes, tin, tout, real, fp64, view_layout=view)
        want = PE.scatter(ref, out_extents(gin, axes, real), tout, PL.LAYOUT_RIGHT)
        assert gather_rel_l2(outs, want) < TOL[fp64], view
        assert gather_rel_l2(backs, ins) < TOL[fp64], view
        plan.destroy()


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("n", [15, 96, 160, 250, 576, 1000])
def test_agrees_with_the_other_kernels(dev, n, fp64):
    """Real lines one by one (per-element kernel; 96 and 160: the power-of-two kernel) and in pairs; a line axis split
    over ranks (per-element kernel) and whole."""
    for gin, axes in (([9, n], [1]), ([n, 9], [0])):
        x = _input(gin, True, fp64)
        pairs = run_gpu_plan(dev, x, gin, axes, [1, 1], [1, 1], True, fp64)
        single = run_gpu_plan(dev, x, gin, axes, [1, 1], [1, 1], True, fp64,
                              configure=lambda p, i, o: (p.set_option("fwd.0.pair", 0), p.set_option("bwd.0.pair", 0)))
        assert rel_l2(pairs[0][0], single[0][0]) < TOL[fp64]
        assert rel_l2(pairs[1][0], single[1][0]) < TOL[fp64]
    x = _input([n, 10], False, fp64)
    split = run_gpu_plan(dev, x, [n, 10], [0], [2, 1], [2, 1], False, fp64)
    whole = run_gpu_plan(dev, x, [n, 10], [0], [1, 1], [1, 1], False, fp64)
    assert rel_l2(np.concatenate(split[0], axis=0), whole[0][0]) < TOL[fp64]
    assert rel_l2(np.concatenate(split[1], axis=0), whole[1][0]) < TOL[fp64]
