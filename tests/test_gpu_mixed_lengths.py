"""Line passes of lengths without a compile-time kernel (products of 2, 3, 5,
7, 11 and 13) against the oracle: every radix alone and in company, lines
along and across the rows, real lines in pairs with an odd one left over,
ragged blocks, and the calls that stay on the per-element kernel."""

import numpy as np
import pytest

from oracle import fft as F
from oracle import planner as PL
from oracle import plan_exec as PE

from helpers import device_array, gather_rel_l2, out_extents, rel_l2, run_gpu_plan, seeded_input

pytestmark = pytest.mark.gpu

# an error of a few rounding units per stage: eps * sqrt(log2 n) with room for
# the twiddle products, n <= 5120
TOL = {True: 4e-15, False: 2e-6}


def _both_ways(dev, gin, axes, real, fp64, **kw):
    x = seeded_input(gin, real, sum(gin) + len(axes))
    x = x.astype((np.float32 if real else np.complex64) if not fp64 else (np.float64 if real else np.complex128))
    tin = kw.pop("tin", [1] * (len(gin) - 1) + [1])
    tout = kw.pop("tout", list(tin))
    outs, backs, ins, plan = run_gpu_plan(dev, x, gin, axes, tin, tout, real, fp64, **kw)
    ref = PE.scatter(F.fftn(x.astype(np.float64 if real else np.complex128), axes, real), out_extents(gin, axes, real),
                     list(tout), PL.LAYOUT_RIGHT)
    assert gather_rel_l2(outs, ref) < TOL[fp64], (gin, axes, real, fp64)
    assert gather_rel_l2(backs, ins) < TOL[fp64], (gin, axes, real, fp64)
    plan.destroy()


SINGLE = [3, 5, 6, 7, 9, 10, 11, 12, 13, 14, 15]
SHORT = [18, 20, 21, 22, 24, 25, 26, 27, 28, 30, 33, 36, 39, 42, 45, 48, 49, 50, 54, 55, 63, 65, 72, 75, 77, 81, 91,
         99, 100, 117, 121, 125, 143, 144, 169]
LONG = [162, 180, 192, 200, 225, 243, 250, 270, 286, 320, 343, 360, 375, 384, 400, 405, 480, 500, 625, 640, 720, 768,
        1000, 1001, 1155, 1280, 1536, 2187, 2401, 3125, 4374, 4802, 5120]


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n", SINGLE + SHORT)
def test_lines_along_and_across(dev, n, real, fp64):
    # axis 1: lanes along the line (contiguous); axis 0: lanes across the lines
    _both_ways(dev, [19, n], [1], real, fp64)
    _both_ways(dev, [n, 19], [0], real, fp64)


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n", LONG)
def test_long_lines_along_and_across(dev, n, real, fp64):
    _both_ways(dev, [7, n], [1], real, fp64)
    _both_ways(dev, [n, 9], [0], real, fp64)


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("gin,tin,tout,axes,view", [
    ([50, 42, 36], [2, 2, 1], [1, 2, 2], [0, 1, 2], None),
    ([45, 30, 21], [3, 1, 1], [1, 3, 1], [0, 1, 2], None),
    ([45, 30, 21], [4, 1, 1], [1, 4, 1], [0, 1, 2], "left"),
    ([24, 33, 260], [2, 1, 1], [1, 2, 1], [0, 1, 2], None),  # R2C rows of 131 entries: padded scratch
    ([60, 20, 250], [2, 1, 1], [1, 2, 1], [0, 1, 2], None),
    ([5, 50, 36], [1, 2, 1], [1, 2, 1], [2], None),
])
def test_plans_of_ragged_extents(dev, gin, tin, tout, axes, view, real, fp64):
    _both_ways(dev, gin, axes, real, fp64, tin=tin, tout=tout, view_layout=view)


@pytest.mark.parametrize("norm", ["forward", "ortho", "none"])
def test_scale_of_the_last_pass(dev, norm):
    gin = [20, 18, 30]
    x = seeded_input(gin, False, 5)
    outs, _, _, _ = run_gpu_plan(dev, x, gin, [0, 1, 2], [2, 1, 1], [1, 2, 1], False, True, norm=norm)
    ref = PE.scatter(F.fftn(x, [0, 1, 2], False, norm), gin, [1, 2, 1], PL.LAYOUT_RIGHT)
    assert gather_rel_l2(outs, ref) < TOL[True]


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
def test_agrees_with_the_per_element_kernel(dev, real, fp64):
    """A line axis split over ranks runs the per-element kernel, a whole one the register kernel."""
    n, w = 60, 14
    x = seeded_input([n, w], real, 3)
    axes = [0]
    split = run_gpu_plan(dev, x, [n, w], axes, [2, 1], [2, 1], real, fp64) if not real else None
    whole = run_gpu_plan(dev, x, [n, w], axes, [1, 1], [1, 1], real, fp64)
    if split is not None:
        a = np.concatenate(split[0], axis=0)
        assert rel_l2(a, whole[0][0]) < TOL[fp64]
    pairs_off = run_gpu_plan(dev, x, [n, w], axes, [1, 1], [1, 1], real, fp64,
                             configure=lambda p, i, o: (p.set_option("fwd.0.pair", 0), p.set_option("bwd.0.pair", 0)))
    assert rel_l2(pairs_off[0][0], whole[0][0]) < TOL[fp64]
    assert rel_l2(pairs_off[1][0], whole[1][0]) < TOL[fp64]


@pytest.mark.parametrize("real", [False, True])
def test_adjoint_of_ragged_plans(dev, real):
    """<F x, y> = <x, F* y> with the half spectrum's weights in the real passes."""
    import torch
    import dfft
    gin, axes, tin, tout = [20, 21, 36], [0, 1, 2], [2, 1, 1], [1, 2, 1]
    gout = out_extents(gin, axes, real)
    x = seeded_input(gin, real, 1)
    y = seeded_input(gout, False, 2)
    ins = [device_array(a, dev, torch.float64 if real else torch.complex128) for a in PE.scatter(x, gin, tin, 0)]
    ys = [device_array(a, dev, torch.complex128) for a in PE.scatter(y, gout, tout, 0)]
    outs = [torch.empty_like(a) for a in ys]
    adj = [torch.empty_like(a) for a in ins]
    plan = dfft.Plan(ins, outs, axes, tin, tout, global_in_extents=gin, global_out_extents=gout)
    dfft.execute(plan, ins, outs, dfft.Direction.forward)
    plan.execute_adjoint(ys, adj, dfft.Direction.forward)
    lhs = sum(float((torch.conj(a) * b).real.sum()) for a, b in zip(outs, ys))
    rhs = sum(float((torch.conj(a) * b).real.sum()) for a, b in zip(ins, adj))
    scale = float(np.linalg.norm(x.ravel()) * np.linalg.norm(y.ravel()) * np.sqrt(np.prod(gin)))
    assert abs(lhs - rhs) < 1e-13 * scale


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
def test_group_members_of_such_lengths(dev, real, fp64):
    import torch
    import dfft
    rdt, cdt = (torch.float64, torch.complex128) if fp64 else (torch.float32, torch.complex64)
    shapes = [[20, 18, 15], [32, 32, 32], [12, 50, 36], [7, 16, 21]]
    xs = [seeded_input(s, real, i) for i, s in enumerate(shapes)]
    ins = [torch.from_numpy(x).to(dev, rdt if real else cdt) for x in xs]
    outs = [torch.empty(out_extents(s, [0, 1, 2], real), dtype=cdt, device=dev) for s in shapes]
    backs = [torch.empty_like(t) for t in ins]
    g = dfft.Group(ins, outs)
    g.execute(ins, outs, dfft.Direction.forward)
    g.execute(outs, backs, dfft.Direction.backward)
    for x, o, b in zip(xs, outs, backs):
        assert rel_l2(o.cpu().numpy(), F.fftn(x, [0, 1, 2], real)) < TOL[fp64]
        assert rel_l2(b.cpu().numpy(), x) < TOL[fp64]
