"""Grouped launches: one block per virtual block against resident blocks
walking them, staged lines against direct ones, and the lengths with a radix 6
or 10 last (96, 160), whose FP64 blocks hold whole 128-byte row segments."""

import numpy as np
import pytest

from oracle import fft as F

from helpers import out_extents, rel_l2, seeded_input

pytestmark = pytest.mark.gpu

# a few rounding units per stage, n <= 160 along each of 3 axes
TOL = {True: 4e-15, False: 2e-6}


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("shapes", [[[160, 160, 9], [3, 160, 160]], [[96, 160, 32], [160, 5, 96], [16, 17, 64]],
                                    [[64, 160, 1], [96, 96, 96]]])
def test_blocks_and_staging(dev, shapes, real, fp64):
    import torch
    import dfft
    rdt, cdt = (torch.float64, torch.complex128) if fp64 else (torch.float32, torch.complex64)
    xs = [seeded_input(s, real, i) for i, s in enumerate(shapes)]
    ins = [torch.from_numpy(x).to(dev, rdt if real else cdt) for x in xs]
    outs = [torch.empty(out_extents(s, [0, 1, 2], real), dtype=cdt, device=dev) for s in shapes]
    backs = [torch.empty_like(t) for t in ins]
    g = dfft.Group(ins, outs)
    refs = [F.fftn(x, [0, 1, 2], real) for x in xs]
    for mult, stage, lanes in ((None, None, None), (1, 1, 256), (0, 1, 64), (0, 0, 128)):
        for key, v in (("grid_mult", mult), ("stage", stage), ("lanes", lanes)):
            if v is not None:
                g.set_option(key, v)
        g.execute(ins, outs, dfft.Direction.forward)
        g.execute(outs, backs, dfft.Direction.backward)
        for x, o, b, r in zip(xs, outs, backs, refs):
            assert rel_l2(o.cpu().numpy(), r) < TOL[fp64], (mult, stage, lanes)
            assert rel_l2(b.cpu().numpy(), x) < TOL[fp64], (mult, stage, lanes)
