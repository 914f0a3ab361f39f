"""The static table area of dfft_group_execute_noalloc holds the records of
2,500 member passes."""

import numpy as np
import pytest

from helpers import rel_l2

pytestmark = pytest.mark.gpu


def test_2500_member_passes(dev):
    import torch
    import dfft
    n = 2500
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (n, 1, 16)) + 1j * rng.uniform(-1, 1, (n, 1, 16))
    a = torch.from_numpy(x).to(dev)
    b = torch.full_like(a, float("nan"))
    ins, outs = list(a), list(b)
    g = dfft.Group(ins, outs, [1])
    g.execute_noalloc(ins, outs, dfft.Direction.forward)
    # a few rounding units per stage
    assert rel_l2(b.cpu().numpy(), np.fft.fft(x, axis=2)) < 4e-15
