"""Real lines of lengths that are no power of two are transformed one by one:
what one line holds (infinities, NaN, values of another magnitude) leaves every
other line as it is, and the rounding errors are those of a complex line."""

import numpy as np
import pytest

from oracle import fft as F

from helpers import rel_l2, run_gpu_plan
from test_gpu_line_errors import TOL, _exact, _lines, _per_element

pytestmark = pytest.mark.gpu

# relative to each line's own norm: a few rounding units per stage, as in the
# tests of the lengths
LINE_TOL = {True: 4e-15, False: 2e-6}
# compiled lengths, with factors 7, and the runtime-radix kernel
LENGTHS = [5, 12, 60, 96, 100, 160, 243, 252, 360, 500, 504, 768, 1001, 1155, 1536]


def _pairs(n, fp64):  # FP32 lines of 96 and 160 points run in pairs, as powers of two do
    return not fp64 and n in (96, 160)


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("n", LENGTHS)
def test_neighbours_of_another_size(dev, n, axis, fp64):
    if _pairs(n, fp64):
        pytest.skip("in pairs")
    rng = np.random.default_rng(n)
    size = np.array([1.0, 1e8, 1e-8, 1.0, 1e6, 1e-6, 1.0])
    x = rng.uniform(-1, 1, (len(size), n)) * size[:, None]
    x[3, n // 2] = np.inf
    x[6, 0] = np.nan
    dirty = (3, 6)
    x = x.astype(np.float64 if fp64 else np.float32)
    y = x if axis == 1 else np.ascontiguousarray(x.T)
    outs, backs, _, plan = run_gpu_plan(dev, y, list(y.shape), [axis], [1, 1], [1, 1], True, fp64)
    plan.destroy()
    got, back = (outs[0], backs[0]) if axis == 1 else (outs[0].T, backs[0].T)
    for k in range(len(size)):
        if k in dirty:
            assert not np.isfinite(got[k]).any()
            continue
        ref = F.fftn(x[k].astype(np.float64)[None], [1], True)[0]
        assert rel_l2(got[k], ref) < LINE_TOL[fp64], (k, size[k])
        assert rel_l2(back[k], x[k]) < LINE_TOL[fp64], (k, size[k])


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("n", [60, 504])
def test_images_of_an_odd_number_of_rows(dev, n, fp64):
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (3, 5, n)).astype(np.float64 if fp64 else np.float32)
    x[1, 2, 3] = np.nan
    outs, backs, _, plan = run_gpu_plan(dev, x, [3, 5, n], [1, 2], [1, 1, 1], [1, 1, 1], True, fp64)
    plan.destroy()
    for k in (0, 2):
        ref = F.fftn(x[k].astype(np.float64), [0, 1], True)
        assert rel_l2(outs[0][k], ref) < LINE_TOL[fp64]
        assert rel_l2(backs[0][k], x[k]) < LINE_TOL[fp64]


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("n", [20, 54, 81, 96, 160, 162, 243, 375, 504, 625, 729, 1155, 1536, 2187, 3125])
def test_forward_errors(dev, n, fp64):
    if _pairs(n, fp64):
        pytest.skip("in pairs")
    x = _lines(n).real.astype(np.float64 if fp64 else np.float32)
    outs, _, _, plan = run_gpu_plan(dev, x, list(x.shape), [0], [1, 1], [1, 1], True, fp64)
    plan.destroy()
    ref = _exact(x)[:n // 2 + 1]
    per_element = _per_element(dev, x.astype(np.complex128 if fp64 else np.complex64), fp64)[:n // 2 + 1]
    assert rel_l2(outs[0], ref) < TOL * rel_l2(per_element, ref)


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("n", [20, 54, 81, 96, 160, 162, 243, 375, 504, 625, 729, 1155, 1536, 2187, 3125])
def test_backward_errors(dev, n, fp64):
    """The per-element kernel runs the Hermitian extension as a complex line; the
    real part of its output is the C2R line.  Of the early stages' errors half
    falls into the imaginary part, which a real output does not keep; the values
    of the last stage lie in the real part, and all of its errors count.  With
    fewer, larger radices that stage has a larger share: 1.25 times the squared
    error allowed (two lines of a pair keep both parts: 2)."""
    if _pairs(n, fp64):
        pytest.skip("in pairs")
    import torch
    import dfft
    cdt, rdt = (np.complex128, np.float64) if fp64 else (np.complex64, np.float32)
    x = _lines(n).real
    full = _exact(x).astype(cdt)
    half = np.ascontiguousarray(full[:n // 2 + 1])
    half[0].imag = 0
    if n % 2 == 0:
        half[-1].imag = 0
    full = np.concatenate([half, np.conj(half[1:(n + 1) // 2][::-1])])
    a = torch.empty(x.shape, dtype=torch.float64 if fp64 else torch.float32, device=dev)
    b = torch.from_numpy(half).to(dev)
    plan = dfft.Plan([a], [b], [0], [1, 1], [1, 1], norm="none", global_in_extents=list(x.shape),
                     global_out_extents=list(half.shape))
    dfft.execute(plan, [b], [a], dfft.Direction.backward)
    got = a.cpu().numpy()
    plan.destroy()
    ref = np.conj(_exact(np.conj(full))).real
    per_element = _per_element(dev, np.conj(full), fp64).real.astype(rdt)
    assert rel_l2(got, ref) < TOL * np.sqrt(1.25) * rel_l2(per_element, ref)


@pytest.mark.parametrize("fp64", [True, False])
@pytest.mark.parametrize("n", [8, 60, 512, 1024])
def test_group_members_launched_on_their_own(dev, n, fp64):
    """Lengths without a grouped kernel, 8, 512 and 1024 among them."""
    import torch
    import dfft
    rdt, cdt = (torch.float64, torch.complex128) if fp64 else (torch.float32, torch.complex64)
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, (5, n))
    x[1] *= 1e8
    x[3, 0] = np.nan
    a = torch.from_numpy(x).to(dev, rdt)
    b = torch.empty((5, n // 2 + 1), dtype=cdt, device=dev)
    c = torch.empty_like(a)
    g = dfft.Group([a], [b], [1])
    g.execute([a], [b], dfft.Direction.forward)
    g.execute([b], [c], dfft.Direction.backward)
    x, got, back = a.cpu().numpy(), b.cpu().numpy(), c.cpu().numpy()
    for k in (0, 1, 2, 4):
        assert rel_l2(got[k], F.fftn(x[k].astype(np.float64)[None], [1], True)[0]) < LINE_TOL[fp64], k
        assert rel_l2(back[k], x[k]) < LINE_TOL[fp64], k
