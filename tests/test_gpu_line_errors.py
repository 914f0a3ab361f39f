"""Rounding errors of the register line kernels, measured against an extended
precision FFT and compared with those of the per-element kernel, which reads
every twiddle from the table and adds whole sums.  It runs the same lines where
the line axis is split over ranks."""

import numpy as np
import pytest

from helpers import rel_l2, run_gpu_plan

pytestmark = pytest.mark.gpu

# The register kernels are to be no further off.  Both errors are root mean
# squares over some 65536 complex values of random lines, whose rounding errors
# are all but independent: their ratio is known to about 1 %; three of these.
TOL = 1.03


def _lines(n):
    w = max(4, 65536 // n // 2 * 2)
    rng = np.random.default_rng(n)
    return rng.uniform(-1, 1, (n, w)) + 1j * rng.uniform(-1, 1, (n, w))


def _exact(x):
    import scipy.fft
    return scipy.fft.fft(x.astype(np.clongdouble), axis=0)


def _per_element(dev, x, fp64):
    outs, _, _, plan = run_gpu_plan(dev, x, list(x.shape), [0], [2, 1], [2, 1], False, fp64)
    plan.destroy()
    return np.concatenate(outs, axis=0)


def _complex_errors(dev, n, fp64):
    x = _lines(n).astype(np.complex128 if fp64 else np.complex64)
    outs, _, _, plan = run_gpu_plan(dev, x, list(x.shape), [0], [1, 1], [1, 1], False, fp64)
    plan.destroy()
    ref = _exact(x)
    return rel_l2(outs[0], ref), rel_l2(_per_element(dev, x, fp64), ref)


@pytest.mark.parametrize("n", [25, 27, 81, 125, 162, 243, 324, 375, 486, 504, 625, 648, 729, 972, 1701, 2187, 3125, 4374])
def test_fp32_lines(dev, n):
    here, per_element = _complex_errors(dev, n, False)
    assert here < TOL * per_element, (here, per_element)


@pytest.mark.parametrize("n", [20, 90, 98, 99, 140, 143, 162, 250, 300, 324, 375, 441, 504, 539, 648, 729, 900, 1000,
                               1001, 1155, 1280, 1536, 1701, 2187, 2401, 3125, 4374, 4802, 5120])
def test_fp64_lines(dev, n):
    here, per_element = _complex_errors(dev, n, True)
    assert here < TOL * per_element, (here, per_element)


@pytest.mark.parametrize("n", [96, 160])
@pytest.mark.parametrize("real", [False, True])
def test_fp64_grouped_lines(dev, n, real):
    """Grouped lines of 96 and 160 points: the power-of-two kernel with a radix 6 or 10."""
    import torch
    import dfft
    x = _lines(n)
    x = np.ascontiguousarray((x.real if real else x).T)
    a = torch.from_numpy(x).to(dev)
    b = torch.empty((x.shape[0], n // 2 + 1 if real else n), dtype=torch.complex128, device=dev)
    g = dfft.Group([a], [b], [1], norm="none")
    g.execute([a], [b], dfft.Direction.forward)
    ref = _exact(x.T)[:b.shape[1]]
    per_element = _per_element(dev, x.T.astype(np.complex128), True)[:b.shape[1]]
    here, there = rel_l2(b.cpu().numpy().T, ref), rel_l2(per_element, ref)
    assert here < TOL * there, (here, there)
