"""The solver's packed state (kept modes in one array of all ranks) against the
state in rank blocks: every way in and out of it, the diagnostics, and the
change of form in the middle of a run."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the same operations on the same modes in both forms; energies and bins sum in another order
TOL = 1e-14
GRIDS = [(8, 1, 1), (16, 2, 2), (32, 3, 1), (32, 1, 4), (64, 2, 4)]


def _solver(n, px, py, kept):
    import dfft_ns
    s = dfft_ns.NavierStokes(n, px, py, lx=2.0, nu=0.01, dt=1e-3)
    s.set_option("kept_modes", kept)
    return s


def _random_spectrum(s, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    y = s.spectral_fields()
    for t in y:
        t.copy_(torch.view_as_complex(torch.rand(list(t.shape) + [2], generator=g, device="cuda", dtype=torch.float64)))
    return y


def _err(a, b):
    num = sum(float((x - y).abs().pow(2).sum()) for x, y in zip(a, b))
    den = sum(float(y.abs().pow(2).sum()) for y in b)
    return np.sqrt(num / den)


@pytest.mark.parametrize("n,px,py", GRIDS)
def test_in_and_out(dev, n, px, py):
    a, b = _solver(n, px, py, 1), _solver(n, px, py, 0)
    assert a.get_option("kept_modes") == 1
    y = _random_spectrum(a, n)  # modes beyond the cutoff too
    a.set_state(y)
    b.set_state(y)
    for u, v in zip(a.get_state(), b.get_state()):
        assert np.array_equal(u.cpu().numpy(), v.cpu().numpy())
    assert abs(a.energy() - b.energy()) <= TOL * b.energy()
    a.init_taylor_green()
    b.init_taylor_green()
    for s in (a, b):
        s.step(2)
    assert _err(a.velocity(), b.velocity()) < TOL
    assert _err(a.vorticity(), b.vorticity()) < TOL
    ea, eb = a.energy_spectrum(10)[0], b.energy_spectrum(10)[0]
    assert np.allclose(ea, eb, rtol=1e-12, atol=1e-12 * max(eb))
    assert _err(a.get_state(), b.get_state()) < TOL


@pytest.mark.parametrize("n,px,py", GRIDS)
def test_change_of_form_in_a_run(dev, n, px, py):
    a, b = _solver(n, px, py, 1), _solver(n, px, py, 0)
    for s in (a, b):
        s.init_taylor_green()
    for kept in (1, 0, 1, 1, 0):
        a.set_option("kept_modes", kept)
        a.step(1, use_graph=True)
        b.step(1, use_graph=True)
    assert _err(a.get_state(), b.get_state()) < TOL
    a.set_option("kept_modes", 1)
    assert _err(a.get_state(), b.get_state()) < TOL
