"""Kept modes at every grid size class of the compiled band kernels that the
other tests leave out, and at 512: steps with the products formed in the
forward transform and apart, and gradients, against the solver on all modes."""

import pytest

pytestmark = pytest.mark.gpu

# the two paths add the same terms (the skipped ones are zeros), in another
# grouping where their kernels' radices differ
TOL = 1e-13


def _solver(n, px, py, kept, fuse=1):
    import dfft_ns
    s = dfft_ns.NavierStokes(n, px, py, lx=2.0, nu=0.01, dt=1e-3, form=dfft_ns.DIVERGENCE)
    s.set_option("kept_modes", kept)
    s.set_option("fuse_products", fuse)
    assert s.get_option("kept_modes") == kept
    return s


def _velocity(s, dev):
    import torch
    out = []
    for r in range(s.nranks):
        e, _ = s.local_extents(r, 0)
        gen = torch.Generator(device=dev).manual_seed(r)
        out.append(torch.rand([3] + list(e), generator=gen, device=dev, dtype=torch.float64) - 0.5)
    return out


def _err(a, b):
    import torch
    num = sum(float(torch.linalg.vector_norm(x - y)) ** 2 for x, y in zip(a, b))
    den = sum(float(torch.linalg.vector_norm(y)) ** 2 for y in b)
    return (num / den) ** 0.5


def _state(n, px, py, kept, fuse, dev):
    s = _solver(n, px, py, kept, fuse)
    s.set_physical(_velocity(s, dev))
    s.step(2)
    y = s.get_state()
    s.destroy()
    return y


@pytest.mark.parametrize("n,px,py", [(54, 2, 1), (80, 1, 1), (108, 2, 2), (144, 1, 2), (162, 2, 1), (180, 1, 1),
                                     (192, 2, 2), (216, 1, 3), (240, 2, 1), (250, 1, 1), (270, 2, 2), (288, 1, 2),
                                     (300, 3, 1), (320, 2, 2), (324, 1, 1), (360, 2, 1), (384, 1, 2), (512, 2, 1)])
def test_steps(dev, n, px, py):
    want = _state(n, px, py, 0, 1, dev)
    assert _err(_state(n, px, py, 1, 1, dev), want) < TOL
    assert _err(_state(n, px, py, 1, 0, dev), want) < TOL


@pytest.mark.parametrize("n,px,py", [(144, 1, 2), (192, 2, 1), (250, 1, 1), (320, 2, 2)])
def test_gradients(dev, n, px, py):
    got = []
    for kept in (1, 0):
        s = _solver(n, px, py, kept)
        got.append(s.gradient(2, _velocity(s, dev), 1))
        s.destroy()
    assert abs(got[0][0] - got[1][0]) < TOL * got[1][0]
    assert _err(got[0][1], got[1][1]) < TOL
