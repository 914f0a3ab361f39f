"""Kept modes of grids of 2^a 3^b 5^c points (compiled kernels that are no power
of two): steps, the products inside the forward transform, tangent, adjoint and
gradient against the solver on all modes."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the two paths add the same terms (the skipped ones are zeros)
TOL = 1e-13
GRIDS = [(36, 1, 1), (40, 2, 2), (48, 1, 3), (50, 3, 2), (60, 2, 1), (72, 1, 1), (90, 2, 2), (96, 2, 2), (100, 1, 2),
         (120, 2, 2), (150, 1, 1), (160, 2, 2), (200, 1, 1)]


def _solver(n, px, py, kept, fuse=1):
    import dfft_ns
    s = dfft_ns.NavierStokes(n, px, py, lx=2.0, nu=0.01, dt=1e-2, form=dfft_ns.DIVERGENCE)
    s.set_option("kept_modes", kept)
    s.set_option("fuse_products", fuse)
    return s


def _velocity(s, seed, dev):
    import torch
    u = np.random.default_rng(seed).standard_normal((3, s.n, s.n, s.n))
    out = []
    for r in range(s.nranks):
        e, st = s.local_extents(r, 0)
        sl = (slice(None),) + tuple(slice(a, a + b) for a, b in zip(st, e))
        out.append(torch.from_numpy(np.ascontiguousarray(u[sl])).to(dev))
    return out


def _err(a, b):
    import torch
    num = sum(float(torch.linalg.vector_norm(x - y)) ** 2 for x, y in zip(a, b))
    den = sum(float(torch.linalg.vector_norm(y)) ** 2 for y in b)
    return (num / den) ** 0.5


@pytest.mark.parametrize("n,px,py", GRIDS)
def test_steps(dev, n, px, py):
    a, b, c = _solver(n, px, py, 1), _solver(n, px, py, 0), _solver(n, px, py, 1, 0)
    assert a.get_option("kept_modes") == 1 and a.get_option("products_fused") == 1
    assert b.get_option("kept_modes") == 0 and c.get_option("products_fused") == 0
    for s in (a, b, c):
        s.set_physical(_velocity(s, n, dev))
        s.step(2, use_graph=True)
    assert _err(a.get_state(), b.get_state()) < TOL
    assert _err(c.get_state(), b.get_state()) < TOL
    assert _err(a.velocity(), b.velocity()) < TOL


@pytest.mark.parametrize("n,px,py", GRIDS[:8])
def test_derivatives(dev, n, px, py):
    a, b = _solver(n, px, py, 1), _solver(n, px, py, 0)
    for s in (a, b):
        s.set_physical(_velocity(s, 1, dev))
    y = b.get_state()
    for s in (a, b):
        s.set_physical(_velocity(s, 2, dev))
    d = b.get_state()
    assert _err(a.rhs(y), b.rhs(y)) < TOL
    assert _err(a.rhs_tangent(y, d), b.rhs_tangent(y, d)) < TOL
    assert _err(a.rhs_adjoint(y, d), b.rhs_adjoint(y, d)) < TOL
    ja, ga = a.gradient(3, _velocity(a, 3, dev), 2)
    jb, gb = b.gradient(3, _velocity(b, 3, dev), 2)
    assert abs(ja - jb) < TOL * jb
    assert _err(ga, gb) < TOL
