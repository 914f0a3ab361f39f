"""The divergence-form solver on the kept modes of the 2/3 rule against the
same solver on all modes: steps, right-hand side, tangent, adjoint, gradient,
with rank blocks that hold both, one or none of the kept runs."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the two paths add the same terms (the skipped ones are zeros)
TOL = 1e-13


def _solver(n, px, py, kept):
    import dfft_ns
    s = dfft_ns.NavierStokes(n, px, py, lx=2.0, nu=0.01, dt=1e-2, form=dfft_ns.DIVERGENCE)
    s.set_option("kept_modes", kept)
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


def _beyond(s, blocks):
    """Largest magnitude among the modes beyond the cutoff."""
    cut = ((s.n // 2) * 2) // 3
    most = 0.0
    for r, b in enumerate(blocks):
        e, st = s.local_extents(r, 1)
        k = [np.arange(st[a], st[a] + e[a]) for a in range(3)]
        for a in range(2):
            k[a] = np.minimum(k[a], s.n - k[a])
        keep = (k[0] <= cut)[:, None, None] & (k[1] <= cut)[None, :, None] & (k[2] <= cut)[None, None, :]
        v = np.abs(b.cpu().numpy())[:, ~keep]
        most = max(most, float(v.max()) if v.size else 0.0)
    return most


GRIDS = [(8, 1, 1), (16, 1, 1), (16, 2, 2), (16, 3, 2), (16, 1, 5), (32, 2, 1), (32, 1, 3), (64, 2, 2), (64, 4, 1),
         (128, 1, 1), (128, 2, 2), (256, 2, 2)]


@pytest.mark.parametrize("n,px,py", GRIDS)
def test_steps(dev, n, px, py):
    a, b = _solver(n, px, py, 1), _solver(n, px, py, 0)
    assert a.get_option("kept_modes") == 1 and b.get_option("kept_modes") == 0
    for s in (a, b):
        s.set_physical(_velocity(s, n, dev))
    assert _err(a.get_state(), b.get_state()) < TOL
    for s in (a, b):
        s.step(2)
        s.step(3, use_graph=True)
    ya, yb = a.get_state(), b.get_state()
    assert _err(ya, yb) < TOL
    assert _beyond(a, ya) == 0.0
    assert abs(a.energy() - b.energy()) < TOL * abs(b.energy())
    # the stored products take the banded forward transform without the fused loads
    a.set_option("fuse_products", 0)
    a.step(1)
    b.step(1)
    assert _err(a.get_state(), b.get_state()) < TOL


@pytest.mark.parametrize("n,px,py", GRIDS[:-1])
def test_derivatives(dev, n, px, py):
    a, b = _solver(n, px, py, 1), _solver(n, px, py, 0)
    u = _velocity(a, n + 1, dev)
    for s in (a, b):
        s.set_physical(u)
    y = b.get_state()
    d = [0.5 * t.flip(0).contiguous() for t in y]
    for out in (lambda s: s.rhs(y), lambda s: s.rhs_tangent(y, d), lambda s: s.rhs_adjoint(y, d)):
        ra, rb = out(a), out(b)
        assert _err(ra, rb) < TOL
        assert _beyond(a, ra) == 0.0
    ja, ga = a.gradient(3, u, checkpoint_every=2)
    jb, gb = b.gradient(3, u, checkpoint_every=2)
    assert abs(ja - jb) < TOL * abs(jb) and _err(ga, gb) < TOL


def test_arguments_with_modes_beyond_the_cutoff(dev):
    """rhs and its derivatives dealias their arguments: what lies beyond the cutoff does not count."""
    import torch
    n = 32
    a, b = _solver(n, 2, 2, 1), _solver(n, 2, 2, 0)
    y = [torch.randn(3, *a.local_extents(r, 1)[0], dtype=torch.complex128, device=dev) for r in range(4)]
    lam = [torch.randn_like(t) for t in y]
    for out in (lambda s: s.rhs(y), lambda s: s.rhs_tangent(y, lam), lambda s: s.rhs_adjoint(y, lam)):
        assert _err(out(a), out(b)) < TOL
    for s in (a, b):
        s.set_state(y)
        s.step(1)
    assert _err(a.get_state(), b.get_state()) < TOL


def test_tuned_plans(dev):
    a, b = _solver(64, 2, 2, 1), _solver(64, 2, 2, 0)
    a.autotune()
    for s in (a, b):
        s.set_physical(_velocity(s, 7, dev))
        s.step(2, use_graph=True)
    assert _err(a.get_state(), b.get_state()) < TOL


def test_where_all_modes_are_handled(dev):
    import dfft
    import dfft_ns
    assert _solver(24, 2, 2, 1).get_option("kept_modes") == 0  # 24-point lines: no such kernel
    assert dfft_ns.NavierStokes(16, 1, 1, form=dfft_ns.ADVECTIVE).get_option("kept_modes") == 0
    with pytest.raises(dfft.DFFTError):
        _solver(16, 1, 1, 2)
