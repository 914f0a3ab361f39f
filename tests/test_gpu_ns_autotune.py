"""NavierStokes.autotune times the kernels that the step launches, and leaves
state and results as they are."""

import pytest

pytestmark = pytest.mark.gpu

# the tuned shapes add the same terms in the same order within a line
TOL = 1e-13


def _solver(n, px, py, kept):
    import dfft_ns
    s = dfft_ns.NavierStokes(n, px, py, lx=2.0, nu=0.01, dt=1e-2, form=dfft_ns.DIVERGENCE)
    s.set_option("kept_modes", kept)
    s.init_taylor_green()
    s.step(1)
    return s


def _err(a, b):
    import torch
    num = sum(float(torch.linalg.vector_norm(x - y)) ** 2 for x, y in zip(a, b))
    den = sum(float(torch.linalg.vector_norm(y)) ** 2 for y in b)
    return (num / den) ** 0.5


@pytest.mark.parametrize("kept", [1, 0])
@pytest.mark.parametrize("n,px,py", [(16, 1, 1), (32, 2, 2), (48, 1, 3), (64, 2, 1)])
def test_results_stay(dev, n, px, py, kept):
    a, b = _solver(n, px, py, kept), _solver(n, px, py, kept)
    b.autotune()
    assert _err(b.get_state(), a.get_state()) == 0.0
    for s in (a, b):
        s.step(2, use_graph=True)
    assert _err(b.get_state(), a.get_state()) < TOL
    assert _err(b.velocity(), a.velocity()) < TOL


def _line_kernels(run):
    """Names of the line kernels `run` launches, up to the kind of memory access."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    run()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        run()
        torch.cuda.synchronize()
    names = {e.key for e in p.key_averages() if "fft_" in e.key}
    assert names
    return names


@pytest.mark.parametrize("n", [32, 48])
def test_the_step_s_kernels_are_timed(dev, n):
    s = _solver(n, 2, 1, 1)
    assert s.get_option("kept_modes") == 1
    s.set_option("fuse_products", 0)  # the products' own instance is not timed
    tuned = _line_kernels(s.autotune)
    assert _line_kernels(lambda: s.step(1)) <= tuned
