"""Poisson integration at the edges of its tiles (64 modes of each parity, 16 per
step, groups of 8 in the elimination), odd and even interiors, against the
sparse LU oracle (1e-6 relative L2, FP64 arithmetic rounded to FP32 once); and
two solves of different sizes in a row on one context, whose workspace is kept."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_grad import gpu_poisson

pytestmark = pytest.mark.gpu


def fields(n):
    rng = np.random.default_rng(n)
    return [rng.standard_normal((n + 1,) * 3).astype(np.float32) for _ in range(2)]


@pytest.mark.parametrize("n", [3, 4, 5, 9, 10, 34, 35, 66, 67])
def test_poisson_sizes(orc, xr, ctx, torch_dev, n):
    g0, g1 = fields(n)
    assert rel_l2(gpu_poisson(xr, ctx, torch_dev, n, g0, g1).reshape(-1), orc.poisson_solve(g0, g1, n).reshape(-1)) <= 1e-6


@pytest.mark.parametrize("n", [130, 131, 133])
def test_poisson_solves_the_system(xr, ctx, torch_dev, n):
    """The 5-point residual in FP64, relative to the right side times the FP32
    rounding of the solution (2^-24) amplified by the stencil (8 |F|)."""
    g0, g1 = fields(n)
    small = gpu_poisson(xr, ctx, torch_dev, 12, *fields(12))
    f = np.asarray(gpu_poisson(xr, ctx, torch_dev, n, g0, g1), np.float64).reshape(n, n, n)
    assert np.array_equal(small, gpu_poisson(xr, ctx, torch_dev, 12, *fields(12)))
    a, b = g0, g1
    rhs = (((a[:n, :n, :n] - a[:n, :n, 1:]) + b[:n, :n, :n]) - b[:n, 1:, :n])[:, 1:-1, 1:-1]
    res = 4 * f[:, 1:-1, 1:-1] - f[:, 2:, 1:-1] - f[:, :-2, 1:-1] - f[:, 1:-1, 2:] - f[:, 1:-1, :-2] - rhs
    assert np.abs(res).max() <= 8 * np.abs(f).max() * 2.0 ** -24
    assert not f[:, 0].any() and not f[:, -1].any() and not f[:, :, 0].any() and not f[:, :, -1].any()
