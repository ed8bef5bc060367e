"""The differentiable scheme on boxes whose axes do not fit the windows of its
kernels (32 positions along x and y, 64 lanes along z): from the smallest box to
axes just below, at and above one and two windows.  The forward is the oracle's to
the bit; the gradient satisfies the dot-product identity with the oracle's
tangent-linear model."""
import numpy as np
import pytest

import pyoracle as O
from fornaxamr_amd import problems as P

pytestmark = pytest.mark.gpu
DOT_TOL = 1e-11     # two sums of some 10^4-10^5 rounded products, ~1e-13 relative


@pytest.mark.parametrize("n", [(4, 4, 4), (5, 33, 7), (29, 6, 61), (31, 28, 62), (57, 61, 9),
                               (8, 17, 125)])
def test_windows(gpu, n):
    import torch
    from fornaxamr_amd.adjoint import AdjointSolver
    rng = np.random.default_rng(sum(n))
    W = np.empty((6,) + n)
    W[0] = 1.0 + 0.1 * rng.standard_normal(n).clip(-3, 3)
    W[1:4] = 0.3 * rng.standard_normal((3,) + n)
    W[4] = 1.5 + 0.1 * rng.standard_normal(n).clip(-3, 3)
    W[5] = 0.1 + 0.01 * rng.standard_normal(n)
    xlim = (0.0, 1.0, 0.0, 1.5, 0.0, 2.0)
    solver = AdjointSolver(n, xlim, 1.4, va_eps2=1e-4, checkpoint_every=2)
    dt, steps = 0.1 / (2.0 * sum(n)), 3
    WT = solver.forward(torch.from_numpy(W).cuda(), steps, dt)
    assert np.array_equal(WT.cpu().numpy(), O.adj_forward(W, xlim, 1.4, 1e-4, dt, steps))
    g = rng.standard_normal(W.shape)
    gW0 = solver.backward(torch.from_numpy(g).cuda()).cpu().numpy()
    d = rng.standard_normal(W.shape)
    _, dWT = O.adj_tlm(W, d, xlim, 1.4, 1e-4, dt, steps)
    a, b = float(np.sum(gW0 * d)), float(np.sum(g * dWT))
    assert abs(a - b) <= DOT_TOL * np.sqrt(np.sum((gW0 * d) ** 2) + np.sum((g * dWT) ** 2)) + DOT_TOL * abs(b)
    solver.close()
