"""The differentiable scheme's forward at the ends of the number range: its short
quotients give way to the division where a numerator or a quotient is next to
underflow, and a numerator next to overflow has a finite quotient.  The oracle's
bits throughout."""
import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu
N = (8, 9, 66)


def state(rho, v, e, ye):
    """Random flow with its variables scaled by powers of two; huge densities need
    uniform pressure and next to no velocity, whose square is taken."""
    rng = np.random.default_rng(abs(rho) + abs(ye))
    W = np.empty((6,) + N)
    W[0] = 1.0 + 0.1 * rng.standard_normal(N).clip(-3, 3)
    W[1:4] = 0.3 * rng.standard_normal((3,) + N)
    W[4] = 1.5 + 0.1 * rng.standard_normal(N).clip(-3, 3)
    W[5] = 0.1 + 0.01 * rng.standard_normal(N)
    if rho > 0:
        W[0], W[4] = 1.0, 31.5
    for q, s in zip((W[0], W[1:4], W[4], W[5]), (rho, v, e, ye)):
        np.multiply(q, 2.0 ** s, out=q)
    return W


@pytest.mark.parametrize("scale", [(0, 0, 0, 0), (0, 0, 0, -930), (0, 0, 0, -962), (0, 0, 0, -1010),
                                   (0, 0, 0, -1060), (-930, 0, 0, 0), (-1000, 0, 0, 0),
                                   (-1035, 0, 0, 0), (0, -1000, 0, 0),
                                   (1000, -520, 0, 0), (1017, -520, 0, 0)])
def test_forward_is_the_oracles(gpu, scale):
    import torch
    from fornaxamr_amd.adjoint import AdjointSolver
    W = state(*scale)
    xlim = sum(((0.0, float(n)) for n in N), ())
    solver = AdjointSolver(N, xlim, 1.4, va_eps2=1e-4, checkpoint_every=2)
    dt, steps = 0.02, 2
    WT = solver.forward(torch.from_numpy(W).cuda(), steps, dt).cpu().numpy()
    solver.close()
    want = O.adj_forward(W, xlim, 1.4, 1e-4, dt, steps)
    assert np.isfinite(want).all()
    assert np.array_equal(WT, want), np.unravel_index(np.argmax(WT != want), WT.shape)
