"""The HLLC face solver's sound speeds take a short form of sqrt(a / b) where
every lane of a wave is well within the exponent range, and the full operations
elsewhere: fluxes bit for bit those of the oracle for states inside the range,
at its edges, outside it, and with one lane of each wave outside."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu
N = 64 * 150 + 37


def states(kind):
    rng = np.random.default_rng(7)
    W = rng.standard_normal((2, N, 6))
    e = {"inside": (-8, 8), "wide": (-140, 140), "edges": (298, 302), "outside": (-500, 500)}
    lo, hi = e.get(kind, e["inside"])
    rho, p = (rng.uniform(1, 2, (2, N)) * 2.0 ** rng.uniform(lo, hi, (2, N)) for _ in range(2))
    if kind == "edges":
        flip = rng.integers(0, 2, (2, N)) == 0
        rho[flip], p[flip] = 1.0 / rho[flip], 1.0 / p[flip]
    if kind == "one_lane":
        at = np.arange(0, N, 64) + rng.integers(0, 64, (N + 63) // 64)
        at = at[at < N]
        p[0, at] = rng.choice([0.0, 5e-324, 1e-310, 1e-95, 1e95, 1e300], at.size)
    W[..., 0] = rho
    W[..., 1:4] *= np.sqrt(p / rho)[..., None]
    W[..., 4] = p / (0.4 * rho)
    d = rng.standard_normal((3, N))
    return W, p, d


@pytest.mark.parametrize("kind", ["inside", "wide", "edges", "outside", "one_lane"])
def test_hllc_over_the_range(gpu, kind):
    import torch
    W, p, d = states(kind)
    g = np.full(N, 1.4)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    args = [dev(W[0].T), dev(W[1].T), dev(p[0]), dev(p[1]), dev(g), dev(g), *map(dev, d)]
    F = torch.empty((6, N), dtype=torch.float64, device="cuda")
    vf = torch.empty((3, N), dtype=torch.float64, device="cuda")
    assert gpu.fx_riemann_hllc_batch(N, *[a.data_ptr() for a in args], F.data_ptr(),
                                     vf.data_ptr(), None) == 0
    torch.cuda.synchronize()
    want = np.empty((N, 6)), np.empty((N, 3))
    ptr = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    lib = O.oracle_lib()
    with np.errstate(all="ignore"):
        for i in range(N):
            lib.fxo_hllc(ptr(W[0, i]), ptr(W[1, i]), p[0, i], p[1, i], 1.4, 1.4,
                         ptr(want[0][i]), ptr(want[1][i]), d[0, i], d[1, i], d[2, i])
    for got, w in ((F, want[0]), (vf, want[1])):
        assert np.array_equal(got.cpu().numpy().T, w, equal_nan=True)
