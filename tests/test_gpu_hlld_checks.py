"""HLLD's checks of both states share one branch, and its star terms are added
under the lane mask: fluxes bit for bit the oracle's wherever it accepts the
face, a status exactly where it refuses, and of several failing checks the first
in the reference's order (left state before right one; density, pressure, gamma)."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu
N = 64 * 90 + 21


def run(gpu, W, p, g, bn):
    import torch
    n = len(bn)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    args = [dev(W[0].T), dev(W[1].T), *map(dev, (p[0], p[1], g[0], g[1], bn))]
    out = [torch.full(s, -7.0, dtype=torch.float64, device="cuda") for s in ((9, n), (3, n), (n,), (n,))]
    st = torch.zeros(n, dtype=torch.int32, device="cuda")
    assert gpu.fx_riemann_hlld_batch(n, *[a.data_ptr() for a in args],
                                     *[o.data_ptr() for o in out], st.data_ptr(), None) == 0
    torch.cuda.synchronize()
    return np.concatenate([o.cpu().numpy().reshape(-1, n) for o in out]), st.cpu().numpy()


# range of the states' exponents, share of faces with zero or refused entries
@pytest.mark.parametrize("spread,share", [(1, 0.0), (6, 0.0), (3, 0.02), (3, 0.3)])
def test_hlld_against_oracle(gpu, spread, share):
    rng = np.random.default_rng(11)
    e = lambda *s: 2.0 ** rng.uniform(-spread, spread, s)
    W = rng.standard_normal((2, N, 9)) * e(2, N, 9)
    W[..., [0, 4]] = np.abs(W[..., [0, 4]])
    p = np.abs(rng.standard_normal((2, N))) * e(2, N)
    g = np.full((2, N), 5.0 / 3.0)
    bn = rng.standard_normal(N) * e(N)
    for a in (W[..., 0], p, g, bn):
        at = rng.random(a.shape) < share
        a[at] = rng.choice([0.0, -1.0], at.sum())
    got, st = run(gpu, W, p, g, bn)
    lib = O.oracle_lib()
    want, code = np.zeros((14, N)), np.zeros(N, dtype=np.int64)
    ptr = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    o = [np.zeros(9), np.zeros(3), np.zeros(1), np.zeros(1)]
    for i in range(N):
        code[i] = lib.fxo_hlld(ptr(W[0, i]), ptr(W[1, i]), p[0, i], p[1, i], g[0, i], g[1, i],
                               bn[i], *map(ptr, o))
        want[:, i] = np.concatenate(o)
    ok = code == 0
    assert np.array_equal(st == 0, ok)
    assert np.array_equal(got[:, ok], want[:, ok])
    assert not got[:, ~ok].any()     # a refused face has zero outputs


def test_first_failing_check(gpu):
    W = np.ones((2, 6, 9))
    p, g, bn = np.ones((2, 6)), np.full((2, 6), 1.4), np.ones(6)
    W[0, 0, 0] = p[0, 0] = -1.0           # left density before left pressure
    p[0, 1] = g[0, 1] = -1.0              # left pressure before left gamma
    g[0, 2] = W[1, 2, 0] = -1.0           # left gamma before right density
    W[1, 3, 0] = p[1, 3] = -1.0           # right density before right pressure
    p[1, 4] = -1.0
    _, st = run(gpu, W, p, g, bn)
    assert st.tolist() == [11, 12, 13, 11, 12, 0]
