"""HLLD's fast speeds take short forms of their divisions and square roots where
every lane of a wave is well within the exponent range: fluxes and statuses those of
the oracle with densities, pressures and fields around the range's ends, zero and
denormal fields, and with one lane of each wave outside."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as O

pytestmark = pytest.mark.gpu
N = 64 * 70 + 9


@pytest.mark.parametrize("kind", ["inside", "ends", "zero_field", "tiny_field", "one_lane"])
def test_hlld_over_the_range(gpu, kind):
    import torch
    rng = np.random.default_rng(5)
    W = rng.standard_normal((2, N, 9))
    W[..., 0] = rng.uniform(0.5, 2, (2, N))
    p = rng.uniform(0.5, 2, (2, N))
    bn = rng.standard_normal(N)
    if kind == "ends":       # rho, p and B^2 scaled together: sound speeds stay near 1
        s = 2.0 ** rng.choice([-302, -301, -300, -299, 298, 299, 300, 301], N)
        W[..., 0] *= s
        p *= s
        W[..., 6:9] *= np.sqrt(s)[:, None]
        bn *= np.sqrt(s)
    if kind in ("zero_field", "tiny_field"):
        f = 0.0 if kind == "zero_field" else 2.0 ** rng.choice([-160, -150, -149, -400, -537], N)
        bn = bn * f
        W[..., 6:9] *= np.asarray(f)[..., None]
    if kind == "one_lane":
        at = np.arange(0, N, 64) + rng.integers(0, 64, (N + 63) // 64)
        at = at[at < N]
        p[1, at] = rng.choice([0.0, 5e-324, 1e-95, 1e95, -1.0], at.size)
        bn[at[::3]] = rng.choice([1e-160, 1e60], at[::3].size)
    W[..., 4] = p / (W[..., 0] * 0.4)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    g = np.full(N, 1.4)
    args = [dev(W[0].T), dev(W[1].T), *map(dev, (p[0], p[1], g, g, bn))]
    out = torch.zeros((14, N), dtype=torch.float64, device="cuda")
    st = torch.zeros(N, dtype=torch.int32, device="cuda")
    assert gpu.fx_riemann_hlld_batch(N, *[a.data_ptr() for a in args],
                                     *[out[k].data_ptr() for k in (0, 9, 12, 13)],
                                     st.data_ptr(), None) == 0
    torch.cuda.synchronize()
    got, st = out.cpu().numpy(), st.cpu().numpy()
    ptr = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    lib = O.oracle_lib()
    want, code = np.zeros((14, N)), np.zeros(N, dtype=np.int64)
    o = [np.zeros(9), np.zeros(3), np.zeros(1), np.zeros(1)]
    for i in range(N):
        code[i] = lib.fxo_hlld(ptr(W[0, i]), ptr(W[1, i]), p[0, i], p[1, i], 1.4, 1.4, bn[i],
                               *map(ptr, o))
        want[:, i] = np.concatenate(o)
    ok = code == 0
    assert ok.any()
    assert np.array_equal(st, code)
    assert np.array_equal(got[:, ok], want[:, ok], equal_nan=True)
