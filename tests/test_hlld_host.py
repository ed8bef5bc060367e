"""The library's HLLD solver, compiled for the host: the oracle's bits and codes,
and no output formed from a variable that was never set, on refused faces either
(the same bits whatever such a variable holds)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import pyoracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def builds(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("clang++ not available")
    d = tmp_path_factory.mktemp("hlld_host")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text("")
    libs = []
    for fill in ("zero", "pattern"):
        so = str(d / f"libhlld_{fill}.so")
        subprocess.run([CLANG, "-std=c++17", "-O1", "-ffp-contract=off", "-fPIC", "-shared",
                        "-DNDEBUG", f"-ftrivial-auto-var-init={fill}", f"-I{d}",
                        os.path.join(HERE, "hlld_host.cpp"), "-o", so], check=True)
        libs.append(C.CDLL(so))
    return libs


def faces(n, seed, spread, share):
    rng = np.random.default_rng(seed)
    e = lambda *s: 2.0 ** rng.uniform(-spread, spread, s)
    W = rng.standard_normal((2, n, 9)) * e(2, n, 9)
    W[..., [0, 4]] = np.abs(W[..., [0, 4]])
    p = np.abs(rng.standard_normal((2, n))) * e(2, n)
    g = np.full((2, n), 5.0 / 3.0)
    bn = rng.standard_normal(n) * e(n)
    for a in (W[..., 0], p, g, bn):
        at = rng.random(a.shape) < share
        a[at] = rng.choice([0.0, -1.0], at.sum())
    # where gamma is next to nothing the contact can outrun the far wave, behind
    # which the double-star state then has no density
    k = n // 4
    b = np.abs(bn[:k]) + 0.1
    bn[:k] = b
    W[:, :k, 0] = 1.0
    W[:, :k, 1] = 0.5 * b
    W[:, :k, 7:] = 0.0
    p[0, :k] = b * b
    p[1, :k] = b * b * rng.uniform(4.0, 7.0, k)
    g[:, :k] = 1e-9
    W[..., 6] = bn
    return W, p, g, bn


@pytest.mark.parametrize("spread,share", [(1, 0.0), (6, 0.0), (3, 0.1)])
def test_against_oracle(builds, spread, share):
    n = 4000
    W, p, g, bn = faces(n, 21, spread, share)
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)
    got = []
    for lib in builds:
        out, st = np.zeros((n, 14)), np.zeros(n, dtype=np.int32)
        lib.fx_test_hlld(n, *map(ptr, (W, p, g, bn, out, st)))
        got.append((out, st))
    assert np.array_equal(got[0][1], got[1][1])
    o = [np.zeros(9), np.zeros(3), np.zeros(1), np.zeros(1)]
    dp = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    code = np.zeros(n, dtype=np.int32)
    want = np.zeros((n, 14))
    for i in range(n):
        code[i] = O.oracle_lib().fxo_hlld(dp(W[0, i]), dp(W[1, i]), p[0, i], p[1, i], g[0, i],
                                          g[1, i], bn[i], *map(dp, o))
        want[i] = np.concatenate(o)
    ok = code == 0
    assert np.array_equal(got[0][1] == 0, ok)
    assert np.array_equal(got[0][0][ok], want[ok])
    star = np.isin(got[0][1], (18, 19))
    assert star.sum() > 20 and ok.sum() > n // 3
    assert got[0][0].tobytes() == got[1][0].tobytes()
