"""The library's host code over a stand-in for the HIP runtime (hip_host.cpp), on
machines without a GPU: in what order a mesh's buffers are cleared.  The scripts
run in a process of their own, where the stand-in is loaded before the library."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

HEAD = """
import ctypes as C, sys
host = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
host.host_pending.argtypes = [C.c_void_p]
host.host_malloc_limit.argtypes = [C.c_size_t]
calls = lambda name: host.host_calls(name.encode())
import numpy as np
from fornaxamr_amd import _native, problems as P
from fornaxamr_amd.mesh import GpuMesh
"""


@pytest.fixture(scope="module")
def host_run(tmp_path_factory):
    from fornaxamr_amd import build
    cxx = shutil.which("g++")
    if cxx is None or not os.path.exists(build.LIB):
        pytest.skip("needs g++ and the built library")
    lib = str(tmp_path_factory.mktemp("hip_host") / "libhip_host.so")
    subprocess.run([cxx, "-O1", "-std=c++17", "-fPIC", "-shared", os.path.join(HERE, "hip_host.cpp"),
                    "-o", lib], check=True)

    def run(script):
        r = subprocess.run([sys.executable, "-c", HEAD + script, lib], cwd=os.path.dirname(HERE),
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


@pytest.mark.parametrize("mhd", [False, True], ids=["hydro", "mhd"])
def test_integrator_clears_in_stream_order(host_run, mhd):
    """Choosing eSSPRK(10,4) leaves no clear of its two further states running (one
    of the null stream would run beside the next step on a non-blocking stream),
    and clears them only when it allocates them."""
    host_run(f"""
m = GpuMesh((32, 32, 32), (0.0, 1.0) * 3, (0,) * 6, 1.4, mhd={mhd})
host.hipDeviceSynchronize()
_native.check(m.lib.fx_mesh_set_stream(m.h, 0x40))
m.set_integrator("essprk10_4")
assert host.host_pending(None) == 0 and host.host_pending(0x40) == 0
fills = calls("hipMemset") + calls("hipMemsetAsync")
m.set_integrator("rk2")
m.set_integrator("essprk10_4")
assert calls("hipMemset") + calls("hipMemsetAsync") == fills
m.close()
""")


def test_created_state_is_clear(host_run):
    """A new mesh or ensemble leaves no clear running that a stream given to it
    afterwards (or the ensemble's own) would not wait for."""
    host_run("""
from fornaxamr_amd.ensemble import GpuEnsemble
for mhd in (False, True):
    m = GpuMesh((32, 32, 32), (0.0, 1.0) * 3, (0,) * 6, 1.4, mhd=mhd)
    assert host.host_pending(None) == 0, mhd
    v = m.view()
    for p in v.W:
        a = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (v.nh * v.vstride,))
        assert not a.any()
    m.close()
host.hipDeviceSynchronize()
h = C.c_void_p()
d = (_native.MeshDesc * 2)()
for i in range(2):
    d[i].n[:] = [16 * (i + 1)] * 3
    d[i].xlim[:] = [0.0, 1.0] * 3
    d[i].gamma = 1.4
lib = _native.load()
_native.check(lib.fx_ensemble_create(2, d, C.byref(h)))
assert host.host_pending(None) == 0
lib.fx_ensemble_destroy(h)
""")


def test_ensemble_out_of_memory(host_run):
    """An ensemble whose states do not all fit is refused with FX_ENOMEM, whichever
    allocation fails."""
    host_run("""
lib = _native.load()
h = C.c_void_p()
n = 40
d = (_native.MeshDesc * n)()
for i in range(n):
    d[i].n[:] = [16 * (i % 3 + 1)] * 3
    d[i].xlim[:] = [0.0, 1.0] * 3
    d[i].gamma = 1.4
for limit in (0, 500, 2000, 10000, 1000000, 2000000):
    host.host_malloc_limit(limit)
    assert lib.fx_ensemble_create(n, d, C.byref(h)) == -4, limit
    assert h.value is None
host.host_malloc_limit(1 << 40)
assert lib.fx_ensemble_create(n, d, C.byref(h)) == 0
lib.fx_ensemble_destroy(h)
""")


def test_transfers_where_staging_memory_is_short(host_run):
    """A transfer that cannot have a larger staging buffer goes through the one
    there is, in more chunks; where there is none, by 2D copies, which leave the
    padding alone and bring the state back to the bit."""
    host_run("""
lib = _native.load()
dp = C.POINTER(C.c_double)
# 2D copies: no staging at all
rng = np.random.default_rng(5)
for mhd in (False, True):
    n = (32, 16, 48)
    m = GpuMesh(n, (0.0, 1.0) * 3, (0,) * 6, 1.4, mhd=mhd)
    host.host_malloc_limit(0)
    W = rng.standard_normal((m.nh,) + n)
    bf = [rng.standard_normal([e + (a == d) for a, e in enumerate(n)]) for d in range(3)]
    m.set_state(W, bf)
    assert calls("hipMemcpy2DAsync") > 0
    v = m.view()
    for s in range(2):
        assert np.array_equal(m.get_prim(s), W)
        if mhd:
            assert all(np.array_equal(a, b) for a, b in zip(m.get_bf(s), bf))
        flat = np.ctypeslib.as_array(C.cast(v.W[s], dp), (m.nh, v.vstride)).copy()
        i = (v.origin + np.arange(n[0])[:, None, None] * v.sx + np.arange(n[1])[:, None] * v.sy
             + np.arange(n[2]))
        assert np.array_equal(flat[:, i], W)
        flat[:, i] = 0.0
        assert not flat.any()
    host.host_malloc_limit(1 << 40)
    m.close()
# a buffer that serves a small instance also serves a large one
d = (_native.MeshDesc * 2)()
for i in range(2):
    d[i].n[:] = [16 + 48 * i] * 3
    d[i].xlim[:] = [0.0, 1.0] * 3
    d[i].gamma = 1.4
h = C.c_void_p()
_native.check(lib.fx_ensemble_create(2, d, C.byref(h)))
W = [rng.standard_normal((6,) + (16 + 48 * i,) * 3) for i in range(2)]
ptr = lambda a: a.ctypes.data_as(dp)
_native.check(lib.fx_ensemble_set_prim(h, 0, ptr(W[0])))
before = calls("hipMemcpy2DAsync"), calls("hipFree")
host.host_malloc_limit(1 << 20)
moved = calls("hipMemcpyAsync")
_native.check(lib.fx_ensemble_set_prim(h, 1, ptr(W[1])))
assert calls("hipMemcpyAsync") - moved == 1 + 64      # the time's reset, and 12.6 MB by 197 kB
_native.check(lib.fx_ensemble_get_prim(h, 1, 0, ptr(W[1])))
_native.check(lib.fx_ensemble_set_prim(h, 0, ptr(W[0])))
assert (calls("hipMemcpy2DAsync"), calls("hipFree")) == before
host.host_malloc_limit(1 << 40)
_native.check(lib.fx_ensemble_set_prim(h, 1, ptr(W[1])))
assert calls("hipFree") == before[1] + 1              # replaced by the larger one
lib.fx_ensemble_destroy(h)
""")
