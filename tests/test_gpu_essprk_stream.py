"""eSSPRK(10,4) on a caller's non-blocking stream, the integrator chosen again
between steps that are still running: cells, faces and dt stay the oracle's, so
no clear of the further states meets a step."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as O
from fornaxamr_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mhd", [False, True], ids=["hydro", "mhd"])
def test_steps_on_a_callers_stream(gpu, mhd):
    import torch
    from fornaxamr_amd.mesh import GpuMesh
    pr = P.random_smooth(n=(48, 32, 32), seed=82, bc=(0 if mhd else 3,) * 6, mhd=mhd)
    stream = torch.cuda.Stream()
    gm = GpuMesh.from_problem(pr, stream=stream.cuda_stream)
    om = O.OracleSim(pr.n, pr.xlim, pr.bc, pr.gamma, mhd=mhd, log_cr=True)
    om.set_state(pr.W, pr.bf) if mhd else om.set_state(pr.W)
    got = C.c_double()
    for s in range(3):
        gm.set_integrator("essprk10_4")
        gm.step_async(pr.cfl)
        gm.set_integrator("essprk10_4")
        dt = om.step_essprk10_4(pr.cfl)
        gm.sync()
        assert gpu.fx_last_dt(gm.h, C.byref(got)) == 0 and got.value == dt, s
        assert np.array_equal(gm.get_prim(0), om.W0), s
        if mhd:
            for a, b in zip(gm.get_bf(0), om.bf0):
                assert np.array_equal(a, b), s
    gm.close()
