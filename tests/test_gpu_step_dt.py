"""On meshes with few recorded CFL maxima stage 1 forms the step's dt itself: the
dts and states of runs, with and without the maxima recorded and with the
growth limit at work, against the oracle, around the largest count that does so and
between calls that set or read dt by other means."""
import numpy as np
import pytest

import pyoracle as O
from fornaxamr_amd import problems as P

pytestmark = pytest.mark.gpu


def pair(n, mhd, riemann="hllc"):
    from fornaxamr_amd.mesh import GpuMesh
    pr = P.random_smooth(n=n, seed=sum(n), bc=(0,) * 6, mhd=mhd)
    gm = GpuMesh.from_problem(pr)
    om = O.OracleSim(pr.n, pr.xlim, pr.bc, pr.gamma, mhd=mhd, log_cr=True, riemann=riemann)
    om.set_state(pr.W, pr.bf) if mhd else om.set_state(pr.W)
    if riemann != "hllc":
        gm.set_riemann(riemann)
    return pr, gm, om


@pytest.mark.parametrize("n,mhd,riemann", [
    ((16, 16, 16), False, "hllc"),
    ((32, 48, 16), False, "hlle"),
    ((112, 48, 80), False, "hllc"),
    ((64, 256, 256), False, "hllc"),     # 1024 blocks
    ((80, 208, 256), False, "hllc"),     # 1040 blocks: a launch of its own
    ((32, 32, 32), True, "hllc"),
    ((64, 64, 64), True, "hllc"),        # 1024 CT parts
])
def test_dts_and_states(gpu, n, mhd, riemann):
    pr, gm, om = pair(n, mhd, riemann)
    big = np.prod(n) > 10**6
    for s in range(2 if big else 4):
        factor = 1.0001 if s > 1 else 1.2       # the limit binds or not
        assert gm.step(pr.cfl, factor) == om.step(pr.cfl, factor), s
    assert np.array_equal(gm.get_prim(0), om.W0)
    if mhd:
        for a, b in zip(gm.get_bf(0), om.bf0):
            assert np.array_equal(a, b)
    gm.close()


@pytest.mark.parametrize("mhd", [False, True], ids=["hydro", "mhd"])
def test_mixed_with_other_calls(gpu, mhd):
    pr, gm, om = pair((32, 48, 32), mhd)
    for s in range(6):
        if s == 2:
            gm.view()                       # drops the recorded maxima
        if s == 4:
            assert gm.calc_dt(pr.cfl) == om.calc_dt(pr.cfl)
        if s == 3:                          # a dt formed on the host
            dt = 0.5 * om.calc_dt(pr.cfl)
            gm.step_dt(dt)
            om.dt = dt
            om.stage(1, dt)
            om.stage(2, dt)
        else:
            assert gm.step(pr.cfl, 1.05) == om.step(pr.cfl, 1.05), s
        assert np.array_equal(gm.get_prim(0), om.W0), s
    gm.close()
