"""Stages whose blocks are split over several workgroups along x, against the
oracle.  The mesh sizes are those at which the rules of a 256-CU GPU take each
number of parts (the edges of the parts fall inside blocks, so a wrong plane at
a part's edge shows in the cells); bit-identical states and dts, as for whole
blocks."""
import numpy as np
import pytest

import pyoracle as O
from fornaxamr_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bc,riemann", [
    ((32, 32, 32), (3,) * 6, "hllc"),               # 16 parts
    ((64, 64, 64), (3, 3, 0, 1, 1, 0), "hllc"),     # 8
    ((48, 112, 80), (1, 0, 3, 3, 1, 1), "hllc"),    # 4, blocks not a multiple of 8
    ((96, 96, 96), (0,) * 6, "hlle"),               # 2
    ((112, 112, 112), (3,) * 6, "hllc"),            # 4, three rounds of workgroups
    ((128, 128, 128), (3,) * 6, "hllc"),            # whole blocks
])
def test_hydro_parts(gpu, n, bc, riemann):
    from fornaxamr_amd.mesh import GpuMesh
    pr = P.random_smooth(n=n, seed=sum(n), bc=bc, gamma=1.4)
    gm = GpuMesh.from_problem(pr)
    om = O.OracleSim(pr.n, pr.xlim, pr.bc, pr.gamma, riemann=riemann)
    om.set_state(pr.W)
    gm.set_riemann(riemann)
    for _ in range(2):   # the second dt comes from the first step's recorded maxima
        assert gm.step(pr.cfl) == om.step(pr.cfl)
        assert np.array_equal(gm.get_prim(0), om.W0)
    gm.close()


@pytest.mark.parametrize("edges", [(32,), (32, 48, 64, 48), (96, 64, 48, 32, 96)])
@pytest.mark.parametrize("schedule", [(0, 0, 1, 0), (1, 0, 1, 0), (1, 64, 1, 1)])
def test_ensemble_parts(gpu, edges, schedule):
    """8, 126 and 531 blocks: 16, 4 and 4 parts in the batched launches."""
    from fornaxamr_amd.ensemble import GpuEnsemble
    probs = [P.random_smooth(n=(e,) * 3, seed=e + i, bc=(3,) * 6, gamma=1.3 + 0.1 * i)
             for i, e in enumerate(edges)]
    e = GpuEnsemble(probs)
    e.set_schedule(*schedule)
    for _ in range(2):
        e.step_async(0.4)
    e.sync()
    dts = e.last_dt()
    for i, pr in enumerate(probs):
        om = O.OracleSim(pr.n, pr.xlim, pr.bc, pr.gamma)
        om.set_state(pr.W)
        om.step(0.4)
        assert om.step(0.4) == dts[i]
        assert np.array_equal(e.get_prim(i), om.W0)
    e.close()


@pytest.mark.parametrize("n,eta", [
    ((32, 32, 16), 0.0),        # flux 16 parts, CT 16
    ((64, 48, 80), 1.0e-3),     # 8, 16; blocks not a multiple of 8
    ((96, 64, 80), 0.0),        # 4, 8
    ((96, 96, 96), 0.0),        # 2, 4
    ((112, 96, 112), 1.0e-3),   # 4, 2
])
def test_mhd_parts(gpu, n, eta):
    from fornaxamr_amd.mesh import GpuMesh
    pr = P.random_smooth(n=n, seed=sum(n), bc=(0,) * 6, mhd=True, eta=eta)
    gm = GpuMesh.from_problem(pr)
    om = O.OracleSim(pr.n, pr.xlim, pr.bc, pr.gamma, mhd=True, eta=eta, log_cr=True)
    om.set_state(pr.W, pr.bf)
    for _ in range(2):
        assert gm.step(pr.cfl) == om.step(pr.cfl)
        assert np.array_equal(gm.get_prim(0), om.W0)
        for a, b in zip(gm.get_bf(0), om.bf0):
            assert np.array_equal(a, b)
    gm.close()
