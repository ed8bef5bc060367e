"""Stages whose blocks are split over several workgroups along x, against the
oracle.  The mesh sizes are those at which the rules of a 256-CU GPU take each
number of parts (the edges of the parts fall inside blocks, so a wrong plane at
a part's edge shows in the cells); bit-identical states and dts, as for whole
blocks."""
import ctypes as C

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


def _blocks_call(lib, mhd, uniq, n):
    """fx_flux_update_blocks over n device blocks, copies of the given ones in
    turn; the outputs as tensors [direction][block]."""
    import torch
    from fornaxamr_amd import _native
    nh = 9 if mhd else 6
    shapes = {"flux": nh * O.RB_CELLS, "v_riemann": 3 * O.RB_CELLS}
    if mhd:
        shapes.update(Bv1=O.RB_CELLS, Bv2=O.RB_CELLS)
    out = {k: torch.full((3, n, m), float("nan"), dtype=torch.float64, device="cuda")
           for k, m in shapes.items()}
    ins = [[torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (slab, eos, *(bf or []))]
           for slab, eos, bf in uniq]
    io = (_native.BlockIO * n)()
    for b in range(n):
        own = ins[b % len(ins)]
        io[b].W, io[b].eosvar, io[b].var_stride = own[0].data_ptr(), own[1].data_ptr(), 2 * O.RB_CELLS
        for d in range(3):
            for k in shapes:
                getattr(io[b], k)[d] = out[k][d, b].data_ptr()
            if mhd:
                io[b].bf[d] = own[2 + d].data_ptr()
    raw = torch.frombuffer(bytearray(bytes(io)), dtype=torch.uint8).cuda()
    status = torch.zeros(8, dtype=torch.int32, device="cuda")
    _native.check(lib.fx_flux_update_blocks(n, C.c_void_p(raw.data_ptr()), mhd,
                                            C.c_void_p(status.data_ptr()),
                                            C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert status.tolist() == [0] * 8
    return out


@pytest.mark.parametrize("mhd", [0, 1], ids=["hydro", "mhd"])
def test_block_parts(gpu, mhd):
    """Per-block fluxes of 1 to 600 blocks in a launch (16 parts down to whole
    blocks) are those of the first call, whose single blocks the reference's
    digests pin."""
    import torch
    uniq = []
    for seed in (11, 12, 13):
        slab, gam, bf = O.block_inputs(seed, bool(mhd))
        uniq.append((slab, O.block_eosvar(slab, 0, gam), bf))
    want = _blocks_call(gpu, mhd, uniq, 3)
    for n in (1, 65, 125, 216, 343, 512, 600):
        got = _blocks_call(gpu, mhd, uniq, n)
        for k in want:
            for b in range(3):
                ref = want[k][:, b].view(torch.int64)
                assert all(torch.equal(got[k][:, c].view(torch.int64), ref)
                           for c in range(b, n, 3)), (n, k, b)
