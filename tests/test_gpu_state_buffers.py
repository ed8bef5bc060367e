"""Where a mesh's state lies in its device buffers, seen through the view's strides
rather than through the transfers themselves: a transfer writes the active cells and
faces of both slots and nothing else, and eSSPRK(10,4) leaves its result in slot 0 and
substep 9 in slot 1, faces included."""
import numpy as np
import pytest

import pyoracle as O
from fornaxamr_amd import problems as P

pytestmark = pytest.mark.gpu
MARK = -77.5


class Array:
    """A device array of the library, for torch."""
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "version": 3,
                                         "data": (ptr, False), "strides": None}


def buffers(m):
    """torch views of both slots' cells and faces, [variable][padded entry]."""
    import torch
    v = m.view()
    at = lambda p, k: torch.as_tensor(Array(p, (k, v.vstride)), device="cuda")
    return [at(p, v.nh) for p in v.W], [at(p, 3) for p in v.bf[:2]] if m.mhd else []


def entries(v, n):
    x, y, z = np.ogrid[:n[0], :n[1], :n[2]]
    return (v.origin + x * v.sx + y * v.sy + z).astype(np.int64)


# 16^3 rows in one chunk; more than the 64 MiB of the staging buffer in several
@pytest.mark.parametrize("n,mhd", [((16, 16, 16), False), ((16, 48, 32), True),
                                   ((112, 128, 144), False), ((160, 96, 80), True)])
def test_transfers_write_active_entries_only(gpu, n, mhd):
    import torch
    from fornaxamr_amd.mesh import GpuMesh
    rng = np.random.default_rng(sum(n))
    m = GpuMesh(n, (0.0, 1.0) * 3, (P.OUTFLOW,) * 6, 1.4, mhd=mhd)
    cells, faces = buffers(m)
    for a in cells + faces:
        a.fill_(MARK)
    torch.cuda.synchronize()
    W = rng.standard_normal((m.nh,) + n)
    bf = [rng.standard_normal([e + (a == d) for a, e in enumerate(n)]) for d in range(3)]
    if mhd:
        for d in range(3):      # cell B is the mean of the faces whatever W holds
            k = n[d]
            W[6 + d] = 0.5 * (bf[d].take(range(k), d) + bf[d].take(range(1, k + 1), d))
    m.set_state(W, bf)
    v = m.view()
    want = np.full((m.nh, v.vstride), MARK)
    want[:, entries(v, n)] = W
    wantb = np.full((3, v.vstride), MARK)
    if mhd:
        for d in range(3):
            wantb[d][entries(v, bf[d].shape)] = bf[d]
    for read in (False, True):
        if read:
            for slot in range(2):
                assert np.array_equal(m.get_prim(slot), W)
                if mhd:
                    assert all(np.array_equal(a, b) for a, b in zip(m.get_bf(slot), bf))
        for a in cells:
            assert np.array_equal(a.cpu().numpy(), want), read
        for a in faces:
            assert np.array_equal(a.cpu().numpy(), wantb), read
    m.close()


@pytest.mark.parametrize("mhd", [False, True], ids=["hydro", "mhd"])
def test_essprk_leaves_substep_9_in_slot_1(gpu, mhd):
    from fornaxamr_amd.mesh import GpuMesh
    pr = P.random_smooth(n=(32, 48, 32), seed=83, bc=(0 if mhd else 3,) * 6, mhd=mhd)
    gm = GpuMesh.from_problem(pr)
    om = O.OracleSim(pr.n, pr.xlim, pr.bc, pr.gamma, mhd=mhd, log_cr=True)
    om.set_state(pr.W, pr.bf) if mhd else om.set_state(pr.W)
    substeps = []
    stage = om.stage

    def record(s, dt):
        stage(s, dt)
        substeps.append((om.W1.copy(), [b.copy() for b in om.bf1] if mhd else []))
    om.stage = record
    gm.set_integrator("essprk10_4")
    for s in range(2):
        del substeps[:]
        assert gm.step(pr.cfl) == om.step_essprk10_4(pr.cfl), s
        for slot, (W, bf) in enumerate([(om.W0, om.bf0 if mhd else []), substeps[8]]):
            assert np.array_equal(gm.get_prim(slot), W), (s, slot)
            if mhd:
                for a, b in zip(gm.get_bf(slot), bf):
                    assert np.array_equal(a, b), (s, slot)
    gm.close()
