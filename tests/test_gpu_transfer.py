"""Host transfers of a mesh's state through the library's staging buffer: what
was set comes back from both slots, to the bit, in one chunk and in several (the
buffer holds 64 MiB), with the padding around it left as it was."""
import numpy as np
import pytest

from fornaxamr_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,mhd", [((16, 16, 16), False), ((16, 48, 32), True),
                                   ((112, 128, 144), False), ((160, 96, 80), True)])
def test_round_trip(gpu, n, mhd):
    from fornaxamr_amd.mesh import GpuMesh
    rng = np.random.default_rng(sum(n))
    m = GpuMesh(n, (0.0, 1.0) * 3, (P.OUTFLOW,) * 6, 1.4, mhd=mhd)
    W = rng.standard_normal((9 if mhd else 6,) + n)
    bf = None
    if mhd:
        bf = [rng.standard_normal([e + (a == d) for a, e in enumerate(n)]) for d in range(3)]
        # cell B is the mean of the faces whatever W holds
        W[6] = 0.5 * (bf[0][:-1] + bf[0][1:])
        W[7] = 0.5 * (bf[1][:, :-1] + bf[1][:, 1:])
        W[8] = 0.5 * (bf[2][:, :, :-1] + bf[2][:, :, 1:])
    m.set_state(W, bf)
    for slot in range(2):
        assert np.array_equal(m.get_prim(slot), W)
        if mhd:
            for a, b in zip(m.get_bf(slot), bf):
                assert np.array_equal(a, b)
    m.close()
