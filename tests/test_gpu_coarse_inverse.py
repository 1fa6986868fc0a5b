"""The dense inverse of the coarsest grid, staged in LDS up to 96 cells and from device memory above, against the
oracle's, to the bit: the smallest, both sides of the line, and a second set-up on the same hierarchy."""
import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from brae_amd import mfv
from test_gpu_amg import channel_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("target", [2, 64, 96, 97, 180])
def test_coarsest_inverse(target):
    S = channel_system(17, 13, 11, seed=3)
    ag = O.brae_agglomeration(S.nC, S.own, S.nei, S.magSf, target=target)
    amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, target)
    n = amg.grid_size(amg.nGrids - 1)[0]
    print("case: coarsest", n, flush=True)
    for a in range(2):
        amg.galerkin(S.dd, S.du, mfv.PREC_FP64)
        r = np.random.default_rng(4).normal(size=S.nC)
        z = G.zeros(S.nC)
        amg.vcycle(G.dev(r), z, 1, 1)
        S.case.sync()
        assert np.array_equal(G.host(z), O.brae_vcycle(ag, S.diag, S.upper, r, 1, 1, single=False))
    amg.close()
