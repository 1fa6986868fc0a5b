"""GAMG's correction scaling with its sums finished by the update (up to 256 partials, 131,072 cells) and by launches
of their own (above) against the context's sequential sums: the same cycles and residual to the sums' rounding."""
import numpy as np
import pytest

import gpu_util as G
from brae_amd import mfv
from test_gpu_amg import channel_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(12, 9, 5), (64, 64, 32), (64, 64, 33)])
def test_scaled_cycles(shape):
    S = channel_system(*shape, seed=2)
    got = []
    for seq in (False, True):
        S.case.ctx.sequential_reduce(seq)
        amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, 10)
        psi = G.zeros(S.nC)
        p = amg.gamg_solve(S.dd, S.du, S.db, psi, tolerance=1e-14, minIter=3, maxIter=3)
        print("case:", shape, "sequential", seq, p.nIterations, p.finalResidual, flush=True)
        got.append((G.host(psi), p.finalResidual))
        amg.close()
    S.case.ctx.sequential_reduce(False)
    # two orders of summing n values differ by at most n eps of their magnitudes; three contracting cycles,
    # and a coarsest solve to 1e-14
    bound = 64 * S.nC * np.finfo(float).eps
    assert np.abs(got[0][0] - got[1][0]).max() <= bound * np.abs(got[1][0]).max()
    assert abs(got[0][1] - got[1][1]) <= bound * max(got[1][1], 1.0)
