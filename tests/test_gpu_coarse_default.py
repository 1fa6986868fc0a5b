"""mfv_amg_coarse_default: the default way of running the coarsest grids can be asked for and returned to after a
mode was set, on one hierarchy, in every precision; the scaled cycle, whose sums the default takes in its own order,
has the same bits before and after."""
import numpy as np
import pytest

import gpu_util as G
from brae_amd import mfv
from test_gpu_amg import channel_system

pytestmark = pytest.mark.gpu


def cycle(S, amg, scale):
    z = G.zeros(S.nC)
    amg.vcycle(S.db, z, 2, 1, scale)
    S.case.sync()
    return G.host(z)


@pytest.mark.parametrize("prec", [mfv.PREC_FP64, mfv.PREC_FP32, mfv.PREC_FP16], ids=["fp64", "fp32", "fp16"])
def test_back_to_the_default(prec):
    S = channel_system(29, 17, 19, seed=4)
    amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, 64)
    amg.galerkin(S.dd, S.du, prec)
    used, first = amg.coarse_default(restore=False)
    print("case: precision", prec, "first grid", first, [amg.grid_size(g)[0] for g in range(amg.nGrids)], flush=True)
    assert used and first >= 1
    assert amg.grid_size(first)[0] <= 8192 < amg.grid_size(first - 1)[0]
    plain, scaled = cycle(S, amg, 0), cycle(S, amg, 1)
    for mode in (0, 1, 2):
        amg.coarse_mode(mode)
        assert amg.coarse_default(restore=False) == (False, first)
        assert np.array_equal(cycle(S, amg, 0), plain)
        cycle(S, amg, 1)
        assert amg.coarse_default() == (True, first)
        assert np.array_equal(cycle(S, amg, 0), plain) and np.array_equal(cycle(S, amg, 1), scaled)
    amg.close()


def test_no_grid_for_it():
    """a hierarchy whose only small grid is its coarsest: nothing for the launch to run"""
    S = channel_system(22, 20, 20, seed=4)
    amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, 900, mergeLevels=4)
    amg.galerkin(S.dd, S.du, mfv.PREC_FP64)
    print("case:", [amg.grid_size(g)[0] for g in range(amg.nGrids)], flush=True)
    assert amg.nGrids == 2 and amg.coarse_default() == (True, -1)
    one = cycle(S, amg, 0)
    amg.coarse_mode(0)
    assert np.array_equal(cycle(S, amg, 0), one)
    amg.close()
