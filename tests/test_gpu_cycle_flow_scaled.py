"""The small grids' launch with the scaled correction, cycle by cycle, against the per-grid kernels; and hierarchies
whose precision changes between captured solves.

The two ways differ in the order of the scaling's two FP64 sums alone. Summed in another order, n terms move a sum by
at most n eps of the sum of their magnitudes, and the cycle is linear in the factor; over the grids and the few
conditions of these sums that stays below 64 n eps in the 2-norm. The factor is rounded to FP32 in the FP32 and FP16
cycles, so there the cycle mostly has the same bits; where the rounding falls the other way once, values move by an
ulp of the stored precision, 2^-23 or 2^-11 of their size."""
import numpy as np
import pytest

import gpu_util as G
from brae_amd import mfv
from test_gpu_amg import channel_system
from test_gpu_cycle_flow import PRECS, systems

pytestmark = pytest.mark.gpu

SWEEPS = [(1, 1), (2, 1), (0, 1), (1, 0), (1, 2), (4, 3)]


@pytest.mark.parametrize("prec", PRECS, ids=["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("name,target,merge", [("small", 64, 1), ("from grid 0", 64, 1), ("at the line", 200, 2),
                                               ("below grid 0", 64, 3), ("wide rows", 300, 1), ("wide rows", 20, 2)])
def test_scaled_cycle(name, target, merge, prec):
    S = systems(name)
    amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, target, mergeLevels=merge)
    amg.galerkin(S.dd, S.du, prec)
    assert amg.coarse_default(restore=False)[1] >= 0
    r = G.dev(np.random.default_rng(22).normal(size=S.nC))
    bound = {mfv.PREC_FP64: 64 * S.nC * np.finfo(float).eps, mfv.PREC_FP32: 2.0 ** -21, mfv.PREC_FP16: 2.0 ** -10}[prec]
    for sweeps in SWEEPS:
        got = []
        for one in (True, False, True):
            if one:
                amg.coarse_default()
            else:
                amg.coarse_mode(0)
            z = G.zeros(S.nC)
            amg.vcycle(r, z, *sweeps, True)
            S.case.sync()
            got.append(G.host(z))
        off = np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])
        print("case: scaled", name, S.nC, "precision", prec, sweeps, "off by", off, "bound", bound, flush=True)
        assert np.isfinite(got[1]).all() and off <= bound
        assert np.array_equal(got[2], got[0])
        unscaled = G.zeros(S.nC)
        amg.coarse_mode(0)
        amg.vcycle(r, unscaled, *sweeps, False)
        S.case.sync()
        # the scaling does something: a factor left out would lie outside the bound (the least here, wide rows in
        # FP16, moves the cycle by 1.6e-2, 16 times the bound; a quarter of that is asked for)
        assert np.linalg.norm(G.host(unscaled) - got[1]) > 4 * bound * np.linalg.norm(got[1])
    amg.close()


@pytest.mark.parametrize("scale", [0, 1])
@pytest.mark.parametrize("name", ["from grid 0", "below grid 0"])
def test_precision_changes_between_captured_solves(name, scale):
    """the launch's words are laid out anew with each precision; a captured cycle must follow them"""
    S = systems(name)

    def solve(amg, prec):
        amg.galerkin(S.dd, S.du, prec)
        psi = G.zeros(S.nC)
        p = amg.solve(S.dd, S.du, S.db, psi, tolerance=1e-9, precision=prec, flexible=1, nPreSweeps=2, nPostSweeps=1,
                      scaleCorrection=scale, captureVcycle=1)
        return G.host(psi), p.nIterations, p.finalResidual

    fresh = {}
    for prec in PRECS:
        amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, 64)
        fresh[prec] = solve(amg, prec)
        amg.close()
    amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, 64)
    F64, F32, F16 = mfv.PREC_FP64, mfv.PREC_FP32, mfv.PREC_FP16
    for prec in [F64, F16, F64, F64, F32, F16, F32, F64]:
        got = solve(amg, prec)
        print("case: precision", prec, name, got[1:], flush=True)
        assert got[1:] == fresh[prec][1:] and np.array_equal(got[0], fresh[prec][0]), prec
    amg.close()
