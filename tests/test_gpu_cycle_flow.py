"""The small grids' cycle in one launch of many waves (cycle_flow.hip, what a hierarchy runs until its coarse mode
is set) against the per-grid kernels (mode 0): the same bits without the scaled correction, in every precision,
whether the launch starts at grid 0 or below it, with rows wider than a batch of entries, agglomerates of more
than four cells, several sweeps either way, and a coarsest grid of several chunks. With the scaled correction its
sums are taken in another order: a whole solve takes the same iterations within one and reaches the tolerance."""
import numpy as np
import pytest

import gpu_util as G
from brae_amd import mfv
from test_gpu_amg import channel_system
from test_gpu_sweep_plans import graph

pytestmark = pytest.mark.gpu

PRECS = [mfv.PREC_FP64, mfv.PREC_FP32, mfv.PREC_FP16]


class Made:
    """a symmetric system on given faces, its off-diagonals the face weights"""

    def __init__(self, label, n, own, nei, bfc, seed):
        rng = np.random.default_rng(seed)
        self.label, self.nC, self.own, self.nei = label, n, own, nei
        self.w = rng.uniform(0.5, 2.0, own.size)
        diag = rng.uniform(0.05, 0.2, n)
        np.add.at(diag, own, self.w)
        np.add.at(diag, nei, self.w)
        self.diag, self.upper, self.b = diag, -self.w, rng.normal(size=n)
        self.case = G.Case(n, own, nei, bfc)
        self.dd, self.du, self.db = G.dev(diag), G.dev(self.upper), G.dev(self.b)
        self.magSf = self.w


def systems(name):
    if name == "wide rows":
        return Made(name, *graph(9000, 14, 11, 700), 1)
    shape = {"small": (9, 7, 5), "from grid 0": (22, 20, 18), "at the line": (32, 16, 16), "below grid 0": (29, 17, 19)}[name]
    return channel_system(*shape, seed=13)


@pytest.mark.parametrize("prec", PRECS, ids=["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("name,target,merge", [("small", 64, 1), ("from grid 0", 64, 1), ("at the line", 200, 2),
                                               ("below grid 0", 64, 3), ("wide rows", 300, 1), ("wide rows", 20, 2)])
def test_same_bits_as_the_per_grid_kernels(name, target, merge, prec):
    S = systems(name)
    one, per = (mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, target, mergeLevels=merge) for _ in range(2))
    print("case:", name, S.nC, "precision", prec, [one.grid_size(g) for g in range(one.nGrids)], flush=True)
    per.coarse_mode(0)
    for a in (one, per):
        a.galerkin(S.dd, S.du, prec)
    r = G.dev(np.random.default_rng(21).normal(size=S.nC))
    for sweeps in [(1, 1), (2, 1), (0, 1), (1, 2), (1, 0), (4, 3)]:
        out = []
        for a in (one, per, one):
            z = G.zeros(S.nC)
            a.vcycle(r, z, *sweeps)
            S.case.sync()
            out.append(G.host(z))
        assert np.isfinite(out[1]).all() and np.abs(out[1]).max() > 0
        assert np.array_equal(out[0], out[1]), (name, sweeps, np.abs(out[0] - out[1]).max())
        assert np.array_equal(out[2], out[1]), (name, sweeps)
    one.close()
    per.close()


@pytest.mark.parametrize("prec", PRECS, ids=["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("name", ["from grid 0", "below grid 0", "wide rows"])
def test_scaled_solve(name, prec):
    S = systems(name)
    got = []
    for mode in (None, 0):
        amg = mfv.Amg(S.case.mesh, S.magSf, mfv.AGG_BRAE, 64)
        if mode is not None:
            amg.coarse_mode(mode)
        amg.galerkin(S.dd, S.du, prec)
        psi = G.zeros(S.nC)
        p = amg.solve(S.dd, S.du, S.db, psi, tolerance=1e-9, precision=prec, flexible=1, nPreSweeps=2, nPostSweeps=1,
                      scaleCorrection=1, captureVcycle=int(mode is None))
        print("case:", name, prec, "mode", mode, p.nIterations, p.finalResidual, flush=True)
        assert p.finalResidual < 1e-9
        got.append((G.host(psi), p.nIterations))
        amg.close()
    assert abs(got[0][1] - got[1][1]) <= 1
    # both solutions are within the tolerance of the system's: their difference is of its order
    assert np.abs(got[0][0] - got[1][0]).max() <= 1e-6 * np.abs(got[1][0]).max()
