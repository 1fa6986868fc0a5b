"""Successive Gauss-Seidel sweeps that follow each other through one workgroup (sweep.hip) against the oracle's host
loop, to the bit: numbers of sweeps that leave the last pass full, with one and with several teams, on meshes
whose teams are many, two (levels of 132 cells) or one, whose neighbours lie one level or many apart, and whose
levels take several steps."""
import ctypes

import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from brae_amd import mfv
from test_gpu_sweep_plans import system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nSweeps", [1, 2, 4, 5, 9, 16])
@pytest.mark.parametrize("name", ["two cells", "chain in LDS", "ragged box", "wide levels", "wide rows in LDS",
                                  "one wide level", "star"])
def test_overlapped_sweeps(name, nSweeps):
    n, own, nei, bfc, diag, up, lo, b, x0 = system(name)
    print("case:", name, n, "cells", nSweeps, "sweeps", flush=True)
    case = G.Case(n, own, nei, bfc)
    A, dx = mfv.ldu(G.dev(diag), G.dev(up)), G.dev(x0)
    case.call("mfv_gauss_seidel", case.mesh.h, ctypes.byref(A), mfv.ptr(G.dev(b)), mfv.ptr(dx), nSweeps)
    case.sync()
    assert np.array_equal(G.host(dx), O.gauss_seidel(n, own, nei, diag, up, b, x0, nSweeps, symmetric=False))
