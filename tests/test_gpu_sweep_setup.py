"""What the first sweep on a mesh pays: the level schedule and the plan of the one-launch sweeps. The schedule is a few
host passes over the faces, as building the mesh is (both about 10 ms here, one thread each), and the plan is laid
out on the device beside it; a plan laid out by the host took five to ten times as long as either."""
import ctypes
import time

import numpy as np
import pytest

import gpu_util as G
from brae_amd import mfv
from test_gpu_sweep_plans import box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fn", ["mfv_dic_precondition", "mfv_gauss_seidel", "mfv_sym_gauss_seidel"])
def test_first_sweep_costs_what_the_mesh_does(fn):
    n, own, nei, bfc = box(128, 128, 64)
    A, b, x = mfv.ldu(G.dev(np.full(n, 7.0)), G.dev(np.full(own.size, -1.0))), G.dev(np.ones(n)), G.zeros(n)
    ctx = mfv.Context(0)
    tail = (3,) if "gauss" in fn else ()
    made, first = [], []
    for _ in range(4):
        t0 = time.perf_counter()
        case = G.Case(n, own, nei, bfc, ctx=ctx)
        case.sync()
        t1 = time.perf_counter()
        case.call(fn, case.mesh.h, ctypes.byref(A), mfv.ptr(b), mfv.ptr(x), *tail)
        case.sync()
        t2 = time.perf_counter()
        made.append(t1 - t0)
        first.append(t2 - t1)
    print("case:", fn, "mesh", min(made), "first sweep", min(first), flush=True)
    assert min(first) < 2.5 * min(made)
