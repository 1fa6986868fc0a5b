"""Per-cell gathers that load a cell's first three owned and three other faces together: meshes whose cells have
fewer (none at all, chains), exactly three and many more of either kind, in both cell orders, against the oracle
to the bit."""
import ctypes

import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from brae_amd import mfv
from test_gpu_sweep_plans import box, graph

pytestmark = pytest.mark.gpu

MESHES = {"one cell": lambda: (1, np.zeros(0, np.int32), np.zeros(0, np.int32), np.zeros(6, np.int32)),
          "chain": lambda: box(257, 1, 1), "box": lambda: box(9, 8, 7), "plane slabs": lambda: box(33, 17, 5),
          "long runs": lambda: graph(3000, 6, 2, 40), "long runs in slabs": lambda: graph(5000, 4, 6, 900)}


@pytest.mark.parametrize("name", MESHES)
def test_gauss_gradient(name):
    n, own, nei, bfc = MESHES[name]()
    rng = np.random.default_rng(8)
    nI, nB = own.size, bfc.size
    print("case:", name, n, nI, nB, flush=True)
    types = rng.integers(0, 3, nB).astype(np.int32)
    vals, Sf, w = rng.normal(size=nB), rng.normal(size=(nI + nB, 3)), rng.uniform(0.2, 0.8, nI)
    V, psi = rng.uniform(0.5, 2.0, n), rng.normal(size=n)
    case = G.Case(n, own, nei, bfc)
    d = [G.dev(a) for a in (types, vals, Sf, w if nI else np.zeros(1), V, psi)]
    g = G.zeros(3 * n)
    case.call("mfv_grad_gauss", case.mesh.h, *[mfv.ptr(a) for a in d], mfv.ptr(g))
    case.sync()
    assert np.array_equal(G.host(g).reshape(n, 3), O.grad_gauss(n, own, nei, bfc, types, vals, Sf, w, V, psi))


@pytest.mark.parametrize("name", MESHES)
def test_face_sums(name):
    """matrix rows (the product and the residual) and sums of face values (the laplacian's and upwind's diagonals)"""
    n, own, nei, bfc = MESHES[name]()
    rng = np.random.default_rng(9)
    nI, nB = own.size, bfc.size
    print("case:", name, n, nI, flush=True)
    case = G.Case(n, own, nei, bfc)
    pad = lambda a: G.dev(a if a.size else np.zeros(1))
    diag, up, lo = rng.uniform(1.0, 2.0, n), rng.normal(size=nI), rng.normal(size=nI)
    x, b, dc, gam, mag = rng.normal(size=n), rng.normal(size=n), rng.normal(size=nI), rng.normal(size=nI), rng.normal(size=nI)
    A, dx, db, dy = mfv.ldu(G.dev(diag), pad(up), pad(lo)), G.dev(x), G.dev(b), G.zeros(n)
    s, r, sums = diag * x, b - diag * x, diag.copy()
    lapD, divD = np.zeros(n), np.zeros(n)
    lap = dc * gam * mag
    dlo = -np.where(dc >= 0.0, 1.0, 0.0) * dc
    dup = dlo + dc
    # each cell's faces in ascending order: the faces' order serves both runs
    for f in range(nI):
        o, e = own[f], nei[f]
        s[o] += up[f] * x[e]
        s[e] += lo[f] * x[o]
        r[o] -= up[f] * x[e]
        r[e] -= lo[f] * x[o]
        lapD[o] -= lap[f]
        lapD[e] -= lap[f]
        divD[o] -= dlo[f]
        divD[e] -= dup[f]
    case.call("mfv_amul", case.mesh.h, ctypes.byref(A), mfv.ptr(dx), mfv.ptr(dy))
    case.sync()
    assert np.array_equal(G.host(dy), s)
    case.call("mfv_residual", case.mesh.h, ctypes.byref(A), mfv.ptr(dx), mfv.ptr(db), mfv.ptr(dy))
    case.sync()
    assert np.array_equal(G.host(dy), r)
    dU, dL = pad(np.zeros(nI)), pad(np.zeros(nI))
    case.call("mfv_laplacian_coeffs", case.mesh.h, mfv.ptr(pad(dc)), mfv.ptr(pad(gam)), mfv.ptr(pad(mag)), mfv.ptr(dy), mfv.ptr(dU),
              mfv.ptr(dL))
    case.sync()
    assert np.array_equal(G.host(dy), lapD)
    case.call("mfv_div_upwind_coeffs", case.mesh.h, mfv.ptr(pad(dc)), mfv.ptr(dy), mfv.ptr(dU), mfv.ptr(dL))
    case.sync()
    assert np.array_equal(G.host(dy), divD)
