"""The one-launch sequential sweeps (sweep.hip) against the oracle's host loops, to the bit: DIC, DILU (through
PBiCGStab with sequential reductions), Gauss-Seidel and symGaussSeidel on meshes at the edges of the plans --
the largest swept in LDS (up to 20,000 cells) and the smallest handed over between waves, one cell per level,
levels wider than a workgroup, rows wider than the entries loaded ahead, and a hub that keeps a launch per
level. A captured sweep replays to the same bits."""
import ctypes

import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from brae_amd import hexmesh, mfv

pytestmark = pytest.mark.gpu


def box(nx, ny, nz):
    m = hexmesh.box_topology(nx, ny, nz)
    nI = m[2].size
    return nx * ny * nz, np.ascontiguousarray(m[1][:nI]), m[2], np.ascontiguousarray(m[1][nI:])


def graph(n, per, seed, reach):
    """random upper-triangular faces: about `per` per cell, to at most `reach` cells on"""
    rng = np.random.default_rng(seed)
    own = np.repeat(np.arange(n), rng.integers(0, 2 * per + 1, n))
    nei = np.minimum(own + rng.integers(1, reach, own.size), n - 1)
    pairs = np.unique(np.stack([own, nei], 1)[nei > own], axis=0)
    return n, pairs[:, 0].astype(np.int32), pairs[:, 1].astype(np.int32), np.array([0], np.int32)


def hub(n):
    """a level of n/4 cells, one of which owns a face to every later cell: no step can hold its entries"""
    q = n // 4
    own = np.concatenate([np.full(n - q, 5), np.delete(np.arange(q), 5)])
    nei = np.concatenate([np.arange(q, n), np.delete(np.arange(q), 5) + q])
    o = np.lexsort([nei, own])
    return n, own[o].astype(np.int32), nei[o].astype(np.int32), np.array([0], np.int32)


def star(n):
    own = np.concatenate([np.zeros(n - 1), np.arange(1, n - 1)]).astype(np.int32)
    nei = np.concatenate([np.arange(1, n), np.full(n - 2, n - 1)]).astype(np.int32)
    return n, own, nei, np.array([0], np.int32)


MESHES = {
    "two cells": lambda: box(2, 1, 1), "chain in LDS": lambda: box(500, 1, 1), "ragged box": lambda: box(13, 7, 5),
    "wide levels": lambda: box(150, 132, 1), "last in LDS": lambda: box(100, 50, 4), "first handed over": lambda: box(3, 59, 113),
    "box handed over": lambda: box(31, 30, 29), "chain handed over": lambda: box(20011, 1, 1),
    "wide rows in LDS": lambda: graph(700, 6, 3, 60), "wide rows handed over": lambda: graph(20500, 5, 4, 900),
    "one wide level": lambda: graph(6000, 1, 5, 5999), "star": lambda: star(3000),
    "hub": lambda: hub(4000),
}


def system(name):
    n, own, nei, bfc = MESHES[name]()
    rng = np.random.default_rng(len(name))
    up = -rng.uniform(0.5, 2.0, own.size)
    lo = -rng.uniform(0.5, 2.0, own.size)
    diag = rng.uniform(0.1, 1.0, n)
    np.add.at(diag, own, np.maximum(-up, -lo))
    np.add.at(diag, nei, np.maximum(-up, -lo))
    return n, own, nei, bfc, diag, up, lo, rng.normal(size=n), rng.normal(size=n)


@pytest.mark.parametrize("name", list(MESHES))
def test_sweeps_bit_exact(name):
    n, own, nei, bfc, diag, up, lo, b, x0 = system(name)
    print("case:", name, n, "cells", own.size, "faces", flush=True)
    case = G.Case(n, own, nei, bfc)
    A = mfv.ldu(G.dev(diag), G.dev(up))
    dw = G.zeros(n)
    for _ in range(2):
        case.call("mfv_dic_precondition", case.mesh.h, ctypes.byref(A), mfv.ptr(G.dev(b)), mfv.ptr(dw))
    assert np.array_equal(G.host(dw), O.dic_precondition(n, own, nei, diag, up, b))
    for fn, sym in (("mfv_gauss_seidel", False), ("mfv_sym_gauss_seidel", True)):
        dx = G.dev(x0)
        case.call(fn, case.mesh.h, ctypes.byref(A), mfv.ptr(G.dev(b)), mfv.ptr(dx), 3)
        case.sync()
        assert np.array_equal(G.host(dx), O.gauss_seidel(n, own, nei, diag, up, b, x0, 3, symmetric=sym)), fn


@pytest.mark.parametrize("name", ["ragged box", "last in LDS", "first handed over", "wide rows handed over", "hub"])
def test_dilu_bit_exact(name):
    n, own, nei, bfc, diag, up, lo, b, x0 = system(name)
    print("case:", name, "PBiCGStab-DILU", flush=True)
    case = G.Case(n, own, nei, bfc)
    case.ctx.sequential_reduce(True)
    A = mfv.ldu(G.dev(diag), G.dev(up), G.dev(lo))
    nB = len(bfc)
    iC, bC = np.full(nB, 0.25), np.full(nB, 0.5)
    dx, perf, ctl = G.dev(x0), mfv.Perf(), mfv.bicg_controls(tolerance=1e-9, maxIter=60)
    case.call("mfv_pbicgstab_solve", case.mesh.h, ctypes.byref(A), mfv.ptr(G.dev(b)), mfv.ptr(G.dev(iC)), mfv.ptr(G.dev(bC)),
              mfv.ptr(dx), ctypes.byref(ctl), ctypes.byref(perf))
    x = x0.copy()
    ref = O.lib().orc_pbicgstab(n, len(own), O.p(O.i32(own)), O.p(O.i32(nei)), O.p(diag), O.p(up), O.p(lo), O.p(b), nB,
                                O.p(O.i32(bfc)), O.p(iC), O.p(bC), O.p(x), 1e-9, 0.0, 60, 0)
    assert perf.nIterations == ref.nIterations and perf.finalResidual == ref.finalResidual
    assert np.array_equal(G.host(dx), x)


@pytest.mark.parametrize("name", ["ragged box", "box handed over"])
def test_captured_sweep_replays(name):
    torch = G.torch_cuda()
    n, own, nei, bfc, diag, up, lo, b, x0 = system(name)
    s = torch.cuda.Stream()
    ctx = mfv.Context(0, stream=s.cuda_stream)
    case = G.Case(n, own, nei, bfc, ctx=ctx)
    A, db, dx, start = mfv.ldu(G.dev(diag), G.dev(up)), G.dev(b), G.dev(x0), G.dev(x0)
    sweep = lambda: case.call("mfv_gauss_seidel", case.mesh.h, ctypes.byref(A), mfv.ptr(db), mfv.ptr(dx), 2)
    ref = O.gauss_seidel(n, own, nei, diag, up, b, x0, 2)
    sweep()                                   # eager: builds the schedule and the plan
    case.sync()
    assert np.array_equal(G.host(dx), ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        dx.copy_(start)
        sweep()
    for _ in range(4):
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(G.host(dx), ref)
        with torch.cuda.stream(s):            # the program's own eager sweep between the replays
            dx.copy_(start)
            sweep()
        torch.cuda.synchronize()
        assert np.array_equal(G.host(dx), ref)
