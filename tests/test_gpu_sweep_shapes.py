"""Sweeps in one launch on meshes unlike a box in its natural order: rows of many faces above the LDS size, and cells
in a few wide levels (colours). Results to the bit against the oracle, and no shape left far slower than the work it
is: a chain of levels in the first case, a stream over the cells in the second."""
import ctypes
import time

import numpy as np
import pytest

import gpu_util as G
import oracle_lib as O
from brae_amd import mfv
from test_gpu_sweep_plans import box, graph

pytestmark = pytest.mark.gpu


def reordered(mesh, place):
    """the mesh with cell c renumbered place[c]"""
    n, own, nei, bfc = mesh
    o, e = np.minimum(place[own], place[nei]), np.maximum(place[own], place[nei])
    k = np.lexsort([e, o])
    return n, o[k].astype(np.int32), e[k].astype(np.int32), place[bfc].astype(np.int32)


def coloured(nx, ny, nz, colours):
    """a box whose cells come colour by colour: at most `colours` levels"""
    c = np.arange(nx * ny * nz)
    i, j, k = c % nx, c // nx % ny, c // (nx * ny)
    colour = (i + j + k) % 2 if colours == 2 else i % 2 + 2 * (j % 2) + 4 * (k % 2)
    place = np.empty(c.size, np.int64)
    place[np.argsort(colour, kind="stable")] = c
    return reordered(box(nx, ny, nz), place)


def hub_and_chain(n):
    """a level of n/4 cells, one of which owns a face to every later cell: no step can hold its entries. The last
    cells are a chain, so there are many levels"""
    q, t = n // 4, n - 300
    own = np.concatenate([np.full(n - q, 5), np.delete(np.arange(q), 5), np.arange(t, n - 1)])
    nei = np.concatenate([np.arange(q, n), np.delete(np.arange(q), 5) + q, np.arange(t + 1, n)])
    o = np.lexsort([nei, own])
    return n, own[o].astype(np.int32), nei[o].astype(np.int32), np.array([0], np.int32)


class Sweeps:
    def __init__(self, mesh):
        self.mesh = mesh
        self.n, self.own, self.nei, bfc = mesh
        rng = np.random.default_rng(6)
        self.up = -rng.uniform(0.5, 2.0, self.own.size)
        self.diag = rng.uniform(0.1, 1.0, self.n)
        np.add.at(self.diag, self.own, -self.up)
        np.add.at(self.diag, self.nei, -self.up)
        self.b, self.x0 = rng.normal(size=self.n), rng.normal(size=self.n)
        self.case = G.Case(self.n, self.own, self.nei, bfc)
        self.A, self.db, self.dw = mfv.ldu(G.dev(self.diag), G.dev(self.up)), G.dev(self.b), G.zeros(self.n)

    def dic(self):
        self.case.call("mfv_dic_precondition", self.case.mesh.h, ctypes.byref(self.A), mfv.ptr(self.db), mfv.ptr(self.dw))
        return self.dw

    def gauss_seidel(self, symmetric):
        dx = G.dev(self.x0)
        self.case.call("mfv_sym_gauss_seidel" if symmetric else "mfv_gauss_seidel", self.case.mesh.h,
                       ctypes.byref(self.A), mfv.ptr(self.db), mfv.ptr(dx), 2)
        self.case.sync()
        return G.host(dx)

    def dic_seconds(self):
        best = 1e9
        for _ in range(6):
            t0 = time.perf_counter()
            self.dic()
            self.case.sync()
            best = min(best, time.perf_counter() - t0)
        return best


MESHES = {"two colours in LDS": lambda: coloured(27, 27, 27, 2), "eight colours in LDS": lambda: coloured(27, 27, 27, 8),
          "eight colours, small": lambda: coloured(12, 12, 12, 8), "two colours": lambda: coloured(40, 40, 40, 2),
          "eight colours": lambda: coloured(40, 40, 40, 8), "eight colours, large": lambda: coloured(80, 80, 80, 8),
          "hub and chain": lambda: hub_and_chain(4000),
          "rows of two batches": lambda: graph(21000, 6, 3, 400), "rows of many": lambda: graph(21000, 14, 3, 3000)}


@pytest.mark.parametrize("name", MESHES)
def test_bits(name):
    S = Sweeps(MESHES[name]())
    print("case:", name, S.n, "cells", S.own.size, "faces", flush=True)
    for _ in range(2):
        assert np.array_equal(G.host(S.dic()), O.dic_precondition(S.n, S.own, S.nei, S.diag, S.up, S.b))
    for symmetric in (False, True):
        assert np.array_equal(S.gauss_seidel(symmetric),
                              O.gauss_seidel(S.n, S.own, S.nei, S.diag, S.up, S.b, S.x0, 2, symmetric=symmetric)), symmetric


def test_two_colours_are_a_stream():
    """1 M cells in 2 levels against the same box in its natural order, 318 levels: 0.15 of its time with a launch per
    level, 0.63 when the waves of the one launch took their chunks one after another"""
    t = [Sweeps(m).dic_seconds() for m in (coloured(128, 128, 64, 2), box(128, 128, 64))]
    print("case: two colours", t, flush=True)
    assert t[0] < 0.35 * t[1]


def test_wide_rows_are_loaded_together():
    """110 levels with rows of up to 25 lower faces against 64^3 cells in 190 levels: 12 times its time, 29 when the
    faces past the first eight were taken one after another"""
    t = [Sweeps(m).dic_seconds() for m in (graph(300000, 4, 4, 30000), box(64, 64, 64))]
    print("case: wide rows", t, flush=True)
    assert t[0] < 20 * t[1]
