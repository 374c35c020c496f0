"""A level's state to the device and back: one gathering kernel for small
levels, chunks through page-locked slots by several threads for larger ones
(the sizes either side of the limit, ragged last chunks).  FP64 storage returns
the doubles, FP32 storage their rounding, with the photon floor kept."""
import ctypes
import dataclasses
import threading

import numpy as np
import pytest

from emma_amd import rt, synth
from emma_amd import tree as T
from emma_amd.params import ATOMIC_TABLES, EMIN, RunParams, static_units
from emma_amd.synth import Fields

pytestmark = pytest.mark.gpu

ROWS = ATOMIC_TABLES["Starburst99_3grpT_3grpS"]


def floor_of(params, g):
    """the photon floor EMIN factgrp / unit_N, in this order of operations"""
    return EMIN * params.factgrp[g] / params.unit_N


def context(level, groups, precision, extra=0, seed=1):
    params = RunParams.from_table(ROWS[:groups], 0.1, (0.0,), **static_units())
    L = T.uniform_level(level)
    levels = [L]
    if extra:  # a finer level of `extra` octs: any number of cells
        levels.append(T.refine(L, np.arange(extra)))
    tree = T.build_tree(levels)
    g = rt.RadGPU(dataclasses.replace(params, lcoarse=level), precision)
    g.load_tree(tree)
    rng = np.random.default_rng(seed)
    F = {l: synth.random_fields(params, np.exp(rng.normal(0.0, 1.0, tree.level(l).ncell)), rng) for l in tree.levels}
    for l in F:  # the floor itself, just above and just below it, in the last cells
        for q in range(groups):
            f = floor_of(params, q)
            F[l].e[q, -3:] = f, np.nextafter(f, 1.0), np.nextafter(f, 0.0)
        F[l].src[:] = rng.random(F[l].src.shape)
    return g, params, tree, F


def stored(params, F, k, precision):
    a = getattr(F, k)
    if precision == rt.FP64 or k in ("nhplus", "eint", "nh", "temp"):
        return a
    with np.errstate(under="ignore"):
        r = a.astype(np.float32)
    if k == "e":
        f = np.array([[floor_of(params, q)] for q in range(params.ngrp)])
        up = np.where(f.astype(np.float32).astype(np.float64) >= f, f.astype(np.float32),
                      np.nextafter(f.astype(np.float32), np.float32(np.inf)))
        r = np.where((a >= f) & (r.astype(np.float64) < f), up, r)
    return r.astype(np.float64)


# cells x (5 G + 4) doubles: below, just below, just above and far above 2^17 of them; ragged finer levels
@pytest.mark.parametrize("level,groups,extra", [(1, 1, 0), (3, 9, 5), (4, 1, 0), (4, 3, 861), (4, 3, 863), (5, 1, 0),
                                                (5, 9, 4097), (6, 3, 0)])
@pytest.mark.parametrize("precision", [rt.FP64, rt.MIXED])
def test_round_trip(gpu_lib, level, groups, extra, precision):
    g, params, tree, F = context(level, groups, precision, extra)
    for l in F:
        g.set(l, 0, F[l])
    for l in F:
        B = g.get(l)
        for k in Fields.NAMES:
            assert np.array_equal(getattr(B, k), stored(params, F[l], k, precision)), (l, k)


def test_some_fields_and_several_threads(gpu_lib):
    """null pointers leave fields out; contexts of different threads at once"""
    cs = [context(6, 1, p, seed=s) for s, p in ((3, rt.FP64), (4, rt.MIXED), (5, rt.FP64))]
    bad = []

    def go(g, params, tree, F):
        for _ in range(4):
            g.set(6, 0, F[6])
            B = Fields.zeros(1, F[6].ncell)
            dp = ctypes.POINTER(ctypes.c_double)
            skip = ("fx", "nh")
            st = g.lib.emma_rt_get_level(g.h, 6, *[None if k in skip else getattr(B, k).ctypes.data_as(dp)
                                                   for k in Fields.NAMES])
            for k in Fields.NAMES:
                want = np.zeros_like(getattr(B, k)) if k in skip else stored(params, F[6], k, g.precision)
                if st != rt.OK or not np.array_equal(getattr(B, k), want):
                    bad.append((st, k))

    th = [threading.Thread(target=go, args=c) for c in cs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
