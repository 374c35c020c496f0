"""The per-cell level step through LDS (one closure per cell, FP64 and the
mixed path's group counts other than 1 and 3) against the persistent kernel's
per-cell items, which read every neighbour from memory: the operations and
their order are the same, so every field is equal bit for bit."""
import dataclasses

import numpy as np
import pytest

from emma_amd import rt, synth
from emma_amd import tree as T
from emma_amd.params import ATOMIC_TABLES, RunParams, static_units
from emma_amd.synth import Fields

pytestmark = pytest.mark.gpu

ROWS = ATOMIC_TABLES["Starburst99_3grpT_3grpS"]


def workload(kind, groups, seed):
    params = RunParams.from_table(ROWS[:groups], 0.1, (0.0,), **static_units())
    rng = np.random.default_rng(seed)
    if kind == "tree":  # ragged last tiles, coarse faces, refluxes, waves with up to 192 halo faces
        W = synth.amr_workload(3, [60, 100, 80], "SB99_equiv_mono_TH", seed=seed, grid=16)
        tree = W.tree
    else:  # one partial tile (8 octs), several full ones (64, 512 octs)
        tree = T.uniform_tree({"part": 2, "two": 3, "full": 4}[kind.split("-")[0]])
    if kind.endswith("-faces"):  # open and reflecting domain faces
        tree = T.with_boundaries(tree, reflect=(0, 2, 4))
    fields = {l: synth.random_fields(params, np.exp(rng.normal(0.0, 1.0, tree.level(l).ncell)), rng)
              for l in range(tree.lmin, tree.lmax + 1)}
    for F in fields.values():
        F.e[:] = np.maximum(F.e, 1e-4)  # well above the floor, so that no cell stops at it
        F.fx *= 0.5
    return dataclasses.replace(params, lcoarse=tree.lmin), tree, fields


@pytest.mark.parametrize("groups", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("kind,variant,mode", [
    ("part", None, rt.RADSTEP), ("two", rt.VARIANT_PERDIR, rt.RADSTEP), ("full", None, rt.RADSTEP),
    ("two-faces", None, rt.RADSTEP), ("two-faces", rt.VARIANT_PERDIR, rt.RADSTEP),
    ("tree", None, rt.RADSTEP), ("tree", None, rt.COARSERAD)])
def test_same_as_per_cell_items(gpu_lib, groups, kind, variant, mode):
    params, tree, fields = workload(kind, groups, 40 + groups)
    for precision in (rt.FP64, rt.MIXED) if groups not in (1, 3) else (rt.FP64,):
        out = []
        for sched in (rt.SCHED_GRAPH, rt.SCHED_PERSISTENT):
            g = rt.RadGPU(params, precision)
            g.setup(params, tree, fields, mode=mode)
            if variant is not None:
                g.set_level_variant(variant)
            g.set_schedule(sched)
            g.coarse_step(1.0, 2)
            out.append({l: g.get(l) for l in fields})
        for l in fields:
            for k in Fields.NAMES:
                a, b = getattr(out[0][l], k), getattr(out[1][l], k)
                assert np.array_equal(a, b), (precision, l, k)
