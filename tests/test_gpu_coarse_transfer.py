"""COARSERAD transfers between the coarse level and the leaves: the gather
(fillrad of the coarse level) against a depth-first sum in the storage type and
the push (the coarse level's radsolver) against a copy, equal bit for bit."""
import dataclasses

import numpy as np
import pytest

from emma_amd import rt, synth
from emma_amd import tree as T
from emma_amd.params import ATOMIC_TABLES, RunParams, static_units

pytestmark = pytest.mark.gpu

ROWS = ATOMIC_TABLES["Starburst99_3grpT_3grpS"]
COMPONENTS = ("e", "fx", "fy", "fz")


def leaves(tree, level, oct_):
    """(level, cell) of the leaves below an oct, depth first, children in order"""
    for cell in range(oct_ * 8, oct_ * 8 + 8):
        ch = tree.level(level).child[cell]
        if ch >= 0:
            yield from leaves(tree, level + 1, ch)
        else:
            yield level, cell


# no split cell; one; more than one wave of them and four levels deep (octs with split and unsplit children)
@pytest.mark.parametrize("counts", [[], [1], [3, 9, 20], [150, 300, 200]])
@pytest.mark.parametrize("groups,precision", [(1, rt.FP64), (3, rt.MIXED), (9, rt.FP64), (9, rt.MIXED)])
def test_gather_and_push(gpu_lib, counts, groups, precision):
    params = RunParams.from_table(ROWS[:groups], 0.1, (0.0,), **static_units())
    rng = np.random.default_rng(60 + groups + len(counts))
    if counts:
        tree = T.amr_tree(3, counts, synth.lognormal_sampler(synth.gaussian_field(8, rng), 1.0), rng)
    else:
        tree = T.uniform_tree(3)
    fields = {}
    for l in range(tree.lmin, tree.lmax + 1):
        fields[l] = synth.random_fields(params, np.exp(rng.normal(0.0, 1.0, tree.level(l).ncell)), rng)
        fields[l].e[:] = np.maximum(fields[l].e, 1e-2)
        fields[l].fx *= 0.5
    params = dataclasses.replace(params, lcoarse=tree.lmin)
    g = rt.RadGPU(params, precision)
    g.setup(params, tree, fields, mode=rt.COARSERAD)
    before = {l: g.get(l) for l in fields}
    g.fillrad(tree.lmin)
    gathered = g.get(tree.lmin)
    g.radsolver(tree.lmin, 1e-3 * params.dt_rad(tree.lmin))
    after = {l: g.get(l) for l in fields}
    g.close()
    R = np.float64 if precision == rt.FP64 else np.float32
    child = tree.level(tree.lmin).child
    for k in COMPONENTS:
        want = getattr(before[tree.lmin], k).reshape(groups, -1).copy()
        for i in np.flatnonzero(child >= 0):
            acc = np.zeros(groups, R)
            for l, cell in leaves(tree, tree.lmin + 1, child[i]):
                x = getattr(before[l], k).reshape(groups, -1)[:, cell].astype(R)
                acc += x * R(8.0 ** (tree.lmin - l))
                top = getattr(after[tree.lmin], k).reshape(groups, -1)[:, i]
                assert np.array_equal(getattr(after[l], k).reshape(groups, -1)[:, cell], top), (k, i, l, cell)
            want[:, i] = acc
        assert np.array_equal(getattr(gathered, k).reshape(groups, -1), want), k
