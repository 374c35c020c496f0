"""Levels whose free tiles (no split cell, no leaf with a finer oct behind a
face) step beside the finer levels: coarse_step, which captures them on a side
stream, against the same launches one after the other (TIMING_LAUNCH), bit for
bit, over several coarse steps, replays and eager work in between."""
import numpy as np
import pytest

from emma_amd import rt, synth
from emma_amd.params import make_params
from emma_amd import tree as T
from emma_amd.synth import Fields

pytestmark = pytest.mark.gpu


def workload(table, lmin, counts, seed):
    params = make_params(table)
    params.lcoarse = lmin
    rng = np.random.default_rng(seed)
    tree = T.amr_tree(lmin, counts, synth.lognormal_sampler(synth.gaussian_field(16, rng), 1.0), rng)
    fields = {}
    for l in range(tree.lmin, tree.lmax + 1):
        F = synth.random_fields(params, np.exp(rng.normal(0.0, 0.5, tree.level(l).ncell)), rng)
        F.e[:] = np.maximum(F.e, 1e-2)  # well above the floor
        F.fx *= 0.5
        fields[l] = F
    return params, tree, fields


# one forked level over a deep chain; two forked levels; a level whose finer launches are too short to fork
@pytest.mark.parametrize("table,lmin,counts", [("Starburst99_1grpT_3grpS", 7, [300, 200, 40]),
                                               ("Starburst99_1grpT_3grpS", 7, [60000, 2000, 300]),
                                               ("SB99_equiv_mono_TH", 7, [500, 100]),
                                               ("Starburst99_1grpT_3grpS", 6, [3000, 900])])
@pytest.mark.parametrize("precision,budget", [(rt.FP64, 0), (rt.MIXED, 0), (rt.MIXED, 2)])
def test_same_as_one_after_the_other(gpu_lib, table, lmin, counts, precision, budget):
    params, tree, fields = workload(table, lmin, counts, 5 + lmin + len(counts))
    out = []
    for timing in (rt.TIMING_LAUNCH, rt.TIMING_OFF):
        g = rt.RadGPU(params, precision)
        g.setup(params, tree, fields)
        g.set_chem_budget(budget)  # > 0: both launches' straggler list
        g.save_state()
        for rep in range(3):
            g.restore_state()
            g.enable_timing(timing)
            g.coarse_step(1.0, 1)
            g.coarse_step(1.0, 1)
            first = g.stats()["cell_updates"], g.stats()["chem_substeps"]
            g.enable_timing(rt.TIMING_OFF)
            g.radsolver(tree.lmax, params.dt_rad(tree.lmax))  # eager work between replays
            g.enable_timing(timing)
            g.coarse_step(1.0, 2)
        out.append((first, {l: g.get(l) for l in fields}))
        g.close()
    assert out[0][0] == out[1][0]
    for l in fields:
        for k in Fields.NAMES:
            assert np.array_equal(getattr(out[0][1][l], k), getattr(out[1][1][l], k)), (l, k)
