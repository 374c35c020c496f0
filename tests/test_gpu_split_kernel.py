"""The small levels' kernel (LATENCY: 64 cells a work-group, a wave per photon
group) against the tiled kernel (PERDIR: 256 cells): the same sums in FP32
with contraction left to the compiler, so the fields agree to FP32 rounding of
a few steps (1e-5), and the counted leaves and the status exactly."""
import dataclasses

import numpy as np
import pytest

from emma_amd import rt, synth
from emma_amd import tree as T
from emma_amd.params import make_params
from test_gpu_parity import field_errors

pytestmark = pytest.mark.gpu

TABLES = {1: "SB99_equiv_mono_TH", 3: "Starburst99_1grpT_3grpS"}


def workload(G, kind, seed):
    params = make_params(TABLES[G])
    rng = np.random.default_rng(seed)
    if kind == "one-oct":  # eight cells of a work-group's 64
        tree = T.uniform_tree(1)
    elif kind.startswith("box"):  # 64 and 512 cells: exactly one and eight work-groups
        tree = T.uniform_tree(int(kind[3]))
    else:  # coarse faces, refluxes, a ragged last work-group
        counts = [int(n) for n in kind.split("-")[1:]]
        tree = T.amr_tree(3, counts, synth.lognormal_sampler(synth.gaussian_field(8, rng), 1.0), rng)
    fields = {}
    for l in range(tree.lmin, tree.lmax + 1):
        fields[l] = synth.random_fields(params, np.exp(rng.normal(0.0, 1.0, tree.level(l).ncell)), rng)
        fields[l].e[:] = np.maximum(fields[l].e, 1e-2)
        fields[l].fx *= 0.5
    return dataclasses.replace(params, lcoarse=tree.lmin), tree, fields


@pytest.mark.parametrize("G", [1, 3])
@pytest.mark.parametrize("kind", ["one-oct", "box2", "box3", "amr-1", "amr-9-17", "amr-60-100-80"])
@pytest.mark.parametrize("mode,faces,budget", [(rt.RADSTEP, False, 0), (rt.RADSTEP, True, 2),
                                               (rt.COARSERAD, False, 0)])
def test_same_as_tiled(gpu_lib, G, kind, mode, faces, budget):
    params, tree, fields = workload(G, kind, 70 + G + len(kind))
    if faces:
        tree = T.with_boundaries(tree, reflect=(0, 2, 4))
    out = []
    for variant in (rt.VARIANT_PERDIR, rt.VARIANT_LATENCY):
        g = rt.RadGPU(params, rt.MIXED)
        g.setup(params, tree, fields, mode=mode)
        g.set_level_variant(variant)
        g.set_chem_budget(budget)
        g.enable_counters(True)
        for _ in range(2):
            g.coarse_step(1.0, 1)
        out.append((g.stats()["cell_updates"], {l: g.get(l) for l in fields}))
        g.close()
    assert out[0][0] == out[1][0]
    for l in fields:
        err = field_errors(out[1][1][l], out[0][1][l], params.cloc())
        assert max(err[k] for k in ("e", "fx", "fy", "fz", "x", "temp", "eint")) < 1e-5, (l, err)
        assert err["src"] == 0 and err["nh"] == 0, (l, err)
