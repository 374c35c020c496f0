"""The small levels' kernel (LATENCY) holds every rounding of the tiled one: each
field equal bit for bit to the per-direction variant (PERDIR), over sizes with
neighbours in the wave, in the same 32-oct tile and beyond it, coarse faces,
domain faces, and chemistry with and without the straggler pass."""
import numpy as np
import pytest

from emma_amd import rt
from emma_amd import tree as T
from emma_amd.synth import Fields
from test_gpu_split_kernel import workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [1, 3])
@pytest.mark.parametrize("kind", ["one-oct", "box2", "box3", "box4", "amr-1", "amr-9-17", "amr-60-100-80"])
@pytest.mark.parametrize("mode,faces,budget", [(rt.RADSTEP, False, 0), (rt.RADSTEP, True, 0), (rt.RADSTEP, False, 2),
                                               (rt.COARSERAD, False, 0)])
def test_equal_to_tiled(gpu_lib, G, kind, mode, faces, budget):
    params, tree, fields = workload(G, kind, 170 + G + len(kind))
    if faces:
        tree = T.with_boundaries(tree, reflect=(0, 2, 4))
    out = []
    for variant in (rt.VARIANT_PERDIR, rt.VARIANT_LATENCY):
        g = rt.RadGPU(params, rt.MIXED)
        g.setup(params, tree, fields, mode=mode)
        g.set_level_variant(variant)
        g.set_chem_budget(budget)
        for _ in range(3):
            g.coarse_step(1.0, 1)
        out.append({l: g.get(l) for l in fields})
        g.close()
    for l in fields:
        for k in Fields.NAMES:
            a, b = getattr(out[0][l], k), getattr(out[1][l], k)
            assert np.array_equal(a, b), (l, k, int((a != b).sum()), a.size)
