"""emma_rt_advance_stencil on page-locked records (read and written in place
by one kernel) against ordinary memory (copied whole to the device buffer and
back): the same records byte for byte, over group counts, REAL types, ragged
last work-groups, split cells and the COARSERAD / chemistry-only modes."""
import numpy as np
import pytest

from emma_amd import rgrid, rt, synth
from emma_amd import tree as T
from emma_amd.params import ATOMIC_TABLES, RunParams, static_units

pytestmark = pytest.mark.gpu


def batch(groups, real, n, seed):
    params = RunParams.from_table(ATOMIC_TABLES["Starburst99_3grpT_3grpS"][:groups], 0.1, (0.0,), **static_units())
    params.lcoarse = 4
    rng = np.random.default_rng(seed)
    L = T.uniform_tree(4).level(4)
    F = synth.random_fields(params, np.exp(rng.normal(0.0, 1.0, L.ncell)), rng)
    F.e[:] = np.maximum(F.e, 1e-4)
    F.src[:, ::7] = rng.random(F.src[:, ::7].shape) * 1e-3
    st = rgrid.gather_complete(L, F, np.sort(rng.permutation(L.noct)[:n]), groups, real)
    st["oct"]["split"][rng.random(st["oct"]["split"].shape) < 0.2] = 1
    st["New"]["rflux"] = 7.0  # what the call does not write stays
    st["New"]["deltaR"]["e"] = 3.0
    return params, st


@pytest.mark.parametrize("groups,real", [(1, 8), (1, 4), (2, 8), (2, 4), (3, 8), (3, 4), (4, 8), (6, 4), (9, 8), (9, 4)])
@pytest.mark.parametrize("n", [1, 3, 8, 9, 67])
@pytest.mark.parametrize("mode,level,chemonly", [(rt.RADSTEP, 4, 0), (rt.RADSTEP, 4, 1), (rt.COARSERAD, 4, 0),
                                                 (rt.COARSERAD, 5, 0)])
def test_same_as_copied(gpu_lib, groups, real, n, mode, level, chemonly):
    params, st = batch(groups, real, n, 100 * groups + n)
    g = rt.RadGPU(params, rt.FP64)
    g.set_mode(mode)
    g.create_radstencil(n + 2, real)
    pinned = g.pinned_stencil(n + 2, real)
    pinned.array[:n] = st
    pinned.array[n:] = st[0]
    rest = pinned.array[n:].tobytes()
    start = st.tobytes()
    out = []
    for a in (st, pinned.array):
        try:
            g.advance_stencil(a, n, 0.5**level, params.dt_rad(level), chemonly=chemonly, level=level)
            status = rt.OK
        except rt.EmmaRTError as e:
            status = e.status
        s = g.stats()
        out.append((status, s["cell_updates"], s["chem_substeps"], a[:n].tobytes()))
    assert out[0][0] == rt.OK
    assert out[0][:3] == out[1][:3]
    a, b = (np.frombuffer(x[3], np.uint8) for x in out)
    pad = np.frombuffer(start, np.uint8)
    assert np.array_equal(a, b), np.nonzero(a != b)[0][:8]
    assert not np.array_equal(a, pad)
    assert pinned.array[n:].tobytes() == rest
    pinned.free()
