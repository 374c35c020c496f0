"""emma_rt_advance_stencil on records in each kind of host memory: page-locked
of the library and of other allocations (coherent or not, aligned to 16 bytes
or off it) against ordinary memory, byte for byte, over several calls with new
inputs in the same memory."""
import ctypes

import numpy as np
import pytest

from emma_amd import rt
from test_gpu_stencil_direct import batch

pytestmark = pytest.mark.gpu

COHERENT, NONCOHERENT = 0x40000000, 0x80000000  # hipHostMalloc's flags


@pytest.mark.parametrize("flags", [0, 1, COHERENT, NONCOHERENT])
@pytest.mark.parametrize("offset", [0, 8])
@pytest.mark.parametrize("groups,real", [(1, 8), (3, 4)])
def test_same_in_any_memory(gpu_lib, flags, offset, groups, real):
    n = 67
    params, st = batch(groups, real, n, 100 * groups + n)
    p = ctypes.c_void_p()
    size = st.nbytes + 64
    # the runtime the library is linked to
    assert gpu_lib.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(size), ctypes.c_uint(flags)) == 0
    raw = np.frombuffer((ctypes.c_uint8 * size).from_address(p.value), np.uint8)
    there = raw[offset : offset + st.nbytes].view(st.dtype)
    g = rt.RadGPU(params, rt.FP64)
    g.create_radstencil(n, real)
    dt = params.dt_rad(4)
    rng = np.random.default_rng(8)
    for call in range(4):
        here = st.copy()
        scale = rng.uniform(0.5, 1.0)
        for state in (here["oct"]["rfield"], here["New"]["rfieldnew"]):
            for k in ("e", "fx", "fy", "fz", "src"):
                state[k] *= scale
        raw[:] = 5
        raw[offset : offset + st.nbytes] = here.view(np.uint8)  # padding bytes too
        g.advance_stencil(here, n, 0.5**4, dt)
        g.advance_stencil(there, n, 0.5**4, dt)
        assert there.tobytes() == here.tobytes(), call
        assert (raw[:offset] == 5).all() and (raw[offset + st.nbytes :] == 5).all()
    g.close()
    assert gpu_lib.hipHostFree(p) == 0
