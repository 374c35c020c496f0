"""The library's host code against a host model of the HIP runtime."""
import ctypes
import dataclasses
import os

import numpy as np

import hip_model as hm
from emma_amd import rgrid, synth
from emma_amd import tree as T
from emma_amd.params import make_params
from hip_model import modelled


def _params(G, level):
    p = make_params({1: "SB99_equiv_mono_TH", 3: "Starburst99_1grpT_3grpS"}[G])
    return dataclasses.replace(p, lcoarse=level)


def _fields(G, tree, seed=1):
    rng = np.random.default_rng(seed)
    p = _params(G, tree.lmin)
    return {l: synth.random_fields(p, np.ones(tree.level(l).ncell), rng) for l in range(tree.lmin, tree.lmax + 1)}


def _tree(lmin, counts, seed=3):
    rng = np.random.default_rng(seed)
    return T.amr_tree(lmin, counts, synth.lognormal_sampler(synth.gaussian_field(8, rng), 1.0), rng)


def _batch(n, G=1, align=16):
    """n records in ordinary memory, their first byte at a multiple of `align` but not of twice that"""
    size = rgrid.rgrid_dtype(G, 8).itemsize * n
    raw = np.zeros(size + 4096, np.uint8)
    at = (-raw.ctypes.data) % 4096 + align % 4096
    st = raw[at : at + size].view(rgrid.rgrid_dtype(G, 8))
    return raw, st


def _stencil_context(rt, n, G=1):
    p = _params(G, 4)
    g = rt.RadGPU(p, rt.FP64)
    g.create_radstencil(n, 8)
    return g, lambda st: g.advance_stencil(st, n, 0.5**4, p.dt_rad(4))


# ---------------------------------------------------------------- batches in place
@modelled
def test_records_not_known_coherent_are_waited_for(m, rt):
    """Results written into page-locked memory by a kernel are the host's to
    read after a runtime synchronisation, or at once if the memory is coherent."""
    g, advance = _stencil_context(rt, 5)
    keep = []  # the model holds on to their ranges
    for flags in (0, hm.PORTABLE, hm.NONCOHERENT):
        raw, st = _batch(5)
        keep.append(raw)
        m.model_lock(raw.ctypes.data, raw.nbytes, flags)
        m.model_forget()
        before = m.model_stream_waits()
        advance(st)
        assert any("stencil_direct_kernel" in k for k in m.launched()), flags
        assert m.model_stream_waits() > before, flags
    pinned = g.pinned_stencil(5, 8)
    pinned.array[:] = st
    m.model_forget()
    before = m.model_stream_waits()
    advance(pinned.array)
    assert any("stencil_direct_kernel" in k for k in m.launched())
    assert m.model_stream_waits() == before


@modelled
def test_own_page_locked_memory_is_coherent(m, rt):
    """the call record is polled while kernels run; transfer slots change hands between host and kernels"""
    tree = T.uniform_tree(5)
    g = rt.RadGPU(_params(1, 5), rt.FP64)
    g.setup(_params(1, 5), tree, _fields(1, tree))
    g.pinned_stencil(3, 8)
    assert m.model_host_blocks() >= 3  # the record, the slots, the batch
    assert m.model_common_flags() & hm.COHERENT


@modelled
def test_batch_between_locked_ranges_is_copied(m, rt):
    """both ends page-locked, the middle not"""
    g, advance = _stencil_context(rt, 5)
    raw, st = _batch(5)
    at = st.ctypes.data
    for a in (at, at + st.nbytes - 4096):
        m.model_lock(a, 4096, hm.COHERENT)
    advance(st)
    assert not any("stencil_direct_kernel" in k for k in m.launched())
    assert any("stencil_kernel" in k for k in m.launched())


@modelled
def test_batch_locked_for_reading_is_copied(m, rt):
    """a kernel may not write there"""
    g, advance = _stencil_context(rt, 5)
    raw, st = _batch(5)
    m.model_lock(raw.ctypes.data, raw.nbytes, hm.REGISTER_READ_ONLY)
    advance(st)
    assert not any("stencil_direct_kernel" in k for k in m.launched())
    assert any("stencil_kernel" in k for k in m.launched())


@modelled
def test_misaligned_batch_is_copied(m, rt):
    g, advance = _stencil_context(rt, 5)
    raw, st = _batch(5, align=8)
    m.model_lock(raw.ctypes.data, raw.nbytes, hm.COHERENT)
    advance(st)
    assert any("stencil_kernel" in k for k in m.launched())


@modelled
def test_ordinary_batch_keeps_what_others_write(m, rt):
    """only rfieldnew and rflux of the records are the call's to write"""
    for n in (1, 700):  # one copy back, several
        g, advance = _stencil_context(rt, n)
        raw, st = _batch(n)
        ours = np.zeros(st.nbytes, bool)
        lay = rgrid.layout(1, 8)
        new, cell, at, end = lay[21], lay[12], lay[15], lay[12]  # New, a cell of it, its rfieldnew up to its end
        for c in range(8):
            ours.reshape(n, -1)[:, new + c * cell + at : new + c * cell + end] = True
        raw8 = st.view(np.uint8)
        old = raw8.copy()

        def meanwhile():
            raw8[~ours] = 77

        f = ctypes.CFUNCTYPE(None)(meanwhile)
        m.model_during(b"stencil_kernel", f)
        advance(st)
        m.model_during(b"none", None)
        assert (raw8[~ours] == 77).all(), n
        assert np.array_equal(raw8[ours], old[ours]), n  # the model runs no kernel


# ---------------------------------------------------------------- devices
@modelled
def test_transfers_from_a_thread_on_another_device(m, rt):
    m.model_device(1)
    tree = T.uniform_tree(5)
    F = _fields(1, tree)
    g = rt.RadGPU(_params(1, 5), rt.FP64)
    g.setup(_params(1, 5), tree, F)
    H = synth.hydro_like(F[5], np.random.default_rng(2))
    m.model_device(0)
    g.set(5, 0, F[5])
    B = g.get(5)
    assert np.array_equal(B.e, F[5].e) and np.array_equal(B.nh, F[5].nh)
    g.set_hydro(5, H)
    assert np.array_equal(g.get_hydro(5)[0], H.p)
    assert m.model_current() == 0


@modelled
def test_coarse_step_from_a_thread_on_another_device(m, rt):
    m.model_device(1)
    tree = _tree(7, [4000, 1500])
    g = rt.RadGPU(_params(3, 7), rt.FP64)
    g.setup(_params(3, 7), tree, {})
    m.model_device(0)
    m.model_forget()
    g.coarse_step(1.0, 1)
    assert sum("transport_kernel" in k for k in m.launched()) == 8  # 1 + 2 + 4 level steps, the first in two parts
    assert m.model_current() == 0


# ---------------------------------------------------------------- forked levels
@modelled
def test_levels_that_fork(m, rt):
    """a level forks where its free tiles are worth it: large levels, by family, and middling ones beside launches
    that leave the chip idle (two launches of each forked level step in a captured coarse step)"""
    rng = np.random.default_rng(97)
    sampler = synth.lognormal_sampler(synth.gaussian_field(32, rng), 1.0)
    small, large = T.amr_tree(6, [40000, 3000], sampler, rng), T.amr_tree(7, [4000, 1500], sampler, rng)
    deep = T.amr_tree(7, [80000, 20000, 3000, 400], sampler, rng)
    kernel = {(1, rt.FP64): "level_step_kernel", (3, rt.FP64): "transport_kernel"}
    for tree, G, precision, forks in ((small, 1, rt.MIXED, 0), (small, 3, rt.MIXED, 0), (small, 1, rt.FP64, 0),
                                      (large, 1, rt.MIXED, 0), (large, 3, rt.MIXED, 1), (large, 1, rt.FP64, 1),
                                      (large, 3, rt.FP64, 1), (deep, 1, rt.MIXED, 0), (deep, 3, rt.MIXED, 1 + 2)):
        g = rt.RadGPU(_params(G, tree.lmin), precision)
        g.setup(_params(G, tree.lmin), tree, {})
        m.model_forget()
        g.coarse_step(1.0, 1)
        name = kernel.get((G, precision), "level_step_")
        steps = 2 ** len(tree.levels) - 1
        assert sum(name in k for k in m.launched()) == steps + forks, (tree.lmin, G, precision, m.launched())
        g.close()


# ---------------------------------------------------------------- failed calls
@modelled
def test_pending_injection_ends_with_a_failed_call(m, rt):
    tree = _tree(3, [20, 30])
    F = _fields(1, tree)
    rng = np.random.default_rng(4)
    for timing in (rt.TIMING_LAUNCH, rt.TIMING_OFF):
        for n in range(8):
            g = rt.RadGPU(_params(1, 3), rt.FP64)
            g.setup(_params(1, 3), tree, F, mode=rt.COARSERAD)
            for l in F:
                g.set_hydro(l, synth.hydro_like(F[l], rng))
            g.set_coupling(True)
            g.enable_timing(timing)
            m.model_set(hm.FAIL_LAUNCH, n)
            try:
                g.coarse_step(1.0, 1)
                assert False, "no launch failed"
            except rt.EmmaRTError:
                pass
            m.model_forget()
            g.fillrad(3)
            assert not any("couple_kernel" in k for k in m.launched()), (timing, n)
            g.coarse_step(1.0, 1)
            g.close()


@modelled
def test_forked_level_after_a_failed_capture(m, rt):
    """a side stream left in a failed capture does not fail later calls"""
    tree = _tree(7, [4000, 1500])
    g = rt.RadGPU(_params(3, 7), rt.FP64)
    g.setup(_params(3, 7), tree, {})
    for n in range(14):
        m.model_set(hm.FAIL_LAUNCH, n)
        try:
            g.coarse_step(1.0, 1)
            assert False, "no launch failed"
        except rt.EmmaRTError:
            pass
        m.model_set(hm.FAIL_LAUNCH, -1)
    g.coarse_step(1.0, 1)


# ---------------------------------------------------------------- the transfers' page-locked memory
def _exact(F):
    """fields that FP32 storage holds exactly"""
    F.e[:] = 0.5
    for k in ("fx", "fy", "fz", "src"):
        getattr(F, k)[:] = np.float32(getattr(F, k))
    return F


@modelled
def test_transfers_keep_few_bounded_blocks(m, rt):
    """one block a transfer, 32 MiB kept at most, 16 between contexts"""
    shapes = [(rt.RadGPU(_params(G, l), precision), T.uniform_tree(l), G)
              for l, G, precision in ((6, 3, rt.FP64), (7, 3, rt.MIXED), (5, 1, rt.FP64))]
    for g, tree, G in shapes:
        g.load_tree(tree)
    record = m.model_host_blocks()
    for g, tree, G in shapes[:1] * 2 + shapes + shapes[:1]:
        l = tree.lmin
        F = _exact(_fields(G, tree)[l])
        g.set(l, 0, F)
        B = g.get(l)
        for k in synth.Fields.NAMES:
            assert g.precision == rt.MIXED or np.array_equal(getattr(B, k), getattr(F, k)), k
        assert m.model_host_blocks() - record <= 2
        assert m.model_host_bytes() <= (32 << 20) + 4096
    for g, tree, G in shapes:
        g.close()
    assert m.model_host_blocks() <= 2 and m.model_host_bytes() <= 16 << 20


@modelled
def test_short_lived_contexts_share_their_blocks(m, rt):
    tree = T.uniform_tree(5)
    F = _fields(3, tree)
    allocs = []
    for _ in range(4):
        g = rt.RadGPU(_params(3, 5), rt.FP64)
        g.setup(_params(3, 5), tree, F)
        g.get(5)
        g.close()
        allocs.append(m.model_host_allocs())
    assert np.array_equal(np.diff(allocs), [1, 1, 1]), allocs  # the call record alone
    m.model_reset()  # of the device: new blocks, and none of the old ones freed
    g = rt.RadGPU(_params(3, 5), rt.FP64)
    g.setup(_params(3, 5), tree, F)
    assert m.model_host_allocs() == allocs[-1] + 2
    for k in synth.Fields.NAMES:
        assert np.array_equal(getattr(g.get(5), k), getattr(F[5], k)), k
    g.close()


@modelled
def test_transfers_with_little_page_locked_memory(m, rt):
    """as many slots as there are, fewer threads with them"""
    tree = T.uniform_tree(6)
    F = _fields(1, tree)[6]
    for free in (2 << 20, 3 << 20, 4 << 20, 9 << 20):
        g = rt.RadGPU(_params(1, 6), rt.FP64)
        g.load_tree(tree)
        m.model_set(hm.HOST_BYTES, m.model_host_bytes() + free)
        g.set(6, 0, F)
        B = g.get(6)
        for k in synth.Fields.NAMES:
            assert np.array_equal(getattr(B, k), getattr(F, k)), (free, k)
        m.model_set(hm.HOST_BYTES, -1)
        g.close()


@modelled
def test_transfers_without_page_locked_memory(m, rt):
    """the runtime's copies serve, converted on the host"""
    for l in (3, 6):
        tree = T.uniform_tree(l)
        F = _exact(_fields(1, tree)[l])
        for precision in (rt.FP64, rt.MIXED):
            g = rt.RadGPU(_params(1, l), precision)
            g.load_tree(tree)
            m.model_set(hm.HOST_BYTES, 0)
            g.set(l, 0, F)
            B = g.get(l)
            for k in synth.Fields.NAMES:
                assert np.array_equal(getattr(B, k), getattr(F, k)), (l, precision, k)
            m.model_set(hm.HOST_BYTES, -1)
            g.close()


# ---------------------------------------------------------------- the wait for a call
@modelled
def test_call_end_clears_what_the_call_used(m, rt):
    """straggler list lengths: one for each level step of this call, however long an earlier one was"""
    tree = _tree(3, [20, 30])
    p = _params(3, 3)
    g = rt.RadGPU(p, rt.MIXED)
    g.setup(p, tree, _fields(3, tree))
    g.set_chem_budget(4)
    g.coarse_step(1.0, 100)
    assert m.model_cleared() == 700
    g.radsolver(5, p.dt_rad(5))
    assert m.model_cleared() == 1
    g.set_chem_budget(0)
    g.radsolver(5, p.dt_rad(5))
    assert m.model_cleared() == 0


@modelled
def test_wait_gives_way(m, rt):
    """a call's wait shares its core with whoever the call waits for"""
    os.sched_setaffinity(0, {min(os.sched_getaffinity(0))})
    tree = T.uniform_tree(3)
    p = _params(1, 3)
    g = rt.RadGPU(p, rt.FP64)
    g.setup(p, tree, _fields(1, tree))
    m.model_set(hm.DELAY_FLAG, 800)
    polled = [0, 0, 0]
    for k in range(60):  # the best of three: the core may be busy with something else
        before = m.model_stream_waits()
        g.radsolver(3, p.dt_rad(3))
        polled[k // 20] += m.model_stream_waits() == before
    assert max(polled) >= 15, polled
