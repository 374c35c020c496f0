"""What the radiation step is asked to do in use, as timed cases.

A pass goes through the entry points of ``emma_amd.rt`` (the mirror of the C
ABI in ``include/emma_rt.h``) the way a host program does:

``run``      a restart point is restored, a run of radiative sub-cycles or
             coarse steps is advanced, and the whole state is read back (the
             host reads the fields once per output or hydro step, after tens
             to hundreds of sub-cycles);
``host``     the host owns the state: it hands every level over, one coarse
             step is advanced, and it takes every level back (a host whose
             hydro runs on the CPU);
``coupled``  as ``run`` on a tree whose hydro state is on the device too:
             FillRad with star particles before every level step, the
             injection into p, dX, E after it; or COARSERAD transport;
``stencil``  one batch of gathered ``struct RGRID`` records: the host refills
             the cells' new state, the batch is advanced in place.

States are drawn per cell from a photo-ionised medium with a lognormal
density, a share of still neutral cells (whose fronts take many chemistry
sub-steps) and point sources, in the units of the synthetic workloads.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from emma_amd import rgrid, rt, synth
from emma_amd import tree as T
from emma_amd.params import make_params

TABLES = {1: "SB99_equiv_mono_TH", 3: "Starburst99_1grpT_3grpS", 9: "Starburst99_3grpT_3grpS"}
PRECISIONS = {"fp64": rt.FP64, "mixed": rt.MIXED}
TPHY = 1e6  # years: the star particles' clock
STAR_LIFE = 1e7

# how a case is advanced: calls = level steps or coarse steps per pass, chunk
# = coarse steps per call of coarse_step (0: radsolver, the level step that
# the reference's recursion calls)
DEFAULTS = {"level": 5, "refined": "", "groups": 1, "precision": "fp64", "steps": 1, "chunk": 0, "records": 0,
            "mode": "radstep", "pinned": True, "real": 8}


def _case(path, name=None, **kw):
    c = {"path": path}
    c.update(DEFAULTS)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest: a 16^3 test box stepped level step by level step, where the latency of a call is what counts
        _case("run", "box16_mixed_g1", level=4, groups=1, precision="mixed", steps=16),
        # the Stromgren test box (32^3, one group, FP64), the host's own time loop
        _case("run", "box32_fp64_g1", level=5, groups=1, precision="fp64", steps=200),
        # the 64^3 one-group FP64 level, sub-cycles batched between outputs
        _case("run", "box64_fp64_g1", level=6, groups=1, precision="fp64", steps=192, chunk=32),
        # FP64 with three groups on a refined tree: a parity-grade AMR run
        _case("run", "amr_fp64_g3", level=6, refined="9000,2500", groups=3, precision="fp64", steps=12, chunk=4),
        # nine groups (three time groups of three): the widest atomic table, in both precisions
        _case("run", "box64_mixed_g9", level=6, groups=9, precision="mixed", steps=96, chunk=32),
        _case("run", "box32_fp64_g9", level=5, groups=9, precision="fp64", steps=64, chunk=32),
        # the 128^3 three-group mixed level, eight times its 32 sub-cycles per output
        _case("run", "box128_mixed_g3", level=7, groups=3, precision="mixed", steps=256, chunk=32),
        # the five-level tree (levels 7 to 11), its run of 40 coarse steps: the largest
        _case("run", "amr7_11_mixed_g3", level=7, refined="80000,25000,6000,1200", groups=3, precision="mixed",
              steps=40, chunk=1),
        # star particles and the hydro state on the device, a coarse step per call
        _case("coupled", "coupled_amr_mixed_g3", level=6, refined="12000,3001", groups=3, precision="mixed", steps=24,
              chunk=1),
        # the host owns the state and hands it over for every coarse step
        _case("host", "host_amr_mixed_g3", level=6, refined="12000,3001", groups=3, precision="mixed", steps=1,
              chunk=1),
        # the drop-in path, batches in page-locked memory as the host allocates them: a full one, and a short ragged
        # one in single precision
        _case("stencil", "stencil8192_fp64_g1", level=6, groups=1, records=8192),
        _case("stencil", "stencil1501_fp32_g3", level=6, groups=3, records=1501, real=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["run", "run", "run", "run", "coupled", "host", "stencil"])
    if path == "stencil":
        g = rng.choice([1, 1, 3])
        return _case("stencil", level=6, groups=g, records=_log_int(rng, 40, 8192 if g == 1 else 4096),
                     real=rng.choice([8, 8, 4]), pinned=rng.random() < 0.8)
    refined = ""
    g = rng.choice([1, 3, 3, 9])
    precision = rng.choice(["mixed", "mixed", "fp64"])
    if path == "run" and rng.random() < 0.5:
        level = rng.choice([3, 4, 5, 6] if g == 9 else [3, 4, 5, 6, 7] if precision == "mixed" else [3, 4, 5, 6])
    else:
        level = rng.choice([4, 5, 6])
        n, counts = 8 ** level, []
        for _ in range(rng.choice([1, 2, 2, 3])):
            n = max(24, int(n * rng.uniform(0.02, 0.09)))
            counts.append(str(n))
            n *= 8
        refined = ",".join(counts)
    # sub-cycles or coarse steps per output: fewer on larger levels
    cells = 8 ** level
    steps = max(4, min(160, _log_int(rng, 8, 64) * max(1, 65536 // cells)))
    if refined:
        steps = max(2, steps // 8)
    if path == "host":
        return _case("host", level=level, refined=refined, groups=g, precision=precision, steps=1, chunk=1)
    if path == "coupled":
        return _case("coupled", level=level, refined=refined, groups=rng.choice([1, 3]), precision=precision,
                     steps=steps, chunk=1, mode=rng.choice(["radstep", "coarserad"]))
    chunk = min(steps, rng.choice([1, 4]) if refined else rng.choice([0, 1, 8, 32]))
    return _case("run", level=level, refined=refined, groups=g, precision=precision,
                 steps=steps // chunk * chunk if chunk else steps, chunk=chunk)


# ---------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=2)
def _tree(level, refined):
    """The mesh of a case (a program builds it once and keeps it): a complete
    level, and refined octs clustered on a smooth random field."""
    counts = [int(x) for x in refined.split(",") if x]
    if not counts:
        return T.uniform_tree(level)
    r = np.random.default_rng(97)
    return T.amr_tree(level, counts, synth.lognormal_sampler(synth.gaussian_field(32, r), 1.0), r)


def _params(case):
    p = make_params(TABLES[case["groups"]], clight=0.1)
    p.lcoarse = case["level"]
    return p


def _fields(params, L, gen, nsrc):
    """One level's state: lognormal density, 97 % photo-ionised cells near
    1e4 K, 3 % neutral ones, photon densities over a decade and a half,
    fluxes up to half the free-streaming limit, point sources."""
    G, n = params.ngrp, L.ncell
    u = lambda lo, hi, *s: torch.rand(*s, generator=gen, dtype=torch.float64).mul_(hi - lo).add_(lo)
    nh = torch.exp(0.5 * torch.randn(n, generator=gen, dtype=torch.float64) - 0.125)
    neutral = torch.rand(n, generator=gen) < 0.03
    x = torch.where(neutral, 10.0 ** u(-4.0, -2.0, n), 1.0 - 10.0 ** u(-5.0, -2.0, n))
    temp = 10.0 ** torch.where(neutral, u(2.5, 3.5, n), u(3.9, 4.3, n))
    e = 10.0 ** u(-1.5, 0.0, G, n)
    mu, phi = u(-1.0, 1.0, G, n), u(0.0, 2.0 * math.pi, G, n)
    mag = u(0.0, 0.5, G, n) * params.cloc() * e
    sin = torch.sqrt(1.0 - mu * mu)
    nh, x, temp = nh.numpy(), x.numpy(), temp.numpy()
    F = synth.Fields(e=e.numpy(), fx=(mag * sin * torch.cos(phi)).numpy(), fy=(mag * sin * torch.sin(phi)).numpy(),
                     fz=(mag * mu).numpy(), src=np.zeros((G, n)), nhplus=x * nh,
                     eint=params.eint_code(nh, x, temp), nh=nh, temp=temp)
    leaves = np.nonzero(L.child < 0)[0]
    if nsrc and leaves.size:
        at = leaves[torch.randperm(leaves.size, generator=gen)[:nsrc].numpy()]
        lum = 10.0 ** u(48.0, 51.0, at.size).numpy()
        F.src[:, at] = params.src_code(lum, 0.5 ** L.level)[None, :]
    return F


def _inputs(case, seed):
    params, tree = _params(case), _tree(case["level"], case["refined"])
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 11)
    fields = {}
    for l in range(tree.lmin, tree.lmax + 1):
        L = tree.level(l)
        fields[l] = _fields(params, L, gen, 64 if l == tree.lmin and case["path"] != "coupled" else 0)
    return params, tree, fields, gen


def _batch(case, seed):
    """records octs of the level, gathered as the host gathers them."""
    params, tree, fields, gen = _inputs(case, seed)
    L = tree.level(case["level"])
    octs = np.sort(torch.randperm(L.noct, generator=gen)[:case["records"]].numpy())
    return params, rgrid.gather_complete(L, fields[case["level"]], octs, case["groups"], case["real"])


def _new_state(rec):
    """rfield and rfieldnew of the batch's centre cells as strided tensors
    over the records' memory."""
    real = rec["New"]["rfield"]["e"].dtype
    flat = torch.from_numpy(rec.view(real).reshape(rec.shape[0], -1))
    n = rec["New"]["rfield"].dtype.itemsize // real.itemsize
    cell = rec["New"].dtype.itemsize // real.itemsize
    base = rec.dtype.fields["New"][1] // real.itemsize
    off = [rec["New"].dtype.fields[k][1] // real.itemsize for k in ("rfield", "rfieldnew")]
    return [torch.as_strided(flat, (rec.shape[0], 8, n), (flat.shape[1], cell, 1), base + o) for o in off]


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    if c["path"] == "stencil":
        params, rec = _batch(c, seed)
        g = rt.RadGPU(params, rt.FP64)
        g.create_radstencil(c["records"], c["real"])
        if c["pinned"]:
            buf = g.pinned_stencil(c["records"], c["real"])
            buf.array[:] = rec
            rec = buf.array
        else:
            buf = None
        now, new = _new_state(rec)
        return {"case": c, "g": g, "rec": rec, "buf": buf, "now": now, "new": new, "dx": 0.5 ** c["level"],
                "dt": params.dt_rad(c["level"])}
    params, tree, fields, gen = _inputs(c, seed)
    g = rt.RadGPU(params, PRECISIONS[c["precision"]])
    s = {"case": c, "g": g, "levels": list(range(tree.lmin, tree.lmax + 1)), "dt": params.dt_rad(tree.lmin)}
    g.setup(params, tree, fields, tphy=TPHY, mode=rt.COARSERAD if c["mode"] == "coarserad" else rt.RADSTEP)
    if c["path"] == "host":
        s["fields"] = fields
        return s
    if c["path"] == "coupled":
        r = np.random.default_rng(int(seed) + 5)
        for l in s["levels"]:
            L = tree.level(l)
            g.set_hydro(l, synth.hydro_like(fields[l], r))
            stars = synth.random_stars(L, max(8, L.ncell // 512), r, params.ngrp_time, TPHY, STAR_LIFE)
            g.set_stars(l, stars)
        g.set_coupling(True)
        # about 1e49 photons/s from a particle of 1e-8 of the box's mass
        g.set_star_sources(1e49 / (1e-8 * params.unit_mass), STAR_LIFE)
    g.save_state()
    return s


# ---------------------------------------------------------------- a pass
def _arrays(F):
    return {k: getattr(F, k) for k in synth.Fields.NAMES}


def run(s):
    c, g = s["case"], s["g"]
    if c["path"] == "stencil":
        s["new"].copy_(s["now"])  # the host's gather: rfieldnew starts as rfield
        g.advance_stencil(s["rec"], c["records"], s["dx"], s["dt"])
        new = s["rec"]["New"]
        return {"rflux": new["rflux"], **{k: new["rfieldnew"][k] for k in synth.Fields.NAMES}}
    if c["path"] == "host":
        for l in s["levels"]:
            g.set(l, 0, s["fields"][l])
        g.coarse_step(1.0, 1)
        return [_arrays(g.get(l)) for l in s["levels"]]
    g.restore_state()
    if c["chunk"] == 0:
        for _ in range(c["steps"]):
            g.radsolver(c["level"], s["dt"])
    else:
        for _ in range(c["steps"] // c["chunk"]):
            g.coarse_step(1.0, c["chunk"])
    out = [_arrays(g.get(l)) for l in s["levels"]]
    if c["path"] == "coupled":
        return [out, [list(g.get_hydro(l)) for l in s["levels"]]]
    return out


# ---------------------------------------------------------------- work
def work(case):
    c = dict(DEFAULTS, **case)
    G, b = c["groups"], 8 if c["precision"] == "fp64" else 4
    # one cell-update: the closure and the three directions' fluxes, one chemistry sub-step with its rate fits
    flops = 150 * G + 40 * G + 250
    if c["path"] == "stencil":
        r, cells = c["real"], 8 * c["records"]
        # in: the centre cells and the facing cells of the six neighbours (N, F and the split flag), the new state;
        # out: the new state and the fluxes
        return {"bytes": cells * r * ((5 * G + 4) + 3 * 4 * G + 2 * (5 * G + 4) + 30 * G), "flops": cells * flops}
    tree = _tree(c["level"], c["refined"])
    done, held = 0, 0
    for l in range(tree.lmin, tree.lmax + 1):
        n = 1 if c["mode"] == "coarserad" else 1 << (l - tree.lmin)
        done += n * tree.leaf_cells(l)
        held += tree.level(l).ncell
    steps = c["steps"]
    update = (9 * G) * b + 48
    if c["path"] == "coupled":
        update += 3 * 8 + 3 * 8  # d, p, dX in, p, dX, E out
    moved = held * (5 * G + 4) * 8 * (2 if c["path"] == "host" else 1)  # the state out to the host (and in)
    return {"bytes": steps * done * update + moved, "flops": steps * done * flops}


# ---------------------------------------------------------------- 64 bits, plain torch
KB, GAMMA, PMIN, EMIN, FRAC = 1.3806e-23, 5.0 / 3.0, 1e-10, 1e-8, 0.25
HNU0 = 13.6 * 1.6022e-19


def _closure(f, e, c):
    """(c^2 E weight of the identity, of n n, and n) of Levermore's M1."""
    norm = torch.sqrt(f[0] * f[0] + f[1] * f[1] + f[2] * f[2])
    some = (e > 0) & (norm > 0)
    n = [torch.where(some, v / norm, torch.zeros_like(v)) for v in f]
    r = torch.where(e > 0, norm / (c * e), torch.zeros_like(e))
    chi = (3.0 + 4.0 * r * r) / (5.0 + 2.0 * torch.sqrt(torch.clamp(4.0 - 3.0 * r * r, min=0.0)))
    return (1.0 - chi) / 2.0 * e * c * c, (3.0 * chi - 1.0) / 2.0 * e * c * c, n


def _pressure(q, d, c, u, sign):
    """One side's share of the Lax-Friedrichs flux through a face normal to d
    (sign +1: the state on the minus side), of E and the three F."""
    diag, arg, n = q
    out = [0.5 * (u[1 + d] + sign * c * u[0])]
    for i in range(3):
        p = arg * n[i] * n[d]
        out.append(0.5 * ((p + diag if i == d else p) + sign * c * u[1 + i]))
    return out


def _rates(t):
    st, lam = torch.sqrt(t), 2.0 * 157807.0 / t
    g = 1.0 + torch.sqrt(t / 1e5)
    a1 = torch.exp(-157809.1 / t) * 2.54e-21 * st / g
    a3 = torch.exp(-118348.0 / t) * 7.5e-19 / g
    a4 = 1.42e-27 * 1.5 * st
    a6 = 3.435e-30 * t * lam ** 1.970 / (1.0 + (lam / 2.250) ** 0.376) ** 3.720
    ab = 2.753e-14 * lam ** 1.5 / (1.0 + (lam / 2.740) ** 0.407) ** 2.242 * 1e-6
    beta = 1.17e-10 * st / g * torch.exp(-157809.0 / t) * 1e-6
    return a1 + a3, a4 + a6, ab, beta


def _chemistry(p, e, fscale, src, x, eint, nh, dt):
    """Adaptive sub-steps of absorption, ionisation and heating, in place:
    e [G, n], fscale [G, n], x and eint [n], code units with a = 1."""
    dev = e.device
    col = lambda v: torch.tensor(list(v), dtype=torch.float64, device=dev)[:, None]
    ae, ai, hnu, fg = col(p.alphae), col(p.alphai), col(p.hnu), col(p.factgrp)
    heat = ae * hnu - ai * HNU0
    energy = p.unit_n * p.unit_d * p.unit_v ** 2
    total = dt * p.unit_t
    floor = PMIN / (GAMMA - 1.0) * energy
    at = torch.arange(x.numel(), device=dev)
    E, X, U, nH = e * p.unit_N, x.clone(), eint * energy, nh * p.unit_N
    S, FS = src * p.unit_N / p.unit_t * fg, torch.ones_like(e)
    t, fudge = torch.zeros_like(x), torch.full_like(x, p.fudgecool)
    while at.numel():
        temp = U / (1.5 * (1.0 + X) * nH * KB)
        cx, cr, ab, beta = _rates(temp)
        n22 = (nH * 1e-6) ** 2 * 0.1
        cool0 = (cx * X * (1.0 - X) + cr * X * X) * n22
        h0 = (heat * E).sum(0) * nH * (1.0 - X)
        d = torch.minimum(fudge * (U / (h0 - cool0)).abs(), total - t)
        w = 1.0 + ai * (1.0 - X) * nH * d
        E1 = (E + S * d) / w
        x1 = 1.0 - (ab * X * X * nH * d + (1.0 - X)) / (1.0 + d * (beta * X * nH + (ai * E1).sum(0)))
        u1 = U + d * ((heat * E1).sum(0) * nH * (1.0 - x1) - (cx * x1 * (1.0 - x1) + cr * x1 * x1) * n22)
        ok = (E1 >= 0).all(0) & (x1 >= 0) & (x1 <= 1) & (u1 >= 0) & ((u1 / U - 1.0).abs() <= FRAC)
        E = torch.where(ok, E1, E)
        FS = torch.where(ok, FS / w, FS)
        X = torch.where(ok, x1, X)
        U = torch.where(ok, torch.clamp(u1, min=floor), U)
        t = torch.where(ok, t + d, t)
        fudge = torch.where(ok, torch.full_like(fudge, p.fudgecool), fudge / 10.0)
        done = t >= total
        if done.any():
            j = at[done]
            e[:, j] = torch.maximum(E[:, done] / p.unit_N, EMIN * fg / p.unit_N)
            fscale[:, j] = FS[:, done]
            x[j], eint[j] = X[done], U[done] / energy
            on = ~done
            at, E, FS, S = at[on], E[:, on], FS[:, on], S[:, on]
            X, U, nH, t, fudge = X[on], U[on], nH[on], t[on], fudge[on]


def _temperature(p, eint, nh, x):
    return eint * (p.unit_n * p.unit_d * p.unit_v ** 2) / (1.5 * nh * p.unit_N * KB * (1.0 + x))


class _Exact:
    """RADSTEP level steps of a tree from its tables, gathers over all cells
    of a level at once."""

    def __init__(self, params, tree, fields, dev):
        self.p, self.lmin, self.c = params, tree.lmin, params.cloc()
        self.lev = []
        for l in range(tree.lmin, tree.lmax + 1):
            L, F = tree.level(l), fields[l]
            t = lambda a: torch.tensor(a, device=dev)
            u = torch.stack([t(F.e), t(F.fx), t(F.fy), t(F.fz)])
            n = L.ncell
            ic, oct_ = np.arange(n) & 7, np.arange(n) >> 3
            faces, below = [], self.lev[-1]["n"] if self.lev else 0
            for f in range(6):
                d, s = f >> 1, f & 1
                no = L.nei_oct[oct_, f].astype(np.int64)
                j = np.where(((ic >> d) & 1) != s, oct_, no) * 8 + (ic ^ (1 << d))
                out = (((ic >> d) & 1) == s) & (no < 0)
                j = np.where(out, n + (-1 - no), j)
                split = np.where(out, False, np.append(L.child, np.zeros(below, np.int32) - 1)[j] >= 0)
                faces.append((t(j), t(1.0 - split), t(np.nonzero(out)[0]), t((-1 - no)[out])))
            sp = np.nonzero(L.child >= 0)[0]
            kids = L.child[sp].astype(np.int64)[:, None] * 8 + np.arange(8)
            self.lev.append({"n": n, "l": l, "u": u, "src": t(F.src), "np": t(F.nhplus), "ei": t(F.eint),
                             "nh": t(F.nh), "te": t(F.temp), "faces": faces, "leaf": t(np.nonzero(L.child < 0)[0]),
                             "split": t(sp), "kids": t(kids), "acc": torch.zeros_like(u)})

    def step(self, k):
        A, c = self.lev[k], self.c
        B = self.lev[k - 1] if k else None
        dt = self.p.dt_rad(A["l"])
        r = dt / 0.5 ** A["l"]
        u = A["u"]
        both = torch.cat([u, B["u"]], 2) if B else u
        q = _closure(both[1:], both[0], c)
        own = (q[0][:, :A["n"]], q[1][:, :A["n"]], [v[:, :A["n"]] for v in q[2]])
        new = u + A["acc"]
        A["acc"].zero_()
        for f, (j, keep, out, cj) in enumerate(A["faces"]):
            d, s = f >> 1, f & 1
            v = both[:, :, j]
            qn = (q[0][:, j], q[1][:, j], [w[:, j] for w in q[2]])
            mine, other = _pressure(own, d, c, u, 1.0 if s else -1.0), _pressure(qn, d, c, v, -1.0 if s else 1.0)
            F = torch.stack([a + b for a, b in zip(mine, other)]) * keep * r
            new += -F if s else F
            if B and out.numel():
                B["acc"].index_add_(2, cj, F[:, :, out] * ((1.0 if s else -1.0) / 8.0))
        i = A["leaf"]
        e, x, ei, nh = new[0][:, i], A["np"][i] / A["nh"][i], A["ei"][i], A["nh"][i]
        fs = torch.ones_like(e)
        _chemistry(self.p, e, fs, A["src"][:, i], x, ei, nh, dt)
        new[0][:, i] = e
        new[1:, :, i] *= fs
        A["np"], A["ei"], A["te"] = A["np"].clone(), A["ei"].clone(), A["te"].clone()
        A["np"][i], A["ei"][i], A["te"][i] = x * nh, ei, _temperature(self.p, ei, nh, x)
        m = A["split"]
        if m.numel():
            C = self.lev[k + 1]
            mean = lambda v: v[..., A["kids"]].mean(-1)
            new[:, :, m] = mean(C["u"])
            A["src"][:, m], A["nh"][m] = mean(C["src"]), mean(C["nh"])
            A["np"][m], A["ei"][m], A["te"][m] = mean(C["np"]), mean(C["ei"]), mean(C["te"])
        A["u"] = new

    def coarse(self, k=0):
        for _ in range(1 if k == 0 else 2):
            if k + 1 < len(self.lev):
                self.coarse(k + 1)
            self.step(k)

    def out(self):
        return [{"e": A["u"][0], "fx": A["u"][1], "fy": A["u"][2], "fz": A["u"][3], "src": A["src"], "nhplus": A["np"],
                 "eint": A["ei"], "nh": A["nh"], "temp": A["te"]} for A in self.lev]


def exact(case, seed):
    c = dict(DEFAULTS, **case)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if c["path"] == "coupled":
        return None
    if c["path"] == "stencil":
        return _exact_batch(c, seed, dev)
    if work(case)["flops"] > 1.2e12:  # minutes in plain torch
        return None
    params, tree, fields, _ = _inputs(c, seed)
    X = _Exact(params, tree, fields, dev)
    for _ in range(c["steps"]):
        X.coarse()
    return X.out()


def _exact_batch(c, seed, dev):
    params, rec = _batch(c, seed)
    G, n, cl = c["groups"], c["records"], params.cloc()
    dt = params.dt_rad(c["level"])
    r = dt / 0.5 ** c["level"]
    t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
    lay = lambda a: t(np.moveaxis(a.reshape(n * a.shape[1], G), 1, 0))  # [G, octs * slots * cells]
    R = rec["oct"]["rfield"]
    u = torch.stack([t(np.moveaxis(R[k].reshape(n * 56, G), 1, 0)) for k in ("e", "fx", "fy", "fz")])
    q = _closure(u[1:], u[0], cl)
    split = rec["oct"]["split"].reshape(-1) != 0
    ic, o = np.arange(n * 8) & 7, np.arange(n * 8) >> 3
    me = torch.tensor(o * 56 + 48 + ic, device=dev)
    pick = lambda i: ((q[0][:, i], q[1][:, i], [w[:, i] for w in q[2]]), u[:, :, i])
    own, mu = pick(me)
    N = rec["New"]["rfieldnew"]
    new = torch.stack([lay(N[k]) for k in ("e", "fx", "fy", "fz")])
    flux = torch.zeros(n * 8, 6, G, 5, dtype=torch.float64, device=dev)
    for f in range(6):
        d, s = f >> 1, f & 1
        slot = np.where(((ic >> d) & 1) != s, 6, f)
        j = o * 56 + slot * 8 + (ic ^ (1 << d))
        qn, v = pick(torch.tensor(j, device=dev))
        mine, other = _pressure(own, d, cl, mu, 1.0 if s else -1.0), _pressure(qn, d, cl, v, -1.0 if s else 1.0)
        F = torch.stack([a + b for a, b in zip(mine, other)]) * t(1.0 - split[j])
        flux[:, f, :, :4] = F.permute(2, 1, 0)
        new += (-F if s else F) * r
    scalar = lambda k: t(N[k].reshape(-1))
    nh, ei = scalar("nh"), scalar("eint")
    e, x, fs = new[0].clone(), scalar("nhplus") / nh, torch.ones_like(new[0])
    _chemistry(params, e, fs, lay(N["src"]), x, ei, nh, dt)
    back = lambda a: a.movedim(0, 1).reshape(n, 8, G)
    out = {"e": back(e), "src": t(N["src"]), "nhplus": (x * nh).reshape(n, 8), "eint": ei.reshape(n, 8),
           "nh": nh.reshape(n, 8), "temp": _temperature(params, ei, nh, x).reshape(n, 8),
           "rflux": flux.reshape(n, 8, 30 * G)}
    for k, v in zip(("fx", "fy", "fz"), new[1:] * fs):
        out[k] = back(v)
    return out
