"""Performance cases of the column step and its solvers, through the package's
public entry points.

Each case stands for a call a model makes: the whole implicit column step of
a global grid or a nest domain, one routine of it, the nested outer step, the
batched column solvers on the reference's level-fastest layout, the polar ring
filter, and the host drop-in a Fortran caller reaches.  Everything is FP64
(the model's precision).  A case is a dict of plain values:

  kind "step"      one column step of a global grid (GlobalState.step) or a nest
                   domain (NestState.step, AUTO scheme); nsub O+ sub-cycles
  kind "routine"   one routine of the step on its own (a model that replaces
                   its routines one at a time)
  kind "nests"     one outer step of a global grid with two nests inside it
                   (NestedStep), replayed as one HIP graph
  kind "trsolv"    trsolv_dev, AUTO scheme: ncol scalar tridiagonal columns
  kind "blktri"    blktri2_dev / blktri3_dev: 2x2 or 3x3 block columns
  kind "filter"    ringfilter_dev: the polar rows of one field
  kind "host"      trsolv_ng on host arrays
"""
import importlib
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = "tiegcm_ng_amd"


def _pkg():
    """The package directory (its name has a dot) as module tiegcm_ng_amd."""
    if PKG not in sys.modules:
        d = os.path.join(ROOT, "tiegcm3.0_ng_amd")
        spec = importlib.util.spec_from_file_location(PKG, os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[PKG] = mod
        spec.loader.exec_module(mod)
        for sub in ("synth", "tgx", "step", "nest"):
            setattr(mod, sub, importlib.import_module(PKG + "." + sub))
    return sys.modules[PKG]


def listed():
    return [
        # the production step at the finest grid, one O+ sub-cycle
        dict(name="step 0.625 deg", kind="step", glb=True, nlon=576, nlat=288, nk=113, nsub=1),
        # the everyday 2.5 deg grid at the model's default of ten O+ sub-cycles
        dict(name="step 2.5 deg", kind="step", glb=True, nlon=144, nlat=72, nk=57, nsub=10),
        # the coarse grid: the smallest step a model takes, bound by latency
        dict(name="step 5 deg", kind="step", glb=True, nlon=72, nlat=36, nk=29, nsub=1),
        # a small nest stepped eagerly, call by call
        dict(name="step nest 100x50", kind="step", glb=False, nlon=100, nlat=50, nk=57, nsub=5),
        # one routine of a 1.25 deg model that keeps its other routines
        dict(name="dt 1.25 deg", kind="routine", routine="dt", glb=True, nlon=288, nlat=144, nk=113, nsub=1),
        # 2.5 deg grid + 0.5 deg nest (2 sub-steps) + 0.1 deg nest (5 per nest-1 step)
        dict(name="nested outer step", kind="nests", nlon=144, nlat=72, nk=57, nlon1=120, nlat1=60, nlon2=100, nlat2=50,
             nstep1=2, nstep2=5),
        # the plain scalar solve: every column of the 0.625 deg and the 5 deg grid
        dict(name="trsolv 0.625 deg", kind="trsolv", ncol=165888, nk=113),
        dict(name="trsolv 5 deg", kind="trsolv", ncol=2592, nk=29),
        # the wind solve's 2x2 rows at 1.25 deg, the O2/O/He 3x3 rows at 2.5 deg
        dict(name="blktri2 1.25 deg", kind="blktri", nblk=2, ncol=41472, nk=113),
        dict(name="blktri3 2.5 deg", kind="blktri", nblk=3, ncol=10368, nk=57),
        # the ring filter of one wind component
        dict(name="filter 0.625 deg", kind="filter", nlon=576, nlat=288, nk=113, order=3, oplus=False),
        # settei's call on a 0.5 deg nest whose arrays live on the host
        dict(name="host trsolv_ng nest", kind="host", nlond=124, nlatd=64, nk=57),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "routine", "nests", "trsolv", "trsolv", "blktri", "blktri", "filter", "host"])
    if kind in ("step", "routine"):
        glb = rng.random() < .6
        if glb:
            nlat = _logint(rng, 30, 200)
            nlon = 12 * max(5, round(nlat / 6 + rng.uniform(-2, 2)))
        else:
            nlon, nlat = _logint(rng, 20, 300), _logint(rng, 20, 150)
        case = dict(kind=kind, glb=glb, nlon=nlon, nlat=nlat, nk=rng.randint(29, 113), nsub=rng.choice([1, 1, 2, 3, 5]))
        if kind == "routine":
            case["routine"] = rng.choice(["dt", "dt", "duv", "minors", "oplus", "comp"])
        return case
    if kind == "nests":
        n = rng.randint(30, 72)
        return dict(kind=kind, nlon=2 * n, nlat=n, nk=rng.randint(29, 64), nlon1=rng.randint(30, 120),
                    nlat1=rng.randint(20, 60), nlon2=rng.randint(30, 100), nlat2=rng.randint(20, 50),
                    nstep1=rng.randint(1, 3), nstep2=rng.randint(2, 5))
    if kind == "trsolv":
        return dict(kind=kind, ncol=_logint(rng, 500, 160000), nk=rng.randint(20, 128))
    if kind == "blktri":
        return dict(kind=kind, nblk=rng.choice([2, 3]), ncol=_logint(rng, 500, 60000), nk=rng.randint(20, 113))
    if kind == "filter":
        nlat = _logint(rng, 30, 280)
        return dict(kind=kind, nlon=12 * max(5, round(nlat / 6)), nlat=nlat, nk=rng.randint(29, 113),
                    order=rng.choice([1, 3]), oplus=rng.random() < .25)
    return dict(kind=kind, nlond=_logint(rng, 24, 160), nlatd=_logint(rng, 24, 80), nk=rng.randint(29, 113))


# ---- grids and states ------------------------------------------------------------
def _chunks(nlon, nlat):
    """A ring filter table for any grid: the model's own where it has one, else
    the outermost seventh of the latitudes, coarse to fine."""
    known = _pkg().tgx.RING_CHUNKS.get((nlon, nlat))
    if known:
        return list(known)
    counts = [c for c in (3, 6, 12, nlon // 4, nlon // 2) if nlon % c == 0]
    rows = max(2, nlat // 7)
    return [counts[min(len(counts) - 1, r * len(counts) // rows)] for r in range(rows)]


def _grid(nlon, nlat, nk, nsub, glb, region=None, opdiffcap=0.):
    synth, tgx = _pkg().synth, _pkg().tgx
    name = "%dx%dx%d%s" % (nlon, nlat, nk, "" if region is None else "n")
    step = 5. * max(1., 288. / nlat)
    synth.CONFIGS[name] = (nlon, nlat, nk, 14. / (nk - 1), step, step, region)
    if glb:
        tgx.RING_CHUNKS.setdefault((nlon, nlat), _chunks(nlon, nlat))
    return synth.make_grid(name, nstep_sub=nsub, glb=glb, opdiffcap=opdiffcap)


def _case_grid(case):
    # a nest domain: 0.2 deg cells at mid latitudes
    region = None if case["glb"] else (30., 80., .2, .2)
    return _grid(case["nlon"], case["nlat"], case["nk"], case["nsub"], case["glb"], region, 0. if case["glb"] else 1e8)


def _fields(case, grid, seed, device="cuda"):
    synth = _pkg().synth
    return (synth.make_global_state if case["glb"] else synth.make_state)(grid, device=device, seed=seed)


ROUTINE_OUT = {
    "oplus": "op op_nm xiop2p xiop2d Fe Fn".split(),
    "minors": "n2d n2d_nm n4s n4s_nm no no_nm ar ar_nm".split(),
    "dt": "tn tn_nm tlbc tlbc_nm".split(),
    "duv": "un un_nm vn vn_nm ulbc vlbc ulbc_nm vlbc_nm".split(),
    "comp": "o2 o2_nm o1 o1_nm he he_nm flx_he".split(),
}


# On a global grid the top level of these holds the model's missing value 1e36.
SPVAL_TOP = "tn tn_nm un un_nm vn vn_nm".split()


def _split_top(out):
    """The missing-value level of a global field apart from the levels below
    it, which it would drown in any comparison of the whole field."""
    for n in SPVAL_TOP:
        if out.get(n) is not None:
            out[n], out[n + "_top"] = out[n][:-1], out[n][-1]
    return out


def _defined(st, names, glb):
    """The points of the outputs that a step writes: all of a nest domain, the
    interior rows of a global grid (views, nothing copied)."""
    if glb:
        return _split_top({n: st.out[n][..., 2:st.nlatd - 2, :st.nlond] for n in names})
    return {n: st.out[n][..., :st.nlond] for n in names}


# ---- column systems --------------------------------------------------------------
def _uniform(gen, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(*shape, generator=gen, dtype=torch.float64, device=gen.device)


def _scalar_system(ncol, nk, seed, device):
    """A conduction-like system: diagonally dominant rows, a Dirichlet bottom
    through the ghost row and a zero-gradient top, a temperature profile on the
    right."""
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    a, c = -_uniform(gen, .5, 2., ncol, nk), -_uniform(gen, .5, 2., ncol, nk)
    b = -(a + c) + _uniform(gen, .1, 1., ncol, nk)
    z = -7. + 14. / (nk - 1) * torch.arange(nk, dtype=torch.float64, device=device)
    f = 1000. - 800. * torch.exp(-(z + 7.) / 2.) + 5. * torch.randn(ncol, nk, generator=gen, dtype=torch.float64, device=device)
    b[:, 0] -= a[:, 0]
    f[:, 0] -= 2. * a[:, 0] * 181.
    a[:, 0] = 0.
    c[:, nk - 2] = 0.
    return a, b, c, f


def _block_system(n, ncol, nk, seed, device):
    """Block rows A, B, C (column-major blocks, as the entry points take them)
    with diffusive couplings and diagonally dominant block rows."""
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    eye = torch.eye(n, dtype=torch.float64, device=device)
    A = -eye * _uniform(gen, .5, 2., ncol, nk, 1, 1) + _uniform(gen, -.1, .1, ncol, nk, n, n)
    C = -eye * _uniform(gen, .5, 2., ncol, nk, 1, 1) + _uniform(gen, -.1, .1, ncol, nk, n, n)
    B = _uniform(gen, -.2, .2, ncol, nk, n, n)
    margin = A.abs().sum((2, 3)) + C.abs().sum((2, 3)) + B.abs().sum((2, 3))
    B = B + eye * (margin + _uniform(gen, .1, 1., ncol, nk))[..., None, None]
    F = 100. * torch.randn(ncol, nk, n, generator=gen, dtype=torch.float64, device=device)
    A[:, 0] = 0.
    C[:, nk - 2] = 0.
    return A, B, C, F


def _filter_field(case, seed, device):
    nk, nlat, nlon = case["nk"], case["nlat"], case["nlon"]
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    ld = _pkg().step.pitch(nlon + 4)
    lon = torch.arange(nlon + 4, dtype=torch.float64, device=device) * (2 * math.pi / nlon)
    f = torch.zeros(nk, nlat + 4, ld, dtype=torch.float64, device=device)
    f[..., :nlon + 4] = 40. * (torch.cos(2 * lon) + .5 * torch.sin(5 * lon + .3)) + 5. * torch.randn(
        nk, nlat + 4, nlon + 4, generator=gen, dtype=torch.float64, device=device)
    return f


# ---- the measured passes ----------------------------------------------------------
def prepare(case, seed):
    p = _pkg()
    kind = case["kind"]
    if kind in ("step", "routine"):
        grid = _case_grid(case)
        F = _fields(case, grid, seed)
        st = p.step.GlobalState(grid, F) if case["glb"] else p.step.NestState(grid, F, scheme="auto")
        if case.get("routine") == "duv":  # it reads this step's TN, Fe and Fn
            st.oplus()
            st.dt()
        return dict(kind=kind, case=case, st=st)
    if kind == "nests":
        grids = [_grid(case["nlon"], case["nlat"], case["nk"], 1, False),
                 _grid(case["nlon1"], case["nlat1"], case["nk"], 1, False, (20., 60., .5, .5), 1e8),
                 _grid(case["nlon2"], case["nlat2"], case["nk"], 1, False, (30., 80., .1, .1), 1e8)]
        doms = [(g, p.synth.make_state(g, device="cuda", seed=seed + 7919 * n)) for n, g in enumerate(grids)]
        ns = p.step.NestedStep(doms, [1, case["nstep1"], case["nstep2"]], scheme="auto", feedback=False)
        ns.capture()
        return dict(kind=kind, ns=ns)
    if kind == "trsolv":
        a, b, c, f = _scalar_system(case["ncol"], case["nk"], seed, "cuda")
        return dict(kind=kind, sys=(a, b, c, f), x=torch.zeros_like(f), k2=case["nk"] - 2)
    if kind == "blktri":
        A, B, C, F = _block_system(case["nblk"], case["ncol"], case["nk"], seed, "cuda")
        mats = tuple(m.transpose(2, 3).contiguous() for m in (A, B, C))
        return dict(kind=kind, sys=mats + (F,), x=torch.zeros_like(F), nrow=case["nk"] - 1, nblk=case["nblk"])
    if kind == "filter":
        return dict(kind=kind, f=_filter_field(case, seed, "cuda"), case=case, chunk=_chunks(case["nlon"], case["nlat"]))
    a, b, c, f = _scalar_system(case["nlond"] * case["nlatd"], case["nk"], seed, "cuda")
    shape = (case["nlatd"], case["nlond"], case["nk"])
    host = [np.ascontiguousarray(t.cpu().numpy().reshape(shape)) for t in (a, b, c, f)]
    return dict(kind=kind, sys=host, x=np.zeros(shape), k2=case["nk"] - 1)


def run(state):
    p = _pkg()
    kind = state["kind"]
    if kind == "step":
        st, glb = state["st"], state["case"]["glb"]
        st.step()
        return _defined(st, p.step.OUT_3D + p.step.OUT_2D, glb)
    if kind == "routine":
        st, case = state["st"], state["case"]
        getattr(st, case["routine"])()
        return _defined(st, ROUTINE_OUT[case["routine"]], case["glb"])
    if kind == "nests":
        ns = state["ns"]
        ns.replay()
        # the prognostic fields of both nests, the outer grid's less the n-1 levels
        names = [n for n in p.step.PROGNOSTIC if n in p.step.OUT_3D]
        return [_defined(st, [n for n in names if d or not n.endswith("_nm")], False) for d, st in enumerate(ns.states)]
    if kind == "trsolv":
        return p.tgx.trsolv_dev(*state["sys"], state["x"], 0, state["k2"])
    if kind == "blktri":
        solve = p.tgx.blktri2_dev if state["nblk"] == 2 else p.tgx.blktri3_dev
        return solve(*state["sys"], state["x"], state["nrow"])
    if kind == "filter":
        c = state["case"]
        return p.tgx.ringfilter_dev(state["f"], c["nlon"], c["nlat"], c["order"], c["oplus"], 2 * math.pi / c["nlon"],
                                    state["chunk"])
    return p.tgx.trsolv_ng(*state["sys"], state["x"], state["k2"])


# Per column and level of one step: the distinct 3-D fields read once and
# written once, and the arithmetic of the assembly and the solves (counted from
# the formulas, a division or a transcendental as one).
STEP_FLOPS = {"oplus": 350, "minors": 700, "dt": 170, "duv": 330, "comp": 900}


def work(case):
    p = _pkg()
    kind = case["kind"]

    def step(nlon, nlat, nk, nsub):
        colev = (nlon + 4) * (nlat + 4) * nk
        nf = len(p.step.IN_3D) + len(p.step.OUT_3D)
        return 8 * nf * colev, (sum(STEP_FLOPS.values()) + 60 * (nsub - 1)) * colev

    if kind == "step":
        by, fl = step(case["nlon"], case["nlat"], case["nk"], case["nsub"])
    elif kind == "routine":
        colev = (case["nlon"] + 4) * (case["nlat"] + 4) * case["nk"]
        by = p.step.alg_bytes_per_column_level(case["routine"]) * colev
        fl = STEP_FLOPS[case["routine"]] * colev
    elif kind == "nests":
        by = fl = 0
        for n, (x, y) in ((1, ("nlon", "nlat")), (case["nstep1"], ("nlon1", "nlat1")),
                          (case["nstep1"] * case["nstep2"], ("nlon2", "nlat2"))):
            b, f = step(case[x], case[y], case["nk"], 1)
            by, fl = by + n * b, fl + n * f
    elif kind == "trsolv":
        by, fl = 40 * case["ncol"] * (case["nk"] - 1), 8 * case["ncol"] * (case["nk"] - 1)
    elif kind == "blktri":
        n, rows = case["nblk"], case["ncol"] * (case["nk"] - 1)
        by, fl = 8 * (3 * n * n + 2 * n) * rows, (6 * n ** 3 + 6 * n * n) * rows
    elif kind == "filter":
        pts = 2 * len(_chunks(case["nlon"], case["nlat"])) * (case["nlon"] + 4) * case["nk"]
        by, fl = 16 * pts, (12 * case["order"] + 12) * pts
    else:
        rows = case["nlond"] * case["nlatd"] * (case["nk"] - 1)
        by, fl = 40 * rows, 8 * rows
    return {"bytes": by, "flops": fl}


# ---- the same in plain torch, 64 bits ----------------------------------------------
def _thomas(a, b, c, f):
    """Rows along the last axis."""
    n = f.shape[-1]
    w, y = [None] * n, [None] * n
    den = b[..., 0]
    y[0] = f[..., 0] / den
    for k in range(1, n):
        w[k - 1] = c[..., k - 1] / den
        den = b[..., k] - a[..., k] * w[k - 1]
        y[k] = (f[..., k] - a[..., k] * y[k - 1]) / den
    for k in range(n - 2, -1, -1):
        y[k] = y[k] - w[k] * y[k + 1]
    return torch.stack(y, -1)


def _block_thomas(A, B, C, F):
    """A, B, C (ncol, rows, n, n) row-major blocks, F (ncol, rows, n)."""
    rows = F.shape[1]
    w, y = [None] * rows, [None] * rows
    den = B[:, 0]
    for k in range(rows):
        rhs = F[:, k]
        if k:
            den = B[:, k] - A[:, k] @ w[k - 1]
            rhs = rhs - (A[:, k] @ y[k - 1][..., None])[..., 0]
        s = torch.linalg.solve(den, torch.cat([C[:, k], rhs[..., None]], -1))
        w[k], y[k] = s[..., :-1].contiguous(), s[..., -1]
    for k in range(rows - 2, -1, -1):
        y[k] = y[k] - (w[k] @ y[k + 1][..., None])[..., 0]
    return torch.stack(y, 1)


def _filter_rows(w, nchunk, order, oplus, dlamda):
    """The ring filter on rows w (..., nlon): the mean and the first harmonics
    are kept, the rest is rebuilt from its chunk averages."""
    nlon = w.shape[-1]
    ang = dlamda * torch.arange(1, nlon + 1, dtype=torch.float64, device=w.device)
    wave = w.mean(-1, keepdim=True).expand_as(w).clone()
    for m in range(1, order + 1):
        for trig in (torch.cos(m * ang), torch.sin(m * ang)):
            wave += 2. / nlon * (w * trig).sum(-1, keepdim=True) * trig
    n = nlon // nchunk
    av = (w - wave).reshape(*w.shape[:-1], nchunk, n).mean(-1)
    nb = {s: torch.roll(av, -s, -1) for s in (-2, -1, 0, 1, 2)}
    left = ((-nb[-2] + 7 * nb[-1] + 7 * nb[0] - nb[1]) / 12.)[..., None]
    right = ((-nb[-1] + 7 * nb[0] + 7 * nb[1] - nb[2]) / 12.)[..., None]
    m = torch.arange(1, n + 1, dtype=torch.float64, device=w.device)
    if oplus:
        c = nb[0][..., None]
        fine = (left + right - 2 * c) / n ** 2 * (3 * m * m - 3 * m + 1) + (3 * c - 2 * left - right) / n * (2 * m - 1) + left
    else:
        fine = (left * (n - m) + right * m) / n
    return fine.reshape(w.shape) + wave


def _filtered(f, nlon, nlat, chunk, order, oplus, dlamda):
    """The polar rows of the field (nk, nlat + 4, >= nlon + 4), their periodic
    points renewed."""
    f = f.clone()
    for r, nc in enumerate(chunk):
        for j in (r + 2, nlat + 1 - r):
            w = _filter_rows(f[:, j, 2:nlon + 2], nc, order, oplus, dlamda)
            f[:, j, :nlon + 4] = torch.cat([w[:, -2:], w, w[:, :2]], -1)
    return f


def _shift(f, s, dim):
    """f displaced by s points along dim, clamped at the ends."""
    n = f.shape[dim]
    return f.index_select(dim, torch.clamp(torch.arange(n, device=f.device) + s, 0, n - 1))


def _where_edge(n, dim, width, device):
    at = torch.arange(n, device=device)
    e = (at < width) | (at >= n - width)
    return e.view(1, -1, 1) if dim == 1 else e.view(1, 1, -1)


def _advect_1d(f, u, dim):
    """u df along dim: fourth order inside, second order on the two outermost
    points, one-sided at the ends."""
    n, dev = f.shape[dim], f.device
    end, two = _where_edge(n, dim, 1, dev), _where_edge(n, dim, 2, dev)
    d1 = _shift(f, 1, dim) - _shift(f, -1, dim)
    d1 = torch.where(end, d1, .5 * d1)
    u1 = torch.where(end, u, .5 * (_shift(u, 1, dim) + _shift(u, -1, dim)))
    d2 = .25 * (_shift(f, 2, dim) - _shift(f, -2, dim))
    u2 = .5 * (_shift(u, 2, dim) + _shift(u, -2, dim))
    return torch.where(two, d1 * u1, 4. / 3. * d1 * u1 - d2 * u2 / 3.)


def _shapiro_1d(f, s, dim):
    n, dev = f.shape[dim], f.device
    m1 = .5 * (_shift(f, 1, dim) + _shift(f, -1, dim))
    m2 = .5 * (_shift(f, 2, dim) + _shift(f, -2, dim))
    gen = f - s * (2. * m2 - 8. * m1 + 6. * f)
    near = f - s * (-8. * m1 + 8. * f)
    return torch.where(_where_edge(n, dim, 1, dev), f, torch.where(_where_edge(n, dim, 2, dev), near, gen))


def _dt(F, g):
    """The TN routine on level planes (nk, lat, lon): advection, heating and
    cooling, heat conduction solved implicitly in z."""
    re, p0, gask, grav, avo = 6.37122e8, 5e-4, 8.314e7, 870., 6.023e23
    nk, dz, dtx = g["nk"], g["dz"], g["dtx2inv"]
    dev = F["tn"].device

    def lev(name):
        return torch.tensor(g[name], dtype=torch.float64, device=dev).view(nk, 1, 1)

    def half(f):  # at the interfaces above, the top extrapolated
        return torch.cat([.5 * (f[:-1] + f[1:]), 1.5 * f[-1:] - .5 * f[-2:-1]])

    tn, un, vn, w = F["tn"], F["un"], F["vn"], F["w_upd"]
    expz, dift = lev("expz"), lev("dift")
    racs = torch.tensor(g["racs"], dtype=torch.float64, device=dev).view(1, -1, 1)
    adv = _advect_1d(tn, un, 2) * racs / g["dlamda"] + _advect_1d(tn, vn, 1) / re / g["dphi"]
    va = torch.cat([((tn[0] - F["t_lbc"]) * w[0] * 2.)[None], (tn[1:-1] - tn[:-2]) * w[1:-1], torch.zeros_like(tn[:1])])
    va = torch.cat([.5 * (va[:-1] + va[1:]), va[-1:]]) / dz
    smooth = _shapiro_1d(_shapiro_1d(F["tn_nm"], g["shapiro"], 1), g["shapiro"], 2)
    cpi = half(F["cp"])
    rhs = cpi * (adv + va - dtx * smooth) * expz

    def shear(u, low):
        s = torch.zeros_like(u)
        s[1:-2] = (u[2:-1] - u[:-3]) / (2. * dz)
        s[0] = (u[0] + u[1] / 3. - 4. / 3. * low) / dz
        s[-2] = s[-3] / 3.
        s[-1] = s[-2] / 3.
        return s

    recomb = 5.11 * 1.602e-12 * F["rkm12"] * (F["xnmbar"] * F["o1"] / 16.) ** 2 * avo / F["mbar"]
    visc = grav * half(F["km"]) / (p0 * F["scht"]) * (shear(un, F["ulbc"]) ** 2 + shear(vn, F["vlbc"]) ** 2) / expz
    rhs = rhs - (half(F["qtotal"]) + F["hdt"] + recomb + F["qji_tn"] + visc) * expz
    tni = torch.cat([F["tlbc"][None], .5 * (tn[:-2] + tn[1:-1]), tn[-2:-1]])
    h = F["schti"]
    rho = p0 * g["expzmid_inv"] / (h * grav) * expz
    gg = grav * (F["kt"] + h * h * rho * F["cp"] * dift) / (p0 * h * dz * dz)
    ff = grav * grav * h * h * rho / (tni * p0 * 2. * dz) * dift
    p = gg - ff
    q = torch.cat([-(gg[1:] - ff[1:] + gg[:-1] + ff[:-1]), -gg[-1:] - ff[-1:]])
    q[-2] = -gg[-2] - ff[-2]
    r = torch.cat([gg[1:] + ff[1:], torch.zeros_like(gg[:1])])
    r[-2] = 0.
    rhs = rhs + F["cool_exp"]
    q = q - (cpi * (dtx + F["cool_imp"]) + half(w) * gask / F["mbar"]) * expz
    q[0] -= p[0]
    rhs[0] -= 2. * p[0] * F["t_lbc"]
    p[0] = 0.
    sol = _thomas(*(t[:-1].movedim(0, -1) for t in (p, q, r, rhs))).movedim(-1, 0)
    top = sol[-1:] ** 2 / sol[-2:-1]
    new = torch.cat([sol, top])
    if g["glb"]:
        new = _filtered(new, g["nlon"], g["nlat"], g["chunk"], 3, False, g["dlamda"])
    else:
        new[:, :, 0], new[:, :, -1] = F["lonb_tn"][:, 0], F["lonb_tn"][:, 1]
        new[:, 0], new[:, -1] = F["latb_tn"][:, 0], F["latb_tn"][:, 1]
    old = .025 * (F["tn_nm"] + new) + .95 * tn
    new = torch.clamp(new, min=100.)
    if g["glb"]:
        nlon = g["nlon"]
        new[-1], old[-1] = 1e36, 1e36
        for t in (new, old):
            t[..., :2], t[..., nlon + 2:] = t[..., nlon:nlon + 2].clone(), t[..., 2:4].clone()
    out = dict(tn=new, tn_nm=old, tlbc=F["t_lbc"], tlbc_nm=F["tlbc"])
    return {n: t[..., 2:-2, :] for n, t in out.items()} if g["glb"] else out


def exact(case, seed):
    """The solvers and the filter on their whole range; of a step the TN part,
    which depends on no other routine's result.  The other routines are the
    model's chemistry and transport at length, None here."""
    p = _pkg()
    kind = case["kind"]
    if kind in ("step", "routine"):
        names = ROUTINE_OUT[case["routine"]] if kind == "routine" else p.step.OUT_3D + p.step.OUT_2D
        if kind == "routine" and case["routine"] != "dt":
            return None
        grid = _case_grid(case)
        got = _dt(_fields(case, grid, seed), grid)
        return _split_top({n: got.get(n) for n in names}) if case["glb"] else {n: got.get(n) for n in names}
    if kind == "nests":
        return None
    if kind == "trsolv":
        k = case["nk"] - 1
        a, b, c, f = _scalar_system(case["ncol"], case["nk"], seed, "cuda")
        x = torch.zeros_like(f)
        x[:, :k] = _thomas(*(t[:, :k] for t in (a, b, c, f)))
        return x
    if kind == "blktri":
        A, B, C, F = _block_system(case["nblk"], case["ncol"], case["nk"], seed, "cuda")
        k = case["nk"] - 1
        x = torch.zeros_like(F)
        x[:, :k] = _block_thomas(*(t[:, :k] for t in (A, B, C, F)))
        return x
    if kind == "filter":
        return _filtered(_filter_field(case, seed, "cuda"), case["nlon"], case["nlat"], _chunks(case["nlon"], case["nlat"]),
                         case["order"], case["oplus"], 2 * math.pi / case["nlon"])
    k = case["nk"] - 1
    a, b, c, f = _scalar_system(case["nlond"] * case["nlatd"], case["nk"], seed, "cuda")
    x = torch.zeros_like(f)
    x[:, :k] = _thomas(*(t[:, :k] for t in (a, b, c, f)))
    return x.reshape(case["nlatd"], case["nlond"], case["nk"]).cpu().numpy()
