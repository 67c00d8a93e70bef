"""The performance cases of the framework: what a program that uses it has it do.

A simulation program calls `tschem` in a time loop and pulls the fields it
writes out into arrays of its own every so many steps, so a pass of most cases
is a run of time steps followed by one output (u, v, w, T, p, the surface's
vertices and the body's log row).  Its arrays are pinned and kept, as such a
program keeps its module arrays; the precision form's values are kept as
float32, which is all they hold.  Every state continues from pass to pass; the Stefan numbers of the small
grids, whose passes are short and many, are low enough that the body lasts.

Kinds:
  melt      a melting, moving body in a periodic box: time loop and output
  fluid     the same without a body (a turbulence precursor run)
  routines  the fluid substep through the routine-by-routine drop-in calls
  ibm       the immersed-boundary calls alone: tagCells and particle
  ensemble  independent simulations of uneven grids advanced together
  diag      the diagnostics of the time loop: cfl, get_dt, divgck, dissipation
  divgck    the allocation-free divergence check on the caller's device arrays
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from melt_ibm_amd import geometry
from melt_ibm_amd.api import FIELD_ID, MeltConfig, MeltContext, load_library
from melt_ibm_amd.ensemble import Ensemble, Member

OUT = ("vx", "vy", "vz", "temp", "pr")
BOX = 2.0 * math.pi
HIT = (0.5, 0.05, 2.5)   # TL, EPSSTAR, KF/KMIN of the benchmark's forcing
CFL = 0.5


def listed():
    return [
        # a monitor inside someone else's loop: one divergence check of a small box, bound by its launches
        dict(name="divgck_64", kind="divgck", n=64, n3=64, f32=False, re=1000.0),
        # the log line of a run (diss.txt and the CFL control) at the benchmark's grid
        dict(name="diag_256", kind="diag", n=256, n3=256, f32=False, re=1000.0),
        # a driver that keeps its own substep and calls the drop-in routines one by one
        dict(name="routines_128", kind="routines", n=128, n3=96, f32=False, steps=3, re=400.0),
        # a turbulence precursor in the precision form, on a grid that is no power of two
        dict(name="fluid_f32_192", kind="fluid", n=192, n3=192, f32=True, steps=30, hit=False, re=800.0),
        # the CPU-runnable reference case: 64^3, 1280 faces; bound by launches
        dict(name="melt_64", kind="melt", n=64, n3=64, f32=False, steps=20, hit=False, graph=False, remesh=False,
             rad=0.6, freq=8, aspect=1.0, st=0.02, re=500.0),
        # a parameter-sweep member at 128^3 in the precision form, the step replayed as a graph
        dict(name="melt_f32_128_graph", kind="melt", n=128, n3=128, f32=True, steps=40, hit=False, graph=True, remesh=False,
             rad=0.6, freq=16, aspect=1.0, st=0.05, re=500.0),
        # the benchmark's workload in FP64, under the reference's CFL control
        dict(name="melt_256_hit", kind="melt", n=256, n3=256, f32=False, steps=10, hit=True, graph=False, remesh=False,
             rad=0.5, freq=32, aspect=1.0, st=0.5, re=1000.0),
        # the same in the precision form
        dict(name="melt_f32_256_hit", kind="melt", n=256, n3=256, f32=True, steps=30, hit=True, graph=False, remesh=False,
             rad=0.5, freq=32, aspect=1.0, st=0.5, re=1000.0),
        # the largest grid of the request stream: a melting spheroid with remeshing
        dict(name="melt_384_remesh", kind="melt", n=384, n3=384, f32=False, steps=4, hit=False, graph=False, remesh=True,
             rad=0.55, freq=44, aspect=2.0, st=0.5, re=800.0),
        # the immersed boundary alone, as a driver with a solver of its own calls it
        dict(name="ibm_128", kind="ibm", n=128, n3=128, f32=False, steps=2, rad=1.0, freq=32, st=0.05, re=800.0),
        # a batch of small simulations of uneven grids on one GPU
        dict(name="ensemble_6", kind="ensemble", grids="48,64,96,128,64,96", steps=4, rad=0.55, st=0.1, re=600.0),
    ]


# Grid sizes the library takes (2^a and 3 2^a, the horizontal sides equal) up to the largest listed.
SIZES = (32, 48, 64, 96, 128, 192, 256, 384)


def draw(rng):
    kind = rng.choice(("divgck", "diag", "routines", "fluid", "melt", "melt", "melt", "melt", "ibm", "ensemble"))
    re = round(math.exp(rng.uniform(math.log(200.0), math.log(1000.0))), 1)
    st = rng.uniform(0.5, 1.5)
    if kind == "ensemble":
        return dict(kind=kind, grids=",".join(str(rng.choice((48, 64, 96, 128))) for _ in range(rng.randint(3, 7))), steps=rng.randint(2, 4),
                    rad=round(rng.uniform(0.45, 0.65), 3), st=round(0.05 * st, 4), re=re)
    top = {"divgck": 384, "diag": 384, "routines": 192, "fluid": 256, "melt": 256, "ibm": 256}[kind]
    n = rng.choice([s for s in SIZES if s <= top])
    n3 = n if rng.random() < 0.6 else rng.choice([s for s in SIZES if n // 2 <= s <= min(2 * n, top)])
    case = dict(kind=kind, n=n, n3=n3, f32=rng.random() < 0.5, re=re)
    cells = n * n * n3
    if kind in ("routines", "fluid", "melt"):
        case["steps"] = rng.randint(2, 4) if cells > 8_000_000 else rng.randint(4, 16)
    if kind in ("fluid", "melt"):
        case["hit"] = rng.random() < 0.4
    if kind == "ibm":
        case["steps"] = rng.randint(1, 2)
    if kind in ("melt", "ibm"):
        # a body of radius 6 h to 30 h, its mean edge between 0.6 h and 1 h, inside the box
        h = BOX / n
        rad = min(1.2, h * math.exp(rng.uniform(math.log(6.0), math.log(30.0))), 0.18 * BOX * n3 / n)
        case.update(rad=round(rad, 4), freq=max(6, min(55, round(1.1 * rad / (h * rng.uniform(0.6, 1.0))))),
                    st=round((0.5 if kind == "melt" else 0.2) * st * (n / 256) ** 2, 5))
    if kind == "melt":
        case.update(aspect=1.0 if rng.random() < 0.6 else round(rng.uniform(1.0, 2.0), 2), remesh=rng.random() < 0.3)
        case["graph"] = not case["hit"] and not case["remesh"] and rng.random() < 0.4
    return case


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _modes(case, gen, kmax):
    """A smooth periodic field: random phases in |k| <= kmax, amplitude 1/|k|^2, of the case's shape [k, j, i]."""
    n3, n2, n1 = case["n3"], case["n"], case["n"]
    f = lambda n: torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device="cuda")  # noqa: E731
    kk = torch.sqrt(f(n3)[:, None, None] ** 2 + f(n2)[None, :, None] ** 2 + torch.arange(n1 // 2 + 1, dtype=torch.float64, device="cuda")[None, None, :] ** 2)
    amp = torch.where((kk <= kmax) & (kk > 0), 1.0 / kk.clamp(min=1.0) ** 2, torch.zeros_like(kk))
    phase = torch.rand(kk.shape, generator=gen, dtype=torch.float64, device="cuda") * (2.0 * math.pi)
    return torch.fft.irfftn(torch.polar(amp, phase), s=(n3, n2, n1), dim=(0, 1, 2))


def _widths(case):
    """1/dx of the three directions (cubic cells: the box is as deep as its planes)."""
    d = case["n"] / BOX
    return d, d, d


def _up(a, axis):
    return torch.roll(a, -1, dims=2 - axis)


def _down(a, axis):
    return torch.roll(a, 1, dims=2 - axis)


def _solenoidal(case, gen, kmax, rms):
    """Staggered components, free of divergence in the discrete sense: the curl of a smooth potential."""
    d = _widths(case)
    a = [_modes(case, gen, kmax) for _ in range(3)]
    fwd = lambda q, ax: (_up(q, ax) - q) * d[ax]  # noqa: E731
    c = [fwd(a[2], 1) - fwd(a[1], 2), fwd(a[0], 2) - fwd(a[2], 0), fwd(a[1], 0) - fwd(a[0], 1)]
    s = rms / torch.sqrt(sum((q * q).mean() for q in c) / 3.0)
    return [(q * s).contiguous() for q in c]


def _inputs(case, seed):
    """Velocity (rms 0.1), a temperature in [0, 1] and a low-mode body force, as the precision stores them."""
    gen = _gen(seed)
    vel = _solenoidal(case, gen, 4.0, 0.1)
    t = _modes(case, gen, 6.0)
    t = 0.5 + 0.5 * t / t.abs().max()
    force = _solenoidal(case, gen, 2.5, 0.05)
    out = dict(zip(("vx", "vy", "vz", "temp", "forcx", "forcy", "forcz"), (*vel, t, *force)))
    return {k: v.float().double() if case["f32"] else v.contiguous() for k, v in out.items()}


def _provisional(case, f):
    """A velocity field before its projection: not free of divergence."""
    v = {q: f[q] * (1.0 + 0.2 * f["temp"]) for q in ("vx", "vy", "vz")}
    return {q: a.float().double() if case["f32"] else a for q, a in v.items()}


def _first_dt(case, f):
    d = _widths(case)
    c = (f["vx"].abs() * d[0] + f["vy"].abs() * d[1] + f["vz"].abs() * d[2]).max().item()
    return CFL / max(c, 6.0 / case["re"] * d[0] ** 2)


# ------------------------------------------------------------------ states
@functools.lru_cache(maxsize=8)
def _mesh(freq, aspect):
    """The surface a program reads from its file: unit volume-equivalent radius."""
    if aspect == 1.0:
        return geometry.icosphere(freq)
    a = aspect ** (-1.0 / 3.0)
    return geometry.spheroid(a, aspect * a, freq)


def _config(case):
    body = case["kind"] in ("melt", "ibm")
    cfg = MeltConfig(n1m=case["n"], n2m=case["n"], n3m=case["n3"], zlen=BOX * case["n3"] / case["n"], ren=case["re"], latheat=1.0 / case.get("st", 1.0),
                     precision=int(case["f32"]), imlsfor=int(body), imlsstr=int(body), imelt=int(body), iremesh=int(case.get("remesh", False)),
                     forcing=int(case.get("hit", False)))
    if cfg.iremesh:
        # the deck's 0.7 h, or a little under the shortest edge of a finer mesh
        m = _mesh(case["freq"], case["aspect"])
        e = m.xyz[m.vert_of_edge[:, 0] - 1] - m.xyz[m.vert_of_edge[:, 1] - 1]
        cfg.perc_ethresh = min(0.7, 0.95 * float(np.sqrt((e * e).sum(axis=1)).min()) * case["rad"] * case["n"] / BOX)
    return cfg


class _State:
    pass


def _host_arrays(s, shape, f32):
    """The program's own arrays: pinned, allocated once."""
    s.host = {q: torch.empty(shape, dtype=torch.float64, pin_memory=True) for q in OUT}
    s.host32 = {q: torch.empty(shape, dtype=torch.float32) for q in OUT} if f32 else None


def _pull(ctx, s):
    """melt_download_field of the output fields into the program's arrays, as a C or Fortran caller pulls them."""
    for q in OUT:
        rc = ctx.lib.melt_download_field(ctx._ctx, FIELD_ID[q], C.c_void_p(s.host[q].data_ptr()), None)
        if rc:
            raise RuntimeError("download of %s: status %d" % (q, rc))
    if s.host32 is None:
        return dict(s.host)
    for q in OUT:
        s.host32[q].copy_(s.host[q])
    return dict(s.host32)


def _log_row(ctx):
    b = ctx.body()
    return np.array([*b.pos_cm[:], *b.vel_cm[:], *b.omega_c[:], b.volume, b.surface])


def prepare(case, seed):
    s = _State()
    s.case = case
    kind = case["kind"]
    if kind == "ensemble":
        grids = [int(g) for g in case["grids"].split(",")]
        members = [Member(n=g, rad=case["rad"] + 0.02 * i, st=case["st"], re=case["re"], seed=int(seed) * 64 + i, level=3 if g <= 64 else 4)
                   for i, g in enumerate(grids)]
        s.ens = Ensemble(members, precision=1, tune=False)
        s.out = []
        for m in members:
            o = _State()
            _host_arrays(o, (m.n, m.n, m.n), True)
            s.out.append(o)
        return s
    f = _inputs(case, seed)
    torch.cuda.synchronize()
    if kind == "divgck":
        s.vel = [a.float() if case["f32"] else a for a in _provisional(case, f).values()]
        s.out = torch.zeros(1, dtype=torch.float64, device="cuda")
        s.lib = load_library()
        torch.cuda.synchronize()
        return s
    s.ctx = ctx = MeltContext(_config(case))
    if kind in ("melt", "ibm"):
        m = _mesh(case["freq"], case.get("aspect", 1.0))
        ctx.set_geometry(m.xyz, m.vert_of_edge, m.edge_of_face, case["rad"])
        ctx.inqpr()
        for q in ("vx", "vy", "vz"):
            ctx.upload_device(q, f[q].data_ptr())
    else:
        if kind == "diag":
            f.update(_provisional(case, f))
            torch.cuda.synchronize()
        for q, a in f.items():
            ctx.upload_device(q, a.data_ptr())
    ctx.set_dt(_first_dt(case, f))
    if kind in ("melt", "ibm"):
        if case.get("hit"):
            ctx.hit_init(*HIT, seed=int(seed))
        ctx.set_tuning(pbuf=4 * case["n"])   # room for a mesh finer than the grid in the first, ray-cast tagging
        ctx.tagCells()
        if case.get("graph"):
            ctx.graph(True)
    if kind == "fluid" and case["hit"]:
        ctx.hit_init(*HIT, seed=int(seed))
    ctx.sync()
    if kind != "diag":
        _host_arrays(s, ctx.cfg.shape, case["f32"])
    return s


# ------------------------------------------------------------------ passes
def _advance(ctx, steps, hit):
    for _ in range(steps):
        if hit:   # forced runs gain energy: the time step follows the CFL number
            ctx.set_dt(ctx.get_dt(CFL))
            ctx.hit_force()
        ctx.tschem()


def _routines(ctx, steps):
    for _ in range(steps):
        for ns in (1, 2, 3):
            ctx.set_stage(ns)
            ctx.hdnl1(); ctx.hdnl2(); ctx.hdnl3(); ctx.hdnlte()  # noqa: E702
            ctx.invtr1(); ctx.invtr2(); ctx.invtr3(); ctx.invtrte()  # noqa: E702
            ctx.divg(); ctx.phcalc(); ctx.updvp(); ctx.prcalc()  # noqa: E702


def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "divgck":
        v = state.vel
        rc = state.lib.melt_divgck_noalloc(*(C.c_void_p(a.data_ptr()) for a in v), case["n"], case["n"], case["n3"], C.c_double(BOX), C.c_double(BOX),
                                           C.c_double(BOX * case["n3"] / case["n"]), v[0].element_size(),
                                           C.c_void_p(torch.cuda.current_stream().cuda_stream), C.c_void_p(state.out.data_ptr()))
        if rc:
            raise RuntimeError("melt_divgck_noalloc: status %d" % rc)
        return state.out
    if kind == "ensemble":
        for _ in range(case["steps"]):
            state.ens.step()
        return [dict(_pull(sim.ctx, o), xyzv=sim.ctx.lag("xyzv")) for sim, o in zip(state.ens.sims, state.out)]
    ctx = state.ctx
    if kind == "diag":
        d = ctx.dissipation()
        return dict(cfl=ctx.cfl(), dt=ctx.get_dt(CFL), div=ctx.divgck(), diss=np.array([d[k] for k in ctx.DISS_KEYS]))
    if kind == "routines":
        _routines(ctx, case["steps"])
        return _pull(ctx, state)
    if kind == "ibm":
        for _ in range(case["steps"]):
            for ns in (1, 2, 3):
                ctx.set_stage(ns)
                ctx.tagCells()
                ctx.particle()
        ctx.sync()
        return dict(_pull(ctx, state), **{k: ctx.lag(k) for k in ("xyzv", "vel_tri", "qw_o", "qw_i", "sur", "tri_nor")}, body=_log_row(ctx))
    _advance(ctx, case["steps"], case["hit"])
    ctx.sync()
    if kind == "fluid":
        return _pull(ctx, state)
    return dict(_pull(ctx, state), xyzv=ctx.lag("xyzv"), body=_log_row(ctx))


# ------------------------------------------------------------------ work
def work(case):
    """Per cell and substep: u, v, w, T, p and the four old explicit terms are read and written, the three forces and the
    volume fraction read (22 values); about 300 operations of the stencils and solves and 4 transform visits of 5 log2 N a
    value pair.  Per face and substep: four shape functions, two spreads and seven probes, about 30 kFLOP, and 2 KB of
    surface data and support values.  The output is written once."""
    kind = case["kind"]
    if kind == "ensemble":
        tot = {"bytes": 0.0, "flops": 0.0}
        for g in (int(x) for x in case["grids"].split(",")):
            w = work(dict(kind="melt", n=g, n3=g, f32=True, steps=case["steps"], freq=8 if g <= 64 else 16))
            tot = {k: tot[k] + w[k] for k in tot}
        return tot
    cells, e = float(case["n"]) ** 2 * case["n3"], 4 if case["f32"] else 8
    if kind == "divgck":
        return {"bytes": 3 * e * cells + 8, "flops": 9 * cells}
    if kind == "diag":   # dissipation reads u, v, w, T, VOFp; the three maxima u, v, w
        return {"bytes": (5 + 3 * 3) * e * cells, "flops": 110 * cells}
    subs = 3 * case["steps"]
    out = len(OUT) * e * cells
    face = 20.0 * case.get("freq", 0) ** 2
    if kind == "ibm":   # the surface and the cells near it; the mean force is taken off u, v, w everywhere
        return {"bytes": subs * (2048 * face + 6 * e * cells) + out, "flops": subs * (30e3 * face + 3 * cells)}
    fft = 5.0 * math.log2(cells)
    return {"bytes": subs * (22 * e * cells + 2048 * face) + out, "flops": subs * ((300 + fft) * cells + 30e3 * face)}


# ------------------------------------------------------------------ exact values
def _lap(q, d):
    return sum((_up(q, a) - 2.0 * q + _down(q, a)) * d[a] ** 2 for a in range(3))


def _eigen(case):
    """2 (1 - cos) of the second difference along each axis, broadcast over the half spectrum [k, j, i]."""
    n3, n = case["n3"], case["n"]
    lam = lambda m, c: 2.0 * (1.0 - torch.cos(2.0 * math.pi * torch.arange(c, dtype=torch.float64, device="cuda") / m))  # noqa: E731
    return lam(n, n // 2 + 1)[None, None, :], lam(n, n)[None, :, None], lam(n3, n3)[:, None, None]


def _exact_fluid(case, f, steps):
    """The RK3 scheme of the fluid (advection, Crank-Nicolson diffusion in factored form, projection) in float64."""
    d, lam = _widths(case), _eigen(case)
    q = [f[k].clone() for k in ("vx", "vy", "vz", "temp")]
    force, length = [f[k] for k in ("forcx", "forcy", "forcz")], (BOX, BOX, BOX * case["n3"] / case["n"])
    p = torch.zeros_like(q[0])
    ru = [torch.zeros_like(p) for _ in range(4)]
    dt, re = _first_dt(case, f), case["re"]
    shape = q[0].shape
    lap = sum(lam[a] * d[a] ** 2 for a in range(3))
    for _ in range(steps):
        for ga, ro in ((8.0 / 15.0, 0.0), (5.0 / 12.0, -17.0 / 60.0), (3.0 / 4.0, -5.0 / 12.0)):
            al = ga + ro
            h = []
            for c in range(3):
                s = torch.zeros_like(p)
                for a in range(3):
                    if a == c:
                        m = (_up(q[c], c) + q[c]) ** 2
                        s -= (m - _down(m, c)) * (0.25 * d[c])
                    else:   # velocity a on the edge below cell c, times velocity c on it
                        m = (q[a] + _down(q[a], c)) * (q[c] + _down(q[c], a))
                        s -= (_up(m, a) - m) * (0.25 * d[a])
                h.append(s + force[c] / length[c])
            s = torch.zeros_like(p)
            for a in range(3):
                m = q[a] * (q[3] + _down(q[3], a))
                s -= (_up(m, a) - m) * (0.5 * d[a])
            h.append(s)
            new = []
            for c in range(4):
                nu = 1.0 / re   # the Prandtl number is 1
                r = ga * h[c] + ro * ru[c] + al * nu * _lap(q[c], d)
                if c < 3:
                    r -= (p - _down(p, c)) * (d[c] * al)
                g = [0.5 * dt * nu * al * d[a] ** 2 for a in range(3)]
                fac = (1.0 + g[0] * lam[0]) * (1.0 + g[1] * lam[1]) * (1.0 + g[2] * lam[2])
                new.append(q[c] + torch.fft.irfftn(torch.fft.rfftn(r * dt) / fac, s=shape))
            q, ru = new, h
            div = sum((_up(q[a], a) - q[a]) * d[a] for a in range(3)) / (dt * al)
            ev = -lap.clone()
            ev[0, 0, 0] = 1.0
            spec = torch.fft.rfftn(div) / ev
            spec[0, 0, 0] = 0.0
            phi = torch.fft.irfftn(spec, s=shape)
            for a in range(3):
                q[a] = q[a] - (phi - _down(phi, a)) * (al * dt * d[a])
            p = p + phi - (al * 0.5 * dt / re) * _lap(phi, d)
    return dict(zip(OUT, (*q, p)))


def _max_div(case, v):
    d = _widths(case)
    return sum((_up(v[a], a) - v[a]) * d[a] for a in range(3)).abs().max().item()


def _exact_diag(case, f):
    d, re = _widths(case), case["re"]
    f = {**f, **_provisional(case, f)}
    u = [f[k] for k in ("vx", "vy", "vz")]
    # one-sided normal gradients, centred cross gradients of the two faces' sum
    grad = [[None] * 3 for _ in range(3)]
    for c in range(3):
        for a in range(3):
            if a == c:
                grad[c][a] = (_up(u[c], c) - u[c]) * d[c]
            elif (c, a) == (1, 0):   # as the diagnostic has them: the outer corner is taken on each side
                grad[c][a] = ((_up(u[1], 0) + _up(_up(u[1], 0), 1)) - (_down(u[1], 0) + _up(_down(u[1], 0), 1))) * (0.25 * d[0])
            else:
                w = u[c] + _up(u[c], c)
                grad[c][a] = (_up(w, a) - _down(w, a)) * (0.25 * d[a])
    tke = sum((u[c] ** 2 + _up(u[c], c) ** 2) for c in range(3)) * 0.25
    dis = sum(grad[c][c] ** 2 for c in range(3)) + 0.5 * ((grad[1][0] + grad[0][1]) ** 2 + (grad[2][0] + grad[0][2]) ** 2 + (grad[2][1] + grad[1][2]) ** 2)
    t = f["temp"]
    chi = sum((0.5 * d[a] * (_up(t, a) - _down(t, a))) ** 2 for a in range(3)) / re
    ken, eps, chi, nu = tke.mean().item(), (dis * 2.0 / re).mean().item(), chi.mean().item(), 1.0 / re
    rms = math.sqrt(2.0 / 3.0 * ken)
    eta, lam = (nu ** 3 / eps) ** 0.25, math.sqrt(15.0 * nu * rms ** 2 / eps)
    row = [eps, ken, rms, eta, lam, ken ** 2 / (nu * eps), rms * lam / nu, ken ** 1.5 / eps, chi, math.pi * d[0] * eta, float(t.numel())]
    mid = sum(((u[a] + _up(u[a], a)) * 0.5 * d[a]).abs() for a in range(3)).max().item()
    adv = sum(u[a].abs() * d[a] for a in range(3)).max().item()
    return dict(cfl=mid, dt=CFL / max(adv, 6.0 / re * d[0] ** 2), div=_max_div(case, u), diss=np.array(row))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("melt", "ibm", "ensemble") or case.get("hit"):
        return None   # the melting body's geometry, or the random forcing
    f = _inputs(case, seed)
    if kind == "divgck":
        return torch.tensor([_max_div(case, list(_provisional(case, f).values()))], dtype=torch.float64)
    if kind == "diag":
        return _exact_diag(case, f)
    return _exact_fluid(case, f, case["steps"])
