"""The work a simulation has this library do, as cases that can be timed.

A case is one stretch of a run between two outputs: some time steps on a state
resident in HBM, then the state (and the dt and conservation sums that the
steps return) handed to the host, as a program that writes snapshots does it.
Each state lives in a library context of its own (rh_ctx_*).

Kinds (case["kind"]):
  level   a uniform periodic 3D box stepped on the device (UniformLevel.run_device)
  tube    a 1D shock tube with outflow boundaries, stepped on the device
  calls   a uniform box through the reference's calls per step (UniformLevel.step:
          rh_cmpdt, rh_set_unew, rh_godunov, rh_set_uold)
  amr     a refined mesh, all levels batched (AmrHierarchy.run_device)
  amrcalls  the same kind of mesh through the reference's calls per level
          (AmrHierarchy.step: rh_cmpdt, rh_set_unew, rh_godunov, rh_set_uold, rh_upload)
  serve   independent jobs of differing sizes advanced together (HipEngine.step)
  flags   the refinement criterion on every level of a refined mesh (HipHydro.hydro_flag)
"""
import ctypes
import functools
import math

import numpy as np
import torch

from ramses2_amd import HydroParams, UniformLevel, UniformMesh, _lib
from ramses2_amd.amr_build import amr_state, build_levels, sedov_profile
from ramses2_amd.hydro import AmrHierarchy, HipHydro
from ramses2_amd.mesh import AmrMesh
from ramses2_amd.serving import HipEngine, job_ic, make_stream

DEV = "cuda"


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest run: the 1024-cell Sod-like tube, where launches are the cost
        dict(name="tube1024", kind="tube", n=1024, steps=100, slope=1, riemann="hllc"),
        # the smallest job size of an ensemble, alone on the device
        dict(name="box32", kind="level", n=32, ic="blast", precision=0, slope=2, riemann="hllc", brick="8,6,8",
             steps=100),
        # an odd number of octs per dimension (no brick shape divides it), with the
        # namelist's default slope and solver (MinMod, LLF)
        dict(name="box90_llf", kind="level", n=90, ic="turbulence", precision=0, slope=1, riemann="llf",
             brick="8,6,8", steps=50),
        # the uniform Sedov blast of 128^3 cells
        dict(name="sedov128", kind="level", n=128, ic="blast", precision=0, slope=2, riemann="hllc", brick="8,6,8",
             steps=100),
        # supersonic turbulence at 256^3, the headline size, in both precisions
        dict(name="turb256", kind="level", n=256, ic="turbulence", precision=0, slope=2, riemann="hllc",
             brick="8,6,16", steps=50),
        dict(name="turb256_mixed", kind="level", n=256, ic="turbulence", precision=1, slope=2, riemann="hllc",
             brick="8,6,16", steps=50),
        # a host code that drives each step through the drop-in calls
        dict(name="calls128", kind="calls", n=128, ic="blast", precision=0, slope=2, riemann="hllc", brick="8,6,8",
             steps=20),
        # the Sedov shell on levels 6-10 and a smaller one in mixed precision, batched
        dict(name="amr6_10", kind="amr", lmin=6, lmax=10, radius=0.3, precision=0, brick="4,4,8", steps=40),
        dict(name="amr5_8_mixed", kind="amr", lmin=5, lmax=8, radius=0.25, precision=1, brick="4,4,4", steps=40),
        # the refined mesh of a host code that calls level by level
        dict(name="amrcalls5_8", kind="amrcalls", lmin=5, lmax=8, radius=0.3, precision=0, brick="4,4,8", steps=10),
        # a dozen resident jobs of 32^3 to 128^3 cells, the load of an ensemble server
        dict(name="serve12", kind="serve", jobs=12, nmin=32, nmax=128, precision=0, brick="8,6,8", steps=100),
        # the refinement criterion before a refine step
        dict(name="flags5_9", kind="flags", lmin=5, lmax=9, radius=0.3),
    ]


PHYSICS = [(2, "hllc"), (2, "hllc"), (1, "hllc"), (1, "llf"), (2, "hll")]
BRICKS = ["8,6,8", "8,6,16", "4,4,8", "7,7,8"]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["level", "level", "level", "tube", "calls", "amr", "amr", "amrcalls", "serve", "flags"])
    slope, riemann = rng.choice(PHYSICS)
    if kind == "tube":
        return dict(kind=kind, n=2 * _log_int(rng, 32, 4096), steps=rng.randint(20, 100), slope=slope,
                    riemann=riemann)
    if kind in ("level", "calls"):
        n = 2 * _log_int(rng, 8, 120 if kind == "level" else 80)
        steps = max(2, min(100, int(4e8 / n ** 3)))
        return dict(kind=kind, n=n, ic=rng.choice(["blast", "turbulence"]), precision=rng.choice([0, 0, 1]),
                    slope=slope, riemann=riemann, brick=rng.choice(BRICKS),
                    steps=steps if kind == "level" else max(2, steps // 5))
    if kind == "serve":
        return dict(kind=kind, jobs=rng.randint(1, 24), nmin=32, nmax=rng.choice([64, 96, 128]),
                    precision=rng.choice([0, 1]), brick=rng.choice(["8,6,8", "8,6,16", "7,7,4"]),
                    steps=rng.randint(20, 100))
    lmin = rng.choice([4, 5, 6])
    case = dict(kind=kind, lmin=lmin, lmax=lmin + rng.randint(1, 3), radius=round(rng.uniform(0.2, 0.35), 3))
    if kind == "flags":
        return case
    return dict(case, precision=rng.choice([0, 0, 1]), brick=rng.choice(["4,4,4", "4,4,8", "8,6,8"]),
                steps=rng.randint(6, 20) if kind == "amr" else rng.randint(3, 8))


def _jobs(case, seed):
    """Jobs of the case's sizes, their initial conditions from the seed."""
    jobs = make_stream(case["jobs"], rate=1.0, nmin=case["nmin"], nmax=case["nmax"], nsteps=case["steps"])
    for j in jobs:
        j.kind, j.ic, j.info = job_ic(j.job_id, j.ncell, 1000 * (1 + seed))
    return jobs


def work(case):
    """80 B per cell and step (the state read and written once) and about 700
    operations per cell and step in 3D; the state once more for the output."""
    kind = case["kind"]
    if kind == "tube":
        c = case["n"]
        return {"bytes": 80.0 * c * case["steps"] + 40.0 * c, "flops": 250.0 * c * case["steps"]}
    if kind in ("level", "calls"):
        c = case["n"] ** 3
    elif kind == "serve":
        c = sum(j.cells for j in _jobs(case, 0))
    else:
        c = 8 * _mesh(case["lmin"], case["lmax"], case["radius"]).ngrid
        if kind == "flags":
            return {"bytes": 44.0 * c, "flops": 60.0 * c}
    return {"bytes": 80.0 * c * case["steps"] + 40.0 * c, "flops": 700.0 * c * case["steps"]}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gamma(case):
    return 5.0 / 3.0 if case.get("ic") == "turbulence" else 1.4


def _params(case):
    return HydroParams(gamma=_gamma(case), courant_factor=0.8 if case["kind"] == "tube" else 0.5,
                       slope_type=case.get("slope", 2), riemann=case.get("riemann", "hllc"))


def _cons(rho, vel, p, gamma):
    ekin = 0.5 * rho * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
    return torch.stack([rho, rho * vel[0], rho * vel[1], rho * vel[2], p / (gamma - 1.0) + ekin])


def _blast(n, seed, gamma):
    """Sedov blast: E in [0.1, 10], ambient p log-uniform in [1e-6, 1e-2], the
    energy in the central 2^3 cells."""
    rng = np.random.default_rng(seed)
    e, p0 = rng.uniform(0.1, 10.0), 10 ** rng.uniform(-6, -2)
    rho = torch.ones((n, n, n), dtype=torch.float64, device=DEV)
    p = torch.full_like(rho, p0)
    lo = n // 2 - 1
    p[lo:lo + 2, lo:lo + 2, lo:lo + 2] = (gamma - 1.0) * e * n ** 3 / 8
    z = torch.zeros_like(rho)
    return _cons(rho, (z, z, z), p, gamma)


def _turbulence(n, seed, gamma, mach=5.0):
    """Solenoidal Gaussian velocities with P(k) ~ k^-2 on 2 <= k <= 8 at rms Mach 5, rho = p = 1."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    k1 = torch.fft.fftfreq(n, d=1.0 / n, dtype=torch.float64, device=DEV)
    kz, ky, kx = torch.meshgrid(k1, k1, k1, indexing="ij")
    kk = torch.sqrt(kx ** 2 + ky ** 2 + kz ** 2)
    amp = torch.where((kk >= 2) & (kk <= 8), 1.0 / (kk ** 2).clamp(min=1.0), torch.zeros_like(kk))
    vk = [torch.complex(torch.randn(kk.shape, generator=g, dtype=torch.float64, device=DEV),
                        torch.randn(kk.shape, generator=g, dtype=torch.float64, device=DEV)) * amp for _ in range(3)]
    div = (kx * vk[0] + ky * vk[1] + kz * vk[2]) / (kk ** 2).clamp(min=1.0)
    vel = [torch.fft.ifftn(v - k * div).real for v, k in zip(vk, (kx, ky, kz))]
    rms = torch.sqrt(sum((v ** 2).mean() for v in vel))
    vel = [v * (mach * math.sqrt(gamma) / rms) for v in vel]
    one = torch.ones_like(kk)
    return _cons(one, vel, one, gamma)


def _tube(n, seed, gamma=1.4):
    """A Riemann problem with Sod's ratios varied by the seed."""
    rng = np.random.default_rng(seed)
    rl, pl = 1.0 + rng.uniform(-0.2, 0.2), 1.0 + rng.uniform(-0.2, 0.2)
    rr, pr = 0.125 * (1 + rng.uniform(-0.2, 0.2)), 0.1 * (1 + rng.uniform(-0.2, 0.2))
    left = torch.arange(n, device=DEV) < n // 2
    f = lambda a, b: torch.where(left, torch.tensor(a, dtype=torch.float64, device=DEV),  # noqa: E731
                                 torch.tensor(b, dtype=torch.float64, device=DEV))
    z = torch.zeros(n, dtype=torch.float64, device=DEV)
    return _cons(f(rl, rr), (z, z, z), f(pl, pr), gamma)


def _cells(case, seed):
    if case["kind"] == "tube":
        return _tube(case["n"], seed)
    return (_blast if case["ic"] == "blast" else _turbulence)(case["n"], seed, _gamma(case))


@functools.lru_cache(maxsize=None)
def _morton(m):
    """Octs (iz, iy, ix flattened) of an m^3 box in Morton order."""
    i = torch.arange(m, dtype=torch.int64)
    spread = torch.zeros_like(i)
    for b in range(10):
        spread |= ((i >> b) & 1) << (3 * b)
    code = (spread[:, None, None] << 2) | (spread[None, :, None] << 1) | spread[None, None, :]
    return torch.argsort(code.reshape(-1)).to(DEV)


def _to_octs(cells):
    """(5, N[, N, N]) cells -> (octs, 5, 2^ndim), octs in Morton order."""
    if cells.dim() == 2:
        return cells.reshape(5, -1, 2).permute(1, 0, 2).contiguous()
    m = cells.shape[1] // 2
    c = cells.reshape(5, m, 2, m, 2, m, 2).permute(1, 3, 5, 0, 2, 4, 6).reshape(m ** 3, 5, 8)
    return c[_morton(m)]


class _OctMesh(UniformMesh):
    """A uniform mesh whose initial state is handed over in the oct layout."""

    def from_cells(self, octs):
        return octs


@functools.lru_cache(maxsize=None)
def _box(ndim, n):
    return _OctMesh.for_cells(ndim, n)


@functools.lru_cache(maxsize=None)
def _mesh(lmin, lmax, radius):
    """The refined mesh, as a checkpoint holds it: the Sedov shell of that radius."""
    return AmrMesh(3, build_levels(lmin, lmax, functools.partial(sedov_profile, radius=radius)))


def _amr_octs(case, seed):
    """The blast on that mesh, with energy and ambient pressure from the seed; for the
    refinement criterion the shock has moved a little since the mesh was made."""
    rng = np.random.default_rng(seed)
    e, p0, moved = rng.uniform(0.5, 2.0), 10 ** rng.uniform(-5, -3), rng.uniform(0.97, 1.03)
    radius = case["radius"] * (moved if case["kind"] == "flags" else 1.0)
    prof = functools.partial(sedov_profile, radius=float(radius), e_blast=float(e), p0=float(p0))
    return amr_state(_mesh(case["lmin"], case["lmax"], case["radius"]), prof)


class Context:
    """A library context and the pinned buffers its state is handed over in."""

    def __init__(self, cid=None):
        if cid is None:
            c = ctypes.c_int32()
            _lib.call("rh_ctx_create", ctypes.byref(c))
            cid = c.value
        self.id = cid
        self.out = None

    def select(self):
        _lib.call("rh_ctx_select", self.id)

    def snapshot(self, noct, ttd=8):
        """The state of the context's first noct octs in its pinned buffer."""
        if self.out is None:
            self.out = torch.empty((noct, 5, ttd), dtype=torch.float64, pin_memory=True)
        self.select()
        _lib.call("rh_transfer_grid_host", ctypes.cast(self.out.data_ptr(), _lib._dp), None, noct, 5, ttd)
        return self.out

    def __del__(self):
        try:
            _lib.call("rh_ctx_destroy", self.id)
        except Exception:
            pass


def _shape(case):
    return tuple(int(b) for b in case["brick"].split(","))


def _upload(case, seed):
    """The context with the case's mesh and initial state."""
    kind = case["kind"]
    if kind in ("amr", "amrcalls", "flags"):
        am, octs = _mesh(case["lmin"], case["lmax"], case["radius"]), _amr_octs(case, seed)
    else:
        mesh, octs = _box(1 if kind == "tube" else 3, case["n"]), _to_octs(_cells(case, seed)).cpu().numpy()
    ctx = Context()
    ctx.select()
    if kind in ("amr", "amrcalls", "flags"):
        bricks = {l: _shape(case) for l in am.levels} if "brick" in case else None
        return ctx, AmrHierarchy(am, octs, _params(case), precision=case.get("precision", 0), bricks=bricks)
    _lib.call("rh_init")
    if kind != "tube":
        HipHydro.set_brick_shape(*_shape(case))
    return ctx, UniformLevel(mesh, octs, _params(case), periodic=kind != "tube")


def prepare(case, seed):
    torch.zeros(1, device=DEV)
    _lib.call("rh_ctx_select", 0)
    _lib.call("rh_init")
    if case["kind"] != "serve":
        ctx, level = _upload(case, seed)
        return {"case": case, "ctx": ctx, "level": level}
    eng = HipEngine(precision=case["precision"], brick=_shape(case))
    specs = _jobs(case, seed)
    jobs = [Context(eng.open(s)) for s in specs]
    eng.close_all()
    return {"case": case, "engine": eng, "specs": specs, "jobs": jobs}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind, steps = case["kind"], case.get("steps", 0)
    if kind == "serve":
        eng = state["engine"]
        ids = [j.id for j in state["jobs"]]
        _lib.call("rh_ctx_select", 0)
        for _ in range(steps):
            eng.step(ids)
        st = [eng.status(i) for i in ids]
        stat = np.array([[s[k] for k in ("t", "dt_next", "mass", "ekin", "eint")] for s in st])
        return [stat] + [j.snapshot((s.ncell // 2) ** 3) for j, s in zip(state["jobs"], state["specs"])]
    lev = state["level"]
    state["ctx"].select()
    if kind == "flags":
        am = lev.am
        return [lev.hh.hydro_flag(am.head[l], am.noct[l], lev.p, 0.1, 0.1)[0] for l in am.levels]
    if kind in ("calls", "amrcalls"):
        for _ in range(steps):
            dt = lev.step(precision=case["precision"]) if kind == "calls" else lev.step()
        return [state["ctx"].snapshot(lev.mesh.noct if kind == "calls" else lev.am.ngrid), dt]
    if kind == "amr":
        dt, t, sums, _ = lev.run_device(steps, use_graph=True)
        return [state["ctx"].snapshot(lev.am.ngrid), dt, t, sums]
    dt, t, sums, _ = lev.run_device(steps, precision=case.get("precision", 0), use_graph=True)
    return [state["ctx"].snapshot(lev.mesh.noct, lev.mesh.ttd), dt, t, sums]


# ---------------------------------------------------------------------------
# The same steps of a uniform box or a tube in plain torch, 64 bits
# ---------------------------------------------------------------------------
SMALLR, SMALLC = 1e-10, 1e-10


def _prim(u, gamma):
    r = u[0].clamp(min=SMALLR)
    v = u[1:4] / r
    e = u[4] - 0.5 * r * (v ** 2).sum(0)
    e = torch.maximum(e, r * (SMALLC ** 2 / gamma / (gamma - 1.0)))
    return torch.cat([r[None], v, ((gamma - 1.0) * e)[None]])


def _dt_sums(u, gamma, cfl, dx, nd):
    r = u[0].clamp(min=SMALLR)
    v = u[1:4] / r
    ke = 0.5 * r * (v ** 2).sum(0)
    p = torch.maximum((gamma - 1.0) * (u[4] - ke), r * (SMALLC ** 2 / gamma))
    ctot = v[:nd].abs().sum(0) + nd * torch.sqrt(gamma * p / r)
    dt = 2.0 * cfl * dx / (float(ctot.max()) * (1.0 + math.sqrt(1.0 + 2.0 * cfl * 1e-4)))
    vol = dx ** nd
    e = float(u[4].sum()) * vol
    return min(dt, cfl * dx / SMALLC), [float(u[0].sum()) * vol, e, float((u[4] - 0.5 * (u[1:4] ** 2).sum(0) / r).sum()) * vol, 0.0]


def _flux(ql, qr, d, gamma, riemann, cap):
    """Flux through the faces of direction d from the states on both sides."""
    n, t1, t2 = 1 + d, 1 + (d + 1) % 3, 1 + (d + 2) % 3
    smallp = SMALLC ** 2 / gamma
    rl, rr = ql[0].clamp(min=SMALLR), qr[0].clamp(min=SMALLR)
    pl, pr = torch.maximum(ql[4], rl * smallp), torch.maximum(qr[4], rr * smallp)
    ul, ur = ql[n], qr[n]
    f = torch.empty_like(ql)
    if riemann == "hllc":
        el = pl / (gamma - 1) + 0.5 * rl * (ql[1:4] ** 2).sum(0)
        er = pr / (gamma - 1) + 0.5 * rr * (qr[1:4] ** 2).sum(0)
        c = torch.sqrt(torch.maximum(gamma * pl / rl, gamma * pr / rr).clamp(min=SMALLC ** 2))
        sl, sr = torch.minimum(ul, ur) - c, torch.maximum(ul, ur) + c
        rcl, rcr = rl * (ul - sl), rr * (sr - ur)
        us = (rcr * ur + rcl * ul + (pl - pr)) / (rcr + rcl)
        ps = (rcr * pl + rcl * pr + rcl * rcr * (ul - ur)) / (rcr + rcl)
        left = (sl > 0) | (us > 0)
        star = ~(sl > 0) & ((us > 0) | (sr > 0))
        s, r, u, p, e = (torch.where(left, a, b) for a, b in ((sl, sr), (rl, rr), (ul, ur), (pl, pr), (el, er)))
        rs = r * (s - u) / (s - us)
        es = ((s - u) * e - p * u + ps * us) / (s - us)
        r, u, p, e = (torch.where(star, a, b) for a, b in ((rs, r), (us, u), (ps, p), (es, e)))
        f[0], f[n], f[4] = r * u, r * u * u + p, (e + p) * u
        f[t1] = r * u * torch.where(left, ql[t1], qr[t1])
        f[t2] = r * u * torch.where(left, ql[t2], qr[t2])
        return f
    cl, cr = torch.sqrt(gamma * pl / rl), torch.sqrt(gamma * pr / rr)
    cons, fl = [], []
    for q in (ql, qr):
        c = torch.cat([q[:1], q[0] * q[1:4], (q[4] / (gamma - 1) + 0.5 * q[0] * (q[1:4] ** 2).sum(0))[None]])
        g = q[n] * c
        g[n] += q[4]
        g[4] += q[n] * q[4]
        cons.append(c)
        fl.append(g)
    if riemann == "llf":
        c = torch.maximum(ul.abs() + cl, ur.abs() + cr).clamp(max=cap)
        return 0.5 * (fl[0] + fl[1] - c * (cons[1] - cons[0]))
    c = torch.maximum(cl, cr)
    sl = (torch.minimum(ul, ur) - c).clamp(max=0.0).clamp(min=-cap)
    sr = (torch.maximum(ul, ur) + c).clamp(min=0.0).clamp(max=cap)
    return (sr * fl[0] - sl * fl[1] + sr * sl * (cons[1] - cons[0])) / (sr - sl)


def _step(u, dt, dx, gamma, cfl, slope, riemann, nd):
    """One MUSCL-Hancock step; in 1D the end cells are repeated outwards."""
    if nd == 1:
        u = torch.cat([u[:, :1], u[:, :1], u, u[:, -1:], u[:, -1:]], 1)
    ax = {d: u.dim() - 1 - d for d in range(nd)}
    q = _prim(u, gamma)
    half = {}
    for d in range(nd):
        qm, qp = torch.roll(q, 1, ax[d]), torch.roll(q, -1, ax[d])
        a, b = q - qm, qp - q
        lim = torch.minimum(a.abs(), b.abs())
        if slope == 2:
            lim = torch.minimum(2 * lim, 0.5 * (a + b).abs())
        h = torch.where((a * b) > 0, 0.5 * torch.sign(a) * lim, torch.zeros_like(a))
        n = 1 + d
        bound = torch.minimum(qm[0] * a[n].abs(), qp[0] * b[n].abs()) / q[0]
        h[n] = torch.sign(h[n]) * torch.minimum(h[n].abs(), bound)
        half[d] = h
        del qm, qp, a, b, lim
    r, v, p = q[0], q[1:4], q[4]
    src = -sum(v[d] * half[d] for d in range(nd))
    div = sum(half[d][1 + d] for d in range(nd))
    src[0] -= div * r
    src[4] -= div * gamma * p
    for d in range(nd):
        src[1 + d] -= half[d][4] / r
    mid = q + src * (dt / dx)
    cap, new = cfl * dx / dt, u.clone()
    for d in range(nd):
        lo, hi = mid - half[d], mid + half[d]
        for s in (lo, hi):
            s[0] = torch.where(s[0] < SMALLR, r, s[0])
            s[4] = torch.where(s[4] < SMALLR * SMALLC ** 2, p, s[4])
        f = _flux(torch.roll(hi, 1, ax[d]), lo, d, gamma, riemann, cap)
        new += (dt / dx) * (f - torch.roll(f, -1, ax[d]))
    return new[:, 2:-2] if nd == 1 else new


def _evolve(u, case, gamma, cfl, n, steps, slope, riemann, nd):
    """(state, dt of the last step, dt of the next, time, sums before the last step, sums after it)."""
    dx, t, dt, before = 1.0 / n, 0.0, 0.0, None
    for _ in range(steps):
        dt, before = _dt_sums(u, gamma, cfl, dx, nd)
        u = _step(u, dt, dx, gamma, cfl, slope, riemann, nd)
        t += dt
    nxt, after = _dt_sums(u, gamma, cfl, dx, nd)
    return u, dt, nxt, t, before, after


def exact(case, seed):
    kind = case["kind"]
    if kind in ("level", "tube", "calls"):
        nd, cfl = (1, 0.8) if kind == "tube" else (3, 0.5)
        u, dt, nxt, t, before, after = _evolve(_cells(case, seed), case, _gamma(case), cfl, case["n"], case["steps"],
                                               case["slope"], case["riemann"], nd)
        octs = _to_octs(u).cpu()
        if kind == "calls":
            return [octs, dt]
        return [octs, dt, t, np.array(before)] if kind == "tube" else [octs, nxt, t, np.array(after)]
    if kind == "serve":
        stat, octs = [], []
        for s in _jobs(case, seed):
            n, a = s.ncell, s.ic
            z = torch.zeros((n, n, n), dtype=torch.float64, device=DEV)
            rho, p = torch.full_like(z, a[0]), torch.full_like(z, a[1])
            if s.kind == 1:
                lo = int(a[3])
                p[lo:lo + 2, lo:lo + 2, lo:lo + 2] = a[2]
            else:
                sl = [slice(None)] * 3
                sl[2 - int(a[4])] = slice(n // 2, None)
                rho[tuple(sl)], p[tuple(sl)] = a[2], a[3]
            u, _, nxt, t, _, after = _evolve(_cons(rho, (z, z, z), p, 1.4), case, 1.4, 0.5, n, case["steps"], 2,
                                             "hllc", 3)
            stat.append([t, nxt] + after[:3])
            octs.append(_to_octs(u).cpu())
        return [np.array(stat)] + octs
    # refined meshes: plain array operations have no short form of the coarse-fine step; flags are whole numbers
    return None
