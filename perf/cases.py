"""The work that users of this framework have it do, as timed cases.

listed() gives the cases, draw(rng) more of the same ranges, prepare(case,
seed) what a program holds before the call, run(state) one pass through the
public entry points, work(case) the bytes and operations of a pass that no
implementation can do without, and exact(case, seed) the outputs in 64 bits
from plain torch.

Kinds of case:
  host      one nvector batch through the Fortran-linkable `unsplit_` on host
            arrays, as godfine1 calls it
  sweep     nvector batches resident in device memory, one launch for the
            whole sweep (`unsplit_device`)
  level     a resident periodic level advanced by whole steps (UniformLevel)
  serve     a closed batch of independent solves (HydroServer)
  amr_sweep courant, set_unew and godunov_fine of one partly refined level
            with its reflux into the coarser one (AmrLevels)
  amr_run   a coarse step over a hierarchy of levels (AmrSolver): `adapt`
            refines and flags on the way, from the same mesh on every pass
"""
import functools
import math

import numpy as np
import torch

import ramses_amd as ra
from ramses_amd import ics
from ramses_amd.amr import AmrLevels, AmrSolver, configure_interpolation, configure_refinement
from ramses_amd.serve import HydroServer, Request
from ramses_amd.tree import OctTree

NV = 32
SMALLR = SMALLC = 1e-10


def listed():
    return [
        # The drop-in's inner call: one batch of godfine1 on host arrays, the
        # gravity array zero (no Poisson solve), all of it latency.
        dict(name="host_batch", kind="host", ngrid=32, riemann="llf", slope=1, gamma=1.4),
        # One sweep of a medium level with self-gravity on: ragged last batch.
        dict(name="sweep_33k_gravity", kind="sweep", groups=1031, last=7, gravity=True, riemann="llf", slope=2,
             precision="fp64", gamma=1.4),
        # The batched boundary at its largest, 2^20 octs, in both precisions.
        dict(name="sweep_1m", kind="sweep", groups=32768, last=32, gravity=False, riemann="hllc", slope=1,
             precision="fp64", gamma=5 / 3),
        dict(name="sweep_262k_fp32", kind="sweep", groups=8192, last=32, gravity=False, riemann="hllc", slope=1,
             precision="fp32", gamma=5 / 3),
        # A Sedov blast on a small level, many steps at a time: launch-bound.
        dict(name="level_64_sedov", kind="level", n=64, steps=16, ic="sedov", mach=0.0, riemann="hllc", slope=1,
             precision="fp64", sums=False, gamma=1.4, cfl=0.8),
        # A side that is no power of two, with the conservation sums of each
        # step and the moncen slopes many production runs take.
        dict(name="level_168_moncen", kind="level", n=168, steps=1, ic="turb", mach=2.0, riemann="llf", slope=2,
             precision="fp64", sums=True, gamma=5 / 3, cfl=0.5),
        # The headline: supersonic turbulence, one step at a time.
        dict(name="level_512", kind="level", n=512, steps=1, ic="turb", mach=5.0, riemann="hllc", slope=1,
             precision="fp64", sums=False, gamma=5 / 3, cfl=0.5),
        dict(name="level_256_fp32", kind="level", n=256, steps=1, ic="turb", mach=5.0, riemann="hllc", slope=1,
             precision="fp32", sums=False, gamma=5 / 3, cfl=0.5),
        # Independent solves of mixed sizes served together to their end times.
        dict(name="serve_12", kind="serve", requests=12, t_end=0.01, riemann="hllc", slope=1, precision="fp32",
             gamma=5 / 3),
        # godunov_fine of a level that covers part of the box.
        dict(name="amr_sweep_7", kind="amr_sweep", levelmin=6, radius=0.3, riemann="hllc", slope=1,
             precision="fp64", gamma=5 / 3),
        # The adaptive Sedov blast: few octs on many levels, subcycled, each
        # coarse step a captured graph.
        dict(name="amr_sedov_6_10", kind="amr_run", adapt=True, graph=True, levelmin=6, levelmax=10, blobs=0,
             riemann="hllc", slope=1, precision="fp64", gamma=1.4),
        # A static hierarchy with most of its octs on the finest level.
        dict(name="amr_static_6_8", kind="amr_run", adapt=False, graph=False, levelmin=6, levelmax=8, blobs=24,
             riemann="hllc", slope=1, precision="fp64", gamma=5 / 3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "sweep", "sweep", "level", "level", "level", "serve", "amr_sweep", "amr_run"])
    c = dict(kind=kind, riemann=rng.choice(["hllc", "hllc", "llf", "hll"]), slope=rng.choice([1, 1, 2]),
             gamma=rng.choice([1.4, 5 / 3]))
    prec = rng.choice(["fp64", "fp32"])
    if kind == "host":
        c.update(ngrid=rng.randint(1, NV))
    elif kind == "sweep":
        c.update(groups=_log(rng, 4, 24000), last=rng.randint(1, NV), gravity=rng.random() < 0.4, precision=prec)
    elif kind == "level":
        n = 8 * _log(rng, 2, 48)
        c.update(n=n, steps=2 * rng.randint(1, 8) if n <= 128 else 1, ic="turb", mach=rng.choice([0.5, 2.0, 5.0]),
                 precision=prec, sums=rng.random() < 0.25, cfl=rng.choice([0.5, 0.8]))
    elif kind == "serve":
        c.update(requests=rng.randint(3, 16), t_end=rng.uniform(0.004, 0.012), precision=prec)
    elif kind == "amr_sweep":
        c.update(levelmin=rng.choice([4, 5, 6]), radius=rng.uniform(0.1, 0.4), precision=prec)
    else:
        adapt = rng.random() < 0.6
        lmin = rng.choice([4, 5, 6])
        c.update(adapt=adapt, graph=rng.random() < 0.5, levelmin=lmin, levelmax=lmin + rng.randint(1, 4 if adapt else 2),
                 blobs=0 if adapt else rng.randint(4, 24), precision=prec)
    return c


# --- what a program has in hand ------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _configure(case):
    ra.configure(gamma=case["gamma"], smallr=SMALLR, smallc=SMALLC, riemann=case["riemann"], slope_type=case["slope"],
                 courant_factor=case.get("cfl", 0.5 if case["kind"] != "amr_run" else 0.8),
                 precision=case.get("precision", "fp64"), nvector=NV)


def _sweep_inputs(case, seed):
    groups = case.get("groups", 1)
    uin, dt = ics.oct_batches(groups * NV, nv=NV, seed=seed, gamma=case["gamma"])
    grav = None
    if case.get("gravity"):
        grav = torch.empty((groups, 3, 6, 6, 6, NV), dtype=torch.float64, device="cuda").normal_(generator=_gen(seed + 1))
    return uin, grav, dt


def _level_ic(n, mach, gamma, seed):
    return ics.turbulent(n, mach, gamma=gamma, rho_sigma=0.5, seed=seed, generator="device")


def _level_inputs(case, seed):
    """Turbulence, or a point blast (its energy from the seed) in a box."""
    if case["ic"] == "sedov":
        return ics.sedov(case["n"], gamma=case["gamma"], e_total=0.5 + (seed % 97) / 97)
    return _level_ic(case["n"], case["mach"], case["gamma"], seed)


def _serve_sizes(case):
    """Sides of the requests, small ones as likely as large ones."""
    sides = (16, 32, 48, 64, 96, 128)
    return [sides[(5 * i + 3 * (i // 6)) % 6] for i in range(case["requests"])]


def _serve_inputs(case, seed):
    return [_level_ic(n, 2.0, case["gamma"], seed * 64 + i) for i, n in enumerate(_serve_sizes(case))]


@functools.lru_cache(maxsize=2)
def _tree(levelmin, levelmax, radius, extra):
    return OctTree(levelmin, levelmax, None if radius == 0.0 else
                   lambda l, x: np.sqrt(((x - 0.5) ** 2).sum(1)) < radius, extra_grids=extra)


def _fields(x, gamma, seed):
    """Smooth periodic conserved fields at positions x (N, 3) in the box."""
    g = torch.Generator()
    g.manual_seed(seed)
    k = torch.randint(1, 4, (5, 3), generator=g).to(x)
    ph = (2 * math.pi * torch.rand((5, 3), generator=g, dtype=torch.float64)).to(x.device)
    s = torch.sin(2 * math.pi * k[:, None, :] * x[None] + ph[:, None, :]).prod(2)
    rho, vel, p = 1.0 + 0.4 * s[0], 0.8 * s[1:4], 1.0 + 0.3 * s[4] + 2.0 * torch.exp(-((x - 0.5) ** 2).sum(1) / 0.01)
    return torch.cat([rho[None], rho * vel, (p / (gamma - 1.0) + 0.5 * rho * (vel * vel).sum(0))[None]])


def _amr_sweep_inputs(case, seed):
    """The tree, and the state over every cell of every level."""
    tree = _tree(case["levelmin"], case["levelmin"] + 1, case["radius"], 0)
    u = torch.ones((5, tree.ncell), dtype=torch.float64)
    for l in range(1, tree.nlevel + 1):
        ic, x = tree.cells_of_level(l)
        u[:, torch.from_numpy(ic) - 1] = _fields(torch.from_numpy(x).cuda(), case["gamma"], seed).cpu()
    return tree, u.numpy()


def _blast(case, seed):
    """A point blast off the box centre; or overdense blobs in a flow."""
    g = torch.Generator()
    g.manual_seed(seed)
    if case["blobs"] == 0:
        center = (0.4 + 0.2 * torch.rand(3, generator=g)).tolist()
        return lambda x, dx: ics.sedov_regions(x, dx, gamma=case["gamma"], center=center)
    at = torch.rand((case["blobs"], 3), generator=g, dtype=torch.float64).cuda()
    size = (0.04 + 0.06 * torch.rand(case["blobs"], generator=g, dtype=torch.float64)).cuda()

    def ic(x, dx):
        u = _fields(x, case["gamma"], seed)
        more = torch.zeros_like(x[:, 0])
        for a, s in zip(at, size):
            r = x - a
            more += 3.0 * torch.exp(-((r - r.round()) ** 2).sum(1) / (s * s))
        return u * (1.0 + more)
    return ic


def _room(case):
    """Octs that a hierarchy may come to hold beyond its coarsest level."""
    return 60000 if case["adapt"] else 400000


def prepare(case, seed):
    _configure(case)
    kind = case["kind"]
    if kind == "host":
        uin, _, dt = _sweep_inputs(case, seed)
        return dict(kind=kind, ngrid=case["ngrid"], dt=dt, uin=uin[0].cpu().numpy(), grav=np.zeros(ra.grav_shape(NV)),
                    pin=np.zeros((6, 6, 6, NV)), flux=np.zeros(ra.flux_shape(NV)), tmp=np.zeros(ra.tmp_shape(NV)))
    if kind == "sweep":
        uin, grav, dt = _sweep_inputs(case, seed)
        out = [torch.zeros((case["groups"],) + s, dtype=torch.float64, device="cuda")
               for s in (ra.flux_shape(NV), ra.tmp_shape(NV))]
        return dict(kind=kind, uin=uin, grav=grav, dt=dt, last=case["last"], flux=out[0], tmp=out[1])
    if kind == "level":
        lvl = ra.UniformLevel(_level_inputs(case, seed), sums=case["sums"])
        lvl.courant()
        if case["steps"] > 1:
            lvl.advance(2)  # captures the pair of steps that advance() replays
        return dict(kind=kind, level=lvl, steps=case["steps"])
    if kind == "serve":
        server = HydroServer(max_slots=16)
        return dict(kind=kind, server=server, ic=_serve_inputs(case, seed), t_end=case["t_end"])
    configure_interpolation(1, 0)
    if kind == "amr_sweep":
        tree, u = _amr_sweep_inputs(case, seed)
        s = AmrLevels(tree, u)
        return dict(kind=kind, mesh=s, level=case["levelmin"] + 1)
    configure_refinement(err_grad_d=0.1, err_grad_p=0.1 if case["adapt"] else -1.0)
    s = AmrSolver(_tree(case["levelmin"], case["levelmin"], 0.0, _room(case)), None, refine=case["adapt"],
                  nlevelmax=case["levelmax"], graph=case["graph"], graph_capacity=max(8 ** (case["levelmin"] - 1), _room(case) // 2))
    s.init_refine(_blast(case, seed))
    s.capture()
    for _ in range(2):  # past the conservation baselines of a run's second step
        s.coarse_step()
    state = dict(kind=kind, solver=s, start=None)
    if case["adapt"]:
        state["start"] = _mesh_copy(s)
    return state


_MESH = ("son", "father", "nbor", "pos", "xg", "ring", "uold", "unew", "flag1", "flag2", "dt", "dtold", "time")


def _mesh_copy(s):
    return dict(arrays=[getattr(s, a).clone() for a in _MESH], lists={l: t.clone() for l, t in s.lists.items()},
                nocts=dict(s.nocts), free=(s.free.head, s.free.numbf, s.free.used_mem))


def _mesh_restore(s, c):
    for a, t in zip(_MESH, c["arrays"]):
        getattr(s, a).copy_(t)
    for l, t in c["lists"].items():
        s.lists[l].copy_(t)
    s.nocts.update(c["nocts"])
    s.free.head, s.free.numbf, s.free.used_mem = c["free"]


def run(state):
    kind = state["kind"]
    if kind == "host":
        dx = 1.0 / 128
        ra.unsplit_fortran(state["uin"], state["grav"], state["pin"], state["flux"], state["tmp"], dx, dx, dx,
                           state["dt"], state["ngrid"])
        return dict(flux=state["flux"], tmp=state["tmp"])
    if kind == "sweep":
        ra.unsplit_device(state["uin"], state["grav"], state["flux"], state["tmp"], 1.0 / 128, state["dt"],
                          ngrid_last=state["last"])
        return dict(flux=state["flux"], tmp=state["tmp"])
    if kind == "level":
        lvl = state["level"]
        if state["steps"] > 1:
            lvl.advance(state["steps"])
        else:
            lvl.step()
        out = dict(u=lvl.u, dt=lvl.dt[0])
        if lvl.sums is not None:
            out["sums"] = lvl.sums
        return out
    if kind == "serve":
        reqs = [Request(i, u.shape[-1], state["t_end"], ic=lambda n, u=u: u, keep_result=True)
                for i, u in enumerate(state["ic"])]
        state["server"].run(reqs)
        return dict(u=[r.result for r in reqs], steps=[r.steps for r in reqs])
    if kind == "amr_sweep":
        s, l = state["mesh"], state["level"]
        s.set_unew(l - 1)
        s.set_unew(l)
        s.courant(l)
        s.godunov(l)
        return dict(unew=s.unew, dt=s.dt[l])
    s = state["solver"]
    if state["start"] is not None:
        _mesh_restore(s, state["start"])
    s.coarse_step()
    return dict(u=s.uold, son=s.son, dt=s.dt, octs=[s.noct(l) for l in range(1, s.nlevelmax + 1)])


# --- what a pass cannot do without ---------------------------------------

# Operations of one cell update: one conversion, three slopes and traces,
# three faces and the update, divisions and roots counted as one each.
_FLOPS = 700.0
_OCT_BYTES = 80 * 5 * 8 + 36 * 7 * 8  # the stencil cells some face depends on, and the 36 faces


def work(case):
    kind = case["kind"]
    if kind in ("host", "sweep"):
        octs = case["ngrid"] if kind == "host" else (case["groups"] - 1) * NV + case["last"]
        grav = 80 * 3 * 8 if case.get("gravity") else 0
        return dict(bytes=float(octs * (_OCT_BYTES + grav)), flops=octs * 36 * 250.0)
    if kind == "level":
        cells = case["n"] ** 3 * case["steps"]
        return dict(bytes=80.0 * cells, flops=_FLOPS * cells)
    if kind == "serve":
        # steps to t_end at the Courant condition of Mach-2 turbulence
        cells = sum(n ** 3 * (1 + case["t_end"] * n * 24) for n in _serve_sizes(case))
        return dict(bytes=80.0 * cells, flops=_FLOPS * cells)
    if kind == "amr_sweep":
        fine = 8 * _tree(case["levelmin"], case["levelmin"] + 1, case["radius"], 0).n_octs(case["levelmin"] + 1)
        coarse = 8.0 ** case["levelmin"]
        return dict(bytes=80.0 * (fine + coarse), flops=_FLOPS * fine)
    # every level once per substep; about as many octs as these meshes come to hold
    cells = 8.0 ** case["levelmin"]
    for l in range(case["levelmin"] + 1, case["levelmax"] + 1):
        share = {7: 0.13 + 0.013 * case["blobs"], 8: 0.002 * case["blobs"]}.get(l, 1.0)
        octs = 1150.0 if case["adapt"] else 8.0 ** (l - 1) * share
        cells += 8 * octs * 2 ** (l - case["levelmin"])
    return dict(bytes=80.0 * cells, flops=_FLOPS * cells)


# --- the outputs in 64 bits ----------------------------------------------

def _prim(u, gamma, grav=None, dt=0.0):
    r = u[0].clamp(min=SMALLR)
    v = [u[d] / r for d in (1, 2, 3)]
    e = u[4] / r - 0.5 * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
    p = (gamma - 1.0) * r * e.clamp(min=SMALLC ** 2 / gamma / (gamma - 1.0))
    if grav is not None:
        v = [v[d] + 0.5 * dt * grav[d] for d in range(3)]
    return torch.stack([r, *v, p])


def _slope(a, b, c, slope):
    lft, rgt = b - a, c - b
    if slope == 1:
        s = torch.where(lft > 0, torch.minimum(lft, rgt), torch.maximum(lft, rgt))
    else:
        cen = 0.5 * (lft + rgt)
        s = torch.sign(cen) * torch.minimum(2.0 * torch.minimum(lft.abs(), rgt.abs()), cen.abs())
    return torch.where(lft * rgt <= 0, torch.zeros_like(s), s)


def _riemann(L, R, gamma, name):
    """Flux of (rho, un, p, ut1, ut2) states: mass, normal momentum, energy,
    two tangential momenta, internal energy."""
    entho, smallp = 1.0 / (gamma - 1.0), SMALLC ** 2 / gamma
    rl, rr = L[0].clamp(min=SMALLR), R[0].clamp(min=SMALLR)
    pl, pr = torch.maximum(L[2], rl * smallp), torch.maximum(R[2], rr * smallp)
    ul, ur = L[1], R[1]
    cl, cr = torch.sqrt(gamma * pl / rl), torch.sqrt(gamma * pr / rr)
    if name == "hllc":
        etl = pl * entho + 0.5 * rl * (ul ** 2 + L[3] ** 2 + L[4] ** 2)
        etr = pr * entho + 0.5 * rr * (ur ** 2 + R[3] ** 2 + R[4] ** 2)
        c = torch.maximum(cl, cr).clamp(min=SMALLC)
        SL, SR = torch.minimum(ul, ur) - c, torch.maximum(ul, ur) + c
        wl, wr = rl * (ul - SL), rr * (SR - ur)
        us = (wr * ur + wl * ul + (pl - pr)) / (wr + wl)
        ps = (wr * pl + wl * pr + wl * wr * (ul - ur)) / (wr + wl)
        left = us > 0
        S, u, r, et, p = (torch.where(left, x, y) for x, y in ((SL, SR), (ul, ur), (rl, rr), (etl, etr), (pl, pr)))
        star = torch.where(left, SL <= 0, SR > 0)
        ro = torch.where(star, r * (S - u) / (S - us), r)
        et = torch.where(star, ((S - u) * et - p * u + ps * us) / (S - us), et)
        eo = torch.where(star, p * entho * (S - u) / (S - us), p * entho)
        uo, po = torch.where(star, us, u), torch.where(star, ps, p)
        m = ro * uo
        return torch.stack([m, m * uo + po, (et + po) * uo, m * torch.where(left, L[3], R[3]),
                            m * torch.where(left, L[4], R[4]), uo * eo])

    def cons(q):
        e = q[2] * entho
        return torch.stack([q[0], q[0] * q[1], e + 0.5 * q[0] * (q[1] ** 2 + q[3] ** 2 + q[4] ** 2), q[0] * q[3],
                            q[0] * q[4], e])
    uL, uR = cons(L), cons(R)
    fL, fR = ul * uL, ur * uR
    for f, q in ((fL, L), (fR, R)):
        f[1] += q[2]
        f[2] += q[1] * q[2]
    if name == "llf":
        return 0.5 * (fL + fR - torch.maximum(ul.abs() + cl, ur.abs() + cr) * (uR - uL))
    SL = (torch.minimum(ul, ur) - torch.maximum(cl, cr)).clamp(max=0)
    SR = (torch.maximum(ul, ur) + torch.maximum(cl, cr)).clamp(min=0)
    return (SR * fL - SL * fR + SR * SL * (uR - uL)) / (SR - SL)


def _at(a, ax, lo, hi):
    """a without `lo` cells at the start and `hi` at the end of axis x, y or z (0, 1, 2); axes are (var, z, y, x, ...)."""
    d = 3 - ax
    return a.narrow(d, lo, a.shape[d] - lo - hi)


def _faces(u, grav, dt, dx, case):
    """Fluxes dt/dx*F of a block (5, z, y, x, ...) with two cells of halo: for
    x, y, z ((rho, mx, my, mz, E) fluxes, (normal velocity, internal energy
    flux)), one more face than cells along the axis."""
    gamma = case["gamma"]
    q = _prim(u, gamma, grav, dt)

    def inner(a, ax):  # one halo cell off both ends of the other two axes
        for o in {0, 1, 2} - {ax}:
            a = _at(a, o, 1, 1)
        return a
    q0 = inner(_at(q, 0, 1, 1), 0)
    D = []
    for ax in range(3):
        t = inner(q, ax)
        D.append(_slope(_at(t, ax, 0, 2), q0, _at(t, ax, 2, 0), case["slope"]))
    r, v, p = q0[0], q0[1:4], q0[4]
    adv = sum(v[d] * D[d] for d in range(3))
    div = sum(D[d][1 + d] for d in range(3))
    src = -adv
    src[0] -= div * r
    src[4] -= div * gamma * p
    for d in range(3):
        src[1 + d] -= D[d][4] / r
    out = []
    for ax in range(3):
        h = 0.5 * dt / dx
        qp, qm = q0 - 0.5 * D[ax] + src * h, q0 + 0.5 * D[ax] + src * h
        for t in (qp, qm):
            t[0] = torch.where(t[0] < SMALLR, q0[0], t[0])
        qp, qm = inner(qp, ax), inner(qm, ax)
        order = [0, 1 + ax, 4] + [1 + o for o in range(3) if o != ax]
        L, R = _at(qm, ax, 0, 1)[order], _at(qp, ax, 1, 0)[order]
        f = _riemann(L, R, gamma, case["riemann"])
        flux = torch.empty_like(f[:5])
        flux[0], flux[4], flux[1 + ax] = f[0], f[2], f[1]
        for k, o in enumerate(o for o in range(3) if o != ax):
            flux[1 + o] = f[3 + k]
        out.append((flux * (dt / dx), torch.stack([0.5 * (L[1] + R[1]), f[5]]) * (dt / dx)))
    return out


def _pad(u):
    for d in (1, 2, 3):
        n = u.shape[d]
        u = torch.cat([u.narrow(d, n - 2, 2), u, u.narrow(d, 0, 2)], d)
    return u


def _step(u, dt, dx, case):
    """One step of a periodic level, in slabs of z planes."""
    n, new = u.shape[1], torch.empty_like(u)
    slab = max(8, min(n, (1 << 25) // (n * n)))
    for z in range(0, n, slab):
        m = min(slab, n - z)
        at = torch.arange(z - 2, z + m + 2, device=u.device) % n
        b = u[:, at]
        for d in (2, 3):
            b = torch.cat([b.narrow(d, n - 2, 2), b, b.narrow(d, 0, 2)], d)
        s = u[:, z:z + m].clone()
        for ax, (f, _) in enumerate(_faces(b, None, dt, dx, case)):
            s += _at(f, ax, 0, 1) - _at(f, ax, 1, 0)
        new[:, z:z + m] = s
    return new


def _courant(u, dx, case, cfl):
    w = 0.0
    for z in range(0, u.shape[1], 64):
        q = _prim(u[:, z:z + 64], case["gamma"])
        c = torch.sqrt(case["gamma"] * torch.maximum(q[4] / q[0], torch.full_like(q[0], SMALLC ** 2 / case["gamma"])))
        w = max(w, float((3.0 * c + q[1].abs() + q[2].abs() + q[3].abs()).max()))
    return torch.tensor(dx / w * (math.sqrt(1.0 + 2e-4 * cfl) - 1.0) / 1e-4, dtype=torch.float64)


def _exact_sweep(case, seed):
    uin, grav, dt = _sweep_inputs(case, seed)
    groups = uin.shape[0]
    last = case["ngrid"] if case["kind"] == "host" else case["last"]
    flux = torch.zeros((groups,) + ra.flux_shape(NV), dtype=torch.float64, device="cuda")
    tmp = torch.zeros((groups,) + ra.tmp_shape(NV), dtype=torch.float64, device="cuda")
    for g in range(0, groups, 1024):
        h = min(groups, g + 1024)
        u = uin[g:h].movedim(0, 4)
        a = None if grav is None else grav[g:h].movedim(0, 4)
        for ax, (f, t) in enumerate(_faces(u, a, dt, 1.0 / 128, case)):
            k, j, i = (3 if ax == o else 2 for o in (2, 1, 0))
            flux[g:h, ax, :, :k, :j, :i] = f.movedim(4, 0)
            tmp[g:h, ax, :, :k, :j, :i] = t.movedim(4, 0)
    flux[-1, ..., last:] = 0
    tmp[-1, ..., last:] = 0
    if case["kind"] == "host":
        return dict(flux=flux[0].cpu().numpy(), tmp=tmp[0].cpu().numpy())
    return dict(flux=flux, tmp=tmp)


def _exact_level(case, seed):
    u = _level_inputs(case, seed)
    dx = 1.0 / case["n"]
    dt = _courant(u, dx, case, case["cfl"])
    for _ in range(case["steps"] + (2 if case["steps"] > 1 else 0)):
        u = _step(u, float(dt), dx, case)
        dt = _courant(u, dx, case, case["cfl"])
    out = dict(u=u, dt=dt)
    if case["sums"]:
        ei = u[4] - 0.5 * (u[1] ** 2 + u[2] ** 2 + u[3] ** 2) / u[0].clamp(min=SMALLR)
        out["sums"] = torch.stack([u[0].sum(), u[4].sum(), ei.sum()]) * dx ** 3
    return out


def _exact_serve(case, seed):
    out = []
    for u in _serve_inputs(case, seed):
        dx, t = 1.0 / u.shape[-1], 0.0
        while t < case["t_end"]:
            dt = min(float(_courant(u, dx, case, 0.5)), case["t_end"] - t)
            u = _step(u, dt, dx, case)
            t += dt
        out.append(u)
    return dict(u=out, steps=[None] * len(out))


def _exact_amr_sweep(case, seed):
    """The fine level on the whole lattice: cells outside its octs take the
    prolongation of the coarser level, and faces of the octs towards coarser
    leaves correct these."""
    tree, u = _amr_sweep_inputs(case, seed)
    l, lc = case["levelmin"] + 1, case["levelmin"]
    n, nc = 2 ** l, 2 ** lc
    u = torch.from_numpy(u).cuda()

    def lattice(level):
        ic, x = tree.cells_of_level(level)
        m = 2 ** level
        at = torch.from_numpy((x * m).astype(np.int64)).cuda()
        return torch.from_numpy(ic).long().cuda() - 1, (at[:, 2] * m + at[:, 1]) * m + at[:, 0]
    cf, xf = lattice(l)
    cc, xc = lattice(lc)
    C = torch.empty((5, nc ** 3), dtype=torch.float64, device="cuda")
    C[:, xc] = u[:, cc]
    C = C.reshape(5, nc, nc, nc)
    U = C
    for d in (1, 2, 3):
        U = U.repeat_interleave(2, d)
    for ax in range(3):
        d = 3 - ax
        s = 0.5 * _slope(C.roll(1, d), C, C.roll(-1, d), 1)
        for e in (1, 2, 3):
            s = s.repeat_interleave(2, e)
        sign = torch.tensor([-0.5, 0.5], dtype=torch.float64, device="cuda").repeat(nc)
        U = U + s * sign.reshape([n if e == d else 1 for e in range(4)])
    U = U.reshape(5, -1)
    U[:, xf] = u[:, cf]
    U = U.reshape(5, n, n, n)
    dx = 1.0 / n
    dt = _courant(u[:, cf].reshape(5, -1, 1, 1), dx, case, 0.5)
    F = _faces(_pad(U), None, float(dt), dx, case)
    new = U.clone()
    fine = torch.zeros(n ** 3, dtype=torch.bool, device="cuda")
    fine[xf] = True
    inside = fine.reshape(n, n, n)[::2, ::2, ::2]  # coarse cells that are refined
    corr = torch.zeros_like(C)
    for ax, (f, _) in enumerate(F):
        d = 3 - ax
        new += _at(f, ax, 0, 1) - _at(f, ax, 1, 0)
        f = _at(f, ax, 0, 1).unfold(d, 1, 2).squeeze(-1)  # the faces on coarse cells' low sides
        for e in {1, 2, 3} - {d}:
            f = f.unfold(e, 2, 2).sum(-1)
        low, high = inside.roll(1, d - 1), inside.roll(-1, d - 1)
        corr += torch.where(low, f, torch.zeros_like(f)) / 8 - torch.where(high, f.roll(-1, d), torch.zeros_like(f)) / 8
    C = torch.where(inside, C, C + corr)
    out = torch.zeros((5, tree.ncell + 1), dtype=torch.float64, device="cuda")
    out[:, 1:] = u
    out[:, 1 + cc] = C.reshape(5, -1)[:, xc]
    out[:, 1 + cf] = new.reshape(5, -1)[:, xf]
    return dict(unew=out, dt=dt)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "sweep"):
        return _exact_sweep(case, seed)
    if kind == "level":
        return _exact_level(case, seed)
    if kind == "serve":
        return _exact_serve(case, seed)
    if kind == "amr_sweep":
        return _exact_amr_sweep(case, seed)
    # the recursion over levels, with its refinement map, is no plain
    # expression; amr_sweep stands for its level sweep
    return None
