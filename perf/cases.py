"""Performance cases of the MI355X assembly library: what a program that uses it runs over and over.

Each case is one pass through the package's public entry points on a synthetic model whose
inputs come from a seed:

frame    Newton assembly (SweepX{0} :iter) of a space frame: jittered lattice nodes, beams along
         x, y and z with lognormal sections, the base clamped by Holds. With `host` the state goes
         up and Lλ and nzval come back, as for a factorization on the host; otherwise the state
         lies on the device and the results stay there.
chains   dynamic assembly (SweepX{1,2} :iter or :step) of catenary mooring lines of uneven
         element counts with inertia, added mass, drag and roll inertia, on the device.
sweep    time steps of such lines (SweepX{2}): the state up, per step a :step and some :iter
         iterations with the device chain solve, the last step's X, X′, X″ back.
solve    the whole call solve(SweepX[0]) of a cantilever's load steps with the device solve.
limit    dg/dA, dg/dU of the top displacements of tensioned risers (LimitStateGradient).
vjp      the adjoint gradients of ΣΛᵀR: static cantilevers under U-loads (OX = 0) or dynamic
         A-scaled lines with a load on every node (OX = 2); Λ up, the gradients back.
direct   one DirectXUA{2,0,0} step of a curved beam with a U-load (AssemblyDirect): gradient and blocks.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "muscade.jl_amd"))

FIELDS = ("t1", "t2", "t3", "r1", "r2", "r3")
DT = 0.05

# EA, EI₂, EI₃, GJ, μ, ι₁, w, then Ca, Cl, Cq along the three axes
STEEL = np.array([2.1e9, 2.1e6, 2.1e6, 2e-5 * 2.1e11 / 2.6, 78.5, 0.157, 0.] + 9 * [0.])
LINE = np.array([5e9, 2e7, 2e7, 1.5e7, 1e3 / 9.81, 0.5, 1e3, 5., 1., 10., 72., 5., 300., 72., 5., 300.])


def listed():
    return [
        # a frame of an ordinary static analysis's size per Newton iteration: latency
        dict(name="frame_small", family="frame", nx=5, ny=4, nz=3, host=True),
        # a building-sized frame, its matrix used on the device
        dict(name="frame_medium", family="frame", nx=33, ny=29, nz=11, host=False),
        # assembly at scale: the 973,400-beam lattice of the repository's benchmark
        dict(name="frame_large", family="frame", nx=100, ny=100, nz=33, host=False),
        # a handful of lines: the first iteration of a step, with its ∂R/∂δr
        dict(name="chains_step", family="chains", OX=2, mission="step", nchain=13, nmin=300, nmax=2100),
        # many long lines: the other iterations
        dict(name="chains_iter_large", family="chains", OX=2, mission="iter", nchain=40, nmin=1000, nmax=20000),
        # first order in time, as for quasi-static lines with damping
        dict(name="chains_iter_first_order", family="chains", OX=1, mission="iter", nchain=24, nmin=100, nmax=4000),
        # one line through four time steps: launches count
        dict(name="sweep_small", family="sweep", nchain=1, nmin=101, nmax=101, steps=4, iters=5),
        # a mooring system's batch through four time steps
        dict(name="sweep_large", family="sweep", nchain=150, nmin=500, nmax=2500, steps=4, iters=5),
        # the whole call of the reference's static case, a 100-beam cantilever in 10 load steps
        dict(name="solve_cantilever", family="solve", nel=100, nstep=10),
        # a reliability search's gradients for a batch of risers
        dict(name="limit_risers", family="limit", nmodel=180, nmin=60, nmax=200),
        # gradients of a batch of static models
        dict(name="vjp_static_batch", family="vjp", OX=0, nmodel=60, nmin=500, nmax=5000),
        # one step of an identification: the blocks of DirectXUA
        dict(name="direct_step", family="direct", nel=230),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    f = rng.choice(("frame", "frame", "chains", "chains", "sweep", "solve", "limit", "vjp", "vjp", "direct"))
    if f == "frame":
        nx, ny, nz = _logint(rng, 3, 60), _logint(rng, 3, 60), _logint(rng, 2, 33)
        return dict(family=f, nx=nx, ny=ny, nz=nz, host=nx * ny * nz < 2000 and rng.random() < 0.5)
    if f == "chains":
        nmax = _logint(rng, 50, 12000)
        return dict(family=f, OX=rng.choice((1, 2, 2)), mission=rng.choice(("iter", "iter", "step")),
                    nchain=_logint(rng, 1, 40), nmin=max(1, nmax // rng.randint(2, 20)), nmax=nmax)
    if f == "sweep":
        nmax = _logint(rng, 50, 2000)
        return dict(family=f, nchain=_logint(rng, 1, 60), nmin=max(20, nmax // rng.randint(1, 8)), nmax=nmax,
                    steps=rng.randint(1, 4), iters=5)
    if f == "solve":
        return dict(family=f, nel=_logint(rng, 10, 150), nstep=rng.randint(3, 12))
    if f == "limit":
        nmax = _logint(rng, 40, 200)
        return dict(family=f, nmodel=_logint(rng, 1, 180), nmin=max(20, nmax // rng.randint(1, 6)), nmax=nmax)
    if f == "vjp":
        nmax = _logint(rng, 60, 5000)
        return dict(family=f, OX=rng.choice((0, 2)), nmodel=_logint(rng, 1, 40), nmin=max(20, nmax // rng.randint(1, 10)),
                    nmax=nmax)
    return dict(family=f, nel=_logint(rng, 10, 400))


# ---------------------------------------------------------------- inputs, from the seed alone
def _smooth(rng, s, length, tangent, amp):
    """A smooth field of small displacements (n, 3) along a line and the rotations that go with it."""
    u, du = np.zeros((s.size, 3)), np.zeros((s.size, 3))
    for k in range(1, 5):
        a, p = rng.normal(0., amp / k ** 2, 3), rng.uniform(0., 2. * np.pi, 3)
        u += a * np.sin(k * np.pi * s[:, None] + p)
        du += a * (k * np.pi / length) * np.cos(k * np.pi * s[:, None] + p)
    return np.concatenate([u, np.cross(tangent, du)], axis=1)


def _line(rng, n, kind, size=1.):
    """One line of n elements: nodes (n+1, 3), its X, X′, X″ per node (3, n+1, 6), `size` times
    the kind's ordinary motion."""
    s = np.linspace(0., 1., n + 1)
    if kind == "catenary":
        length = rng.uniform(500., 2000.)
        x = np.stack([0.8 * length * s, 0. * s, 0.5 * length * (np.cosh(1.5 * s) - 1.) / (np.cosh(1.5) - 1.)], axis=1)
        amp = (0.05, 0.1, 0.1)
    elif kind == "riser":                       # vertical, elements of 2 m
        length = 2. * n
        x = np.stack([0. * s, 0. * s, length * s], axis=1)
        amp = (0.002 * length, 0., 0.)
    else:                                       # a cantilever along x, elements of 0.05 m
        length = 0.05 * n
        x = np.stack([length * s, 0. * s, 0. * s], axis=1)
        amp = (0.001 * length, 0., 0.)
    t = np.gradient(x, s, axis=0) if n > 1 else np.repeat(x[1:] - x[:1], 2, axis=0)
    t /= np.linalg.norm(t, axis=1)[:, None]
    return x, np.stack([_smooth(rng, s, length, t, size * a) for a in amp])


class _Inputs:
    """xyz (nodes), pairs (beam end nodes), o2, sec, node states X (3, nnod, 6); holds (field →
    nodes); per-element U-node (or None) and A-node numbers counted from 0."""


def _inputs(case, seed):
    rng = np.random.default_rng([seed, 77])
    q, f = _Inputs(), case["family"]
    q.u = q.a = q.tops = None
    if f == "frame":
        n = (case["nx"], case["ny"], case["nz"])
        g = np.stack(np.meshgrid(*[np.arange(m) for m in n], indexing="ij"), axis=-1).transpose(2, 1, 0, 3).reshape(-1, 3)
        nid = lambda c: c[:, 0] + n[0] * (c[:, 1] + n[1] * c[:, 2])   # noqa: E731
        q.xyz = g + rng.uniform(-0.01, 0.01, g.shape)
        pairs, o2 = [], []
        for axis in range(3):
            a = g[g[:, axis] < n[axis] - 1]
            pairs.append(np.stack([nid(a), nid(a + np.eye(3, dtype=int)[axis])], axis=1))
            o2.append(np.tile([[0., 1., 0.], [0., 0., 1.], [0., 1., 0.]][axis], (len(a), 1)))
        q.pairs, q.o2 = np.concatenate(pairs), np.concatenate(o2)
        q.sec = np.tile(STEEL, (len(q.pairs), 1))
        q.sec[:, :4] *= rng.lognormal(0., 0.2, (len(q.pairs), 4))
        base = nid(g[g[:, 2] == 0])
        q.holds = [(k, base) for k in range(6)]
        X = rng.normal(0., 1e-3, (len(g), 6))
        X[:, 3:] *= 10.
        q.X = np.stack([X, 0. * X, 0. * X])
        return q
    kind = {"chains": "catenary", "sweep": "catenary", "limit": "riser"}.get(f)
    if kind is None:
        kind = "catenary" if f == "vjp" and case["OX"] else "cantilever"
    if f == "direct":
        ne = [case["nel"]]
    else:
        size = case.get("nchain", case.get("nmodel"))     # the same uneven counts for every seed
        ne = np.random.default_rng(size).integers(case["nmin"], case["nmax"] + 1, size=size).tolist()
    xyz, X, pairs, first, last, at = [], [], [], [], [], 0
    for c, n in enumerate(ne):
        x, st = _line(rng, n, kind, 0.1 if f == "sweep" else 1.)   # time steps: motions that converge in each step
        x[:, 1] += 50. * c
        if f == "direct":
            x[:, 2] += 0.02 * x[:, 0] ** 2
        xyz.append(x)
        X.append(st)
        pairs.append(np.stack([at + np.arange(n), at + 1 + np.arange(n)], axis=1))
        first.append(at)
        last.append(at + n)
        at += n + 1
    q.xyz, q.X, q.pairs = np.concatenate(xyz), np.concatenate(X, axis=1), np.concatenate(pairs)
    first, last = np.array(first), np.array(last)
    q.tops, q.ne = last, ne
    ntot = len(q.pairs)
    q.o2 = np.tile([0., 1., 0.], (ntot, 1))
    q.sec = np.tile(STEEL if kind == "cantilever" else LINE, (ntot, 1))
    rep = np.repeat(np.arange(len(ne)), ne)
    within = np.concatenate([np.arange(n) for n in ne])
    frac = within / np.repeat(ne, ne)
    if f in ("limit", "vjp", "direct"):
        q.holds = [(k, first) for k in range(6)]
    else:
        q.holds = [(k, first) for k in range(3)]
    if f == "limit":
        q.sec[:, 6:] = 0.
        q.holds += [(5, last)]
        q.u = rep * 8 + np.minimum((frac * 8).astype(int), 7)
        q.a = rep * 16 + np.minimum((frac * 16).astype(int), 15)
        q.X[0, :, 2] = q.xyz[:, 2] * (1e6 / LINE[0])          # the taut riser
        length = 2. * np.repeat(ne, 8)
        q.U = rng.normal(0., 0.1, (8 * len(ne), 3))
        q.U[:, 0] += 1.
        q.U *= (0.04 * 1e6 / length)[:, None]
        q.A = rng.normal(0., 0.1 / np.log(10.), 16 * len(ne))
    elif f == "vjp" and case["OX"]:
        q.u, q.U = q.pairs[:, 0], rng.normal(100., 50., (len(q.xyz), 3))
        q.a, q.A = rep * 16 + np.minimum((frac * 16).astype(int), 15), rng.normal(0., 0.05, 16 * len(ne))
    elif f == "vjp":
        q.sec[:, :4] *= np.repeat(rng.lognormal(0., 0.1, len(ne)), ne)[:, None]
        q.u, q.U = rep * 8 + np.minimum((frac * 8).astype(int), 7), rng.normal(0., 1e3, (8 * len(ne), 3))
    elif f == "direct":
        q.sec = np.tile(LINE, (ntot, 1))
        q.u, q.U = np.zeros(ntot, int), rng.normal(0., 1e2, (1, 3))
    q.lam = rng.normal(0., 1., (len(q.xyz), 6))
    return q


def _topload(t, F0=1e5, T=10.):
    return F0 * np.sin(2. * np.pi * t / T)


def _tension(t, T=1e6):
    return T


def _number(q):
    """First-encounter X numbering of the nodes along the elements: rank of each node."""
    flat = q.pairs.ravel()
    u, first = np.unique(flat, return_index=True)
    rank = np.full(len(q.xyz), -1)
    rank[u[np.argsort(first)]] = np.arange(u.size)
    return rank


def _vector(q, rank, values, nlam):
    """Node values (nnod, 6) as an X vector, the multipliers zero."""
    x = np.zeros(6 * len(q.xyz) + nlam)
    x[:-nlam if nlam else None].reshape(-1, 6)[rank] = values
    return x


def _model(case, q):
    """The model of the inputs and its initial state, by the package's own calls."""
    import muscade_amd as mc
    model = mc.Model(case["family"])
    mc.addnode(model, q.xyz)
    nodes = q.pairs + 1
    El = mc.EulerBeam3D
    kw = dict(mat=q.sec, orient2=q.o2)
    if q.u is not None:
        El = mc.EulerBeam3DU
        if len(q.U) == len(q.xyz):
            nodes = np.concatenate([nodes, nodes[:, :1]], axis=1)
        else:
            u0 = mc.addnode(model, np.zeros((len(q.U), 3)) - 10.)
            nodes = np.concatenate([nodes, u0[q.u][:, None]], axis=1)
    if q.a is not None:
        El = mc.EulerBeam3DAU
        a0 = mc.addnode(model, np.zeros((len(q.A), 3)) - 20.)
        nodes = np.concatenate([nodes, a0[q.a][:, None]], axis=1)
        kw.update(scaled=("EA", "EI₂", "EI₃", "GJ"), afield="Ξk")
    mc.addelement(model, El, nodes, **kw)
    for k, held in q.holds:
        mc.addelement(model, mc.Hold, (held + 1).reshape(-1, 1), field=FIELDS[k])
    if case["family"] in ("chains", "sweep"):
        mc.addelement(model, mc.DofLoad, (q.tops + 1).reshape(-1, 1), field="t1", value=_topload)
    if case["family"] == "limit":
        mc.addelement(model, mc.DofLoad, (q.tops + 1).reshape(-1, 1), field="t3", value=_tension)
    state = mc.initialize(model, nXder=3, time=0.)
    q.nlam = sum(len(h) for _, h in q.holds)
    q.rank = _number(q)
    for d in range(3):
        state.X[d][:] = _vector(q, q.rank, q.X[d], q.nlam)
    if q.u is not None:
        dn = model.dofnode("U")
        ids = np.stack([model.getdofID("U", FIELDS[k]) for k in range(3)], axis=1) - 1
        first = 0 if len(q.U) == len(q.xyz) else u0[0] - 1
        for k in range(3):
            state.U[0][ids[:, k]] = q.U[dn[ids[:, k]] - first, k]
    if q.a is not None:
        state.A[:] = q.A[model.dofnode("A") - (a0[0] - 1)]
    return mc, model, state


class _View:
    """An array of the library's as torch takes it; the tensor holds this, and this its owner."""

    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=2)


def _device_results(mc, asm):
    """The assembled Lλ and Lλx.nzval where they lie on the device."""
    r, k = ctypes.POINTER(ctypes.c_double)(), ctypes.POINTER(ctypes.c_double)()
    asm.ctx.check(mc.lib.mh_device_outputs(asm.ctx.h, ctypes.byref(r), ctypes.byref(k)), "device outputs")
    return [torch.as_tensor(_View(asm, ctypes.cast(p, ctypes.c_void_p).value, n), device="cuda")
            for p, n in ((r, asm.nX), (k, asm.nnz))]


def prepare(case, seed):
    f = case["family"]
    if f == "solve":
        return _prepare_solve(case, seed)
    q = _inputs(case, seed)
    mc, model, state = _model(case, q)
    s = dict(case=case, mc=mc, state=state)
    if f == "frame":
        asm = s["asm"] = mc.AssemblySweepX(0, model, state.dis, graph=True)
        if not case["host"]:
            asm.set_state(state, state.time)
            s["out"] = _device_results(mc, asm)
    elif f == "chains":
        asm = s["asm"] = mc.AssemblySweepX(case["OX"], model, state.dis, graph=True)
        asm.c = mc.Newmarkβcoefficients(case["OX"], DT)
        asm.set_state(state, state.time)
        s["out"] = _device_results(mc, asm)
    elif f == "sweep":
        from muscade_amd.chainsolve import ChainSolver
        asm = s["asm"] = mc.AssemblySweepX(2, model, state.dis, graph=True)
        s["solver"] = ChainSolver(asm)
    elif f == "limit":
        s["grad"] = mc.LimitStateGradient(model, state.dis)
        s["grad"].out.set_state(state, state.time)
        tip = np.array([6 * q.rank[n] + 1 for n in q.tops], np.int64)
        s["dgdX"] = (tip, np.ones(tip.size))
    elif f == "vjp":
        asm = s["asm"] = mc.AssemblySweepX(case["OX"], model, state.dis, graph=True)
        asm.set_state(state, state.time)
        s["lam"] = _vector(q, q.rank, q.lam, q.nlam)
    else:
        s["asm"] = mc.AssemblyDirect(2, 0, 0, model, state.dis)
        s["lam"] = _vector(q, q.rank, q.lam, q.nlam)
    return s


def _prepare_solve(case, seed):
    import muscade_amd as mc
    rng = np.random.default_rng([seed, 78])
    n = case["nel"]
    model = mc.Model("cantilever")
    x = np.linspace(0., 10., n + 1)
    mc.addnode(model, np.stack([x, 0. * x, 0. * x], axis=1))
    nodes = np.stack([np.arange(1, n + 1), np.arange(2, n + 2)], axis=1)
    sec = np.tile(STEEL, (n, 1))
    sec[:, :4] *= rng.lognormal(0., 0.1, (n, 4))
    mc.addelement(model, mc.EulerBeam3D, nodes, mat=sec, orient2=np.array([0., 1., 0.]))
    for k in FIELDS:
        mc.addelement(model, mc.Hold, [1], field=k)
    F = float(rng.uniform(4e4, 6e4)) / 10
    mc.addelement(model, mc.DofLoad, [n + 1], field="t3", value=lambda t: F * t)
    return dict(case=case, mc=mc, state=mc.initialize(model, time=0.))


def run(s):
    case, mc = s["case"], s["mc"]
    f = case["family"]
    if f == "frame" and case["host"]:
        return s["asm"].assemble(s["state"], "iter")
    if f in ("frame", "chains"):
        s["asm"].assemble(s["state"], case.get("mission", "iter"), fetch=False, upload=False)
        return s["out"]
    if f == "sweep":
        asm, solver = s["asm"], s["solver"]
        for step in range(1, case["steps"] + 1):
            asm.c = mc.Newmarkβcoefficients(2, DT)
            asm.set_state(s["state"], step * DT, X=step == 1)
            c6 = asm.c.array()
            for it in range(case["iters"]):
                norms = solver.iteration_graph(2, it == 0, c6)
        out = s["state"].copy()
        solver.fetch_X(out, 2)
        return out.X
    if f == "solve":
        out = mc.solve(mc.SweepX[0], initialstate=s["state"], time=np.arange(1., case["nstep"] + 1.), maxΔx=1e-8,
                       verbose=False, catcherror=False, linsolve="device")
        return [o.X[0] for o in out]
    if f == "limit":
        gA, gU, _ = s["grad"](s["state"], s["dgdX"], upload=False, check=False)
        return gA, gU
    if f == "vjp":
        return s["asm"].vjp(s["state"], s["lam"], upload=False)
    L1, L2 = s["asm"].assemble(s["state"], s["lam"], "matrices", 1.0)
    return ([L1[c][0] for c in ("Λ", "X", "U")], [m.data for m in L2[("Λ", "X")][0]], [m[0].data for m in L2[("X", "Λ")]],
            L2[("Λ", "U")][0][0].data, L2[("U", "Λ")][0][0].data)


def _counts(case):
    f = case["family"]
    if f == "frame":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        nodes = nx * ny * nz
        beams = (nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1)
        return nodes, beams, 6 * nx * ny
    if f in ("solve", "direct"):
        return case["nel"] + 1, case["nel"], 6
    n = case.get("nchain", case.get("nmodel"))
    beams = n * (case["nmin"] + case["nmax"]) // 2
    return beams + n, beams, n * {"limit": 7, "vjp": 6}.get(f, 3)


def work(case):
    """Each input read once (state, node coordinates, and per beam its two nodes, orientation and
    section) and each output written once; operations of a closed-form element of each kind."""
    f = case["family"]
    nodes, beams, holds = _counts(case)
    nX = 6 * nodes + holds
    nnz = 36 * (nodes + 2 * beams) + 3 * holds
    OX = case.get("OX", {"sweep": 2, "direct": 2}.get(f, 0))
    read = (OX + 1) * 8 * nX + 24 * nodes + beams * (8 + 24 + (128 if OX else 40))
    flops = beams * (12000. if OX else 2500.)
    if f in ("frame", "chains"):
        return dict(bytes=read + 8 * (nX + nnz), flops=flops)
    solve = 6 ** 3 * 8. * nodes
    if f in ("sweep", "solve"):
        n = case["steps"] * case["iters"] if f == "sweep" else 5 * case["nstep"]
        return dict(bytes=n * (read + 8 * nnz + 8 * (OX + 1) * nX), flops=n * (flops + solve))
    if f == "limit":
        return dict(bytes=read + 8 * nnz + 8 * nX, flops=2 * flops + solve)
    if f == "vjp":
        return dict(bytes=read + 8 * nX + 8 * (OX + 1) * nX, flops=flops)
    return dict(bytes=read + 8 * nX + 8 * 6 * nnz, flops=3 * flops)


# ---------------------------------------------------------------- the element in plain torch, 64 bits
# Jets: lists of the time levels of a quantity (value, first and second time derivative).
def _add(a, b):
    return [x + y for x, y in zip(a, b)]


def _sub(a, b):
    return [x - y for x, y in zip(a, b)]


def _scl(c, a):
    return [c * x for x in a]


def _mul(a, b):
    r = [a[0] * b[0]]
    if len(a) > 1:
        r.append(a[1] * b[0] + a[0] * b[1])
    if len(a) > 2:
        r.append(a[2] * b[0] + 2. * a[1] * b[1] + a[0] * b[2])
    return r


def _poly(c, a):
    r = [torch.full_like(a[0], c[-1])] + [torch.zeros_like(a[0]) for _ in a[1:]]
    for x in c[-2::-1]:
        r = _mul(r, a)
        r[0] = r[0] + x
    return r


# sin θ/θ in θ², and θ² = acos²(1−u) in u (twice the series of arcsin² at √(u/2))
_SINC = [(-1.) ** k / math.factorial(2 * k + 1) for k in range(14)]
_ACOS2 = [0.] + [2. * 2. ** n / (n * n * math.comb(2 * n, n)) for n in range(1, 45)]


def _rodrigues(v):
    """I + sinc(θ)S + ½sinc²(θ/2)S², the square by the reference's power rule on time levels
    (the second level keeps only s·s̈: src/Adiff.jl:230)."""
    x, y, z = v
    t = _add(_add(_mul(x, x), _mul(y, y)), _mul(z, z))
    a, s = _poly(_SINC, t), _poly(_SINC, _scl(0.25, t))
    b = [0.5 * s[0] * s[0]] + ([s[0] * s[1]] if len(s) > 1 else []) + ([s[0] * s[2]] if len(s) > 2 else [])
    xx, yy, zz = _mul(x, x), _mul(y, y), _mul(z, z)
    one = lambda q: [q[0] + 1.] + q[1:]   # noqa: E731
    off = lambda p, w, sg: _add(_scl(sg, _mul(a, w)), _mul(b, p))   # noqa: E731
    return [[one(_scl(-1., _mul(b, _add(yy, zz)))), off(_mul(x, y), z, -1.), off(_mul(x, z), y, 1.)],
            [off(_mul(x, y), z, 1.), one(_scl(-1., _mul(b, _add(xx, zz)))), off(_mul(y, z), x, -1.)],
            [off(_mul(x, z), y, -1.), off(_mul(y, z), x, 1.), one(_scl(-1., _mul(b, _add(xx, yy))))]]


def _mm(A, B):
    return [[_add(_add(_mul(A[i][0], B[0][j]), _mul(A[i][1], B[1][j])), _mul(A[i][2], B[2][j])) for j in range(3)]
            for i in range(3)]


def _tr(A):
    return [[A[j][i] for j in range(3)] for i in range(3)]


def _mv(A, v):
    return [_add(_add(_mul(A[i][0], v[0]), _mul(A[i][1], v[1])), _mul(A[i][2], v[2])) for i in range(3)]


def _log(M):
    """Rodrigues⁻¹: spin⁻¹(M)/sinc(acos((tr M − 1)/2))."""
    u = _scl(-0.5, _add(_add(M[0][0], M[1][1]), M[2][2]))
    u[0] = u[0] + 1.5
    sc = _poly(_SINC, _poly(_ACOS2, u))
    inv = [1. / sc[0]]
    if len(sc) > 1:
        inv.append(-sc[1] * inv[0] ** 2)
    if len(sc) > 2:
        inv.append((2. * sc[1] ** 2 * inv[0] - sc[2]) * inv[0] ** 2)
    return [_mul(_scl(0.5, _sub(M[i][j], M[j][i])), inv) for i, j in ((2, 1), (0, 2), (1, 0))]


class _Beams:
    """R of a slice of beams with its graph: X (levels of (n, 12)), U (n, 3), a (n,)."""

    def __init__(self, q, sl, OX, dev, dofs):
        T = lambda v: torch.as_tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)   # noqa: E731
        p = q.pairs[sl]
        n = len(p)
        self.X = [T(q.X[d][p].reshape(n, 12)).requires_grad_() for d in range(OX + 1)]
        self.U = T(q.U[q.u[sl]]).requires_grad_() if q.u is not None else torch.zeros(n, 3, dtype=torch.float64, device=dev)
        self.a = T(q.A[q.a[sl]]).requires_grad_() if q.a is not None else torch.zeros(n, dtype=torch.float64, device=dev)
        sec = T(q.sec[sl])
        k = 10. ** self.a
        EA, EI2, EI3, GJ = (sec[:, i] * k for i in range(4))
        c1, c2, o2 = T(q.xyz[p[:, 0]]), T(q.xyz[p[:, 1]]), T(q.o2[sl])
        tg = c2 - c1
        L = tg.norm(dim=1)
        t = tg / L[:, None]
        o2 = o2 / o2.norm(dim=1)[:, None]
        nn = o2 - (o2 * t).sum(1)[:, None] * t
        nn = nn / nn.norm(dim=1)[:, None]
        rm = torch.stack([t, nn, torch.linalg.cross(t, nn)], dim=2)
        s30, s65 = math.sqrt(30.), math.sqrt(6. / 5.)
        z1, z2 = 0.5 * math.sqrt(3. / 7. + 2. / 7. * s65), 0.5 * math.sqrt(3. / 7. - 2. / 7. * s65)
        zg = (-z1, -z2, z2, z1)
        wg = ((18. - s30) / 72., (18. + s30) / 72., (18. + s30) / 72., (18. - s30) / 72.)
        kin = self._kinematics(self.X, rm, tg, L, zg)
        rsm, cs, ul, vl, xg = kin
        # loads at the Gauss points from the time levels, then R = ∂Π/∂X₀ with the loads held
        r0 = [[rsm[i][j][0] for j in range(3)] for i in range(3)]
        lev = lambda q_, d: q_[d] if d <= OX else torch.zeros_like(L)   # noqa: E731
        mu, iota, w = sec[:, 4], sec[:, 5], sec[:, 6]
        fe = []
        for g in range(4):
            xd, xdd = [lev(xg[g][i], 1) for i in range(3)], [lev(xg[g][i], 2) for i in range(3)]
            l1 = [sum(r0[i][j] * xd[i] for i in range(3)) for j in range(3)]
            l2 = [sum(r0[i][j] * xdd[i] for i in range(3)) for j in range(3)]
            b = [sec[:, 7 + 3 * j] * l2[j] + sec[:, 8 + 3 * j] * l1[j] + sec[:, 9 + 3 * j] * l1[j] * l1[j].abs()
                 for j in range(3)]
            fe.append(torch.stack([mu * xdd[i] + sum(r0[i][j] * b[j] for j in range(3)) + (w if i == 2 else 0.) - self.U[:, i]
                                   for i in range(3)], dim=1))
        r2 = [[lev(rsm[i][j], 2) for j in range(3)] for i in range(3)]
        m1 = 0.5 * iota * sum(r0[i][2] * r2[i][1] - r0[i][1] * r2[i][2] for i in range(3))
        self.loads = [torch.stack(fe, dim=1), torch.stack([r0[i][0] * m1 for i in range(3)], dim=1)]
        held = self.held = [x.detach().requires_grad_() for x in self.loads]
        # the same kinematics at the value level alone
        rsm, cs, ul, vl, xg = self._kinematics(self.X[:1], rm, tg, L, zg) if OX else kin
        ax = ul[0][0] + 0.5 * L
        eps = (ax * ax + ul[1][0] ** 2 + ul[2][0] ** 2).sqrt() * 2. / L - 1.
        E = 0.5 * EA * eps * eps * L
        for g in range(4):
            dL, z = wg[g] * L, zg[g]
            ku, kv = -24. * z / L ** 2, 2. / L
            k1, k2, k3 = kv * vl[0][0], ku * ul[1][0] + kv * vl[2][0], ku * ul[2][0] - kv * vl[1][0]
            E = E + dL * 0.5 * (GJ * k1 * k1 + EI3 * k2 * k2 + EI2 * k3 * k3)
            E = E + dL * sum(held[0][:, g, i] * xg[g][i][0] for i in range(3))
        if OX:
            vs = _log([[rsm[i][j][:1] for j in range(3)] for i in range(3)])
            E = E + L * sum(held[1][:, i] * vs[i][0] for i in range(3))
        self.R = torch.autograd.grad(E.sum(), self.X[0], create_graph=True)[0]
        self.OX, self.n = OX, n
        self.idx = torch.as_tensor(dofs[p].reshape(n, 12), device=dev)

    @staticmethod
    def _kinematics(X, rm, tg, L, zg):
        c = lambda k: [x[:, k] for x in X]   # noqa: E731
        u1, v1, u2, v2 = [c(k) for k in range(3)], [c(k) for k in range(3, 6)], [c(k) for k in range(6, 9)], [c(k) for k in range(9, 12)]
        R1, R2 = _rodrigues(v1), _rodrigues(v2)
        dv = [_scl(0.5, p) for p in _log(_mm(R2, _tr(R1)))]
        R1m = [[_add(_add(_scl(rm[:, 0, j], R1[i][0]), _scl(rm[:, 1, j], R1[i][1])), _scl(rm[:, 2, j], R1[i][2]))
                for j in range(3)] for i in range(3)]
        rsm = _mm(_rodrigues(dv), R1m)
        cs = [_scl(0.5, _add(u1[k], u2[k])) for k in range(3)]
        dd = [_sub(u2[k], cs[k]) for k in range(3)]
        dd = [[dd[k][0] + 0.5 * tg[:, k]] + dd[k][1:] for k in range(3)]
        ul, vl = _mv(_tr(rsm), dd), _mv(_tr(rsm), dv)
        ul[0] = [ul[0][0] - 0.5 * L] + ul[0][1:]
        xg = []
        for z in zg:
            ya, yu, yv = 2. * z, -4. * z ** 3 + 3. * z, (z * z - 0.25) * L
            p = [_scl(ya, ul[0]), _add(_scl(yu, ul[1]), _scl(yv, vl[2])), _sub(_scl(yu, ul[2]), _scl(yv, vl[1]))]
            p[0] = [p[0][0] + L * z] + p[0][1:]
            x = _mv(rsm, p)
            xg.append([_add(x[k], cs[k]) for k in range(3)])
        return rsm, cs, ul, vl, xg

    def pull(self, w):
        """The derivatives of Σ w·R in X (all levels), U and a."""
        g = torch.autograd.grad((w * self.R).sum(), [self.X[0]] + self.held + [self.a] * self.a.requires_grad,
                                retain_graph=True, allow_unused=True)
        z = lambda v, x: torch.zeros_like(x) if v is None else v   # noqa: E731
        ins = self.X + [self.U] * self.U.requires_grad
        outs = [(l, z(h, l)) for l, h in zip(self.loads, g[1:3]) if l.requires_grad]
        dX, dU = [torch.zeros_like(x) for x in self.X], torch.zeros_like(self.U)
        if outs:
            h = torch.autograd.grad([o for o, _ in outs], ins, [v for _, v in outs], retain_graph=True, allow_unused=True)
            dX = [z(v, x) for v, x in zip(h, self.X)]
            dU = z(h[len(self.X)], self.U) if self.U.requires_grad else dU
        dX[0] = dX[0] + g[0]
        return dX, dU, z(g[3], self.a) if self.a.requires_grad else torch.zeros_like(self.a)

    def jacobians(self):
        """∂R/∂X⁽ᵈ⁾ (n, 12, 12) of every level and ∂R/∂U (n, 12, 3)."""
        J, JU = [[] for _ in self.X], []
        for i in range(12):
            w = torch.zeros_like(self.R)
            w[:, i] = 1.
            dX, dU, _ = self.pull(w)
            for d, v in enumerate(dX):
                J[d].append(v)
            JU.append(dU)
        return [torch.stack(j, dim=1) for j in J], torch.stack(JU, dim=1)


def _slices(n, size):
    return [slice(a, min(a + size, n)) for a in range(0, n, size)]


def exact(case, seed):
    f = case["family"]
    if f in ("sweep", "solve"):     # trajectories of Newton iterations: no closed value
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    q = _inputs(case, seed)
    rank = _number(q)
    dofs = 6 * rank[:, None] + np.arange(6)
    lamd, nX = [], 6 * len(q.xyz)
    for k, h in q.holds:
        lamd.append((dofs[h, k], nX + np.arange(len(h))))
        nX += len(h)
    ne = len(q.pairs)
    T = lambda v: torch.as_tensor(v, dtype=torch.float64, device=dev)   # noqa: E731
    I = lambda v: torch.as_tensor(v, device=dev)   # noqa: E731
    OX = case.get("OX", 2 if f == "direct" else 0)
    x0 = T(_vector(q, rank, q.X[0], nX - 6 * len(q.xyz)))
    if f in ("frame", "chains", "direct"):
        rhs, keys, vals, ukeys, uvals = torch.zeros(nX, dtype=torch.float64, device=dev), [], [[] for _ in range(OX + 1)], [], []
        step = f == "chains" and case["mission"] == "step"
        gam, bet = 0.5, 0.25
        if OX == 1:
            a1, a2, a3, b1, b2, b3 = 1. / (gam * DT), 1. / gam, 0., 0., 0., 0.
        else:
            a1, a2, a3 = gam / (bet * DT), gam / bet, (gam / (2. * bet) - 1.) * DT
            b1, b2, b3 = 1. / (bet * DT ** 2), 1. / (bet * DT), 1. / (2. * bet)
        for sl in _slices(ne, 120000 if OX else 250000):
            e = _Beams(q, sl, OX, dev, dofs)
            J, JU = e.jacobians()
            r = e.R.detach()
            if step:
                X = [x.detach() for x in e.X] + [0.]
                r = r - (J[1] @ (a2 * X[1] + a3 * X[2])[:, :, None])[:, :, 0]
                if OX == 2:
                    r = r - (J[2] @ (b2 * X[1] + b3 * X[2])[:, :, None])[:, :, 0]
            rhs.index_add_(0, e.idx.reshape(-1), r.reshape(-1))
            if f == "chains":
                J = [J[0] + a1 * J[1] + (b1 * J[2] if OX == 2 else 0.)]
            # column by column: key = column · nX + row
            keys.append((e.idx[:, None, :] * nX + e.idx[:, :, None]).reshape(-1))
            for v, j in zip(vals, J):
                v.append(j.reshape(-1))
            if f == "direct":
                ukeys.append((torch.arange(3, device=dev)[None, None, :] * nX + e.idx[:, :, None]).reshape(-1))
                uvals.append(JU.reshape(-1))
            del e, J, JU
        gX = torch.zeros_like(rhs)
        lam = T(_vector(q, rank, q.lam, nX - 6 * len(q.xyz))) if f == "direct" else None
        for h, l in lamd:
            h, l = I(h), I(l)
            rhs[h] -= x0[l]
            rhs[l] -= x0[h]
            one = torch.ones(len(h), dtype=torch.float64, device=dev)
            keys += [h * nX + h, l * nX + h, h * nX + l, l * nX + l]
            for d, v in enumerate(vals):
                v += [0. * one, -one * (d == 0), -one * (d == 0), 0. * one]
            if f == "direct":
                gX[h] -= lam[l]
                gX[l] -= lam[h]
        if f == "chains":
            rhs[I(dofs[q.tops, 0])] -= _topload(0.)
        keys = torch.cat(keys)
        u, inv = torch.unique(keys, return_inverse=True)
        nz = []
        for v in vals[:1 if f == "chains" else None]:
            nz.append(torch.zeros(u.numel(), dtype=torch.float64, device=dev).index_add_(0, inv, torch.cat(v)))
        if f != "direct":
            return [rhs, nz[0]]
        # the transposed blocks: the entry (row, column) of the pattern holds the value of (column, row)
        at = torch.searchsorted(u, (u % nX) * nX + torch.div(u, nX, rounding_mode="floor"))
        uu, uinv = torch.unique(torch.cat(ukeys), return_inverse=True)
        un = torch.zeros(uu.numel(), dtype=torch.float64, device=dev).index_add_(0, uinv, torch.cat(uvals))
        # (U, Λ): column-major over the dofs, three rows each
        order = torch.argsort((uu % nX) * 3 + torch.div(uu, nX, rounding_mode="floor"))
        return ([rhs, gX, torch.zeros(3, dtype=torch.float64, device=dev)], nz, [v[at] for v in nz], un, un[order])
    nU, nA = q.U.size, len(q.A) if q.a is not None else 0
    # U and A are numbered as the elements meet them: their own order here, but for the last node of a line
    meet = lambda v: np.unique(v)[np.argsort(np.unique(v, return_index=True)[1])]   # noqa: E731
    gU = torch.zeros(q.U.shape, dtype=torch.float64, device=dev)
    gA = torch.zeros(nA, dtype=torch.float64, device=dev)
    if f == "vjp":
        gX = torch.zeros(OX + 1, nX, dtype=torch.float64, device=dev)
        for sl in _slices(ne, 120000):
            e = _Beams(q, sl, OX, dev, dofs)
            dX, dU, da = e.pull(T(q.lam[q.pairs[sl]].reshape(-1, 12)))
            for d in range(OX + 1):
                gX[d].index_add_(0, e.idx.reshape(-1), dX[d].reshape(-1))
            gU.index_add_(0, I(q.u[sl]), dU)
            if nA:
                gA.index_add_(0, I(q.a[sl]), da)
        lam = T(_vector(q, rank, q.lam, nX - 6 * len(q.xyz)))
        for h, l in lamd:
            gX[0][I(h)] -= lam[I(l)]
            gX[0][I(l)] -= lam[I(h)]
        return (list(gX), gU[I(meet(q.u))].reshape(-1), gA[I(meet(q.a))] if nA else gA)
    # limit: K μ = ∂g/∂X riser by riser (held dofs fixed), then −μᵀ ∂R/∂(A, U)
    held = np.zeros(nX, bool)
    for h, _ in lamd:
        held[h] = True
    mu = torch.zeros(nX, dtype=torch.float64, device=dev)
    e = _Beams(q, slice(0, ne), 0, dev, dofs)
    K = e.jacobians()[0][0].detach()
    e0 = 0
    for m, n in enumerate(q.ne):
        ix = e.idx[e0:e0 + n]
        d0, nd = int(ix.min()), 6 * (n + 1)
        A = torch.zeros(nd * nd, dtype=torch.float64, device=dev)
        A.index_add_(0, ((ix[:, :, None] - d0) * nd + (ix[:, None, :] - d0)).reshape(-1), K[e0:e0 + n].reshape(-1))
        A = A.reshape(nd, nd)
        free = I(np.nonzero(~held[d0:d0 + nd])[0])
        A = A[free][:, free]
        b = torch.zeros(nX, dtype=torch.float64, device=dev)
        b[int(dofs[q.tops[m], 0])] = 1.
        b = b[d0:d0 + nd][free]
        LU, piv = torch.linalg.lu_factor(A)
        x = torch.linalg.lu_solve(LU, piv, b[:, None])
        for _ in range(2):
            x = x + torch.linalg.lu_solve(LU, piv, b[:, None] - A @ x)
        mu[free + d0] = x[:, 0]
        e0 += n
    _, dU, da = e.pull(-mu[e.idx])
    gU.index_add_(0, I(q.u), dU)
    gA.index_add_(0, I(q.a), da)
    return gA[I(meet(q.a))], gU[I(meet(q.u))].reshape(-1)
