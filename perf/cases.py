"""Performance cases: the runs a user of the framework does, through its public entry points.

One pass advances a prepared solver (or batch, or coupled pair) by the steps
between two outputs and takes its state to the host, as a driver's output
loop does; the adjoint cases evaluate an objective and its gradient through
``torch.autograd``.  The state goes through the C ABI into pinned memory that
the program keeps.

Families (sizes, options and parameters are those of ``hom3_amd.cases``, of
``hom3_amd.batch`` and of the tests and the benchmark):

* ``vortex``   2D Euler, MUSCL, periodic, full uniform grids: the reference's
  own verification case, run from coarse grids (launch latency) to 4 M cells;
* ``tgv``      3D Navier-Stokes Taylor-Green vortex, full uniform grids: the
  production flow solve, FP64 and FP32 stage states;
* ``blast``    3D Euler blast on 2:1 refined grids: ragged leaf counts from
  some ten thousand to 5 M, zero-gradient boundaries;
* ``batch``    many independent refined 2D Riemann problems of uneven size in
  one batch: parameter studies;
* ``channel``  conjugate heat transfer: fluid channel over a heated block,
  both solvers coupled every step, walls, inflow and outflow;
* ``adjoint``  the same case's wall heat flux and its gradient with respect
  to the solid's sources (reverse mode, stored, checkpointed or binomial).

``exact`` evaluates the same schemes in plain torch, FP64, without the
framework: dense arrays for the uniform grids, gathered neighbours on a tree
built here for the refined ones, torch's autograd for the gradient.
"""
import ctypes
import functools
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import hom3_amd as H
from hom3_amd import adjoint, batch, cases
from hom3_amd import _lib as L

GAMMA, GM1 = 1.4, 0.4
SUTHERLAND = 110.4 / 273.15
TR0 = 0.01       # ratio of the solid's to the fluid's diffusive time scale
KRATIO = 100.0   # conductivity ratio of the channel case


def listed():
    return [
        # coarse grids: a step is a few launches of microseconds each
        dict(name="vortex 256^2", family="vortex", level=8, precision="fp64", steps=100),
        dict(name="tgv 32^3", family="tgv", level=5, precision="fp64", steps=50),
        # grids that fill the GPU
        dict(name="vortex 2048^2 fp32", family="vortex", level=11, precision="fp32", steps=40),
        dict(name="tgv 128^3 fp32", family="tgv", level=7, precision="fp32", steps=50),
        # the largest production solve
        dict(name="tgv 256^3", family="tgv", level=8, precision="fp64", steps=40),
        # refined grids: the thin shell (0.8 M leaves) and the refined ball (5 M)
        dict(name="blast shell", family="blast", base=6, extra=2, band=0.025, precision="fp64", steps=60),
        dict(name="blast ball fp32", family="blast", base=6, extra=2, band=0.2, precision="fp32", steps=40),
        # parameter studies: a few instances, and enough for the whole GPU
        dict(name="batch 12", family="batch", count=12, low=6, high=8, precision="fp64", steps=40),
        dict(name="batch 48 fp32", family="batch", count=48, low=6, high=9, precision="fp32", steps=30),
        # the coupled step, and its gradient with every step kept or recomputed
        dict(name="channel 128", family="channel", level=7, precision="fp64", steps=60),
        dict(name="adjoint 64", family="adjoint", level=6, ckpt=0, steps=40),
        dict(name="adjoint 128 checkpointed", family="adjoint", level=7, ckpt=10, steps=30),
    ]


def draw(rng):
    family = rng.choice(["vortex", "tgv", "blast", "batch", "channel", "adjoint"])
    precision = rng.choice(["fp64", "fp32"])
    if family == "vortex":
        return dict(family=family, level=rng.randint(5, 11), precision=precision, steps=rng.randint(10, 60))
    if family == "tgv":
        return dict(family=family, level=rng.randint(3, 7), precision=precision, steps=rng.randint(10, 60))
    if family == "blast":
        return dict(family=family, base=rng.randint(4, 6), extra=rng.randint(1, 2),
                    band=round(math.exp(rng.uniform(math.log(0.02), math.log(0.2))), 4), precision=precision,
                    steps=rng.randint(10, 40))
    if family == "batch":
        low = rng.randint(5, 7)
        return dict(family=family, count=rng.randint(2, 40), low=low, high=rng.randint(low, 9), precision=precision,
                    steps=rng.randint(10, 30))
    if family == "channel":
        return dict(family=family, level=rng.randint(5, 7), precision=precision, steps=rng.randint(10, 60))
    return dict(family=family, level=rng.randint(4, 6), ckpt=rng.choice([0, 5, 10, -4]), steps=rng.randint(10, 40))


# ---- inputs, from the seed alone -------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _uniform(seed, *shape):
    dev = _device()
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    return torch.rand(*shape, generator=g, device=dev, dtype=torch.float64)


def _conserved(u, rho, p):
    """(rho u.., rho, rho E) stacked along the first axis."""
    e = p / GM1 + 0.5 * rho * sum(c * c for c in u)
    return torch.stack([rho * c for c in u] + [rho, e])


@functools.lru_cache(maxsize=4)
def _morton(level, nd):
    """Cells of a uniform grid in solver (Morton) order: (nd, n) integer coordinates."""
    m = np.arange(1 << (nd * level), dtype=np.int64)
    c = np.zeros((nd, m.size), np.int64)
    for b in range(level):
        for d in range(nd):
            c[d] |= ((m >> (nd * b + d)) & 1) << b
    return c


def _flat(coords, shape):
    """Index into a dense array of `shape`, flattened, of every cell."""
    i = np.zeros(coords.shape[1], np.int64)
    for c, n in zip(coords, shape):
        i = i * n + c
    return torch.from_numpy(i).to(_device())


def _infinity(mach):
    T = 1.0 / (1.0 + 0.5 * GM1 * mach * mach)
    return mach * math.sqrt(T), T ** (1.0 / GM1), T ** (GAMMA / GM1) / GAMMA


def _vortex_field(level, seed):
    """Isentropic vortex with a centre and a strength of its own, [0, 10]^2."""
    n = 1 << level
    r = np.random.default_rng(seed)
    centre, beta = r.uniform(3.0, 7.0, 2), r.uniform(4.0, 5.0)
    x = (torch.arange(n, device=_device(), dtype=torch.float64) + 0.5) * (10.0 / n)
    dx, dy = torch.meshgrid(x - centre[0], x - centre[1], indexing="ij")
    f = torch.exp(1.0 - dx * dx - dy * dy)
    rho = (1.0 - GM1 * beta * beta * f * f / (16.0 * GAMMA * math.pi ** 2)) ** (1.0 / GM1)
    return _conserved([1.0 - beta * f * dy / (2 * math.pi), 1.0 + beta * f * dx / (2 * math.pi)], rho, rho ** GAMMA)


def _tgv_field(level, seed):
    """Taylor-Green vortex, Mach 0.1, with 1% noise on the density."""
    n = 1 << level
    v0, rho, p = _infinity(0.1)
    x = (torch.arange(n, device=_device(), dtype=torch.float64) + 0.5) * (2 * math.pi / n)
    X, Y, Z = torch.meshgrid(x, x, x, indexing="ij")
    u = [v0 * X.sin() * Y.cos() * Z.cos(), -v0 * X.cos() * Y.sin() * Z.cos(), torch.zeros_like(X)]
    p = p + rho * v0 * v0 / 16.0 * ((2 * X).cos() + (2 * Y).cos()) * ((2 * Z).cos() + 2.0)
    return _conserved(u, rho * (1.0 + 0.01 * (2.0 * _uniform(seed, n, n, n) - 1.0)), p)


def _blast_cells(x, seed):
    """Blast of radius 0.2 in the unit cube at the cell centres x (3, n), 1% noise on the density."""
    inside = ((x - 0.5) ** 2).sum(0).sqrt() < 0.2
    one = torch.ones_like(x[0])
    rho = torch.where(inside, one, 0.125 * one) * (1.0 + 0.01 * (2.0 * _uniform(seed, x.shape[1]) - 1.0))
    zero = torch.zeros_like(one)
    return _conserved([zero, zero, zero], rho, torch.where(inside, 10.0 * one, 0.1 * one))


def _channel_shape(level):
    n = 1 << level
    return (n, n // 2, n // 2), (n // 4, n // 8, n // 4)


def _channel_fields(level, seed):
    """Fluid at the inflow state with 1% velocity noise, solid at the fluid's temperature with 1% noise, sources U[0,1]."""
    fluid, solid = _channel_shape(level)
    u, rho, p = _infinity(0.2)
    noise = 0.02 * u * (_uniform(seed, 3, *fluid) - 0.5)
    one = torch.ones(fluid, device=_device(), dtype=torch.float64)
    T = GAMMA * p / rho * (1.0 + 0.02 * (_uniform(seed + 1, *solid) - 0.5))
    return _conserved([u + noise[0], noise[1], noise[2]], rho * one, p * one), T, _uniform(seed + 2, *solid)


@functools.lru_cache(maxsize=4)
def _channel_order(level):
    """Dense flat index of every fluid and solid cell in solver order."""
    n = 1 << level
    c = _morton(level, 3)
    out = []
    for lo, shape in zip(((0, n // 4, 0), (3 * n // 8, n // 8, n // 8)), _channel_shape(level)):
        k = np.all([(c[d] >= lo[d]) & (c[d] < lo[d] + shape[d]) for d in range(3)], axis=0)
        out.append(_flat(c[:, k] - np.array(lo)[:, None], shape))
    return out


def _instances(case, seed):
    """The study's grids (drawn once), and the four states of every instance from the seed."""
    levels = tuple(range(case["low"], case["high"] + 1))
    grids = H.four_quadrant_instances(2024, case["count"], levels=levels)
    states = H.four_quadrant_instances(seed, case["count"], levels=levels)
    return [dict(g, ic=s["ic"]) for g, s in zip(grids, states)]


# ---- what a user's program holds before the call ------------------------------------------

def _set_state(solver, q):
    """q: (nvars, internal cells) in solver order; the ghosts are filled by the solver."""
    n, first_ghost = solver.counts()
    full = np.empty((solver.nvars, n))
    full[:, :first_ghost] = q.cpu().numpy()
    full[:, first_ghost:] = full[:, :1]
    solver.set_lhs(full)


def _pinned(*shape):
    return torch.empty(*shape, dtype=torch.float64, pin_memory=torch.cuda.is_available())


def _pointer(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))


def _read(solver, out):
    """The solver's cells into the program's buffer; the internal ones are the result."""
    L.check(L.lib().hom3g_solver_download_state(solver.ctx.h, solver.id, _pointer(out), out.shape[1]))
    return out[:, : solver.first_gc]


def prepare(case, seed):
    family = case["family"]
    ctx = H.Context(0)
    if family in ("vortex", "tgv"):
        build = cases.vortex if family == "vortex" else cases.tgv
        nd = 2 if family == "vortex" else 3
        g, s = build(H, case["level"], precision=case["precision"], ctx=ctx)
        q = (_vortex_field if family == "vortex" else _tgv_field)(case["level"], seed)
        _set_state(s, q.reshape(nd + 2, -1)[:, _flat(_morton(case["level"], nd), q.shape[1:])])
        return dict(case=case, ctx=ctx, solver=s, out=_pinned(s.nvars, s.ncells))
    if family == "blast":
        g, s, _ = cases.blast(H, base=case["base"], extra=case["extra"], band=case["band"], amp=0.0, ctx=ctx,
                              precision=case["precision"])
        x = np.ascontiguousarray(s.topology()["x_center"][:, : s.first_gc])
        _set_state(s, _blast_cells(torch.from_numpy(x).to(_device()), seed))
        return dict(case=case, ctx=ctx, solver=s, out=_pinned(s.nvars, s.ncells))
    if family == "batch":
        solvers = [batch.build_instance(H, p, ctx=ctx) for p in _instances(case, seed)]
        b = H.Batch(solvers, case["precision"])
        for s in solvers:
            s.close()
        b.autotune()
        return dict(case=case, ctx=ctx, batch=b, out=[_pinned(b.nvars, n) for n in b.n_int])
    order = _channel_order(case["level"])
    fluid, solid, source = _channel_fields(case["level"], seed)
    precision = case.get("precision", "fp64")
    g, cns, heat, _ = cases.channel_cht(H, level=case["level"], kratio=KRATIO, ctx=ctx, precision=precision)
    _set_state(cns, fluid.reshape(5, -1)[:, order[0]])
    _set_state(heat, solid.reshape(1, -1)[:, order[1]])
    source = source.reshape(-1)[order[1]]
    heat.set_source(source.cpu().numpy())
    if family == "channel":
        return dict(case=case, ctx=ctx, cns=cns, heat=heat, out=[_pinned(s.nvars, s.ncells) for s in (cns, heat)])
    start = adjoint.Snapshot(cns, heat)
    _, dts = adjoint.cht_objective(cns, heat, TR0, case["steps"])
    return dict(case=case, ctx=ctx, cns=cns, heat=heat, start=start, dts=dts, flux=adjoint.WallHeatFlux(),
                source=source.detach().clone().requires_grad_(True))


def run(state):
    case = state["case"]
    family = case["family"]
    if family in ("vortex", "tgv", "blast"):
        s = state["solver"]
        s.solve(case["steps"])
        return dict(q=_read(s, state["out"]), time=s.time())
    if family == "batch":
        b = state["batch"]
        b.solve(case["steps"])
        for i, out in enumerate(state["out"]):
            L.check(L.lib().hom3g_batch_download_state(b.ctx.h, b.id, i, _pointer(out), out.shape[1]))
        return dict(q=state["out"])
    if family == "channel":
        H.coupling.apply_and_step(TR0, state["cns"], state["heat"], case["steps"])
        return dict(fluid=_read(state["cns"], state["out"][0]), solid=_read(state["heat"], state["out"][1]),
                    time=state["cns"].time())
    source = state["source"]
    source.grad = None
    J = state["flux"].apply(source, state["cns"], state["heat"], TR0, state["dts"], state["start"], case["ckpt"])
    J.backward()
    return dict(J=J.detach(), grad=source.grad)


# ---- what one pass cannot do without --------------------------------------------------------

def work(case):
    """Bytes: every SSP-RK3 stage reads its input (and U^n) and writes its output once, FP64 or FP32 stage states;
    flops: the face fluxes (about 60 flops for AUSM, 150 more for the viscous part, 60 for MUSCL) and the update."""
    family, steps = case["family"], case["steps"]
    fp32 = case.get("precision") == "fp32"
    if family == "adjoint":
        fluid, solid = (math.prod(s) for s in _channel_shape(case["level"]))
        # forward (stage states kept) and reverse: state and adjoint, read and written
        return dict(bytes=3 * steps * (5 * fluid + solid) * 8 * (8 / 3 + 4), flops=3 * steps * 3 * 210 * fluid * 4)
    if family == "channel":
        fluid, solid = (math.prod(s) for s in _channel_shape(case["level"]))
        return dict(bytes=3 * steps * (5 * fluid + solid) * (16 if fp32 else 64 / 3), flops=3 * steps * 3 * 210 * fluid)
    if family == "vortex":
        cells, nd, face = 4 ** case["level"], 2, 120
    elif family == "tgv":
        cells, nd, face = 8 ** case["level"], 3, 210
    elif family == "blast":
        cells, nd, face = _tree(3, case["base"], case["extra"], (0.5, 0.5, 0.5), 0.2, case["band"])["n"], 3, 60
    else:
        # the mean base grid, and the refinement of a disc of radius 0.2 by one level on average
        levels = range(case["low"], case["high"] + 1)
        cells, nd, face = int(1.6 * case["count"] * sum(4 ** k for k in levels) / len(levels)), 2, 60
    nv = nd + 2
    return dict(bytes=3 * steps * cells * nv * (16 if fp32 else 64 / 3), flops=3 * steps * cells * (nd * face + 10 * nv))


# ---- the same schemes in plain torch, FP64 -----------------------------------------------------

def _prims(q):
    nd = q.shape[0] - 2
    u = q[:nd] / q[nd]
    p = GM1 * (q[nd + 1] - 0.5 * q[nd] * (u * u).sum(0))
    return u, p, (GAMMA * p / q[nd]).sqrt()


def _ausm(qL, qR, d):
    """Liou-Steffen flux along d; leading axis: the conserved variables."""
    nd = qL.shape[0] - 2
    (uL, pL, aL), (uR, pR, aR) = _prims(qL), _prims(qR)

    def split(M, s):
        out = M.abs() > 1.0
        m = torch.where(out, 0.5 * (M + s * M.abs()), s * 0.25 * (M + s) ** 2)
        p = torch.where(out, 0.5 * (1.0 + s * torch.sign(M)), 0.25 * (M + s) ** 2 * (2.0 - s * M))
        return m, p

    mL, wL = split(uL[d] / aL, 1.0)
    mR, wR = split(uR[d] / aR, -1.0)
    m = mL + mR
    left = m >= 0.0
    f = torch.where(left, torch.cat([qL[: nd + 1], (qL[nd + 1] + pL)[None]]) * aL,
                    torch.cat([qR[: nd + 1], (qR[nd + 1] + pR)[None]]) * aR) * m
    momentum = [f[k] + (wL * pL + wR * pR) if k == d else f[k] for k in range(nd)]
    return torch.stack(momentum + [f[nd], f[nd + 1]])


def _viscous(qL, qR, G, d, Re0, Pr):
    """Three-point viscous flux along d; G[sd]: gradient of the conserved variables along sd at the face."""
    nd = qL.shape[0] - 2
    qs = 0.5 * (qL + qR)
    rho, u = qs[nd], qs[:nd] / qs[nd]
    p = GM1 * (qs[nd + 1] - 0.5 * rho * (u * u).sum(0))
    du = [[(G[sd][c] - G[sd][nd] * u[c]) / rho for sd in range(nd)] for c in range(nd)]
    dp = GM1 * (G[d][nd + 1] - 0.5 * (G[d][nd] * (u * u).sum(0) + 2.0 * rho * sum(u[c] * du[c][d] for c in range(nd))))
    T = GAMMA * 0.5 * (_prims(qL)[1] + _prims(qR)[1]) / rho
    mu = T ** 1.5 * (1.0 + SUTHERLAND) / (T + SUTHERLAND)
    heat = -mu * GAMMA / (GM1 * Pr * rho) * (dp - p / rho * G[d][nd])
    div = 2.0 / 3.0 * sum(du[c][c] for c in range(nd))
    t = [-mu * (du[d][i] + du[i][d] - (div if i == d else 0.0)) for i in range(nd)]
    energy = sum(u[i] * t[i] for i in range(nd)) + heat
    return torch.stack(t + [torch.zeros_like(rho), energy]) / Re0


def _min_dt(q, h, cfl, visc=None):
    u, p, a = _prims(q)
    dt = cfl * h / (u.abs().amax(0) + a)
    if visc:
        Re0, Pr = visc
        T = a * a
        s = T ** 1.5 * (1.0 + SUTHERLAND) / (T + SUTHERLAND) / (q[-2] * h)
        dt = torch.minimum(dt, cfl * h / (2.0 * s * max(1.0 / Re0, 1.0 / (Re0 * Pr * GM1))))
    return dt.amin()


def _rk3(q, rhs):
    """SSP-RK3 with increments rhs(stage input)."""
    s = q + rhs(q)
    s = 0.75 * q + 0.25 * (s + rhs(s))
    return q / 3.0 + (2.0 / 3.0) * (s + rhs(s))


def _minmod(a, b):
    return torch.where(a * b <= 0.0, torch.zeros_like(a), torch.where(a.abs() < b.abs(), a, b))


def _vortex_exact(case, seed):
    q, h = _vortex_field(case["level"], seed), 10.0 / (1 << case["level"])
    time = 0.0
    for _ in range(case["steps"]):
        dt = _min_dt(q, h, 0.5)
        time += float(dt)

        def rhs(s):
            out = torch.zeros_like(s)
            for d in range(2):
                up = s.roll(-1, 1 + d)
                lim = _minmod(s - s.roll(1, 1 + d), up - s)
                f = _ausm(s + 0.5 * lim, (s - 0.5 * lim).roll(-1, 1 + d), d)
                out += f.roll(1, 1 + d) - f
            return dt / h * out

        q = _rk3(q, rhs)
    return dict(q=q.reshape(4, -1)[:, _flat(_morton(case["level"], 2), q.shape[1:])].cpu(), time=time)


def _cut(a, d, lo, hi):
    """a[lo:hi] along spatial axis d (negative hi: from the end; 0: to the end)."""
    n = a.shape[1 + d]
    return a.narrow(1 + d, lo, (n + hi if hi <= 0 else hi) - lo)


def _cns_increment(q, ghosts, wall, h, dt, visc):
    """dt/h times the Navier-Stokes fluxes into every cell of a box.  ghosts[d]: the layers below and above along d;
    wall[d]: per side, the factor on the momenta of the ghost's tangential slope (1, or 0 where the face sums
    opposite slopes: walls), a number or an array over the layer."""
    Re0, Pr = visc
    pad = [torch.cat([ghosts[d][0], q, ghosts[d][1]], 1 + d) for d in range(3)]
    slope = [(_cut(pad[d], d, 2, 0) - _cut(pad[d], d, 0, -2)) / (2.0 * h) for d in range(3)]
    out = torch.zeros_like(q)
    for d in range(3):
        qL, qR = _cut(pad[d], d, 0, -1), _cut(pad[d], d, 1, 0)
        G = [None] * 3
        for sd in range(3):
            if sd == d:
                G[sd] = (qR - qL) / h
                continue
            s = slope[sd]
            if wall is None:
                G[sd] = 0.5 * (torch.cat([_cut(s, d, s.shape[1 + d] - 1, 0), s], 1 + d) +
                               torch.cat([s, _cut(s, d, 0, 1)], 1 + d))
                continue
            ends = []
            for side in range(2):
                e = _cut(s, d, 0, 1) if side == 0 else _cut(s, d, s.shape[1 + d] - 1, 0)
                ends.append(torch.cat([e[:3] * wall[d][side], e[3:]]))
            G[sd] = torch.cat([ends[0], 0.5 * (_cut(s, d, 0, -1) + _cut(s, d, 1, 0)), ends[1]], 1 + d)
        f = _ausm(qL, qR, d) + _viscous(qL, qR, G, d, Re0, Pr)
        out = out + (_cut(f, d, 0, -1) - _cut(f, d, 1, 0))
    return dt / h * out


def _re0(mach, re):
    u, rho, p = _infinity(mach)
    T = GAMMA * p / rho
    return re * T ** 1.5 * (1.0 + SUTHERLAND) / (T + SUTHERLAND) / (rho * u)


def _tgv_exact(case, seed):
    q, h = _tgv_field(case["level"], seed), 2 * math.pi / (1 << case["level"])
    visc = (_re0(0.1, 1600.0), 0.71)
    time = 0.0
    for _ in range(case["steps"]):
        dt = _min_dt(q, h, 0.5, visc)
        time += float(dt)
        q = _rk3(q, lambda s: _cns_increment(
            s, [(_cut(s, d, s.shape[1 + d] - 1, 0), _cut(s, d, 0, 1)) for d in range(3)], None, h, dt, visc))
    return dict(q=q.reshape(5, -1)[:, _flat(_morton(case["level"], 3), q.shape[1:])].cpu(), time=time)


@functools.lru_cache(maxsize=2)
def _tree(nd, base, extra, centre, radius, band):
    """Leaves of the unit box in solver order: `base` levels everywhere, `extra` more where the sphere's surface is
    within `band`, 2:1 balanced.  Neighbours, and the finer cells behind a face, as index arrays."""
    coords = [_morton(base, nd).T]
    level = [np.full(coords[0].shape[0], base)]
    refined = [np.zeros(coords[0].shape[0], bool)]
    dense = {l: np.full((1 << l,) * nd, -1, np.int32) for l in range(base, base + extra + 1)}
    dense[base][tuple(coords[0].T)] = np.arange(coords[0].shape[0])
    child = np.array([[(k >> d) & 1 for d in range(nd)] for k in range(1 << nd)])

    def table():
        return np.concatenate(coords), np.concatenate(level), np.concatenate(refined)

    def refine(flag):
        c, l, r = table()
        k = np.nonzero(flag)[0]
        r[k] = True
        new = (2 * c[k][:, None, :] + child[None]).reshape(-1, nd)
        lev = np.repeat(l[k] + 1, 1 << nd)
        coords[:], level[:], refined[:] = [c, new], [l, lev], [r, np.zeros(len(new), bool)]
        for q in np.unique(lev):
            dense[q][tuple(new[lev == q].T)] = len(c) + np.nonzero(lev == q)[0]
        return len(k)

    while True:
        c, l, r = table()
        h = 0.5 ** l
        dist = np.sqrt(sum(((c[:, d] + 0.5) * h - centre[d]) ** 2 for d in range(nd))) - radius
        if not refine(~r & (l < base + extra) & (np.abs(dist) <= band + 0.5 * h * math.sqrt(nd))):
            break
    while True:
        c, l, r = table()
        flag = np.zeros(len(c), bool)
        for q in range(base + 1, base + extra):
            for k in range(2 * nd):
                n = c[r & (l == q)].copy()
                n[:, k // 2] += 1 if k % 2 else -1
                n = n[((n >= 0) & (n < 1 << q)).all(1)]
                n = n[dense[q][tuple(n.T)] < 0]
                for up in range(q - 1, base - 1, -1):
                    n = n >> 1
                    at = dense[up][tuple(n.T)]
                    flag[at[at >= 0]] = True
                    n = n[at < 0]
        if not refine(flag & ~r):
            break
    c, l, r = table()
    leaf = np.nonzero(~r)[0]
    cell = np.full(len(c), -1, np.int64)
    cell[leaf] = np.arange(len(leaf))
    c, l = c[leaf], l[leaf]
    first = {q: np.nonzero(l == q)[0] for q in np.unique(l)}
    nghbr = np.tile(np.arange(len(leaf)), (2 * nd, 1))  # a zero-gradient ghost holds the cell itself
    fine = []
    for k in range(2 * nd):
        d, step = k // 2, 1 if k % 2 else -1
        cells, subs = [], []
        for q, i in first.items():
            n = c[i].copy()
            n[:, d] += step
            ok = (n[:, d] >= 0) & (n[:, d] < 1 << q)
            i, n = i[ok], n[ok]
            at = dense[q][tuple(n.T)]
            same = at >= 0
            nghbr[k, i[same]] = cell[at[same]]
            if q > base:
                up = dense[q - 1][tuple((n[~same] >> 1).T)]
                nghbr[k, i[~same]] = cell[up]
            inner = same.copy()
            inner[same] = cell[at[same]] < 0
            if inner.any():
                facing = child[child[:, d] == (0 if k % 2 else 1)]
                sub = 2 * n[inner][:, None, :] + facing[None]
                cells.append(i[inner])
                subs.append(cell[dense[q + 1][tuple(sub.reshape(-1, nd).T)]].reshape(-1, len(facing)))
                nghbr[k, i[inner]] = i[inner]
        fine.append((np.concatenate(cells), np.concatenate(subs)) if cells else None)
    return dict(n=len(leaf), x=((c + 0.5) * (0.5 ** l)[:, None]).T.copy(), h=0.5 ** l, nghbr=nghbr, fine=fine)


def _refined_exact(tree, q, steps, cfl):
    """First-order Euler on a tree's leaves."""
    dev = q.device
    h = torch.from_numpy(tree["h"]).to(dev)
    nb = [torch.from_numpy(k).to(dev) for k in tree["nghbr"]]
    fine = [None if f is None else (torch.from_numpy(f[0]).to(dev), torch.from_numpy(f[1]).to(dev)) for f in tree["fine"]]
    time = 0.0
    for _ in range(steps):
        dt = _min_dt(q, h, cfl)
        time += float(dt)

        def rhs(s):
            out = torch.zeros_like(s)
            for k, n in enumerate(nb):
                d, upper = k // 2, k % 2
                f = _ausm(s, s[:, n], d) if upper else _ausm(s[:, n], s, d)
                if fine[k] is not None:
                    c, sub = fine[k]
                    own, other = s[:, c][:, :, None].expand(-1, -1, sub.shape[1]), s[:, sub]
                    f[:, c] = (_ausm(own, other, d) if upper else _ausm(other, own, d)).mean(2)
                out += -f if upper else f
            return dt / h * out

        q = _rk3(q, rhs)
    return q.cpu(), time


def _blast_exact(case, seed):
    tree = _tree(3, case["base"], case["extra"], (0.5, 0.5, 0.5), 0.2, case["band"])
    q, time = _refined_exact(tree, _blast_cells(torch.from_numpy(tree["x"]).to(_device()), seed), case["steps"], 0.1)
    return dict(q=q, time=time)


def _batch_exact(case, seed):
    out = []
    for p in _instances(case, seed):
        half = 0.5 * p["radius"]
        tree = _tree(2, p["level"], p["extra"], tuple(p["centre"]), half, half if p["extra"] else -1e9)
        x = torch.from_numpy(tree["x"]).to(_device())
        # the cell mean of the four states by two Gauss points per axis: a quadrant edge is always a cell edge
        k = (x[0] >= 0.5).long() + 2 * (x[1] >= 0.5).long()
        pv = torch.tensor(p["ic"][2:], dtype=torch.float64, device=x.device).reshape(4, 4)[k].T
        out.append(_refined_exact(tree, _conserved([pv[0], pv[1]], pv[2], pv[3]), case["steps"], 0.4)[0])
    return dict(q=out)


class _Channel:
    """The channel over the heated block in dense arrays: fluid (5, n, n/2, n/2), solid (n/4, n/8, n/4)."""

    def __init__(self, level):
        n = 1 << level
        self.h, self.mach = 1.0 / n, 0.2
        self.visc = (_re0(0.2, 1000.0), 0.71)
        u, rho, p = _infinity(0.2)
        self.inflow, self.p_out = (u, 0.0, 0.0, rho), p
        self.x, self.z = slice(3 * n // 8, 5 * n // 8), slice(n // 8, 3 * n // 8)  # the block's top, in fluid cells
        self.scaling = TR0 * self.visc[1] * self.visc[0]

    def interface(self, fluid, solid):
        """Temperature of the conjugate interface from the cells on its two sides."""
        q = fluid[:, self.x, 0, self.z]
        Tf = GAMMA * _prims(q)[1] / q[3]
        return (Tf + KRATIO * solid[:, -1]) / (1.0 + KRATIO)

    def ghosts(self, q, Ts):
        def state(b, u, rho, p):
            return _conserved(u, rho, p)

        def wall(b):
            return torch.cat([-b[:3], b[3:]])

        ends = [(_cut(q, d, 0, 1), _cut(q, d, q.shape[1 + d] - 1, 0)) for d in range(3)]
        b = ends[0][0]
        u, p, _ = _prims(b)
        I = self.inflow
        inflow = _conserved([2.0 * I[k] - u[k] for k in range(3)], 2.0 * I[3] - b[3], p)
        b = ends[0][1]
        u, p, _ = _prims(b)
        outflow = _conserved(list(u), b[3], 2.0 * self.p_out - p)
        lower = wall(ends[1][0])
        b = q[:, self.x, 0, self.z]
        u, p, _ = _prims(b)
        top = _conserved([-c for c in u], 2.0 * p * GAMMA / Ts - b[3], p)
        lower = torch.cat([lower[:, : self.x.start], torch.cat(
            [lower[:, self.x, :, : self.z.start], top[:, :, None, :], lower[:, self.x, :, self.z.stop:]], 3),
            lower[:, self.x.stop:]], 1)
        return [(inflow, outflow), (lower, wall(ends[1][1])), (wall(ends[2][0]), wall(ends[2][1]))]

    def fluid_step(self, fluid, solid, dt):
        Ts = self.interface(fluid, solid)
        slip = [(1.0, 1.0), (0.0, 0.0), (0.0, 0.0)]
        return _rk3(fluid, lambda s: _cns_increment(s, self.ghosts(s, Ts), slip, self.h, dt, self.visc))

    def solid_step(self, fluid, solid, source, dt):
        Ts = self.interface(fluid, solid)

        def rhs(T):
            out = torch.zeros_like(T)
            for d in range(3):
                first, last = T.narrow(d, 0, 1), T.narrow(d, T.shape[d] - 1, 1)
                pad = torch.cat([first, T, (2.0 * Ts[:, None] - last) if d == 1 else last], d)
                f = pad.diff(dim=d) / self.h
                out = out + f.diff(dim=d)
            return dt / self.h * out + dt * source

        return _rk3(solid, rhs)

    def dt(self, fluid):
        heat = 0.3 * 0.5 * self.h * self.h
        return torch.clamp(_min_dt(fluid, self.h, 0.4, self.visc), max=heat / self.scaling)

    def flux(self, fluid, solid, dt):
        return dt * self.scaling * (self.h * 2.0 * (solid[:, -1] - self.interface(fluid, solid))).sum()


def _channel_exact(case, seed):
    C = _Channel(case["level"])
    order = _channel_order(case["level"])
    fluid, solid, source = _channel_fields(case["level"], seed)
    if case["family"] == "channel":
        time = 0.0
        for _ in range(case["steps"]):
            dt = C.dt(fluid)
            time += float(dt)
            fluid = C.fluid_step(fluid, solid, dt)
            solid = C.solid_step(fluid, solid, source, dt * C.scaling)
        return dict(fluid=fluid.reshape(5, -1)[:, order[0]].cpu(), solid=solid.reshape(1, -1)[:, order[1]].cpu(),
                    time=time)
    source = source.requires_grad_(True)

    def step(fluid, solid, dt):
        fluid = C.fluid_step(fluid, solid, dt)
        solid = C.solid_step(fluid, solid, source, dt * C.scaling)
        return fluid, solid, C.flux(fluid, solid, dt)

    J = 0.0
    for _ in range(case["steps"]):
        dt = C.dt(fluid.detach())
        fluid, solid, q = checkpoint(step, fluid, solid, dt, use_reentrant=False)
        J = J + q
    grad, = torch.autograd.grad(J, source)
    return dict(J=J.detach().cpu(), grad=grad.reshape(-1)[order[1]].cpu())


def exact(case, seed):
    family = case["family"]
    if family == "vortex":
        return _vortex_exact(case, seed)
    if family == "tgv":
        return _tgv_exact(case, seed)
    if family == "blast":
        return _blast_exact(case, seed)
    if family == "batch":
        return _batch_exact(case, seed)
    return _channel_exact(case, seed)
