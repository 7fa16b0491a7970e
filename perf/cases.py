"""The work a solver program has this framework do, as measurable cases.

A case is one run segment of a program on a patch grid, the way
``drnum_amd/apps/drnum_run.cpp`` is written: hand the field to the device
(updateDevice), advance it some Runge-Kutta steps, fetch every patch's field
(updateHost).  The grid, its donor tables and its device context are kept
between segments, as such a program keeps them; the fields are new each time.

``mode`` says how the program steps:
  step    one rk_step call per step (HIP_RungeKutta, drnum_run's ``hip``)
  graph   rk_graph_run (``graph``)
  loop    copyField, copyDonorData, compute and the post operation as separate
          calls (RungeKutta over the virtual iterator interface, ``rk``)
  cfl     rk_step, then the diagnostics of the new field, from which the next
          time step is chosen (``cfl=<target>``)
  output  no steps: what a program writes at an output interval (the
          post-processing variables of every patch, the conservation sums, the
          diagnostics and the last step's density change)
``tune`` says whether the program called autotune once after setting up its
grid, as bench.py does, or takes the default work list, as drnum_run does.

The inputs are smooth random disturbances, other ones for every seed, on each
configuration's initial flow.
"""
import collections
import math

import numpy as np
import torch

from drnum_amd import configs, hip, host

GAMMA, R_GAS, CP, CV = 1.4, 287.2, 1004.5, 717.5
ALPHA = (0.25, 0.5, 1.0)
CFL_TARGET = 0.25  # of the x axis alone, as diagnostics gives it; the jet runs along z
# the largest number of global cells times stages that exact() evaluates (about 15 s)
EXACT_CELL_STAGES = 5.5e9


def _case(name, flow, core, blocks, dtype, mode, steps, tune=False):
    case = {"flow": flow, "core": core, "blocks": blocks, "dtype": dtype, "mode": mode, "steps": steps, "tune": tune}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a grid for debugging a set-up: every launch is smaller than the chip, latency alone counts
        _case("jet8_tiny_f64", "jet", 8, 2, "f64", "step", 3),
        # the Sod tube of the validation suite: one patch in double precision, 100 replayed steps
        _case("sod64_f64", "sod", 64, 1, "f64", "graph", 100),
        # a small production grid of odd block size
        _case("jet27_odd_f32", "jet", 23, 3, "f32", "step", 60),
        # the subsonic jet on 64 patches, the main application: 200 steps between two outputs
        _case("jet64_f32", "jet", 64, 4, "f32", "step", 200),
        # the same jet started with the time step under CFL control
        _case("jet64_cfl_f32", "jet", 48, 4, "f32", "cfl", 60),
        # double precision on a mid-size jet grid, work list tuned once
        _case("jet27_f64", "jet", 48, 3, "f64", "step", 40, True),
        # the largest: a periodic shear-layer box in few large patches, tuned, replayed steps
        _case("kh8_large_f32", "kh", 192, 2, "f32", "graph", 100, True),
        # the periodic box through the reference's own stage loop, call by call
        _case("kh27_loop_f32", "kh", 40, 3, "f32", "loop", 60),
        # the viscous shear layer
        _case("shear64_visc_f32", "shear", 32, 4, "f32", "step", 100),
        # bodies in a free stream: a level-set fill and a second exchange in every stage
        _case("spheres12_f32", "spheres", 64, 3, "f32", "step", 100),
        # an uneven batch with nested refined patches: interpolating, multi-donor exchange
        _case("uneven60_f32", "uneven", 96, 60, "f32", "step", 60),
        # the output interval of the jet
        _case("jet64_output_f32", "jet", 48, 4, "f32", "output", 0),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    flow = rng.choice(("jet", "jet", "kh", "sod", "shear", "spheres", "uneven"))
    dtype = rng.choice(("f32", "f32", "f32", "f64"))
    tune = rng.random() < 0.3
    if flow == "sod":
        core, blocks = log_int(12, 160), 1
    elif flow == "spheres":
        core, blocks = log_int(24, 72), rng.choice((2, 3))
    elif flow == "uneven":
        core, blocks = log_int(32, 96), log_int(8, 60)
    else:
        blocks = rng.choice((1, 2, 3, 4)) if flow != "jet" else rng.choice((2, 3, 4))
        core = log_int(8, {1: 200, 2: 120, 3: 80, 4: 56}[blocks])
    mode = rng.choice(("step", "step", "graph", "loop", "cfl", "output"))
    cells = (core * blocks) ** 3 if flow not in ("uneven", "spheres") else core ** 3 * blocks * 4
    steps = 0 if mode == "output" else max(3, min(log_int(20, 150), int(1.2e9 / cells)))
    if dtype == "f64" and steps > 40:
        steps = 40
    return _case("", flow, core, blocks, dtype, mode, steps, tune)


# ---------------------------------------------------------------------------
# the grid and its device context, kept between a program's segments
# ---------------------------------------------------------------------------

def _workload(case):
    core, b = case["core"], case["blocks"]
    if case["flow"] == "jet":
        # a radius between two rings of cell centres: no centre lies on the edge
        return configs.jet(core=core, blocks=b, radius_cells=round(core * b / 16) + 0.37)
    if case["flow"] == "kh":
        return configs.kelvin_helmholtz(core=core, blocks=b)
    if case["flow"] == "shear":
        return configs.viscous_shear(core=core, blocks=(b, b, b))
    if case["flow"] == "spheres":
        return configs.levelset_spheres(core=core, blocks=(b, 2, 2), n_spheres=8,
                                        r_range=(core * 6.0 / 64.0, core * 14.0 / 64.0))
    if case["flow"] == "uneven":
        return configs.uneven_batch(n_patches=b, size_range=(16, core))
    return configs.sod(core)


_GRIDS = collections.OrderedDict()


def _grid(case):
    """(workload, context) of a case's grid; the last two grids are kept."""
    key = tuple(case[k] for k in ("flow", "core", "blocks", "dtype", "tune"))
    if key not in _GRIDS:
        while len(_GRIDS) >= 2:
            _GRIDS.popitem(last=False)
        w = _workload(case)
        dtype = np.float32 if case["dtype"] == "f32" else np.float64
        hg = host.HostGrid.from_workload(w, fp64_geometry=True)
        hg.compute_dependencies(w.periodic)
        ctx = hip.Context(dtype)
        ctx.set_operator(w.recon, w.limiter, w.viscous)
        hg.to_device(ctx)
        hg.upload_exchange(ctx)
        if w.spheres is not None:
            hg.levelset_spheres(w.spheres, w.ls_inner_layers, 0, w.ls_min_inner_rel)
            hg.upload_levelset(ctx)
        if case["tune"]:
            for p in range(len(w.patches)):
                ctx.upload(p, 0, w.initial_state(p, dtype))
            ctx.autotune()
        _GRIDS[key] = (w, ctx)
    _GRIDS.move_to_end(key)
    return _GRIDS[key]


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _extent(w):
    return [max(P.origin[a] + P.length[a] - (P.seek[2 * a + 1] * P.dx(a) if w.periodic[a] else 0.0) for P in w.patches)
            for a in range(3)]


def _disturbance(w, seed):
    """disturb(axes) -> (5, nx, ny, nz): smooth fields of amplitude about 1 from the
    seed, sums of four products of sines with whole periods in the box."""
    rng = np.random.RandomState(seed % (1 << 31))
    ext = _extent(w)
    modes = [[(rng.randint(1, 4, 3), rng.uniform(0.0, 2.0 * math.pi, 3)) for _ in range(4)] for _ in range(5)]

    def disturb(axes):
        out = []
        for q in range(5):
            tot = 0.0
            for wave, phase in modes[q]:
                s = [torch.sin(2.0 * math.pi * float(wave[a]) / ext[a] * axes[a] + float(phase[a])) for a in range(3)]
                tot = tot + 0.5 * s[0][:, None, None] * s[1][None, :, None] * s[2][None, None, :]
            out.append(tot)
        return torch.stack(out)

    return disturb


def _patch_state(w, case, P, disturb, dtype):
    """Conserved variables (5, ni, nj, nk) of patch P's first field, in the state type."""
    axes = [P.origin[a] + (np.arange(n) + 0.5) * P.dx(a) for a, n in enumerate((P.ni, P.nj, P.nk))]
    axes = [torch.tensor(x, dtype=torch.float64, device=_device()) for x in axes]
    d = disturb(axes)
    x, y = axes[0][:, None, None], axes[1][None, :, None]
    one = torch.ones_like(d[0])
    p, rho, u, v, wv = configs.P_AMB * one, one, 0.0 * one, 0.0 * one, 0.0 * one
    vel = 1.0  # the speed the disturbance is a fraction of
    if case["flow"] == "sod":
        left = (x < 0.5) & (one > 0)
        p, rho, vel = torch.where(left, 1.0, 0.1) * one, torch.where(left, 1.0, 0.125) * one, 0.0
    elif case["flow"] == "kh":
        inside = ((y % 1.0 > 0.25) & (y % 1.0 < 0.75)) & (one > 0)
        rho, u = torch.where(inside, 2.0, 1.0) * one, torch.where(inside, 0.5, -0.5) * one
    elif case["flow"] == "shear":
        L = _extent(w)[1]
        yy, vel = y % L, 30.0
        u = torch.where(yy < 0.5 * L, 30.0 * torch.tanh((yy - 0.25 * L) * 16.0 / L),
                        -30.0 * torch.tanh((yy - 0.75 * L) * 16.0 / L)) * one
        p, rho = 1.0e5 * one, 1.0e5 / (R_GAS * 300.0) * one
    elif case["flow"] == "spheres":
        u = 0.3 * one
    elif case["flow"] == "uneven":
        u = 0.5 * one
    p, rho = p * (1.0 + 0.01 * d[0]), rho * (1.0 + 0.01 * d[1])
    u, v, wv = u + 0.02 * vel * d[2], v + 0.02 * vel * d[3], wv + 0.02 * vel * d[4]
    e = p * (CV / R_GAS) + 0.5 * rho * (u * u + v * v + wv * wv)
    return torch.stack([rho, rho * u, rho * v, rho * wv, e]).to(dtype)


def prepare(case, seed):
    w, ctx = _grid(case)
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
    disturb = _disturbance(w, seed)
    fields = [_patch_state(w, case, P, disturb, dtype).reshape(5, -1).cpu().numpy() for P in w.patches]
    if case["mode"] == "output":
        # the program's last two fields are on the device when it comes to write
        before = [(f * (1.0 + 1.0e-3 * np.sin(1.0 + seed % 97))).astype(f.dtype) for f in fields]
        return {"case": dict(case), "w": w, "ctx": ctx, "fields": fields, "before": before}
    return {"case": dict(case), "w": w, "ctx": ctx, "fields": fields}


# ---------------------------------------------------------------------------
# one segment
# ---------------------------------------------------------------------------

def run(state):
    case, w, ctx = state["case"], state["w"], state["ctx"]
    patches = range(len(w.patches))
    for p in patches:
        ctx.upload(p, 0, state["fields"][p])
    mode, steps, dt = case["mode"], case["steps"], w.dt
    if mode == "output":
        for p in patches:
            ctx.upload(p, 1, state["before"][p])
        change = [ctx.variable_difference(p, 0, 0, 1, 0) for p in patches]
        out = [np.stack(list(ctx.post_variables(p, ("Ma", "p", "rho")).values())) for p in patches[::2]]
        d = ctx.diagnostics(0, dt)
        return {"fields": out, "sums": ctx.core_sums(0), "change": np.array(change),
                "diag": [d["cfl"], d["rho_min"], d["rho_max"], d["nonfinite"], ctx.cfl_axes(0, dt)]}
    if mode == "graph":
        ctx.rk_graph_run(dt, ALPHA, steps)
    elif mode == "loop":
        for _ in range(steps):
            ctx.exchange(0)
            ctx.copy_field(0, 1)
            for s, a in enumerate(ALPHA):
                if s > 0:
                    ctx.exchange(0)
                ctx.stage(0, 1, 2, a * dt)
                ctx.swap_fields(0, 2)
                ctx.exchange(0)
                if w.spheres is not None:
                    ctx.levelset_fill(0)
    else:
        for _ in range(steps):
            ctx.rk_step(dt, ALPHA)
            if mode == "cfl":
                dt *= CFL_TARGET / ctx.diagnostics(0, dt)["cfl"]
    return [ctx.download(p, 0) for p in patches]


def work(case):
    w = _workload(case)
    es = 4 if case["dtype"] == "f32" else 8
    stored, core = w.total_cells, w.core_cells
    if case["mode"] == "output":
        half = sum(P.cells for P in w.patches[::2])
        return {"bytes": float((2 * 5 * stored + 3 * half) * es), "flops": float(100 * stored)}
    # a three-stage step reads the old field once and then, per later stage, the old and the
    # last stage's field, and writes a field per stage; the field comes and goes once
    per_step = core * (10 + 15 * (len(ALPHA) - 1)) * es
    # 300 operations per cell and stage of the convective flux, twice that with the viscous one
    flops = core * len(ALPHA) * case["steps"] * (600 if w.viscous else 300)
    return {"bytes": float(per_step * case["steps"] + 2 * 5 * stored * es), "flops": float(flops)}


# ---------------------------------------------------------------------------
# the same in 64 bits, on the whole box instead of on patches
# ---------------------------------------------------------------------------

def _prim(U):
    ir = 1.0 / U[0]
    u, v, w = U[1] * ir, U[2] * ir, U[3] * ir
    T = (U[4] * ir - 0.5 * (u * u + v * v + w * w)) / CV
    return u, v, w, T, U[0] * R_GAS * T


def _limited(d1, d2):
    """van Albada: lim(d2 / d1) * d1, the divisor kept 1e-10 from zero"""
    s = torch.where(d1 < 0, torch.clamp(d1, max=-1e-10), torch.clamp(d1, min=1e-10))
    r = d2 / s
    return (r * r + r) / (r * r + 1.0) * d1


def _side(U, axis):
    """Density, velocity, normal velocity, pressure, sound speed and total enthalpy of a face side."""
    u, v, w, T, p = _prim(U)
    return U[0], (u, v, w), (u, v, w)[axis], p, torch.sqrt(GAMMA * R_GAS * T), (U[4] + p) / U[0]


def _mach_split(M, s):
    sup = M.abs() >= 1.0
    m1 = 0.5 * (M + s * M.abs())
    m2, m2o = 0.25 * s * (M + s) ** 2, -0.25 * s * (M - s) ** 2
    m4 = torch.where(sup, m1, m2 * (1.0 - 2.0 * s * m2o))
    p5 = torch.where(sup, m1 / torch.where(sup, M, 1.0), m2 * ((2.0 * s - M) - 3.0 * s * M * m2o))
    return m4, p5


def _ausm(UL, UR, axis):
    """AUSM+ flux per unit area through the faces between the sides UL and UR."""
    rl, vl, nl, pl, al, hl = _side(UL, axis)
    rr, vr, nr, pr, ar, hr = _side(UR, axis)
    a = 0.5 * (al + ar)
    m4l, p5l = _mach_split(nl / a, 1.0)
    m4r, p5r = _mach_split(nr / a, -1.0)
    M = m4l + m4r
    f0 = a * (rl * torch.clamp(M, min=0.0) + rr * torch.clamp(M, max=0.0))
    fp, fm = torch.clamp(f0, min=0.0), torch.clamp(f0, max=0.0)
    F = [f0] + [fp * vl[c] + fm * vr[c] for c in range(3)] + [fp * hl + fm * hr]
    F[1 + axis] = F[1 + axis] + (p5l * pl + p5r * pr)
    return torch.stack(F)


def _gradient(U, axis, h):
    """Central difference along a periodic axis (0, 1 or 2)."""
    return (torch.roll(U, -1, axis + 1) - torch.roll(U, 1, axis + 1)) * (0.5 / h)


def _viscous(U, axis, h):
    """Viscous flux per unit area through the face between every cell and the next one on a periodic axis."""
    nxt = torch.roll(U, -1, axis + 1)
    var = 0.5 * (U + nxt)
    g = []
    for b in range(3):
        if b == axis:
            g.append((nxt - U) / h[b])
        else:
            gb = _gradient(U, b, h[b])
            g.append(0.5 * (gb + torch.roll(gb, -1, axis + 1)))
    ir = 1.0 / var[0]
    T = (var[4] * ir - 0.5 * ir * ir * (var[1] ** 2 + var[2] ** 2 + var[3] ** 2)) / CV
    mu = 1.781e-5 * (T / 300.55) ** 1.5 * (300.55 + 111.0) / (T + 111.0)
    dvel = [[(g[b][1 + c] - g[b][0] * var[1 + c] * ir) * ir for b in range(3)] for c in range(3)]
    gn = g[axis]
    dT = 0.4 * ir * ir * (gn[4] * var[0] - gn[0] * var[4] - var[1] * gn[1] - var[2] * gn[2] - var[3] * gn[3]
                          + gn[0] * ir * (var[1] ** 2 + var[2] ** 2 + var[3] ** 2))
    tau = []
    for c in range(3):
        if c == axis:
            o = [b for b in range(3) if b != c]
            tau.append(0.6666666 * mu * (2.0 * dvel[c][c] - dvel[o[0]][o[0]] - dvel[o[1]][o[1]]))
        else:
            tau.append(mu * (dvel[c][axis] + dvel[axis][c]))
    q = mu * CP / 0.7 / R_GAS * dT
    work_done = (tau[0] * var[1] + tau[1] * var[2] + tau[2] * var[3]) * ir
    return torch.stack([torch.zeros_like(tau[0])] + [-t for t in tau] + [-(work_done + q)])


def _mix(x):
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))


def _jet_inflow(n, radius_cells, mach=0.9, noise=0.01, seed=1234, coflow=0.1):
    """Velocity (3, n, n) of the z = 0 face: the top hat with its noise, the co-flow around it."""
    gi, gj = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    key = (gi.astype(np.uint64) << np.uint64(32)) | gj.astype(np.uint64)
    base = _mix(key ^ _mix(np.array([seed], np.uint64))[0])
    r = []
    for c in range(3):
        with np.errstate(over="ignore"):
            h = _mix(base + np.uint64(c))
        r.append(((h >> np.uint64(40)).astype(np.int64) - 8388608) / 8388608.0)
    hot = (gi + 0.5 - 0.5 * n) ** 2 + (gj + 0.5 - 0.5 * n) ** 2 < radius_cells ** 2
    vel = [np.where(hot, mach * noise * r[0], 0.0), np.where(hot, mach * noise * r[1], 0.0),
           np.where(hot, mach * (1.0 + noise * r[2]), coflow)]
    return torch.tensor(np.stack(vel), device=_device())


def _wall(case, w, U, axis, plus, n):
    """Flux per unit area through a domain face next to the cells U (5, m, m)."""
    u, v, wv, T, p = _prim(U)
    F = torch.zeros_like(U)
    if case["flow"] == "sod" and axis > 0:
        F[1 + axis] = p  # a slip wall
    elif case["flow"] == "jet" and axis == 2 and not plus:
        vel = _jet_inflow(n, round(n / 16) + 0.37)
        T_in = configs.P_AMB / R_GAS
        F[0] = p / (R_GAS * T_in) * vel[2]
        for c in range(3):
            F[1 + c] = F[0] * vel[c]
        F[3] = F[3] + p
        F[4] = F[0] * (CP * T_in + 0.5 * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2))
    else:  # transmissive: the flux of the cell itself
        m = U[1 + axis]
        for q in range(4):
            F[q] = m * U[q] / U[0]
        F[1 + axis] = F[1 + axis] + p
        F[4] = m * (U[4] + p) / U[0]
    return F


def _residual(case, w, U, h, periodic, n):
    res = torch.zeros_like(U)
    for axis in range(3):
        a = axis + 1
        m = U.shape[a]
        if periodic:
            d = torch.roll(U, -1, a) - U
            dm = torch.roll(d, 1, a)
            slope = 0.5 * _limited(dm, d)
            left, right = U + slope, U - 0.5 * _limited(d, dm)
            F = _ausm(left, torch.roll(right, -1, a), axis)
            if w.viscous:
                F = F + _viscous(U, axis, h)
            res += (torch.roll(F, 1, a) - F) / h[axis]
            continue
        d = U.narrow(a, 1, m - 1) - U.narrow(a, 0, m - 1)
        left, right = U.narrow(a, 0, m - 1).clone(), U.narrow(a, 1, m - 1).clone()
        dl, dr = d.narrow(a, 0, m - 2), d.narrow(a, 1, m - 2)
        left.narrow(a, 1, m - 2).add_(0.5 * _limited(dl, dr))
        right.narrow(a, 0, m - 2).sub_(0.5 * _limited(dr, dl))
        F = _ausm(left, right, axis)
        lo = _wall(case, w, U.select(a, 0), axis, False, n)
        hi = _wall(case, w, U.select(a, m - 1), axis, True, n)
        F = torch.cat([lo.unsqueeze(a), F, hi.unsqueeze(a)], a)
        res += (F.narrow(a, 0, m) - F.narrow(a, 1, m)) / h[axis]
    return res


def _cells_of(w, U, periodic):
    """The patches' fields, seek layers included, out of the box field U."""
    out = []
    for P in w.patches:
        V = U
        for a, size in enumerate((P.ni, P.nj, P.nk)):
            idx = torch.arange(P.gidx[a], P.gidx[a] + size, device=U.device) % U.shape[a + 1]
            V = V.index_select(a + 1, idx)
        out.append(V.reshape(5, -1))
    return out


def exact(case, seed):
    if case["flow"] in ("spheres", "uneven"):
        return None  # mirror images and nested interpolation have no form without donor tables
    w = _workload(case)
    n = case["core"] * case["blocks"]
    if float(n) ** 3 * 3 * case["steps"] * (2 if w.viscous else 1) > EXACT_CELL_STAGES:
        return None
    dtype = torch.float32 if case["dtype"] == "f32" else torch.float64
    disturb = _disturbance(w, seed)
    U = torch.empty((5, n, n, n), dtype=torch.float64, device=_device())
    fields = []
    for P in w.patches:
        f = _patch_state(w, case, P, disturb, dtype)
        fields.append(f)
        s = P.seek
        lo = [P.gidx[a] + s[2 * a] for a in range(3)]
        hi = [P.gidx[a] + m - s[2 * a + 1] for a, m in enumerate((P.ni, P.nj, P.nk))]
        U[:, lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] = f[:, s[0]:P.ni - s[1], s[2]:P.nj - s[3], s[4]:P.nk - s[5]]
    h = [w.patches[0].dx(a) for a in range(3)]
    dt = w.dt
    if case["mode"] == "output":
        return _exact_output(case, seed, w, U, fields, h, dt)
    periodic = w.periodic[0] > 0
    for _ in range(case["steps"]):
        base = U
        for a in ALPHA:
            U = base + a * dt * _residual(case, w, U, h, periodic, n)
        if case["mode"] == "cfl":
            u, _, _, T, _ = _prim(U)
            s = torch.sqrt(GAMMA * R_GAS * T)
            dt *= CFL_TARGET / float((torch.maximum((u + s).abs(), (u - s).abs()) * dt / h[0]).max())
    return [f.cpu().numpy() for f in _cells_of(w, U, periodic)]


def _exact_output(case, seed, w, U, fields, h, dt):
    factor = 1.0 + 1.0e-3 * np.sin(1.0 + seed % 97)
    out, change, cfl_x, cfl_3, rmin, rmax = [], [], 0.0, 0.0, math.inf, -math.inf
    for q, f in enumerate(fields):
        before = torch.tensor((f.cpu().numpy() * factor).astype(f.cpu().numpy().dtype), device=f.device).double()
        V = f.double()
        d = before[0] - V[0]
        change.append([float(d.abs().max()), float(d.square().sum().sqrt())])
        u, v, wv, T, p = _prim(V)
        s = torch.sqrt(GAMMA * R_GAS * T)
        if q % 2 == 0:
            Ma = torch.sqrt((u * u + v * v + wv * wv) / (GAMMA * R_GAS * T))
            out.append(torch.stack([Ma, p, V[0]]).reshape(3, -1).cpu().numpy())
        cfl_x = max(cfl_x, float((torch.maximum((u + s).abs(), (u - s).abs()) * dt / h[0]).max()))
        cfl_3 = max([cfl_3] + [float(((c.abs() + s) * dt / h[a]).max()) for a, c in enumerate((u, v, wv))])
        rmin, rmax = min(rmin, float(V[0].min())), max(rmax, float(V[0].max()))
    sums = U.sum(dim=(1, 2, 3)).cpu().numpy() * (h[0] * h[1] * h[2])
    return {"fields": out, "sums": sums, "change": np.array(change), "diag": [cfl_x, rmin, rmax, 0.0, cfl_3]}
