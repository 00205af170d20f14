"""Performance cases: what a program that uses this framework has it do, through its public entry points.

`listed()` names the cases, `draw(rng)` gives more of the same ranges, `prepare(case, seed)` makes what
such a program has in hand before the call, `run(state)` is one pass, `work(case)` what a pass cannot do
without and `exact(case, seed)` the same outputs in 64 bits, where plain numpy can give them in a few
seconds.

Every case starts from a jittered lattice (+-0.1 dr), as the benchmark and the tests do.  The kinds:

  step    one step! of a flow in progress (StepDesc, device resident): the Taylor-Green vortex, the
          lid-driven cavity, the Gresho vortex and the Rayleigh-Taylor instability, with the solvers
          their configurations use
  lloyd   iterations of populate_lloyd! (remesh!, x = centroid) on seeds in place: initial conditions,
          and remeshing on its own
  frame   reading one frame of a run back to the host: the mesh (CSR) and fields
  probe   point_value at host query points: centreline profiles, maps, tracers
  mls     the moving-least-squares expansion of a field at every polygon
  train   one step of training the learned preconditioner on an assembled pressure system
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

lv = load_package()

DR_JITTER = 0.1
STEP_FIELDS = ("x", "v", "rho", "mass", "momentum", "e", "energy", "P", "D")


def listed():
    return [
        # the cavity example's centreline profile: 100 points on a 100 x 100 run, the smallest call there is
        dict(name="probe_centreline", kind="probe", nx=100, ny=100, m=100, field="v[1]"),
        # a map of a field on a regular raster's worth of points, for a picture or a transfer to another grid
        dict(name="probe_map", kind="probe", nx=512, ny=512, m=200003, field="P"),
        # gradients and curvature of the pressure at every particle of a middle-sized walled run (h = 3 dr, as a
        # quadratic fit needs in the corners)
        dict(name="mls_quadratic", kind="mls", nx=317, ny=251, order=2, reach=3, field="P"),
        # one output frame of a middle-sized run: polygons, labels and two fields on the host
        dict(name="frame_500", kind="frame", nx=500, ny=500, periodic=True),
        # initial conditions: a few Lloyd iterations of a walled domain with odd sides
        dict(name="lloyd_701", kind="lloyd", nx=701, ny=601, periodic=False, iterations=3),
        # the learned preconditioner's training runs on 32..64 a side systems, 20,000 of them
        dict(name="train_48", kind="train", nx=48, ny=48, nprobe=8),
        # the reference's cavity example (N = 100), 10,001 of these steps make its run
        dict(name="step_cavity_100", kind="step", flow="cavity", nx=100, solver="amg", tol=1e-10),
        # the Gresho vortex configuration: 100 x 100, incompressible, plain FP64 conjugate gradients
        dict(name="step_gresho_100", kind="step", flow="gresho", nx=100, solver="pcg64", tol=1e-10),
        # Rayleigh-Taylor with gravity, ideal gas and the multiphase projection, a quarter of rt1024's side
        dict(name="step_rt_256", kind="step", flow="rt", nx=256, solver="amg", tol=1e-10),
        # a middle-sized compressible run whose side is no multiple of anything
        dict(name="step_tg_515", kind="step", flow="tg", nx=515, solver="amg", tol=1e-10),
        # a large incompressible walled run (the ldc family), where the coarse levels do the work
        dict(name="step_cavity_1000", kind="step", flow="cavity", nx=1000, solver="amg", tol=1e-10),
        # the benchmark: Taylor-Green 2048 x 2048 to 1e-8
        dict(name="step_tg_2048", kind="step", flow="tg", nx=2048, solver="amg", tol=1e-8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("probe", "mls", "frame", "lloyd", "train", "step", "step", "step"))
    if kind == "probe":
        side = _log_int(rng, 48, 1024)
        return dict(kind=kind, nx=side, ny=max(32, int(side * rng.uniform(0.6, 1.4))), m=_log_int(rng, 1, 500000),
                    field=rng.choice(("P", "v[1]", "v[2]", "rho")))
    if kind == "mls":
        side = _log_int(rng, 48, 600)
        order = rng.choice((1, 2))
        return dict(kind=kind, nx=side, ny=max(32, int(side * rng.uniform(0.6, 1.4))), order=order,
                    reach=3 if order == 2 else rng.choice((2, 3)), field=rng.choice(("P", "v[1]", "v[2]")))
    if kind == "frame":
        side = _log_int(rng, 48, 700)
        return dict(kind=kind, nx=side, ny=max(32, int(side * rng.uniform(0.6, 1.4))), periodic=rng.random() < 0.5)
    if kind == "lloyd":
        side = _log_int(rng, 48, 1100)
        return dict(kind=kind, nx=side, ny=max(32, int(side * rng.uniform(0.6, 1.4))), periodic=rng.random() < 0.5,
                    iterations=rng.randint(1, 5))
    if kind == "train":
        return dict(kind=kind, nx=rng.randint(32, 80), ny=rng.randint(32, 80), nprobe=8)
    flow = rng.choice(("tg", "tg", "cavity", "gresho", "rt"))
    solver = {"tg": rng.choice(("amg", "amg", "pcg64")), "cavity": "amg", "gresho": "pcg64", "rt": "amg"}[flow]
    hi = {"amg": 1300, "pcg64": 420}[solver]
    return dict(kind=kind, flow=flow, nx=_log_int(rng, 48, 700 if flow == "rt" else hi), solver=solver,
                tol=rng.choice((1e-8, 1e-10)) if flow == "tg" else 1e-10)


# ---- inputs ----------------------------------------------------------------------------------------


def _lattice(nx, ny, dr, seed):
    """SoA planes double[2 n] of an nx by ny lattice with +-0.1 dr jitter; particle p = j nx + i"""
    n = nx * ny
    d = np.random.default_rng(seed).uniform(-DR_JITTER, DR_JITTER, size=(2, n))
    x = np.empty(2 * n)
    x[:n] = (np.tile(np.arange(nx, dtype=np.float64), ny) + 0.5 + d[0]) * dr
    x[n:] = (np.repeat(np.arange(ny, dtype=np.float64), nx) + 0.5 + d[1]) * dr
    return x


def _smooth(x, name):
    """the smooth fields the interpolation cases read, by name, at SoA positions x"""
    n = x.size // 2
    X, Y = 2 * math.pi * x[:n], 2 * math.pi * x[n:]
    if name == "P":
        return 0.25 * (np.cos(2 * X) + np.cos(2 * Y)) + 3.0 * x[:n]
    if name == "v[1]":
        return np.sin(X) * np.cos(Y)
    if name == "v[2]":
        return -np.cos(X) * np.sin(Y)
    return 1.0 + 0.1 * np.sin(X + Y)


def _queries(case, seed, dr):
    """m points inside the domain (planes 2 x m)"""
    q = np.random.default_rng([seed, 1]).uniform(0.0, 1.0, size=(case["m"], 2))
    return q * np.array([case["nx"] * dr, case["ny"] * dr])


class _DeviceField:
    """a field's device memory as torch's array interface sees it; keeps the grid alive"""

    def __init__(self, grid, ptr, shape, typestr):
        self.grid = grid
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(ptr, False), version=2, strides=None)


def _device_field(grid, name):
    import ctypes

    fid, comps = lv.FIELDS[name]
    p = ctypes.c_void_p()
    rc = lv.lib().lv_field_device_ptr(grid.ctx, fid, ctypes.byref(p))
    if rc != 0:
        raise RuntimeError("lv_field_device_ptr(%s): status %d" % (name, rc))
    return torch.as_tensor(_DeviceField(grid, p.value, (comps * grid.n,), "<f8"), device="cuda")


def _flow(case, seed):
    """a flow in progress: (grid, step descriptor), two steps from the initial condition"""
    flow, K = case["flow"], case["nx"]
    dr = 1.0 / K
    ny = 2 * K if flow == "rt" else K
    periodic = flow in ("tg", "gresho")
    x = _lattice(K, ny, dr, seed)
    grid = lv.VoronoiGrid(lv.Rectangle((0.0, 0.0), (1.0, ny * dr)), dr, xperiodic=periodic, yperiodic=periodic,
                          positions=x)
    lv.remesh(grid)
    area = grid.get("area")
    kw = {}
    if flow == "tg":
        ic = lv.inputs.taylor_green(x, area)
        dt = 2.5e-4 * (2048.0 / K)  # c0 dt / dr of the benchmark at every size
        keys = ("v", "rho", "mass", "P", "e", "mu")
        kw.update(eos="stiffened", gamma=ic["gamma"], P0=ic["P0"])
    elif flow == "gresho":
        ic = lv.inputs.gresho(x, area)
        dt = 0.1 * dr
        keys = ("v", "rho", "mass", "P", "e", "c2")
        kw.update(eos="rho", viscous=False)
    elif flow == "rt":
        ic = lv.inputs.rayleigh_taylor(x, area)
        dt = 0.1 * dr
        keys = ("v", "rho", "mass", "P", "e", "mu", "phase")
        kw.update(eos="ideal", gamma=1.4, gravity=(0.0, -1.0), artificial_viscosity=True,
                  multiphase=lv.MultiphaseSolver(grid))
    else:
        ic = lv.inputs.cavity(x, area, mu=1e-2)
        dt = min(0.1 * dr, 10.0 * dr * dr)
        keys = ("v", "rho", "mass", "mu", "c2")
        kw.update(eos="rho", friction={lv.BDARY_UP: (1.0, 0.0)})
    for k in keys:
        grid.set_soa(k, ic[k])
    amg = case["solver"] == "amg"
    solver = lv.PressureSolver(grid, method=case["solver"], tol=case["tol"], itmax=4000,
                               picard_window=8 if amg else 0, picard_carry=1 if amg else 0)
    desc = lv.make_step_desc(dt, solver=solver, **kw)
    for _ in range(2):
        lv.step_fused(grid, desc)
    return grid, desc


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        grid, desc = _flow(case, seed)
        return dict(kind=kind, grid=grid, desc=desc, out={k: _device_field(grid, k) for k in STEP_FIELDS})
    nx, ny = case["nx"], case["ny"]
    dr = 1.0 / nx
    periodic = case.get("periodic", kind == "train")
    x = _lattice(nx, ny, dr, seed)
    grid = lv.VoronoiGrid(lv.Rectangle((0.0, 0.0), (nx * dr, ny * dr)), dr, xperiodic=periodic, yperiodic=periodic,
                          positions=x)
    lv.remesh(grid)
    if kind == "lloyd":
        return dict(kind=kind, grid=grid, iterations=case["iterations"],
                    out={k: _device_field(grid, k) for k in ("x", "area", "centroid")})
    if kind == "train":
        ic = lv.inputs.taylor_green(x, grid.get("area"))
        for k in ("v", "rho", "mass", "P", "e", "mu"):
            grid.set_soa(k, ic[k])
        lv.stiffened_eos(grid, ic["gamma"], ic["P0"])
        lv.spai.set_params(grid, lv.spai.load_params())
        return dict(kind=kind, grid=grid, solver=lv.PressureSolver(grid), dt=2.5e-4 * (2048.0 / nx),
                    nprobe=case["nprobe"], step=0)
    grid.set("v", np.stack([_smooth(x, "v[1]"), _smooth(x, "v[2]")], 1))
    grid.set("P", _smooth(x, "P"))
    grid.set("rho", _smooth(x, "rho"))
    if kind == "probe":
        return dict(kind=kind, grid=grid, q=_queries(case, seed, dr), field=case["field"])
    if kind == "mls":
        return dict(kind=kind, grid=grid, order=case["order"], field=case["field"], h=case["reach"] * dr)
    return dict(kind=kind, grid=grid)


def run(state):
    kind, grid = state["kind"], state["grid"]
    if kind == "step":
        stats = lv.step_fused(grid, state["desc"])
        return dict(state["out"], nsolves=stats["nsolves"])
    if kind == "lloyd":
        rc = lv.lib().lv_lloyd(grid.ctx, state["iterations"])
        if rc != 0:
            raise RuntimeError("lv_lloyd: status %d" % rc)
        return state["out"]
    if kind == "frame":
        ptr, labels, verts = grid.mesh()
        return dict(ptr=ptr, labels=labels, verts=verts, v=grid.get("v"), P=grid.get("P"))
    if kind == "probe":
        return lv.point_value(grid, state["q"], state["field"])
    if kind == "mls":
        return lv.movingls(state["order"], grid, state["field"], h=state["h"])
    # train: the step's system, one Adam step on it, and the parameters the next system starts from
    state["step"] += 1
    state["solver"].assemble(state["dt"])
    loss = lv.spai.train_step(grid, lr=2e-4, nprobe=state["nprobe"], seed=1000003 + 17 * state["step"])
    return dict(loss=loss, theta=lv.spai.get_params(grid))


# ---- what a pass cannot do without -------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    n = case["nx"] * (2 * case["nx"] if case.get("flow") == "rt" else case.get("ny", case["nx"]))
    edges = 6 * n
    mesh = 36 * edges + 4 * n  # labels and vertices of every polygon
    if kind == "step":
        # the 22 planes of the state in and out, two meshes written, and ten Picard solves that each read
        # the operator's couplings and columns (12 B), its diagonal, right-hand side and guess once
        return dict(bytes=2 * 22 * 8 * n + 2 * mesh + 10 * (12 * edges + 4 * 8 * n), flops=2 * 5600 * n)
    if kind == "lloyd":
        # each iteration reads the seeds and writes the mesh, areas and centroids
        return dict(bytes=(case["iterations"] + 1) * (16 * n + mesh + 24 * n),
                    flops=(case["iterations"] + 1) * 5600 * n)
    if kind == "frame":
        return dict(bytes=2 * (mesh + 24 * n), flops=0)  # read on the device, written on the host
    if kind == "probe":
        near = min(n, 13 * case["m"])  # the seeds and values within h of the queries
        return dict(bytes=24 * case["m"] + 24 * near, flops=13 * 40 * case["m"])
    if kind == "mls":
        k = {1: 2, 2: 5}[case["order"]]
        near = 13 if case["reach"] == 2 else 28
        return dict(bytes=24 * n + 8 * k * n, flops=near * (2 * k * k + 4 * k + 30) * n)
    # train: three layers forward (2 E 192 64) and backward (twice that), the states read and written once
    return dict(bytes=6 * 2 * 64 * 2 * edges + 16 * 36000, flops=3 * 3 * 2 * edges * 192 * 64)


# ---- the same outputs in 64 bits ---------------------------------------------------------------------


def _offsets(reach):
    return [(a, b) for b in range(-reach, reach + 1) for a in range(-reach, reach + 1) if a or b]


def _linear_or_quadratic(case, x, f, i, order, reach):
    """movingls at the seeds i of the walled jittered lattice x: Gaussian weights at h = reach dr over the
    seeds nearer than h, which lie at most `reach` lattice steps away (one more is at least 0.8 dr too far)"""
    nx, ny = case["nx"], case["ny"]
    n, h = nx * ny, reach * (1.0 / nx)
    N = {1: 2, 2: 5}[order]
    ii, jj = i % nx, i // nx
    a, R = np.zeros((i.size, N)), np.zeros((i.size, N, N))
    for da, db in _offsets(reach):
        p, q = ii + da, jj + db
        ok = (p >= 0) & (p < nx) & (q >= 0) & (q < ny)
        j = np.where(ok, p + q * nx, i)
        d1, d2 = x[j] - x[i], x[n + j] - x[n + i]
        r = np.sqrt(d1 * d1 + d2 * d2)
        w = np.where(ok & (r < h), np.exp(-0.5 * (r / h) ** 2), 0.0)
        d1, d2 = d1 / h, d2 / h  # scaled, for the conditioning of the normal equations
        P = np.stack([d1, d2] if order == 1 else [d1, d2, d1 * d1, d1 * d2, d2 * d2], 1)
        a += (w * (f[j] - f[i]))[:, None] * P
        R += w[:, None, None] * P[:, :, None] * P[:, None, :]
    c = np.linalg.solve(R, a[:, :, None])[:, :, 0]
    c[:, :2] /= h
    c[:, 2:] /= h * h
    return c


def _clip_cells(x, nx, ny, dr, periodic):
    """area and centroid of the Voronoi cell of every seed of a (nearly regular) lattice whose Voronoi
    neighbours lie at most two lattice steps away: half-plane clipping of all cells at once"""
    n, W, H = nx * ny, nx * dr, ny * dr
    i = np.arange(n)
    ii, jj = i % nx, i // nx
    x1, x2 = x[:n], x[n:]
    M = 12
    big = 3.0 * dr
    lo1, hi1, lo2, hi2 = -big * np.ones(n), big * np.ones(n), -big * np.ones(n), big * np.ones(n)
    if not periodic:
        lo1, hi1 = np.maximum(lo1, -x1), np.minimum(hi1, W - x1)
        lo2, hi2 = np.maximum(lo2, -x2), np.minimum(hi2, H - x2)
    V = np.zeros((M, 2, n))  # vertices relative to the seed, counter-clockwise
    for k, (a, b) in enumerate(((lo1, lo2), (hi1, lo2), (hi1, hi2), (lo1, hi2))):
        V[k, 0], V[k, 1] = a, b
    cnt = np.full(n, 4)
    for da, db in sorted(_offsets(2), key=lambda o: o[0] ** 2 + o[1] ** 2):
        p, q = ii + da, jj + db
        ok = np.ones(n, bool) if periodic else (p >= 0) & (p < nx) & (q >= 0) & (q < ny)
        j = np.where(ok, (p % nx) + (q % ny) * nx, i)
        d1, d2 = x1[j] - x1, x2[j] - x2
        if periodic:
            d1, d2 = d1 - W * np.round(d1 / W), d2 - H * np.round(d2 / H)
        F = V[:, 0] * d1 + V[:, 1] * d2 - 0.5 * (d1 * d1 + d2 * d2)
        live = np.arange(M)[:, None] < cnt
        hit = np.nonzero(ok & ((F > 0) & live).any(0))[0]
        if hit.size == 0:
            continue
        Vh, Fh, ch = V[:, :, hit], F[:, hit], cnt[hit]
        out, m = np.zeros_like(Vh), np.zeros(hit.size, int)
        col = np.arange(hit.size)
        for k in range(int(ch.max())):
            nxt = np.where(k + 1 < ch, k + 1, 0)
            f0, f1 = Fh[k], Fh[nxt, col]
            on = k < ch
            keep = on & (f0 <= 0)
            out[m[keep], :, col[keep]] = Vh[k][:, keep].T
            m += keep
            cross = on & ((f0 <= 0) != (f1 <= 0))
            c = col[cross]
            t = f0[cross] / (f0[cross] - f1[cross])
            A, B = Vh[k][:, cross], Vh[nxt[cross], :, c].T
            out[m[cross], :, c] = (A + t * (B - A)).T
            m += cross
        V[:, :, hit], cnt[hit] = out, m
    area, c1, c2 = np.zeros(n), np.zeros(n), np.zeros(n)
    for k in range(int(cnt.max())):
        nxt = np.where(k + 1 < cnt, k + 1, 0)
        on = k < cnt
        a, b = V[k], np.stack([V[nxt, 0, i], V[nxt, 1, i]])
        h = np.where(on, 0.5 * (a[0] * b[1] - a[1] * b[0]), 0.0)
        area += h
        c1 += h * (a[0] + b[0]) / 3.0
        c2 += h * (a[1] + b[1]) / 3.0
    return area, np.concatenate([x1 + c1 / area, x2 + c2 / area])


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("probe", "mls", "lloyd"):
        # a step's outputs carry its iterative solves, a training step's its 16-bit network: no closed form
        return None
    nx, ny = case["nx"], case["ny"]
    n, dr = nx * ny, 1.0 / nx
    x = _lattice(nx, ny, dr, seed)
    if kind == "lloyd":
        if n * (case["iterations"] + 1) > 2_000_000:
            return None
        for _ in range(case["iterations"]):
            x = _clip_cells(x, nx, ny, dr, case["periodic"])[1]
        area, cent = _clip_cells(x, nx, ny, dr, case["periodic"])
        return dict(x=x, area=area, centroid=cent)
    f = _smooth(x, case["field"])
    if kind == "mls":
        return _linear_or_quadratic(case, x, f, np.arange(n), case["order"], case["reach"])
    q = _queries(case, seed, dr)
    ci = np.clip((q[:, 0] / dr).astype(int), 0, nx - 1)
    cj = np.clip((q[:, 1] / dr).astype(int), 0, ny - 1)
    best, at = np.full(case["m"], np.inf), np.zeros(case["m"], int)
    for da, db in [(0, 0)] + _offsets(1):
        p, r = ci + da, cj + db
        ok = (p >= 0) & (p < nx) & (r >= 0) & (r < ny)
        j = np.where(ok, p + r * nx, 0)
        d = np.where(ok, (x[j] - q[:, 0]) ** 2 + (x[n + j] - q[:, 1]) ** 2, np.inf)
        at, best = np.where(d < best, j, at), np.minimum(d, best)
    L = _linear_or_quadratic(case, x, f, at, 1, 2)
    return f[at] + L[:, 0] * (q[:, 0] - x[at]) + L[:, 1] * (q[:, 1] - x[n + at])
