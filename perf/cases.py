"""The work a user of this framework has it do, as cases with their inputs.

A simulation program builds a case's tables, creates a context, uploads the
initial state and runs the pre-loop (prepare); then it advances the solve from
one output time to the next and takes the new state down to write it (run):
`steps` time steps, each a replay of the captured step (`graph`) or launched
eagerly as the Fortran driver does, the device's status check, and the
download.  A case evolves from pass to pass, as a simulation does.

Fields of an FP64 solve are returned as they are.  The FP32-mixed form sums
pairs in FP32, which every field follows within a step: its fields are
returned in the single precision a results file holds.

Keys of a case: kind ("3d", "2d", "batch", "dbsph"), mixed, rk1, steps, graph,
jitter (of the lattice, in dx), dx, the tank and the column (tx ty tz cx cy cz),
vx (an initial velocity along x), obstacle, outlet, wallfn, moving.
"""
import functools
import math

import numpy as np
import torch

from sphera_amd import case2d, serve
from sphera_amd import runtime as rt
from sphera_amd.case import DamBreak3D, build
from sphera_amd.dbsph import DBSPHParams

FIELDS = ("coord", "vel", "acc", "dens", "pres", "dden", "vpres")


def _3d(name, dx, tank, column, **kw):
    c = dict(kind="3d", mixed=True, rk1=False, steps=40, graph=True, jitter=0.01, dx=dx, vx=0.0,
             tx=tank[0], ty=tank[1], tz=tank[2], cx=column[0], cy=column[1], cz=column[2])
    c.update(kw)
    return dict(name=name, **c) if name else c


def listed():
    big, water = (1.6, 0.6, 0.6), (0.4, 0.6, 0.3)
    return [
        # the smallest solve the tests and a first deck run: launches and latency count
        _3d("tank_1k_mixed", 0.01, (0.4, 0.2, 0.3), (0.12, 0.1, 0.12), graph=False),
        # the 2D dam break of the reference's configurations, FP64 as the Fortran driver steps it
        dict(name="plane_5k_fp64", kind="2d", mixed=False, rk1=False, steps=100, graph=False, jitter=0.01,
             dx=0.01, tx=3.22, tz=1.8, cx=1.0, cz=0.5),
        # the same tank refined, an odd spacing, replayed steps
        dict(name="plane_61k_mixed", kind="2d", mixed=True, rk1=False, steps=40, graph=True, jitter=0.03,
             dx=0.00287, tx=3.22, tz=1.8, cx=1.0, cz=0.5),
        # one served request of the ensemble's middle size, ragged column sides, stepped eagerly
        _3d("request_25k_mixed", 0.0131, big, (0.383, 0.571, 0.257), graph=False, jitter=0.0),
        # the tutorial-sized dam break in FP64
        _3d("dam_72k_fp64", 0.01, big, water, mixed=False),
        # a larger request of the ensemble
        _3d("request_190k_mixed", 0.00813, big, (0.412, 0.537, 0.451)),
        # the headline benchmark, both precisions
        _3d("dam_576k_mixed", 0.005, big, water),
        _3d("dam_576k_fp64", 0.005, big, water, mixed=False),
        # explicit RK1, a sill on the floor, an open end, rough walls: the deck options in use
        _3d("flume_rk1_mixed", 0.0079, (0.6, 0.5, 0.5), (0.31, 0.5, 0.33), rk1=True, vx=0.8, jitter=0.04,
            obstacle=True, outlet=True, wallfn=True),
        # eight requests of the served ensemble as one segmented batch
        dict(name="batch_8_mixed", kind="batch", mixed=True, rk1=False, steps=40, graph=True, jitter=0.01,
             seed0=0, count=8),
        # DB-SPH walls, the moving tank of the DB-SPH benchmark, and a small static one
        dict(name="dbsph_70k_moving", kind="dbsph", mixed=False, rk1=True, steps=40, graph=True, jitter=0.01,
             dx=0.01, tx=1.6, ty=0.6, tz=0.6, cx=0.4, cy=0.6, cz=0.3, moving=True),
        dict(name="dbsph_2k", kind="dbsph", mixed=False, rk1=True, steps=40, graph=False, jitter=0.01,
             dx=0.02, tx=0.8, ty=0.3, tz=0.4, cx=0.3, cy=0.3, cz=0.2, moving=False),
    ]


def draw(rng):
    """One more case: a dam break of log-uniform size, its form and options as used."""
    kind = rng.choice(("3d", "3d", "3d", "3d", "2d", "2d", "batch", "dbsph"))
    mixed = rng.random() < 0.6
    jit = round(rng.choice((0.0, 0.01, 0.03)) + 0.02 * rng.random(), 5)
    steps, graph = rng.randrange(20, 41), rng.random() < 0.6
    if kind == "2d":
        n = math.exp(rng.uniform(math.log(1500), math.log(100000)))
        cx, cz = round(rng.uniform(0.5, 1.4), 4), round(rng.uniform(0.3, 0.9), 4)
        return dict(kind="2d", mixed=mixed, rk1=rng.random() < 0.2, steps=steps, graph=graph, jitter=jit,
                    dx=round(math.sqrt(cx * cz / n), 6), tx=3.22, tz=1.8, cx=cx, cz=cz)
    if kind == "batch":
        return dict(kind="batch", mixed=mixed, rk1=False, steps=steps, graph=graph, jitter=jit,
                    seed0=rng.randrange(0, 500), count=rng.randrange(2, 5))
    tank = (1.6, 0.6, 0.6)
    col = [round(rng.uniform(0.2, 0.6), 4) for _ in range(3)]
    if kind == "dbsph":
        n = math.exp(rng.uniform(math.log(1200), math.log(20000)))
        return dict(kind="dbsph", mixed=False, rk1=True, steps=steps, graph=graph, jitter=jit,
                    dx=round(max(0.014, (col[0] * col[1] * col[2] / n) ** (1 / 3)), 5), tx=0.8, ty=0.6, tz=0.6,
                    cx=col[0], cy=col[1], cz=col[2], moving=rng.random() < 0.5)
    n = math.exp(rng.uniform(math.log(1200), math.log(500000 if mixed else 300000)))
    opt = rng.random()
    kw = dict(obstacle=True, outlet=True, wallfn=True) if opt < 0.15 else {}
    return _3d(None, round((col[0] * col[1] * col[2] / n) ** (1 / 3), 6), tank, col, mixed=mixed,
               rk1=rng.random() < 0.2, steps=steps, graph=graph, jitter=jit, vx=round(rng.uniform(0, 0.5), 4)
               if opt < 0.4 else 0.0, **kw)


# ---- inputs ------------------------------------------------------------------
MOVING = dict(kinematics=((0.0,) * 7, (0.01, 0.5, 0.0, 0.0, 0.0, 0.0, 1.0), (100.0, 0.5, 0.0, 0.0, 0.0, 0.0, 1.0)),
              rotation_centre=(0.8, 0.3, 0.0))


@functools.lru_cache(maxsize=2)
def _tables(key):
    """The set-up tables of a case (the deck's, whatever the initial state)."""
    c = dict(key)
    if c["kind"] == "batch":
        return [build(serve.ensemble_case(c["seed0"] + k)) for k in range(c["count"])]
    ts = 0 if c["rk1"] else 1
    if c["kind"] == "2d":
        return [case2d.build(case2d.DamBreak2D(tank=(c["tx"], c["tz"]), column=(c["cx"], c["cz"]), dx=c["dx"],
                                               time_split=ts))]
    kw = {}
    if c["kind"] == "dbsph":
        kw["dbsph"] = DBSPHParams(**(MOVING if c["moving"] else {}))
    if c.get("obstacle"):
        kw["obstacle"] = (c["cx"] + 4 * c["dx"], c["cx"] + 12 * c["dx"], 0.2 * c["cz"])
    if c.get("outlet"):
        kw["outlet"] = True
    if c.get("wallfn"):
        kw.update(slip_mode=2, roughness=(0.0005, 0.0015))
    return [build(DamBreak3D(tank=(c["tx"], c["ty"], c["tz"]), column=(c["cx"], c["cy"], c["cz"]), dx=c["dx"],
                             time_split=ts, **kw))]


def _inputs(case, seed):
    """Per solve: its tables, the jittered lattice and the initial velocity."""
    tbs = _tables(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    rng = np.random.default_rng(seed)
    got = []
    for tb in tbs:
        c = tb.particles["coord"]
        # a served request starts on its lattice: there the seed moves it by less than a thousandth of dx
        j = rng.uniform(-1.0, 1.0, c.shape) * max(case["jitter"], 5e-4) * tb.case.dx
        if case["kind"] == "2d":
            j[:, 1] = 0.0
        v = np.zeros_like(c)
        v[:, 0] = case.get("vx", 0.0)
        got.append((tb, c + j, v))
    return got


def prepare(case, seed):
    ins = _inputs(case, seed)
    prec = rt.FP32_MIXED if case["mixed"] else rt.FP64
    if case["kind"] == "batch":
        d = rt.SphBatch([tb for tb, _, _ in ins], precision=prec)
        d.upload(coords=[x for _, x, _ in ins])
    else:
        tb, x, v = ins[0]
        d = rt.SphContext(tb, precision=prec)
        d.upload(coord=x, vel=v)
    d.preloop()
    return dict(ctx=d, case=case)


def run(state):
    d, case = state["ctx"], state["case"]
    if case["graph"]:
        for _ in range(case["steps"]):
            d.step_graph(1)
        d.sync()
    else:
        d.step(case["steps"])
    if case["kind"] == "batch":
        return [_out(d.seg_state(k), case) for k in range(case["count"])]
    out = _out(d.state(), case)
    if case["kind"] == "dbsph":
        out.update(d.dbsph_state())
    return out


def _out(st, case):
    t = np.float32 if case["mixed"] else np.float64
    return {f: st[f].astype(t, copy=False) for f in FIELDS}


def work(case):
    """Per step: every particle's state (position, velocity, density, pressure,
    mass) read once and the new state with its rates written once; per pair the
    four pair sums and the kernel values (about 160 operations)."""
    if case["kind"] == "batch":
        n, pairs = sum(len(tb.particles["coord"]) for tb, _, _ in _inputs(case, 0)), 78
    elif case["kind"] == "2d":
        n, pairs = case["cx"] * case["cz"] / case["dx"] ** 2, 20
    else:
        n, pairs = case["cx"] * case["cy"] * case["cz"] / case["dx"] ** 3, 78
    return {"bytes": case["steps"] * n * 8 * (9 + 13), "flops": case["steps"] * n * pairs * 160}


# ---- the step in 64 bits -------------------------------------------------------
# Weakly compressible SPH with semi-analytic walls in a box, written out in
# torch over the list of pairs: cubic spline, Monaghan and Morris viscosity,
# leapfrog, velocity and pressure smoothing, linear equation of state.

def _lists(x, lo, dcd, ncd, r2max):
    """Ordered pairs (i, j), i included, within the cut-off."""
    c = torch.ceil((x - lo) / dcd).long() - 1
    key = (c[:, 2] * ncd[1] + c[:, 1]) * ncd[0] + c[:, 0]
    order = torch.argsort(key)
    cells = int(ncd.prod())
    cnt = torch.bincount(key, minlength=cells)
    start = torch.cumsum(cnt, 0) - cnt
    I, J = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                q = c + torch.tensor([dx, dy, dz], device=x.device)
                ok = ((q >= 0) & (q < ncd)).all(1)
                k = torch.where(ok, (q[:, 2] * ncd[1] + q[:, 1]) * ncd[0] + q[:, 0], 0)
                m = torch.where(ok, cnt[k], 0)
                i = torch.repeat_interleave(torch.arange(len(x), device=x.device), m)
                first = torch.cumsum(m, 0) - m
                j = order[start[k][i] + torch.arange(len(i), device=x.device) - first[i]]
                near = ((x[i] - x[j]) ** 2).sum(1) <= r2max
                I.append(i[near])
                J.append(j[near])
    return torch.cat(I), torch.cat(J)


def _radial(case):
    """Tables over r/h of the volume integrals of the spline (41 rows)."""
    h = case.h
    t = np.linspace(0.0, 2.0, 41)
    near, d = t < 1.0, 2.0 - t
    ks = 0.31830989
    w = np.where(near, 0.25 - (0.333333333333333 - 0.3 * t ** 2 + 0.125 * t ** 3) * t ** 3,
                 (0.0625 * t ** 2 + 0.025 * d * t + 4.16666666666667e-03 * d * d) * d ** 4) / 3.14159265358979
    j1 = np.where(near, -0.75 + (1 - 0.5625 * t) * t ** 3, -1 + (1.5 - t + 0.1875 * t * t) * t * t) * ks / (h * h)
    j2 = np.where(near, -0.7 + (0.75 - 0.45 * t) * t ** 4, -0.8 + (1 - 0.75 * t + 0.15 * t * t) * t ** 3) * ks / h
    j3 = np.where(near, -0.75 + (0.6 - 0.375 * t) * t ** 5, -0.8 + (0.75 - 0.6 * t + 0.125 * t * t) * t ** 4) * ks
    out = np.stack([w, j1, j2, j3], 1)
    out[-1] = 0.0
    return out


def _directions(h):
    """The 8 x 32 rays of the half sphere: offset, solid angle, unit vector."""
    pi = 3.14159265358979
    dfi, dte = pi / 16, pi / 16
    fi = (np.arange(8) + 0.5) * dfi
    te = (np.arange(32) + 0.5) * dte
    F, T = np.meshgrid(fi, te, indexing="ij")
    u = np.stack([np.sin(F) * np.cos(T), np.sin(F) * np.sin(T), -np.cos(F)], -1).reshape(-1, 3)
    da = (dte * 2 * math.sin(0.5 * dfi) * np.sin(F)).reshape(-1)
    return u, da


def _walls(case, x, tab, u, da):
    """Per wall (floor, x = 0, x = X, y = 0, y = Y): the particles within 2h of
    it, and their integrals: W dV, dW/r dV, grad, dW/r z^2 dV, the tensor."""
    h, zmin = case.h, 0.05 * case.h
    X, Y, Z = case.tank
    got = []
    for ax, side in ((2, 0.0), (0, 0.0), (0, X), (1, 0.0), (1, Y)):
        z = x[:, ax] - side if side == 0.0 else side - x[:, ax]
        idx = torch.nonzero((z >= 0) & (z < 2 * h))[:, 0]
        if not len(idx):
            continue
        e1, e2 = [a for a in range(3) if a != ax]
        size = (X, Y, Z)
        p, q = x[idx, e1], x[idx, e2]
        inside = (p >= 0) & (p <= size[e1]) & (q >= 0) & (q <= size[e2])
        L = torch.clamp(z[idx], min=zmin)
        a = torch.zeros(len(idx), 13, dtype=x.dtype, device=x.device)
        for k in range(len(da)):
            ux, uy, uz = (float(v) for v in u[k])
            t = L / -uz
            hx, hy = p + ux * t, q + uy * t
            keep = (t <= 2 * h) & (hx >= 0) & (hx <= size[e1]) & (hy >= 0) & (hy <= size[e2])
            rob = t / h
            r0 = torch.clamp((rob / 0.05).long(), max=39)
            f = (rob - 0.05 * r0) / 0.05
            J = (tab[r0] + f[:, None] * (tab[r0 + 1] - tab[r0])) * float(da[k]) * keep[:, None]
            J = torch.where((rob < 0.05)[:, None], tab[0] * float(da[k]) * keep[:, None], J)
            a[:, 0] += J[:, 0]
            a[:, 1] += J[:, 1]
            a[:, 2] += uz * uz * J[:, 1]
            for m, w in enumerate((ux, uy, uz)):
                a[:, 3 + m] += w * J[:, 2]
            for m, w in enumerate((ux * ux, ux * uy, ux * uz, uy * uy, uy * uz, uz * uz)):
                a[:, 6 + m] += w * J[:, 3]
        a[:, 0] = torch.where(L == zmin, 0.5 * inside, a[:, 0])
        e = torch.zeros(3, 3, dtype=x.dtype, device=x.device)  # rows: the two wall axes, the inward normal
        e[0, e1], e[1, e2], e[2, ax] = 1.0, 1.0, 1.0 if side == 0.0 else -1.0
        got.append((idx, z[idx], inside, a, e))
    return got


def _advance(tb, x, v, rho, p, m, steps):
    C, s = tb.case, tb.scalars
    h, c0, nu = C.h, math.sqrt(C.bulk / C.rho0), C.mu / C.rho0
    dev, T = x.device, lambda a: torch.as_tensor(np.asarray(a, np.float64), device=x.device)  # noqa: E731
    lo, dcd = T(tb.grid.extr_lo), T(tb.grid.dcd)
    ncd = torch.as_tensor(np.asarray(tb.grid.ncd, np.int64), device=dev)
    r2max = (2 * h) * (2 * h)
    grav, tab = T(C.grav), T(_radial(C))
    u, da = _directions(h)
    eta, eta2 = 1e-3 * h, 1e-2 * h * h
    n = len(x)

    def pairs():
        I, J = _lists(x, lo, dcd, ncd, r2max)
        return I, J

    def geometry(I, J):
        R = x[I] - x[J]
        r2 = (R * R).sum(1)
        r = torch.sqrt(r2)
        q = r / h
        d = 2.0 - q
        w = torch.where(q < 1, 0.666666667 + q * q * (0.5 * q - 1), d ** 3 * 0.166666666667) * (0.477464 / h ** 3)
        k1 = torch.where(q < 1, -2 * q + 1.5 * q * q, 2 * q - 0.5 * q * q - 2) * (0.477464 / h ** 4) / (r + eta)
        k3 = (-12.0 - 3 * q * q + 12 * q) * (0.074603 / h ** 4) / (r + eta)
        far = q >= 2
        return R, r2, *(torch.where(far, 0.0, k) for k in (w, k1, k3))

    def add(I, t):
        return torch.zeros((n,) + t.shape[1:], dtype=x.dtype, device=dev).index_add_(0, I, t)

    def rate(U):
        return (C.cfl * 2 * h / (c0 + torch.sqrt((U * U).sum(1)))).min()

    dt_vis = C.vsc_coeff * h * h / (0.5 * nu)
    dt = min(float(rate(v)), dt_vis)
    I, J = pairs()
    W = _walls(C, x, tab, u, da)
    a = dd = vp = None
    for _ in range(steps):
        old, dt = dt, min(float(rate(v)), dt_vis)
        # momentum
        R, r2, w, k1, k3 = geometry(I, J)
        k2, sym = k1 / (r2 + eta2), p[I] / rho[I] ** 2 + p[J] / rho[J] ** 2
        dv = v[J] - v[I]
        mon = C.alfa_mon * 2 * c0 * h / (rho[I] + rho[J]) * (-(dv * R).sum(1))
        vis = 4 * nu * nu / (nu * rho[I] + nu * rho[J] + 1e-3) * k2 * r2
        a = add(I, m[J][:, None] * ((mon * k2 - sym * k3)[:, None] * R - vis[:, None] * dv)) + grav
        for idx, z, inside, B, e in W:
            M = torch.stack([B[:, [6, 7, 8]], B[:, [7, 9, 10]], B[:, [8, 10, 11]]], 1)
            vn = 2.0 * (v[idx] @ e[2])
            loc = (M * (e @ grav)[None, None, :]).sum(2) + (2 * p[idx] / rho[idx])[:, None] * B[:, 3:6]
            t = (loc[:, :, None] * e[None]).sum(1) + (C.alfa_mon * c0 * h * vn * B[:, 2])[:, None] * e[2]
            a[idx] += torch.where((z > 0)[:, None], t, 0.0)
            hit = (z < 0.25 * C.dx) & inside & (vn < 0)
            push = -c0 * c0 * torch.log((h + z - 0.25 * C.dx) / h) / h
            a[idx] += torch.where(hit, push, 0.0)[:, None] * e[2]
        v = v + 0.5 * (dt + old) * a
        # velocity smoothing and positions
        s1 = add(I, (v[J] - v[I]) * (m[J] * w / rho[J])[:, None])
        for idx, z, inside, B, e in W:
            s1[idx] += (-2.0 * (v[idx] @ e[2]) * B[:, 0])[:, None] * e[2]
        v = v + C.teta_v * c0 * dt / h * s1
        x = x + dt * v
        # new lists, continuity, equation of state, pressure smoothing
        I, J = pairs()
        W = _walls(C, x, tab, u, da)
        R, r2, w, k1, k3 = geometry(I, J)
        dd = -rho * add(I, m[J] / rho[J] * k1 * ((v[J] - v[I]) * R).sum(1))
        for idx, z, inside, B, e in W:
            t = 2.0 * (v[idx] @ e[2]) * (e[2] * (B[:, 3:6] @ e)).sum(1)
            dd[idx] -= torch.where(z > 0, rho[idx] * t, 0.0)
        rho = rho + dt * dd
        p = C.bulk / C.rho0 * (rho - C.rho0) + C.p_ref
        pes = m[J] * w / rho[J]
        app, som = add(I, pes), add(I, (p[J] - p[I]) * pes)
        for idx, z, inside, B, e in W:
            app[idx] += torch.where(z > 0, B[:, 0], 0.0)
        vp = torch.where(app < 0.95, som + (C.p_ref - p) * (1 - app), som / app)
        p = p + C.teta_p * c0 * dt / h * vp
        rho = C.rho0 * (1 + (p - C.p_ref) / C.bulk)
    return dict(coord=x, vel=v, acc=a, dens=rho, pres=p, dden=dd, vpres=vp)


def exact(case, seed):
    """Box tanks with leapfrog and smooth walls; the other forms have none."""
    if case["kind"] not in ("3d", "batch") or case["rk1"] or case.get("obstacle"):
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    got = []
    for tb, x, v in _inputs(case, seed):
        P = tb.particles
        st = [torch.as_tensor(np.ascontiguousarray(q), dtype=torch.float64, device=dev)
              for q in (x, v, P["dens"], P["pres"], P["mass"])]
        out = _advance(tb, *st, case["steps"])
        got.append({k: out[k].cpu().numpy() for k in FIELDS})
    return got if case["kind"] == "batch" else got[0]
