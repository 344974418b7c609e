"""The workloads the solver's speed is measured on, each through the public Python interface.

``listed()`` names them, ``draw(rng)`` gives another of the same ranges, ``prepare`` builds
what a program holds before the call (the solver of a job, or the solvers of a batch),
``run`` is one pass, ``work`` the bytes and operations a pass cannot do without and
``exact`` the same pass in 64-bit torch.

A case is a mesh kind with its cell counts, a precision and a use:

* kinds: ``block`` (isotropic aluminium block), ``water`` (the block driven by three stress
  sources on its top face, the water-column form), ``plate`` (16-ply CFRP laminate with
  through-holes and a surface crack), ``bracket`` (cracked Ti-6Al-4V L-bracket), ``graded``
  (block whose stiffness varies from cell to cell, so no two cells share a material) and
  ``batch`` (independent isotropic boxes of mixed sizes);
* uses: ``run`` (an inspection solve: its sensor traces and final energies), ``interval``
  (a driver's write interval: the steps, then every state field), ``single`` (the same with
  one ``solve()`` per step, as the drivers call it), ``restart`` (a checkpoint written into
  the solver, the steps, the new checkpoint) and ``batch`` (all instances advanced together,
  each one's traces and energies).

Meshes are numbered as the case makers number them: x outermost, z innermost.
"""
from __future__ import annotations

import math

import numpy as np
import torch

CIJ = [(i, j) for i in range(6) for j in range(i, 6)]
CORNERS = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
LAYUP = [0, 45, 90, -45, 0, 45, 90, -45, -45, 90, 45, 0, -45, 90, 45, 0]
MATERIALS = {"al": (2700.0, 51.0e9, 26.0e9), "ti": (4430.0, 90.0e9, 44.0e9)}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest job of the smoke run: a few hundred cells, where only launches count
        dict(name="smallest-block-fp64", kind="block", nx=10, ny=8, nz=6, precision="fp64", use="interval", steps=40),
        # the aluminium block of the reference's own example, its whole 500 steps
        dict(name="al-block-fp64", kind="block", nx=40, ny=40, nz=20, precision="fp64", use="interval", steps=500),
        # the same block as the drivers run it: one solve() per step, written every 50 steps
        dict(name="al-block-steps-fp64", kind="block", nx=40, ny=40, nz=20, precision="fp64", use="single", steps=50),
        # a water-column job of ordinary size, with odd cell counts
        dict(name="water-column-fp64", kind="water", nx=51, ny=47, nz=35, precision="fp64", use="interval",
             steps=100),
        # one box of the middle of the batch range, solved alone in FP32
        dict(name="box-fp32", kind="block", nx=71, ny=64, nz=57, precision="fp32", use="run", steps=500),
        # a part whose stiffness varies from cell to cell (per-cell coefficient arrays)
        dict(name="graded-fp64", kind="graded", nx=100, ny=90, nz=50, precision="fp64", use="interval", steps=100),
        # a checkpoint of a million cells resumed for one write interval
        dict(name="restart-fp64", kind="block", nx=128, ny=128, nz=64, precision="fp64", use="restart", steps=50),
        # the laminate plate of the benchmark: one write interval, and stretches of an inspection
        dict(name="plate-interval-fp64", kind="plate", nx=256, ny=256, nz=64, precision="fp64", use="interval",
             steps=50),
        dict(name="plate-fp64", kind="plate", nx=256, ny=256, nz=64, precision="fp64", use="run", steps=500),
        dict(name="plate-fp32", kind="plate", nx=256, ny=256, nz=64, precision="fp32", use="run", steps=500),
        # the largest: the bracket of 9.4 M cells
        dict(name="bracket-fp32", kind="bracket", nx=512, ny=96, nz=96, precision="fp32", use="run", steps=300),
        # independent boxes of 32^3 to 128^3 cells in one batch
        dict(name="batch-fp32", kind="batch", count=16, lo=32768, hi=2097152, precision="fp32", use="batch",
             steps=300),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    precision = rng.choice(["fp64", "fp32"])
    kind = rng.choice(["block", "block", "plate", "bracket", "water", "graded", "batch"])
    if kind == "batch":
        hi = _log_int(rng, 131072, 2097152)
        return dict(kind=kind, count=rng.randint(4, 16), lo=32768, hi=hi, precision=precision, use="batch",
                    steps=rng.randint(50, 120))
    if kind == "plate":
        n = _log_int(rng, 24, 256)
        dims = dict(nx=n, ny=max(24, int(n * rng.uniform(0.8, 1.0))), nz=16 * rng.randint(1, 4))
    elif kind == "bracket":
        w = rng.randint(12, 72)
        dims = dict(nx=int(round(w * rng.uniform(3.0, 16 / 3))), ny=w, nz=max(8, int(w * rng.uniform(0.7, 1.0))))
    else:
        cells = _log_int(rng, 480, 6.0e5 if kind == "graded" else 2.1e6)
        a, b = math.exp(rng.uniform(-0.4, 0.4)), math.exp(rng.uniform(-0.4, 0.4))
        m = cells ** (1 / 3)
        dims = dict(nx=max(5, int(round(m * a))), ny=max(5, int(round(m * b))), nz=max(5, int(round(m / (a * b)))))
    cells = dims["nx"] * dims["ny"] * dims["nz"]
    use = rng.choice(["run", "interval", "single", "restart"])
    steps = rng.randint(30, 70) if use in ("single", "restart") else rng.randint(40, 500 if cells < 1 << 18 else 200)
    if use == "restart" and cells > 1 << 20:
        use = "interval"
    return dict(kind=kind, precision=precision, use=use, steps=steps, **dims)


# ------------------------------------------------------------------ the jobs

def _isotropic(lam, mu):
    c = np.zeros((6, 6))
    c[:3, :3] = lam
    c[np.arange(3), np.arange(3)] += 2 * mu
    c[np.arange(3, 6), np.arange(3, 6)] = mu
    return c


def _ply(degrees):
    """The CFRP ply's stiffness with its fibres turned by ``degrees`` about z."""
    c = np.zeros((6, 6))
    c[0, 0], c[1, 1], c[2, 2] = 135e9, 9.5e9, 9.5e9
    c[0, 1] = c[1, 0] = c[0, 2] = c[2, 0] = 4.5e9
    c[1, 2] = c[2, 1] = 4.2e9
    c[3, 3], c[4, 4], c[5, 5] = 2.6e9, 5.0e9, 5.0e9
    s, a = math.sin(math.radians(degrees)), math.cos(math.radians(degrees))
    # stress transformation of a rotation about z, Voigt order xx yy zz yz xz xy
    t = np.array([[a * a, s * s, 0, 0, 0, -2 * a * s], [s * s, a * a, 0, 0, 0, 2 * a * s], [0, 0, 1, 0, 0, 0],
                  [0, 0, 0, a, s, 0], [0, 0, 0, -s, a, 0], [a * s, -a * s, 0, 0, 0, a * a - s * s]])
    c = t @ c @ t.T
    return 0.5 * (c + c.T)


def _grid(nx, ny, nz, d, keep2d=None, crack=None):
    """Nodes and cells of the kept columns of a grid.  ``crack`` = (i, j0, j1, k0): the nodes of
    plane i with j0 < j < j1 and k > k0 get a copy that the cells from i on use."""
    keep = np.ones((nx, ny, nz), dtype=bool) if keep2d is None else np.repeat(keep2d[:, :, None], nz, axis=2)
    used = np.zeros((nx + 1, ny + 1, nz + 1), dtype=bool)
    for a, b, c in CORNERS:
        used[a:a + nx, b:b + ny, c:c + nz] |= keep
    ijk = np.nonzero(used)
    nid = np.full(used.shape, -1, dtype=np.int32)
    nid[used] = np.arange(ijk[0].shape[0], dtype=np.int32)
    xyz = [q * d for q in ijk]
    cells = np.empty((int(keep.sum()), 8), dtype=np.int32)
    far = None
    if crack is not None:
        i, j0, j1, k0 = crack
        solid = np.ones((nx, ny), dtype=bool) if keep2d is None else keep2d
        cut = np.zeros_like(used)
        for j in range(j0 + 1, j1):  # not at the rim of a hole: both copies keep cells of their own
            cut[i, j, k0 + 1:] = solid[i - 1:i + 1, j - 1:j + 1].all()
        copied = np.nonzero(cut)
        far = nid.copy()
        far[cut] = ijk[0].shape[0] + np.arange(copied[0].shape[0], dtype=np.int32)
        xyz = [np.concatenate([q, c * d]) for q, c in zip(xyz, copied)]
    for v, (a, b, c) in enumerate(CORNERS):
        col = nid[a:a + nx, b:b + ny, c:c + nz]
        if far is not None:
            col = col.copy()
            col[crack[0]:] = far[a + crack[0]:a + nx, b:b + ny, c:c + nz]
        cells[:, v] = col[keep]
    return xyz, cells, keep


def _burst(freq, cycles, dt):
    n = int(math.ceil((cycles / freq) / dt))
    t = np.arange(n) * dt
    v = np.sin(2 * np.pi * freq * t) * np.hanning(n)
    return t, v / v.max()


def _job(case, rng):
    """One job from its generator: mesh, materials, sources, sensors, dt."""
    kind, nx, ny, nz = case["kind"], case["nx"], case["ny"], case["nz"]
    d = 5.0e-5 if kind in ("plate", "bracket") else 1.0e-4
    keep2d, crack = None, None
    lx, ly = nx * d, ny * d
    if kind == "plate":
        xc, yc = np.meshgrid((np.arange(nx) + 0.5) * d, (np.arange(ny) + 0.5) * d, indexing="ij")
        keep2d = np.ones((nx, ny), dtype=bool)
        holes = np.random.default_rng(nx * 4099 + ny)  # the part's shape: the case's, not the seed's
        for k in range(5):
            r = holes.uniform(0.08, 0.2) * min(lx, ly) / 2
            ang = (k + holes.uniform(0.2, 0.8)) * 2 * math.pi / 5
            hx, hy = lx / 2 + 0.33 * lx * math.cos(ang), ly / 2 + 0.33 * ly * math.sin(ang)
            keep2d &= (xc - hx) ** 2 + (yc - hy) ** 2 >= r * r
        center = (rng.uniform(0.45, 0.55) * lx, rng.uniform(0.45, 0.55) * ly)
        crack = (nx // 4, ny // 3, 2 * ny // 3, nz // 2)
    elif kind == "bracket":
        keep2d = np.zeros((nx, ny + nx), dtype=bool)
        keep2d[:, :ny] = True
        keep2d[:ny, :] = True
        center = (rng.uniform(0.25, 0.4) * lx, 0.5 * ly)
        crack = (int(rng.uniform(0.55, 0.8) * nx), ny // 4, 3 * ny // 4, nz // 2)
    else:
        center = (rng.uniform(0.4, 0.6) * lx, rng.uniform(0.4, 0.6) * ly)
    xyz, cells, keep = _grid(nx, keep2d.shape[1] if keep2d is not None else ny, nz, d, keep2d, crack)
    nc = cells.shape[0]
    shift = 1 + rng.uniform(-0.05, 0.05)  # each job's own material sample
    if kind == "plate":
        rho, c6 = 1580.0 * shift, np.stack([_ply(a) for a in LAYUP])
        mat = (np.nonzero(keep)[2] // (nz // 16)).astype(np.int64)
        freq, cycles, radius = 2.0e6, 5, 2.0e-3 * min(lx, ly) / 12.8e-3
    else:
        rho, lam, mu = MATERIALS["ti" if kind == "bracket" else case.get("material", "al")]
        rho, c6, mat = rho * shift, _isotropic(lam, mu)[None], None
        freq, cycles, radius = (10.0e6 if kind == "bracket" else 5.0e6), 3, min(2.0e-3, 0.3 * min(lx, ly))
    speed = math.sqrt(max(float(c6[:, q, q].max()) for q in range(3)) / rho)
    scale = None
    if kind == "graded":  # stiffness of a part whose temperature varies from place to place
        centre = [q[cells].mean(axis=1) for q in xyz]
        scale = 1 - 0.2 * np.sin(40 * centre[0] + 0.3) ** 2 * np.cos(30 * centre[1]) ** 2 - 0.05 * centre[2] / (nz * d)
        scale *= 1 - 1e-3 * rng.random(nc)
    dt = 0.9 / (speed * 3.0 / d)
    t, v = _burst(freq, cycles, dt)
    top = np.nonzero(np.abs(xyz[2] - nz * d) < 0.25 * d)[0]
    sensors = np.sort(rng.choice(top, size=min(16, top.shape[0]), replace=False)).astype(np.int32)
    at = (center[0], center[1], nz * d)
    discs = [(0, v), (1, 0.5 * v), (2, -0.25 * v)] if kind == "water" else [(2, v)]
    return dict(xyz=xyz, cells=cells, rho=rho, c6=c6, mat=mat, scale=scale, dt=dt, d=d, sensors=sensors, at=at,
                radius=radius, t=t, discs=discs, moment=kind == "water")


def _boxes(case, rng):
    """Jobs of a batch: log-uniform cell counts between lo and hi, seeded proportions."""
    shapes = np.random.default_rng(case["count"] * 7919 + case["hi"])  # sizes are the case's, not the seed's
    jobs = []
    for k in range(case["count"]):
        cells = math.exp(shapes.uniform(math.log(case["lo"]), math.log(case["hi"])))
        a = np.exp(shapes.uniform(-0.5, 0.5, size=3))
        n = np.maximum(8, np.round(a / a.prod() ** (1 / 3) * cells ** (1 / 3))).astype(int)
        jobs.append(_job(dict(kind="block", nx=int(n[0]), ny=int(n[1]), nz=int(n[2]),
                              material="ti" if k % 2 else "al"), rng))
    return jobs


def _jobs(case, seed):
    rng = np.random.default_rng(seed)
    return _boxes(case, rng) if case["kind"] == "batch" else [_job(case, rng)]


def _checkpoint(job, seed):
    """A wave field to resume from: a few plane waves in velocity and stress."""
    rng = np.random.default_rng(seed + 1)
    xyz, ext = job["xyz"], [max(float(q.max()), job["d"]) for q in job["xyz"]]

    def fields(points, count, size):
        out = np.empty((count, points[0].shape[0]))
        for f in range(count):
            k = rng.uniform(2, 8, size=3) * 2 * np.pi / np.array(ext)
            out[f] = size * np.sin(k[0] * points[0] + k[1] * points[1] + k[2] * points[2] + rng.uniform(0, 6))
        return out

    corner = [q[job["cells"][:, 0]] for q in xyz]
    return fields(xyz, 3, 1e-6), fields(corner, 6, 20.0)


def _solver(job, precision):
    from pannde_amd import cases, rsg

    c6, mat, scale = job["c6"], job["mat"], job["scale"]
    nc = job["cells"].shape[0]
    if scale is not None:
        cij = [cases.Field(cases.FIELD_CELL, c6[0, i, j] * scale) for i, j in CIJ]
    elif mat is not None:
        cij = [cases.Field(cases.FIELD_CELL, c6[:, i, j][mat]) for i, j in CIJ]
    else:
        cij = [cases.Field(cases.FIELD_CONSTANT, c6[:, i, j].copy()) for i, j in CIJ]
    discs = [cases.Disc(k, job["at"], job["radius"], job["d"], job["t"], v) for k, v in job["discs"]]
    return rsg.DeviceSolver(*job["xyz"], job["cells"], cases.Field(cases.FIELD_CELL, np.full(nc, job["rho"])), cij,
                            job["dt"], force=[] if job["moment"] else discs, moment=discs if job["moment"] else [],
                            moment_form=int(job["moment"]), sensors=job["sensors"],
                            precision=rsg.RSG_FP32 if precision == "fp32" else rsg.RSG_FP64)


def prepare(case, seed):
    jobs = _jobs(case, seed)
    state = dict(case, done=0, solvers=[_solver(j, case["precision"]) for j in jobs])
    if case["use"] == "restart":
        state["V"], state["S"] = _checkpoint(jobs[0], seed)
    return state


# ------------------------------------------------------------------ one pass

def run(state):
    steps, first = state["steps"], state["done"]
    state["done"] += steps
    if state["use"] == "batch":
        return _run_batch(state, steps, first)
    s = state["solvers"][0]
    if state["use"] == "restart":
        s.set_state(state["V"], state["S"])
    if state["use"] == "single":
        for _ in range(steps):
            t = s.solve()
    else:
        t = s.solve(steps)
    out = dict(time=t, traces=s.traces(first, steps))
    if state["use"] == "run":
        out["kinetic"], out["strain"] = s.energy()
    else:
        out["V"], out["S"] = s.get_state()
    return out


def _run_batch(state, steps, first):
    from pannde_amd import rsg

    b = rsg.Batch(state["solvers"][0].precision)
    slots = [b.add(s, steps) for s in state["solvers"]]
    b.run(10 ** 6)
    b.synchronize()
    out = []
    for slot in slots:
        s = b.remove(slot)
        out.append(dict(traces=s.traces(first, steps), energy=list(s.energy())))
    b.close()
    return out


def _sizes(case):
    """(cells, nodes) of each job, holes and cracks left out of the count."""
    if case["kind"] == "batch":
        shapes = np.random.default_rng(case["count"] * 7919 + case["hi"])
        out = []
        for _ in range(case["count"]):
            cells = math.exp(shapes.uniform(math.log(case["lo"]), math.log(case["hi"])))
            a = np.exp(shapes.uniform(-0.5, 0.5, size=3))
            n = np.maximum(8, np.round(a / a.prod() ** (1 / 3) * cells ** (1 / 3))).astype(int)
            out.append((int(n.prod()), int((n + 1).prod())))
        return out
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    columns = nx * ny + (nx - ny) * ny if case["kind"] == "bracket" else nx * ny
    if case["kind"] == "bracket":
        columns = nx * ny + ny * nx
    return [(columns * nz, int((columns + nx + ny + 1) * (nz + 1)))]


def work(case):
    """A step reads and writes the state once (3 values a node, 6 a cell); about 190 operations a
    cell and 100 a node.  A graded part's 21 coefficients a cell are read every step too; a
    checkpoint or a written state crosses once as FP64."""
    elt = 4 if case["precision"] == "fp32" else 8
    total = flops = 0
    for cells, nodes in _sizes(case):
        step = 2 * elt * (3 * nodes + 6 * cells) + (21 * elt * cells if case["kind"] == "graded" else 0)
        total += case["steps"] * step
        flops += case["steps"] * (190 * cells + 100 * nodes)
        if case["use"] in ("interval", "single", "restart"):
            total += 8 * (3 * nodes + 6 * cells) * (2 if case["use"] == "restart" else 1)
    return dict(bytes=total, flops=flops)


# ------------------------------------------------------------------ the pass in 64-bit torch

FWD = ([1, 2, 5, 6], [2, 3, 6, 7], [4, 5, 6, 7])
BWD = ([0, 3, 4, 7], [0, 1, 4, 5], [0, 1, 2, 3])


def _amplitude(job, v, t):
    """The burst at time t, the last value held after its end, on the 8 corners' weight."""
    return 0.125 * float(np.interp(t, job["t"], v))


def _exact_job(case, job, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    f64 = dict(dtype=torch.float64, device=dev)
    cells = torch.from_numpy(job["cells"]).to(dev).long()
    xyz = torch.from_numpy(np.stack(job["xyz"])).to(dev)
    nc, nn, d, dt = cells.shape[0], xyz.shape[1], job["d"], job["dt"]
    around = torch.full((nn, 8), nc, dtype=torch.long, device=dev)  # entry nc: no cell there
    ids = torch.arange(nc, device=dev)
    for v in range(8):
        around[cells[:, v], v ^ 6] = ids
    rho = job["rho"] * (around < nc).sum(dim=1).to(torch.float64) / 8
    at = torch.tensor(job["at"], **f64)[:, None]
    points = xyz if job["moment"] else xyz[:, cells].mean(dim=2)
    inside = ((points[2] - at[2]).abs() <= 0.75 * d) & (((points - at) ** 2).sum(dim=0).sqrt() < job["radius"])
    if job["moment"]:
        hits = inside.to(torch.float64)[cells].sum(dim=1)
    else:
        hits = torch.cat([inside.to(torch.float64), torch.zeros(1, **f64)])[around].sum(dim=1)
    c6 = torch.from_numpy(job["c6"]).to(dev)
    plies = None if job["mat"] is None else [torch.from_numpy(np.nonzero(job["mat"] == m)[0]).to(dev)
                                             for m in range(c6.shape[0])]
    scale = None if job["scale"] is None else torch.from_numpy(job["scale"]).to(dev)
    V, S = torch.zeros(3, nn, **f64), torch.zeros(6, nc + 1, **f64)
    if case["use"] == "restart":
        v0, s0 = _checkpoint(job, seed)
        V, S[:, :nc] = torch.from_numpy(v0).to(dev), torch.from_numpy(s0).to(dev)

    def diff(f, links, axis):
        return sum(f[links[:, a]] - f[links[:, b]] for a, b in zip(FWD[axis], BWD[axis])) * (0.25 / d)

    def apply(matrices, e):
        if plies is None:
            return matrices[0] @ e
        s = torch.empty_like(e)
        for m, ply in zip(matrices, plies):
            s[:, ply] = m @ e[:, ply]
        return s

    rows = ((0, 5, 4), (5, 1, 3), (4, 3, 2))  # Voigt index of stress (i, j)
    sensors = torch.from_numpy(job["sensors"]).to(dev).long()
    traces, t = [], 0.0
    for _ in range(case["steps"]):
        f = [sum(diff(S[rows[i][j]], around, j) for j in range(3)) for i in range(3)]
        if not job["moment"]:
            for comp, v in job["discs"]:
                f[comp] = f[comp] + hits * _amplitude(job, v, t)
        V = V + torch.stack(f) * (dt / rho)
        traces.append(V[:, sensors].T)
        g = [[diff(V[k], cells, i) for k in range(3)] for i in range(3)]  # g[i][k] = d V_k / d x_i
        e = torch.stack([g[0][0], g[1][1], g[2][2], g[1][2] + g[2][1], g[0][2] + g[2][0], g[0][1] + g[1][0]])
        r = apply(c6, e) if scale is None else apply(c6, e) * scale
        if job["moment"]:
            for comp, v in job["discs"]:
                r[comp] += hits * _amplitude(job, v, t)
        S[:, :nc] += dt * r
        t += dt
    kinetic = 0.5 * d ** 3 * (rho * (V * V).sum(dim=0)).sum()
    s = S[:, :nc]
    e = apply(torch.linalg.inv(c6), s)
    if scale is not None:
        e = e / scale
    strain = 0.5 * d ** 3 * (s * e).sum()
    return dict(time=t, traces=torch.stack(traces).cpu().numpy(), kinetic=float(kinetic), strain=float(strain),
                V=V.cpu().numpy(), S=s.cpu().numpy())


def exact(case, seed):
    outs = [_exact_job(case, j, seed) for j in _jobs(case, seed)]
    if case["use"] == "batch":
        return [dict(traces=o["traces"], energy=[o["kinetic"], o["strain"]]) for o in outs]
    keys = ("time", "traces", "kinetic", "strain") if case["use"] == "run" else ("time", "traces", "V", "S")
    return {k: outs[0][k] for k in keys}
