"""The work a user of this package has it do, as cases to be timed.

Three kinds of pass, each through the package's public entry points:

  check  one residual check interval of a load step on one handle:
         ``EffPlast2D.iterate(iters)`` and ``residual``; the state stays on the
         GPU, and the pass ends with its U and V fields and the residual
  solve  one whole ``ComputeEffModuli`` call: every load step to its residual
         target, with the records and the moduli at the end
  batch  a kept ``Batch`` engine that is given a set of requests, runs them and
         hands back their results

Inputs are drawn as ``effplast2d_amd.workloads`` draws its requests: pore
count, porosity, yield stress and a preload of random size and direction.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

MAX_CELL_ITERS = 20 * 1024 * 1024 * 1500.0   # the largest listed case


def listed():
    return [
        # the smallest grid the package ships a CLI for, one short check
        # interval: launches and latency
        dict(name="check-64-fp64", kind="check", nX=64, mode="fp64", iters=100, pores=1, tasks=3),
        # the default grid of derive_params (32 nGrid, nGrid = 4): a whole
        # elastoplastic solve, three load steps
        dict(name="solve-128-fp64", kind="solve", nX=128, mode="fp64", iters=20000, check=500,
             tasks=3, pores=1),
        # the reference's kernel structure on the elastic problem
        dict(name="solve-128-plain", kind="solve", nX=128, mode="plain", iters=20000, check=500,
             tasks=1, pores=1),
        # an odd grid, several pores
        dict(name="check-333-split", kind="check", nX=333, mode="split", iters=300, pores=3,
             tasks=3),
        # a mid-size sample of the serving mix, in FP64
        dict(name="check-512-fp64", kind="check", nX=512, mode="fp64", iters=500, pores=2,
             tasks=3),
        # the grid and scheme of the drop-in class and its CLI (NGRID = 32)
        dict(name="check-1024-fp64", kind="check", nX=1024, mode="fp64", iters=500, pores=1,
             tasks=3),
        # the same grid in the split scheme
        dict(name="check-1024-split", kind="check", nX=1024, mode="split", iters=500, pores=1,
             tasks=3),
        # the largest grid of the serving mix
        dict(name="check-2048-split", kind="check", nX=2048, mode="split", iters=300, pores=2,
             tasks=3),
        # the 16-pore grid of the precision comparison, the largest one
        dict(name="check-4096-split", kind="check", nX=4096, mode="split", iters=200, pores=4,
             tasks=3),
        # the benchmark's batch, with the iterations of a step cut short
        dict(name="batch-20x1024-split", kind="batch", nX=1024, count=20, mixed=False,
             mode="split", iters=500, check=500, tasks=3),
        # the batched sweep over grids of 128 to 1024
        dict(name="batch-mixed-64-split", kind="batch", nX=1024, count=64, mixed=True,
             mode="split", iters=1000, check=500, tasks=3),
        # an FP64 batch
        dict(name="batch-12x1024-fp64", kind="batch", nX=1024, count=12, mixed=False,
             mode="fp64", iters=250, check=250, tasks=3),
    ]


def draw(rng):
    kind = rng.choice(["check", "check", "check", "solve", "batch"])
    mode = rng.choice(["fp64", "split"])
    if kind == "check":
        n = int(round(math.exp(rng.uniform(math.log(24), math.log(4096)))))
        if rng.random() < 0.4:
            n = max(32, (n + 16) // 32 * 32)
        if rng.random() < 0.1:
            mode, n = "plain", min(n, 1024)
        iters = int(round(math.exp(rng.uniform(math.log(50), math.log(1000)))))
        iters = max(20, min(iters, int(0.15 * MAX_CELL_ITERS / (n * n))))
        return dict(kind="check", nX=n, mode=mode, iters=iters, pores=rng.randint(1, 4),
                    tasks=rng.choice([1, 2, 3, 3]))
    if kind == "solve":
        n = int(round(math.exp(rng.uniform(math.log(48), math.log(400)))))
        return dict(kind="solve", nX=n, mode=mode, iters=8000, check=rng.choice([200, 500]),
                    tasks=rng.choice([1, 2, 3]), pores=rng.randint(1, 3))
    n = int(round(math.exp(rng.uniform(math.log(100), math.log(1200)))))
    count = rng.randint(4, 40)
    iters = rng.choice([200, 300, 500])
    while count * n * n * 3.0 * iters > 0.8 * MAX_CELL_ITERS:
        count -= 1
    return dict(kind="batch", nX=n, count=max(1, count), mixed=rng.random() < 0.5, mode=mode,
                iters=iters, check=iters, tasks=rng.choice([1, 2, 3]))


def work(case):
    """A pass reads the displacement and velocity fields once and writes them
    once; the stencil's arithmetic is counted per cell and iteration: strains
    and trial stress 25, the two yield invariants 24, velocity and
    displacement 24."""
    vb = 4 if case["mode"] == "split" else 8
    flops = 49 + (24 if case["tasks"] > 1 else 0)
    if case["kind"] == "check":
        cells, iters = case["nX"] ** 2, case["iters"]
    elif case["kind"] == "solve":
        # the preload takes about seven iterations per grid line, a small
        # increment about five
        n = case["nX"]
        cells = n * n
        per = (7, 12, 17)[case["tasks"] - 1] * n
        iters = min(max(per, case["check"]), case["iters"] * case["tasks"])
    else:
        cells = sum(n * n for n in _sizes(case))
        iters = case["iters"] * case["tasks"]
    return {"bytes": 2.0 * cells * (16 + 2 * vb), "flops": float(flops) * cells * iters}


# -- inputs --------------------------------------------------------------------
LX = 20.0
K0, G0, RHO0, CFL = 1.0, 0.5, 1.0, 0.5


def _sizes(case):
    if not case["mixed"]:
        return [case["nX"]] * case["count"]
    steps = (8, 4, 2, 1)
    return [max(16, case["nX"] // steps[k % 4]) for k in range(case["count"])]


def _sample(rng, n, pores):
    """One RVE: parameter vector (get_sigma_2D.m:3-32) and preload."""
    phi = rng.uniform(0.005, 0.05)
    Y = rng.uniform(1e-3, 5e-3)
    mag = rng.uniform(1e-3, 5e-3)
    u = [rng.gauss(0.0, 1.0) for _ in range(3)]
    s = math.sqrt(sum(x * x for x in u))
    dX = LX / (n - 1)
    dt = CFL * dX / math.sqrt((K0 + 4.0 * G0 / 3.0) / RHO0)
    damp = 4.0 / dt / n
    rad = math.sqrt(phi * LX * LX / (math.pi * pores * pores))
    pa = np.array([dX, dX, dt, K0, G0, RHO0, damp, damp, Y * math.sqrt(2.0), rad, float(pores)])
    return pa, -mag, [x / s for x in u]


def _elastic_load(case, load, lt):
    # the elastic problem is loaded within the elastic range, isotropically
    return (1e-2 * load, [1.0, 1.0, 0.0]) if case["tasks"] == 1 else (load, lt)


class _Field:
    """A device buffer of a handle, for torch.as_tensor (no copy); it keeps
    the handle, which owns the buffer."""

    def __init__(self, owner, ptr, shape, f32):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "strides": None,
                                         "typestr": "<f4" if f32 else "<f8", "version": 2}


def _field(g, name):
    m, n = g.field_shape(name)
    f32 = g.mode == "split" and name in ("Vx", "Vy")
    buf = _Field(g, g.device_ptr(name), (n, m), f32)
    t = torch.as_tensor(buf, device="cuda")
    t.owner = buf
    return t


def prepare(case, seed):
    from effplast2d_amd import Batch, EffPlast2D
    rng = random.Random(f"{seed}")
    if case["kind"] == "batch":
        eng = Batch(mode=case["mode"], checkInterval=case["check"])
        reqs = []
        for k, n in enumerate(_sizes(case)):
            pa, load, lt = _sample(rng, n, rng.randint(1, 3))
            load, lt = _elastic_load(case, load, lt)
            reqs.append(dict(pa=pa, nX=n, nTasks=case["tasks"], nIter=case["iters"], eIter=1e-8,
                             initLoad=load, loadType=lt, shearLoadType=[0.0, 0.0, 1.0], tag=k))
        return dict(case=case, eng=eng, reqs=reqs)
    pa, load, lt = _sample(rng, case["nX"], case["pores"])
    load, lt = _elastic_load(case, load, lt)
    if case["kind"] == "solve":
        g = EffPlast2D(pa, case["nX"], nTasks=case["tasks"], nIter=case["iters"], eIter=1e-8,
                       checkInterval=case["check"], mode=case["mode"],
                       shearLoadType=[0.0, 0.0, 1.0])
        return dict(case=case, g=g, load=load, lt=lt)
    g = EffPlast2D(pa, case["nX"], nTasks=case["tasks"], mode=case["mode"])
    e = [load * x for x in lt]
    g.apply_affine(e[0], e[1], e[2], e[2])
    return dict(case=case, g=g, strain=e)


def _moduli(res):
    return {k: [res["num"][k], res["num_per"][k]] for k in ("Kphi", "Kd", "G")} | {
        "Gxy": [res["Gxy"], res["GxyPer"]]}


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        eng = state["eng"]
        for rq in state["reqs"]:
            eng.submit(**rq)
        eng.run()
        out = sorted(eng.poll(), key=lambda r: r["tag"])
        return {"status": np.array([r["status"] for r in out], dtype=np.int64),
                "iters": np.array([r["result"]["totalIters"] for r in out], dtype=np.int64),
                "moduli": np.array([sum(_moduli(r["result"]).values(), []) for r in out])}
    g = state["g"]
    if case["kind"] == "check":
        g.iterate(case["iters"])
        err, bad = g.residual(state["strain"])
        return {"residual": err, "bad": bad,
                "U": [_field(g, "Ux"), _field(g, "Uy")], "V": [_field(g, "Vx"), _field(g, "Vy")]}
    res = g.ComputeEffModuli(state["load"], state["lt"])
    recs = g.records()
    return {"iters": np.array([int(r["iters"]) for r in recs], dtype=np.int64),
            "sigma": np.array([list(r["sigma"])[:3] for r in recs]),
            "pore": np.array([[r["deltaP"], r["dPhi"]] for r in recs]),
            "moduli": {k: _moduli(res)[k][0] for k in ("Kphi", "Kd")},
            "U": [_field(g, "Ux"), _field(g, "Uy")]}


# -- the same in plain torch, FP64 ----------------------------------------------
class _Exact:
    """get_sigma_2D.m:45-166 with the CUDA path's edge averages, fields [j, i]."""

    def __init__(self, pa, n, plastic):
        (self.dX, self.dY, self.dt, k0, g0, rho, dampx, dampy, self.coh, self.rad,
         self.N) = [float(v) for v in pa]
        self.n, self.plastic = n, plastic
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        dX, dY, N = self.dX, self.dY, int(self.N)
        i = torch.arange(n, dtype=torch.float64, device=self.dev)
        lx, ly = dX * (n - 1), dY * (n - 1)
        x, y = -0.5 * lx + dX * i, -0.5 * ly + dY * i
        vx, vy = (-0.5 * dX * (n - 2) + dX * i)[:-1], (-0.5 * dY * (n - 2) + dY * i)[:-1]

        def inside(a, b):
            m = torch.zeros((b.numel(), a.numel()), dtype=torch.bool, device=self.dev)
            for k in range(N):
                for q in range(N):
                    ca = a - 0.5 * lx * (1.0 - 1.0 / N) + (lx / N) * k
                    cb = b - 0.5 * ly * (1.0 - 1.0 / N) + (ly / N) * q
                    m |= torch.sqrt(ca[None, :] ** 2 + cb[:, None] ** 2) < self.rad
            return m

        self.cell, self.vert = inside(x, y), inside(vx, vy)
        one = torch.ones((n, n), dtype=torch.float64, device=self.dev)
        self.K = torch.where(self.cell, 0.01 * k0 * one, k0 * one)
        self.G = torch.where(self.cell, 0.01 * g0 * one, g0 * one)
        G = self.G
        self.Gv = 0.25 * (G[:-1, :-1] + G[:-1, 1:] + G[1:, :-1] + G[1:, 1:])
        self.vdx, self.vdy, self.dr = 1.0 - self.dt * dampx, 1.0 - self.dt * dampy, self.dt / rho
        z = lambda a, b: torch.zeros((a, b), dtype=torch.float64, device=self.dev)  # noqa: E731
        self.Ux, self.Uy, self.Vx, self.Vy = z(n, n + 1), z(n + 1, n), z(n, n + 1), z(n + 1, n)

    def affine(self, exx, eyy, exy):
        n, dX, dY = self.n, self.dX, self.dY
        a = lambda m: torch.arange(m, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.Ux += ((-0.5 * dX * n + dX * a(n + 1)) * exx)[None, :] + \
            ((-0.5 * dY * (n - 1) + dY * a(n)) * exy)[:, None]
        self.Uy += ((-0.5 * dY * n + dY * a(n + 1)) * eyy)[:, None] + \
            ((-0.5 * dX * (n - 1) + dX * a(n)) * exy)[None, :]

    def stress(self):
        Ux, Uy = self.Ux, self.Uy
        exx, eyy = (Ux[:, 1:] - Ux[:, :-1]) / self.dX, (Uy[1:] - Uy[:-1]) / self.dY
        d = exx + eyy
        P = (-self.K * d).masked_fill_(self.cell, 0.0)
        txx = (2.0 * self.G * (exx - d / 3.0)).masked_fill_(self.cell, 0.0)
        tyy = (2.0 * self.G * (eyy - d / 3.0)).masked_fill_(self.cell, 0.0)
        txy = self.Gv * ((Ux[1:, 1:-1] - Ux[:-1, 1:-1]) / self.dY +
                         (Uy[1:-1, 1:] - Uy[1:-1, :-1]) / self.dX)
        txy.masked_fill_(self.vert, 0.0)
        if self.plastic:
            av4 = lambda t: 0.25 * (t[:-1, :-1] + t[:-1, 1:] + t[1:, :-1] + t[1:, 1:])  # noqa: E731
            av = torch.nn.functional.pad(av4(txy)[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
            J2 = torch.sqrt(txx * txx + tyy * tyy + 2.0 * av * av)
            Jv = torch.sqrt(av4(txx) ** 2 + av4(tyy) ** 2 + 2.0 * txy * txy)
            s = torch.where(J2 > self.coh, self.coh / J2, torch.ones_like(J2))
            sv = torch.where(Jv > self.coh, self.coh / Jv, torch.ones_like(Jv))
            txx, tyy, txy = txx * s, tyy * s, txy * sv
        return P, txx, tyy, txy

    def iterate(self, iters):
        n = self.n
        for _ in range(iters):
            self.last = P, txx, tyy, txy = self.stress()
            a, b = txx - P, tyy - P
            self.Vx[1:-1, 1:n] = self.Vx[1:-1, 1:n] * self.vdx + self.dr * (
                (a[1:-1, 1:] - a[1:-1, :-1]) / self.dX + (txy[1:] - txy[:-1]) / self.dY)
            self.Vy[1:n, 1:-1] = self.Vy[1:n, 1:-1] * self.vdy + self.dr * (
                (b[1:, 1:-1] - b[:-1, 1:-1]) / self.dY + (txy[:, 1:] - txy[:, :-1]) / self.dX)
            self.Ux[:, :n] += self.Vx[:, :n] * self.dt
            self.Uy[:n] += self.Vy[:n] * self.dt

    def residual(self, e):
        n = self.n
        return (float(self.Vx.abs().max()) / (self.dX * (n - 1)) +
                float(self.Vy.abs().max()) / (self.dY * (n - 1))) * self.dt / \
            max(abs(e[0]), e[1], e[2])

    # the volume averages, boundary mean and hole area of a load step
    def record(self, nu0):
        n, (P, txx, tyy, txy) = self.n, self.last
        c = slice(1, n - 1)
        s0, s1 = float((txx - P)[c, c].sum()), float((tyy - P)[c, c].sum())
        s2 = float((txy[1:, 1:] + nu0 * (txx + tyy - 2.0 * P)[c, c]).sum())
        sig = [s0 / (n * n), s1 / (n * n), s2 / ((n - 1) * (n - 1))]
        q = txx + tyy - 2.0 * P
        dP = -0.125 * (float(q[0, c].sum() + q[n - 1, c].sum()) / (n - 2) +
                       float(q[c, 0].sum() + q[c, n - 1].sum()) / (n - 2))
        return sig, dP, self._hole()

    def _hole(self):
        n, N, rad = self.n, int(self.N), self.rad
        dX, dY, lx, ly = self.dX, self.dY, self.dX * (n - 1), self.dY * (n - 1)
        Ux, Uy = self.Ux.cpu().numpy().ravel(), self.Uy.cpu().numpy().ravel()

        def inside(uy, i, j):
            x = (-0.5 * lx if uy else -0.5 * dX * n) + dX * i
            y = (-0.5 * dY * n if uy else -0.5 * ly) + dY * j
            return any(math.hypot(x - 0.5 * lx * (1 - 1 / N) + lx / N * k,
                                  y - 0.5 * ly * (1 - 1 / N) + ly / N * q) < rad
                       for k in range(N) for q in range(N))

        def signed(uy, flats):
            m, best = (n if uy else n + 1), 0.0
            for f in flats:
                v = 0.0 if inside(uy, f % m, f // m) else float((Uy if uy else Ux)[f])
                if abs(v) > abs(best):
                    best = v
            return best

        area = 0.0
        for k in range(N):
            for q in range(N):
                cx = 0.5 * (n - 1) * (1 - 1 / N) - (n - 1) / N * k
                cy = 0.5 * (n - 1) * (1 - 1 / N) - (n - 1) / N * q
                row = int(cy + 0.5 * (n - 1)) * (n + 1)
                r0, r1 = int(cx - rad / dX + 0.5 * n), int(cx + rad / dX + 0.5 * n)
                col = int(cx + 0.5 * (n - 1))
                b0, b1 = int(cy - rad / dY + 0.5 * n), int(cy + rad / dY + 0.5 * n)
                dx = -0.5 * (signed(False, [row + r0 - 1 + t for t in range(5)]) -
                             signed(False, [row + r1 - 2 + t for t in range(5)]))
                dy = -0.5 * (signed(True, [(b0 - 1 + t) * n + col for t in range(5)]) -
                             signed(True, [(b1 - 2 + t) * n + col for t in range(5)]))
                area += (rad + dx) * (rad + dy)
        return 3.1415926 * abs(area - rad * rad * N * N) / (lx * ly)


def exact(case, seed):
    if case["kind"] == "batch":
        return None
    rng = random.Random(f"{seed}")
    pa, load, lt = _sample(rng, case["nX"], case["pores"])
    load, lt = _elastic_load(case, load, lt)
    s = _Exact(pa, case["nX"], case["tasks"] > 1)
    if case["kind"] == "check":
        e = [load * x for x in lt]
        s.affine(*e)
        s.iterate(case["iters"])
        return {"residual": s.residual(e), "bad": 0, "U": [s.Ux, s.Uy], "V": [s.Vx, s.Vy]}
    inc, sph = 0.005, 0.5 * (lt[0] + lt[1])
    steps = [[load * x for x in lt], [load * inc * sph, load * inc * sph, 0.0],
             [0.0, 0.0, load * inc]][:case["tasks"]]
    nu0 = (1.5 * K0 - G0) / (3.0 * K0 + G0)
    e, its, recs = [0.0, 0.0, 0.0], [], []
    for de in steps:
        e = [a + b for a, b in zip(e, de)]
        s.affine(*de)
        done = 0
        while done < case["iters"]:
            c = min(case["check"], case["iters"] - done)
            s.iterate(c)
            done += c
            if c == case["check"] and s.residual(e) < 1e-8:
                break
        its.append(done)
        recs.append(s.record(nu0) + (e,))
    b = 0 if case["tasks"] == 1 else 1
    zero = ([0.0, 0.0, 0.0], 0.0, 0.0, [0.0, 0.0, 0.0])
    r0, r1 = (recs[0], recs[1]) if b else (zero, recs[0])
    kphi = (r1[1] - r0[1]) / (r1[2] - r0[2])
    kd = 0.33333333 * sum(p - q for p, q in zip(r1[0], r0[0])) / (r1[3][0] + r1[3][1] - r0[3][0] - r0[3][1])
    return {"iters": np.array(its, dtype=np.int64), "sigma": np.array([r[0] for r in recs]),
            "pore": np.array([[r[1], r[2]] for r in recs]),
            "moduli": {"Kphi": kphi, "Kd": kd}, "U": [s.Ux, s.Uy]}
