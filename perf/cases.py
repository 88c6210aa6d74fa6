"""The work that a program has this library do, as measurable cases.

A case is one pass of a program's loop through the public entry points of
`sphugo_amd`: some steps of a simulation and the pull of its fields that the
program draws or stores (the Animator of the reference pulls x, y, rho and h
of every frame), a force pass, a neighbour readback, a batch of independent
simulations, or a burst of jobs through the serve loop.

Layouts (seeded NumPy draws of the layouts in sphugo_amd/ics.py and of the
reference's example configurations):
  uniform    periodic unit box, at rest, e = 1
  blast      70 % uniform, 30 % in a Gaussian at the centre, e = 10 inside it
  clustered  80 % in 16 Gaussians (sigma 0.02), v ~ N(0, 0.1^2) per axis
  speedtest  the reference's timing harness: open axes, mass 1, DeltaTHalf
             0.02, gravity (0, 0.2)
  tube       the reference's second example: open axes with three walls,
             Wendland, gamma 4.666, mass 1e5, DeltaTHalf 0.00424

In the FP32-compensated form the pair sums are computed in 32 bits, and a
program keeps what it pulls as float32; plain FP64 stays float64.
"""
import math
import random

import numpy as np
import torch

from sphugo_amd import _lib as L

FRAME = ("x", "y", "rho", "h")                       # what a frame of the Animator shows
STATE = ("x", "y", "vx", "vy", "e", "rho", "h")      # what a served job returns
FORCES = ("rho", "h", "ax", "ay", "edot")
OPEN = (-L.DBL_MAX, L.DBL_MAX)
NO_WALLS = (-L.DBL_MAX, L.DBL_MAX, -L.DBL_MAX, L.DBL_MAX)


def listed():
    return [
        # a viewer that steps once and draws: the smallest call there is
        dict(name="frame-uniform-2200", kind="steps", layout="uniform", n=2200, k=32,
             kernel="monaghan", prec="fp64", steps=1, graph=False),
        # the same box run for a while between two pulls, replayed from a graph
        dict(name="run-uniform-2200", kind="steps", layout="uniform", n=2200, k=32,
             kernel="monaghan", prec="fp64", steps=50, graph=True),
        # one small served job: the reference's second example configuration
        # (open axes, walls), from its initial condition
        dict(name="job-tube-4700", kind="serve", layout="tube", count=1, lo=4700, hi=4700, draw=0,
             kernel="wendland", prec="fp64", steps_lo=20, steps_hi=20),
        # CalculateForces on the input of the reference's timing harness
        dict(name="forces-open-100000", kind="forces", layout="speedtest", n=100000, k=32,
             kernel="monaghan", prec="fp64"),
        # CalculateForces in the reference's own summation order
        dict(name="forces-bitwise-30011", kind="forces", layout="clustered", n=30011, k=32,
             kernel="monaghan", prec="bitwise"),
        # a frame that also shows neighbours (NearestNeighbours, NNDists, NNPos)
        dict(name="neighbours-50021", kind="neighbours", layout="uniform", n=50021, k=32,
             kernel="monaghan", prec="fp64"),
        # an odd size and an odd neighbour count in the FP32-compensated form
        dict(name="run-wendland-77777", kind="steps", layout="uniform", n=77777, k=19,
             kernel="wendland", prec="fp32c", steps=10, graph=False),
        # the blast of 262,144 particles
        dict(name="blast-262144", kind="steps", layout="blast", n=262144, k=32,
             kernel="monaghan", prec="fp64", steps=20, graph=False),
        # a million particles in plain FP64
        dict(name="clustered-1M", kind="steps", layout="clustered", n=1048576, k=64,
             kernel="monaghan", prec="fp64", steps=20, graph=False),
        # the headline size: 4M clustered, FP32-compensated
        dict(name="clustered-4M", kind="steps", layout="clustered", n=4194304, k=64,
             kernel="monaghan", prec="fp32c", steps=20, graph=False),
        # independent simulations stepped together
        dict(name="batch-32", kind="batch", count=32, lo=1024, hi=65536, draw=4, k=32,
             kernel="monaghan", prec="fp32c", steps=10, graph=True),
        # jobs of mixed size, k and length through the serve loop
        dict(name="serve-12", kind="serve", layout="", count=12, lo=1024, hi=131072, draw=5,
             kernel="monaghan", prec="fp64", steps_lo=10, steps_hi=60),
    ]


def draw(rng):
    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return n | 1 if rng.random() < 0.5 else n

    kind = rng.choice(["steps"] * 6 + ["forces", "neighbours", "batch", "serve"])
    c = dict(kind=kind, kernel=rng.choice(["monaghan", "monaghan", "wendland"]),
             prec=rng.choice(["fp64", "fp32c"]))
    if kind == "steps":
        c["layout"] = rng.choice(["uniform", "blast", "clustered"])
        c["n"] = size(2000, 1 << 20)
        c["k"] = rng.choice([16, 19, 32, 32, 47, 64])
        c["steps"] = rng.choice([1, 5, 10, 20])
        c["graph"] = rng.random() < 0.3
    elif kind == "forces":
        c["layout"] = rng.choice(["uniform", "blast", "clustered", "speedtest"])
        c["n"] = size(2000, 1 << 17)
        c["k"] = rng.choice([16, 32, 33, 64])
        c["prec"] = rng.choice(["bitwise", "fp64", "fp32c"])
    elif kind == "neighbours":
        c["layout"] = rng.choice(["uniform", "blast"])
        c["n"] = size(2000, 1 << 17)
        c["k"] = rng.choice([16, 32, 33])
        c["prec"] = "fp64"
    elif kind == "batch":
        c.update(count=rng.randrange(8, 49), lo=1024, hi=65536, draw=rng.randrange(1 << 16),
                 k=rng.choice([16, 32, 40]), steps=rng.choice([5, 10]), graph=rng.random() < 0.7)
    else:
        c.update(layout=rng.choice(["", "", "speedtest", "tube"]), count=rng.randrange(1, 13),
                 lo=1024, hi=131072, draw=rng.randrange(1 << 16), steps_lo=10, steps_hi=60)
        if c["layout"]:  # fixed half steps: as long as the reference's harness runs
            c.update(hi=8192 if c["layout"] == "tube" else 131072, steps_hi=20)
    return c


# --------------------------------------------------------------------------
# inputs

def _layout(name, n, g):
    """Positions, velocities, energies of one simulation from generator g."""
    vx = vy = np.zeros(n)
    e = np.ones(n)
    if name in ("uniform", "speedtest"):
        x, y = g.random(n), g.random(n)
        if name == "speedtest":
            e = np.full(n, 0.01)
    elif name == "blast":
        nb = int(0.3 * n)
        x, y = g.random(n), g.random(n)
        x[n - nb:] = 0.5 + 0.05 * g.standard_normal(nb)
        y[n - nb:] = 0.5 + 0.05 * g.standard_normal(nb)
        e[(x - 0.5) ** 2 + (y - 0.5) ** 2 < 0.05 ** 2] = 10.0
    elif name == "clustered":
        nc = int(0.8 * n)
        cx, cy = g.random(16), g.random(16)
        which = np.arange(nc) % 16
        x, y = g.random(n), g.random(n)
        x[:nc] = cx[which] + 0.02 * g.standard_normal(nc)
        y[:nc] = cy[which] + 0.02 * g.standard_normal(nc)
        vx, vy = 0.1 * g.standard_normal(n), 0.1 * g.standard_normal(n)
    else:  # tube: a long and a tall rectangle
        n0 = n * 40 // 47
        x, y = 0.3 + 0.4 * g.random(n), g.random(n)
        y[:n0] = 0.3 + 0.1 * y[:n0]
        y[n0:] = 0.3 + 0.2 * y[n0:]
        e = np.full(n, 0.01)
    if name in ("blast", "clustered"):
        x, y = x - np.floor(x), y - np.floor(y)
        x[x >= 1.0] = 0.0
        y[y >= 1.0] = 0.0
    return dict(x=x, y=y, vx=vx, vy=vy, e=e)


def _physics(layout, n):
    """What a program sets in the configuration of such a simulation."""
    p = dict(gamma=5 / 3, mass=1.0 / n, dt_half=0.0, cfl=0.3, accel=(0.0, 0.0), hor=(0.0, 1.0),
             vert=(0.0, 1.0), refl=NO_WALLS, visc_alpha=1.0, visc_beta=2.0, visc_eta2=0.01)
    if layout == "speedtest":
        p.update(gamma=1.66666, mass=1.0, dt_half=0.02, accel=(0.0, 0.2), hor=OPEN, vert=OPEN,
                 visc_alpha=0.75, visc_beta=1.5)
    elif layout == "tube":
        p.update(gamma=4.666, mass=1e5, dt_half=0.00424, accel=(0.0, 0.05), hor=OPEN, vert=OPEN,
                 refl=(0.2, L.DBL_MAX, 0.25, 0.5), visc_alpha=0.75, visc_beta=1.5)
    return p


def _plan(case):
    """Size, k, steps and layout of each simulation of a case."""
    if case["kind"] not in ("batch", "serve"):
        return [(case["n"], case["k"], case.get("steps", 1), case["layout"])]
    r = random.Random(case["draw"])
    out = []
    for _ in range(case["count"]):
        n = round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]))))
        k, steps, layout = case.get("k"), case.get("steps"), "blast"
        if case["kind"] == "serve":
            k, steps = r.choice([32, 64]), r.randint(case["steps_lo"], case["steps_hi"])
            layout = r.choice(["blast", "clustered"])
            if case["layout"]:  # the reference's configurations, with its NN_SIZE
                k, layout = 32, case["layout"]
        out.append((n, k, steps, layout))
    return out


def _sims(case, seed):
    """The simulations of a case: (state, physics, k, steps) each."""
    return [(_layout(layout, n, np.random.default_rng([seed, i])), _physics(layout, n), k, steps)
            for i, (n, k, steps, layout) in enumerate(_plan(case))]


def _params(case, phys, k):
    return L.default_params(
        k=k, kernel=L.KERNEL_WENDLAND if case["kernel"] == "wendland" else L.KERNEL_MONAGHAN,
        precision=L.PREC_FP32C if case["prec"] == "fp32c" else L.PREC_FP64,
        flags=L.FLAG_BITWISE if case["prec"] == "bitwise" else 0, **phys)


def prepare(case, seed):
    sims = _sims(case, seed)
    kind = case["kind"]
    state = dict(case=case)
    if kind == "batch":
        state["sim"] = L.Batch([_params(case, ph, k) for _, ph, k, _ in sims],
                               [st for st, _, _, _ in sims])
    elif kind == "serve":
        total = sum(len(st["x"]) for st, _, _, _ in sims)
        state["server"] = L.Server(total + 4096, max_jobs=len(sims), kmax=64,
                                   precision=_params(case, sims[0][1], 32).precision)
        state["jobs"] = [(_params(case, ph, k), st, steps) for st, ph, k, steps in sims]
    else:
        st, ph, k, _ = sims[0]
        state["sim"] = L.Sim(_params(case, ph, k), st["x"], st["y"], st["vx"], st["vy"], st["e"])
        if kind == "forces":  # CalculateForces reads the predicted state
            state["sim"].set("vpx", st["vx"])
            state["sim"].set("vpy", st["vy"])
            state["sim"].set("epred", st["e"])
    if case.get("graph"):
        L.set_graph(state["sim"], True)
    return state


# --------------------------------------------------------------------------
# one pass

def _kept(case, a):
    return a.astype(np.float32) if case["prec"] == "fp32c" else a


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "serve":
        srv = state["server"]
        ids = [srv.submit(p, st, steps) for p, st, steps in state["jobs"]]
        out = []
        for j in ids:
            srv.wait(j)
            out.append({f: _kept(case, srv.result(j, f)) for f in ("x", "y", "vx", "rho", "h")})
            srv.release(j)
        return out
    sim = state["sim"]
    if kind == "forces":
        sim.calculate_forces()
        return {f: _kept(case, sim.get(f)) for f in FORCES}
    if kind == "neighbours":
        sim.step(1)
        ids, d2 = sim.neighbours()
        px, py = sim.neighbour_pos()
        return dict(x=sim.get("x"), y=sim.get("y"), h=sim.get("h"), ids=ids.view(np.int32), d2=d2,
                    px=px, py=py)
    sim.step(case["steps"])
    fields = STATE if kind == "batch" else FRAME
    return {f: _kept(case, sim.get(f)) for f in fields}


def work(case):
    """Own state read and written once per step, what is pulled written once;
    per neighbour about 10 operations of density, 35 of force, 5 of distance."""
    byts = flops = 0.0
    passes = 1 if case["kind"] in ("forces", "neighbours") else None
    for n, k, steps, _ in _plan(case):
        s = passes or steps
        byts += s * n * 2 * 8 * 8.0
        flops += s * n * k * 50.0
        fields = {"forces": 5, "neighbours": 3, "batch": 7, "serve": 5}.get(case["kind"], 4)
        byts += n * fields * 8.0
        if case["kind"] == "neighbours":
            byts += n * k * (4 + 3 * 8.0)
    return {"bytes": byts, "flops": flops}


# --------------------------------------------------------------------------
# the same in 64 bits, in plain torch

def exact(case, seed):
    plan = _plan(case)
    if case["kind"] != "serve" and sum(n * (s + 1) for n, _, s, _ in plan) > 6e6:
        return None
    out = []
    budget = 4e6
    for (st, ph, k, steps), (n, _, _, _) in zip(_sims(case, seed), plan):
        if case["kind"] == "serve":
            budget -= n * (steps + 1)
            if budget < 0:
                out.append(None)
                continue
        r = _Exact(st, ph, k, case["kernel"])
        if case["kind"] == "forces":
            r.forces()
        else:
            r.run(steps)
        out.append(r)
    if case["kind"] == "serve":
        return [None if r is None else {f: r.get(f) for f in ("x", "y", "vx", "rho", "h")}
                for r in out]
    if case["kind"] == "batch":
        return {f: np.concatenate([r.get(f) for r in out]) for f in STATE}
    r = out[0]
    if case["kind"] == "forces":
        return {f: r.get(f) for f in FORCES}
    if case["kind"] == "neighbours":
        # rows are pulled after the step's last drift, and show its pass: they
        # are held to the pass's own positions
        return dict(x=r.get("x"), y=r.get("y"), h=r.get("h"), ids=None,
                    d2=r.d2.cpu().numpy(), px=(r.xp[:, None] - r.rx).cpu().numpy(),
                    py=(r.yp[:, None] - r.ry).cpu().numpy())
    return {f: r.get(f) for f in FRAME}


class _Exact:
    """One simulation of the reference's scheme: exact k nearest neighbours
    over the periodic images, density, force, drift-kick-drift."""

    def __init__(self, st, ph, k, kernel):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        for f in ("x", "y", "vx", "vy", "e"):
            setattr(self, f, torch.tensor(st[f], dtype=torch.float64, device=self.dev))
        self.p, self.k, self.wendland = ph, k, kernel == "wendland"
        self.vpx, self.vpy, self.ep = self.vx, self.vy, self.e
        self.open = (ph["hor"] == OPEN, ph["vert"] == OPEN)
        self.dt = ph["dt_half"]

    def get(self, f):
        return getattr(self, f).cpu().numpy()

    def run(self, steps):
        self.forces()
        for _ in range(steps):
            self.step()

    def _span(self, axis):
        return 0.0 if self.open[axis] else self.p["hor" if axis == 0 else "vert"][1] - \
            self.p["hor" if axis == 0 else "vert"][0]

    def knn(self):
        """ids, squared distances (ascending) and p_i - (p_j - o) of the k nearest."""
        x, y, k, n = self.x, self.y, self.k, len(self.x)
        lx, ly = self._span(0), self._span(1)
        ox = [0.0] if self.open[0] else [-lx, 0.0, lx]
        oy = [0.0] if self.open[1] else [-ly, 0.0, ly]
        ix = torch.arange(n, device=self.dev)
        cx = torch.cat([x - a for a in ox for _ in oy])
        cy = torch.cat([y - b for _ in ox for b in oy])
        cj = ix.repeat(len(ox) * len(oy))
        # queries in Morton order, so that a run of them is compact
        gx = ((x - x.min()) / (x.max() - x.min()) * 65535).long()
        gy = ((y - y.min()) / (y.max() - y.min()) * 65535).long()
        key = torch.zeros_like(gx)
        for b in range(16):
            key |= ((gx >> b) & 1) << (2 * b) | ((gy >> b) & 1) << (2 * b + 1)
        order = torch.argsort(key)
        ids = torch.empty((n, k), dtype=torch.long, device=self.dev)
        d2 = torch.empty((n, k), dtype=torch.float64, device=self.dev)
        rx, ry = torch.empty_like(d2), torch.empty_like(d2)
        run_ = 1024
        for a in range(0, n, run_):
            q = order[a:a + run_]
            qx, qy = x[q], y[q]
            x0, x1, y0, y1 = (float(v) for v in torch.stack(
                [qx.min(), qx.max(), qy.min(), qy.max()]).cpu())
            reach = math.sqrt(3.0 * k / math.pi * max((x1 - x0) * (y1 - y0), 1e-12) / len(q))
            while True:
                near = ((cx >= x0 - reach) & (cx <= x1 + reach) & (cy >= y0 - reach) &
                        (cy <= y1 + reach)).nonzero().squeeze(1)
                if len(near) <= k:
                    reach *= 1.7
                    continue
                ex = qx[:, None] - cx[near][None]
                ey = qy[:, None] - cy[near][None]
                dd = ex * ex + ey * ey
                dd.masked_fill_(cj[near][None] == q[:, None], math.inf)
                v, w = torch.topk(dd, k, dim=1, largest=False, sorted=True)
                far = float(v[:, -1].max().sqrt())
                if far <= reach:
                    break
                reach = min(far * 1.001, reach * 3.0)
            ids[q] = cj[near][w]
            d2[q] = v
            rx[q] = ex.gather(1, w)
            ry[q] = ey.gather(1, w)
        return ids, d2, rx, ry

    def forces(self):
        p = self.p
        self.ids, self.d2, self.rx, self.ry = self.knn()
        self.xp, self.yp = self.x, self.y
        h = self.d2[:, -1].sqrt()
        d = self.d2.sqrt()
        q = d / h[:, None]
        a = 1 - q
        if self.wendland:
            F, DF = a ** 4 * (1 + 4 * q), -10 * q * a ** 3
            fpref, dfpref = 7 / math.pi, 14 / math.pi
        else:
            F = torch.where(q < 0.5, q ** 3 - q ** 2 + 1 / 6, a ** 3 / 3)
            DF = torch.where(q < 0.5, 3 * q * q - 2 * q, -a * a)
            fpref = dfpref = 240 / (7 * math.pi)
        rho = fpref * p["mass"] * F.sum(1) / (h * h)
        c = torch.sqrt(p["gamma"] * (p["gamma"] - 1) * self.ep)
        B = c * c / (p["gamma"] * rho)
        j = self.ids
        rx, ry = -self.rx, -self.ry
        vx, vy = self.vpx[j] - self.vpx[:, None], self.vpy[j] - self.vpy[:, None]
        dot = vx * rx + vy * ry
        mu = dot * 0.5 * (h[:, None] + h[j]) / (self.d2 + p["visc_eta2"])
        pi = (-p["visc_alpha"] * 0.5 * (c[:, None] + c[j]) * mu + p["visc_beta"] * mu * mu) / \
            (0.5 * (rho[:, None] + rho[j]))
        pi = torch.where(dot < 0, pi, torch.zeros_like(pi))
        w = (pi + B[:, None] + B[j]) * DF / d
        fac = p["mass"] * dfpref / h ** 3
        self.ax = (rx * w).sum(1) * fac + p["accel"][0]
        self.ay = (ry * w).sum(1) * fac + p["accel"][1]
        self.edot = B * (dot * DF).sum(1) * p["mass"]
        self.rho, self.h, self.c = rho, h, c
        self._next_dt()

    def _next_dt(self):
        if self.p["dt_half"] <= 0:
            v = torch.sqrt(self.vx ** 2 + self.vy ** 2)
            self.dt = 0.5 * self.p["cfl"] * float((0.5 * self.h / (self.c + v)).min())

    def step(self):
        p, dt = self.p, self.dt
        self.x, self.y = self.x + self.vx * dt, self.y + self.vy * dt
        self.vpx, self.vpy = self.vx + self.ax * dt, self.vy + self.ay * dt
        self.ep = self.e + self.edot * dt
        self.forces()
        self.vx, self.vy = self.vx + self.ax * 2 * dt, self.vy + self.ay * 2 * dt
        self.e = self.e + self.edot * 2 * dt
        x, y = self.x + self.vx * dt, self.y + self.vy * dt
        # the wrap of y is skipped where x wraps
        done = torch.zeros_like(x, dtype=torch.bool)
        if not self.open[0]:
            lo, hi = x < p["hor"][0], x > p["hor"][1]
            x = x + (lo.double() - hi.double()) * self._span(0)
            done = lo | hi
        if not self.open[1]:
            lo, hi = (y < p["vert"][0]) & ~done, (y > p["vert"][1]) & ~done
            y = y + (lo.double() - hi.double()) * self._span(1)
        left, right, up, down = p["refl"]
        for lim, low in ((left, True), (right, False)):
            out = x < lim if low else x > lim
            x, self.vx = torch.where(out, torch.full_like(x, lim), x), torch.where(out, -self.vx, self.vx)
        for lim, low in ((up, True), (down, False)):
            out = y < lim if low else y > lim
            y, self.vy = torch.where(out, torch.full_like(y, lim), y), torch.where(out, -self.vy, self.vy)
        self.x, self.y = x, y
        self._next_dt()
