"""The framework's work as its users have it done, case by case.

A user of the engine keeps a lattice (or a batch of lattices), advances it a
number of time steps, and reads what a log line and a field file hold: the
Globals of the last step and the velocity and pressure (density) fields.
One pass here is one such stretch: `iterate(steps)` with the Globals on the
last step, then the Globals and both fields.  The state stays on the GPU
and goes on from pass to pass, as in a run.

Inputs of a seed: the obstacles (discs, spheres) and the viscosity, the
inlet or initial velocity, the force or the lid's velocity.
"""
import math
import random

import numpy as np
import torch

import tclb_amd
from tclb_amd import cases as C

STORED = {"f64": 8, "f32": 4, "f32s": 4, "f16s": 2, "bf16s": 2}
Q = {"d2q9_SRT": 9, "d2q9_SRT_drag": 9, "d2q9": 9, "d2q9_drag": 9, "d3q19": 19, "d3q19_lid": 19, "d3q27": 27,
     "d3q27_cumulant": 27}
# additions, multiplications and divisions of one node's collision
FLOPS = {"d2q9_SRT": 130, "d2q9_SRT_drag": 130, "d2q9": 150, "d2q9_drag": 150, "d3q19": 430, "d3q19_lid": 430,
         "d3q27": 480, "d3q27_cumulant": 900}


def _case(name, model, storage, nx, ny, nz, steps, boxes=0, sr=False):
    c = {"model": model, "storage": storage, "nx": nx, "ny": ny, "nz": nz, "steps": steps, "boxes": boxes, "sr": sr}
    return dict({"name": name}, **c) if name else c


def listed():
    return [
        # the smallest call: a coarse 2D channel with a disc, logged every 10
        # steps, as a case file with a small <Log Iterations> does
        _case("channel_128x32_f64", "d2q9_SRT", "f64", 128, 32, 1, 10),
        # the cylinder channel with drag and lift, logged every 1000 steps
        _case("cylinder_1024x128_f64", "d2q9_SRT_drag", "f64", 1024, 128, 1, 1000),
        # a 2D channel of uneven size in the 16-bit format (MRT collision)
        _case("channel_1501x333_f16s", "d2q9", "f16s", 1501, 333, 1, 1000),
        # a large 2D domain in full precision: its snapshots fill several caches
        _case("channel_4096x2048_f64", "d2q9_SRT", "f64", 4096, 2048, 1, 800),
        # a parameter sweep: many cylinder channels of uneven sizes in one batch
        _case("sweep_24_f16s", "d2q9_drag", "f16s", 1024, 256, 1, 700, boxes=24),
        # a small porous box, as the small requests of a solve server are
        _case("porous_61x48x57_f64", "d3q19", "f64", 61, 48, 57, 200),
        # the porous channel, double precision: the headline workload
        _case("porous_256_f64", "d3q19", "f64", 256, 256, 256, 300),
        # the same in the 16-bit storage format
        _case("porous_256_f16s", "d3q19", "f16s", 256, 256, 256, 800),
        # a batch of porous boxes of uneven sizes: the requests a solve
        # server advances together
        _case("requests_6_f16s", "d3q19", "f16s", 256, 256, 256, 400, boxes=6),
        # a lid-driven cavity, shifted single precision
        _case("cavity_192x176x160_f32s", "d3q19_lid", "f32s", 192, 176, 160, 500),
        # the 27-velocity models: channels with obstacles, one of uneven size
        _case("cumulant_160x128x96_f16s", "d3q27_cumulant", "f16s", 160, 128, 96, 500),
        _case("d3q27_129x97x113_f32", "d3q27", "f32", 129, 97, 113, 400),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    """Another run of the same kinds: any of the models and storage formats,
    sizes spread over the range (its logarithm), with a number of steps that
    keeps the pass below the largest listed one."""
    kind = rng.choice(["2d", "2d", "3d", "3d", "27", "batch2d", "batch3d"])
    st = rng.choice(["f64", "f64", "f32", "f32s", "f16s", "f16s", "bf16s"])
    if kind == "2d":
        model = rng.choice(["d2q9_SRT", "d2q9_SRT_drag", "d2q9", "d2q9_drag"])
        nx, ny = _log_uniform(rng, 100, 4000), _log_uniform(rng, 32, 2000)
        steps = _log_uniform(rng, 10, max(12, min(2000, int(2e9 / (nx * ny)))))
        return _case("", model, st, nx, ny, 1, steps, sr=st in ("f16s", "bf16s") and rng.random() < 0.4)
    if kind == "3d":
        model = rng.choice(["d3q19", "d3q19", "d3q19_lid"])
        nx, ny, nz = (_log_uniform(rng, 32, 256) for _ in range(3))
        steps = _log_uniform(rng, 10, max(12, min(500, int(2e9 / (nx * ny * nz)))))
        return _case("", model, st, nx, ny, nz, steps, sr=st in ("f16s", "bf16s") and rng.random() < 0.4)
    if kind == "27":
        model = rng.choice(["d3q27", "d3q27_cumulant"])
        nx, ny, nz = (_log_uniform(rng, 32, 160) for _ in range(3))
        steps = _log_uniform(rng, 10, max(12, min(200, int(4e8 / (nx * ny * nz)))))
        return _case("", model, st, nx, ny, nz, steps)
    if kind == "batch2d":
        return _case("", "d2q9_drag", st, rng.randint(200, 1024), rng.randint(64, 256), 1, _log_uniform(rng, 20, 300),
                     boxes=rng.randint(4, 24))
    return _case("", "d3q19", st, *(_log_uniform(rng, 60, 200) for _ in range(3)), _log_uniform(rng, 20, 150),
                 boxes=rng.randint(2, 6))


# ---------------------------------------------------------------- inputs ---
def _discs(rng, nx, ny):
    """Discs in the channel: one for each square of its height, at most 40."""
    solid = np.zeros((ny, nx), dtype=bool)
    x, y = np.arange(nx) + 0.5, np.arange(ny) + 0.5
    for _ in range(min(40, max(1, nx // (4 * ny)))):
        r = rng.uniform(0.06, 0.13) * min(ny, nx / 2)
        cx, cy = rng.uniform(0.2, 0.8) * nx, rng.uniform(0.35, 0.65) * ny
        xs = slice(max(0, int(cx - r) - 1), min(nx, int(cx + r) + 2))
        ys = slice(max(0, int(cy - r) - 1), min(ny, int(cy + r) + 2))
        solid[ys, xs] |= (x[xs] - cx) ** 2 + (y[ys, None] - cy) ** 2 < r * r
    return solid


def _spheres(rng, nx, ny, nz):
    """Spheres of radius 4 to 12 (less in a small box), about 10% solid."""
    solid = np.zeros((nz, ny, nx), dtype=bool)
    side = min(nx, ny, nz)
    left = 0.1 * nx * ny * nz
    while left > 0:
        r = rng.uniform(min(4.0, side / 12), min(12.0, side / 6))
        cx, cy, cz = rng.uniform(0, nx), rng.uniform(r, ny - r), rng.uniform(0, nz)
        xs, ys, zs = (np.arange(int(c - r) - 1, int(c + r) + 2) for c in (cx, cy, cz))
        ys = ys[(ys >= 0) & (ys < ny)]
        ball = ((zs + 0.5 - cz) ** 2)[:, None, None] + ((ys + 0.5 - cy) ** 2)[:, None] + (xs + 0.5 - cx) ** 2 < r * r
        at = np.ix_(zs % nz, ys, xs % nx)
        solid[at] |= ball
        left -= 4.19 * r ** 3
    return solid


def _shapes(case):
    """The lattice sizes of the pass: the case's own, or those of its boxes
    (the same for every seed)."""
    if not case["boxes"]:
        return [(case["nx"], case["ny"], case["nz"])]
    rng = np.random.default_rng([case["nx"], case["ny"], case["nz"], case["boxes"]])
    out = []
    for _ in range(case["boxes"]):
        if case["nz"] == 1:   # sides uniform up to the case's, in steps of 16
            out.append((128 + 16 * int(rng.integers(0, max(1, (case["nx"] - 128) // 16 + 1))),
                        64 + 16 * int(rng.integers(0, max(1, (case["ny"] - 64) // 16 + 1))), 1))
        else:                 # sides log-uniform from 48 up to the case's
            out.append(tuple(int(round(math.exp(rng.uniform(math.log(48), math.log(case[k]))))) for k in ("nx", "ny", "nz")))
    return out


def _inputs(case, shape, seed, k):
    """What a run is given: the solid nodes and the physical parameters."""
    nx, ny, nz = shape
    rng = np.random.default_rng([seed, k])
    p = {"u0": rng.uniform(0.01, 0.03), "nu": rng.uniform(0.03, 0.08), "force": rng.uniform(1e-6, 1e-5)}
    if Q[case["model"]] == 9:
        bands = min(ny - 2, 500)   # rows of one inlet velocity each: the zones
        band = (np.arange(1, ny - 1) - 1) * bands // (ny - 2)
        row = np.array([np.flatnonzero(band == b)[0] + 1.0 for b in range(bands)])
        p["band"], p["inlet"] = band, p["u0"] * 6 * (row - 0.5) * (ny - 1.5 - row) / (ny - 2) ** 2
        p["solid"] = _discs(rng, nx, ny)
        p["wall"] = np.zeros((ny, nx), dtype=bool)
        p["wall"][[0, -1]] = True
    elif case["model"] == "d3q19_lid":
        p["wall"] = np.zeros((nz, ny, nx), dtype=bool)
        p["wall"][:, :, [0, -1]] = p["wall"][:, 0] = p["wall"][[0, -1]] = True
        p["lid"] = np.zeros((nz, ny, nx), dtype=bool)
        p["lid"][:, -1] = True
        p["wall"] &= ~p["lid"]
        p["solid"] = _spheres(rng, nx, ny, nz) & ~p["wall"] & ~p["lid"]
    else:
        p["solid"] = _spheres(rng, nx, ny, nz)
        p["wall"] = np.zeros((nz, ny, nx), dtype=bool)
        p["wall"][:, [0, -1]] = True
    return p


def _as_case(case, shape, p):
    """The run as the framework's Case: NodeType map, settings, zonal settings."""
    model = case["model"]
    m = tclb_amd.Model(model)
    nx, ny, nz = shape
    if Q[model] == 9:
        srt = model.startswith("d2q9_SRT")
        vx = "Velocity_x" if srt else "VelocityX"
        fluid = m.flag("BGK" if srt else "MRT")
        zone = m.group("SETTINGZONE")[1]
        flags = np.full((1, ny, nx), fluid, dtype=np.uint16)
        flags[0, 1:-1, 0] = m.flag("WVelocity") | fluid | ((1 + p["band"]) << zone)
        flags[0, 1:-1, -1] = m.flag("EPressure") | fluid
        flags[0][p["solid"]] = m.flag("Solid")
        flags[0][p["wall"]] = m.flag("Wall")
        settings = [("nu", p["nu"]), ("Density", 1.0)] if srt else [("Viscosity", p["nu"])]
        zonal = [(vx, 0, p["u0"])] + [(vx, 1 + b, float(v)) for b, v in enumerate(p["inlet"])]
        return C.Case("channel", model, nx, ny, 1, flags, settings=settings, zonal=zonal)
    flags = np.full((nz, ny, nx), m.flag("MRT"), dtype=np.uint16)
    flags[p["solid"]] = m.flag("Solid" if Q[model] == 19 else "Wall")
    flags[p["wall"]] = m.flag("Wall")
    settings, zonal = [("nu", p["nu"]), ("ForceX", p["force"])], []
    if model == "d3q19_lid":
        flags[p["lid"]] = m.flag("MovingWall")
        settings = [("nu", p["nu"]), ("MovingWallVelocityX", p["u0"])]
    elif Q[model] == 19:
        settings.append(("InletVelocity", p["u0"]))   # the initial velocity
    else:
        zonal.append(("Velocity", -1, p["u0"]))       # the initial velocity
    return C.Case("porous", model, nx, ny, nz, flags, settings=settings, zonal=zonal)


def prepare(case, seed):
    shapes = _shapes(case)
    runs = [_as_case(case, s, _inputs(case, s, seed, k)) for k, s in enumerate(shapes)]
    scalar = "Rho" if Q[case["model"]] == 9 else "P"
    if not case["boxes"]:
        lat = runs[0].build(case["storage"])
        if case["sr"]:
            lat.set_stochastic_rounding(True, seed=1)
        return {"lattice": lat, "steps": case["steps"], "scalar": scalar}
    probe = tclb_amd.Batch(case["model"], case["storage"], 1 << 20)
    room = sum(probe.case_bytes(*s) for s in shapes) + (16 << 20)
    probe.close()
    batch = tclb_amd.Batch(case["model"], case["storage"], capacity_bytes=room)
    return {"batch": batch, "ids": [batch.add(r) for r in runs], "steps": case["steps"]}


def run(state):
    if "lattice" in state:
        lat = state["lattice"]
        lat.iterate(state["steps"])
        return {"globals": lat.globals, "u": lat.quantity("U"), "rho": lat.quantity(state["scalar"])}
    b = state["batch"]
    b.iterate(state["steps"])
    return {"globals": np.stack([b.globals(i) for i in state["ids"]]), "u": [b.quantity(i, "U") for i in state["ids"]]}


def work(case):
    """What the pass cannot do without: the state and the NodeTypes read
    once, the state and the fields written once; every step's collisions."""
    q, s = Q[case["model"]], STORED[case["storage"]]
    n = sum(a * b * c for a, b, c in _shapes(case))
    fields = 3 if case["boxes"] else 4
    return {"bytes": n * (2 * q * s + 2 + 8 * fields), "flops": n * case["steps"] * FLOPS[case["model"]]}


# ------------------------------------------- the same in 64 bits, in torch ---
_E9 = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 0, 0), (0, -1, 0), (1, 1, 0), (-1, 1, 0), (-1, -1, 0), (1, -1, 0)]
_E19 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, 1, 0), (1, -1, 0),
        (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1), (0, -1, -1)]
_E27 = [(i % 3 - 1, i // 3 % 3 - 1, i // 9 - 1) for i in range(27)]


def _weight(e, q):
    k = sum(abs(v) for v in e)
    return {9: (4 / 9, 1 / 9, 1 / 36), 19: (1 / 3, 1 / 18, 1 / 36), 27: (8 / 27, 2 / 27, 1 / 54, 1 / 216)}[q][k]


class _Exact:
    """One lattice in 64 bits: f[q, z, y, x], plain torch."""

    def __init__(self, model, shape, p):
        self.model, self.p, self.q = model, p, Q[model]
        nx, ny, nz = shape
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        kw = {"dtype": torch.float64, "device": dev}
        self.es = {9: _E9, 19: _E19, 27: _E27}[self.q]
        self.opp = torch.tensor([self.es.index(tuple(-v for v in e)) for e in self.es], device=dev)
        self.w = torch.tensor([_weight(e, self.q) for e in self.es], **kw)
        self.e = torch.tensor(self.es, **kw)
        as_mask = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).reshape(nz, ny, nx)  # noqa: E731
        self.solid, self.wall = as_mask(p["solid"] & ~p["wall"]), as_mask(p["wall"])
        self.lid = as_mask(p["lid"]) if "lid" in p else None
        self.bounce = self.solid | self.wall if self.lid is None else self.solid | self.wall | self.lid
        self.fluid = ~self.bounce
        u0 = 0.0 if model == "d3q19_lid" else p["u0"]
        u = torch.full((nz, ny, nx), u0, **kw)
        if self.q == 9:
            inlet = torch.tensor(p["inlet"], **kw)[torch.from_numpy(np.asarray(p["band"])).to(dev)]
            self.inlet = inlet
            rows = self.fluid[0, 1:-1, 0]
            u[0, 1:-1, 0] = torch.where(rows, inlet, u[0, 1:-1, 0])
        if model in ("d2q9", "d2q9_drag", "d3q27_cumulant"):   # their walls start at rest
            u[self.wall | (self.solid if self.q == 27 else False)] = 0.0
        self.force = p["force"] if self.q > 9 and model != "d3q19_lid" else 0.0
        self.tau = 3 * p["nu"] + 0.5
        if self.q == 19:
            self.basis19(kw)
        self.f = self.feq(torch.ones_like(u), u, torch.zeros_like(u), torch.zeros_like(u))

    def basis19(self, kw):
        """The orthogonal moments of the 19 velocities: polynomials of the
        velocity, and their relaxation rates at omega = 1/tau."""
        x, y, z = (self.e[:, i] for i in range(3))
        c = x * x + y * y + z * z
        m = [torch.ones_like(x), 19 * c - 30, (21 * c * c - 53 * c + 24) / 2, x, (5 * c - 9) * x, y, (5 * c - 9) * y, z,
             (5 * c - 9) * z, 3 * x * x - c, (3 * c - 5) * (3 * x * x - c), y * y - z * z, (3 * c - 5) * (y * y - z * z),
             x * y, y * z, x * z, (y * y - z * z) * x, (z * z - x * x) * y, (x * x - y * y) * z]
        self.m = torch.stack(m)
        self.minv = (self.m / (self.m * self.m).sum(1, keepdim=True)).T.contiguous()
        om = 1 / self.tau
        g1, g2 = 1 - om, 1 - 8 * (2 - om) / (8 - om)
        self.gamma = torch.tensor([0, g1, g1, 0, g2, 0, g2, 0, g2] + [g1] * 7 + [g2] * 3, **kw)

    def feq(self, rho, jx, jy, jz):
        """Equilibrium of density rho and momentum j, second order in j (19
        velocities: of the model's equilibrium moments)."""
        if self.q == 19:
            zero = torch.zeros_like(rho)
            m = self.req19([rho, zero, zero, jx, zero, jy, zero, jz])
            return (self.minv @ m.reshape(19, -1)).reshape(m.shape)
        out = []
        j2 = (jx * jx + jy * jy + jz * jz) / rho
        for e, w in zip(self.es, self.w):
            ej = e[0] * jx + e[1] * jy + e[2] * jz
            out.append(w * (rho + 3 * ej + 4.5 * ej * ej / rho - 1.5 * j2))
        return torch.stack(out)

    def pulled(self):
        return torch.stack([torch.roll(self.f[i], (e[2], e[1], e[0]), (0, 1, 2)) if any(e) else self.f[i]
                            for i, e in enumerate(self.es)])

    def momentum(self, f):
        return [sum(e[a] * f[i] for i, e in enumerate(self.es) if e[a]) for a in range(3)] if self.q > 9 else \
            [sum(e[a] * f[i] for i, e in enumerate(self.es) if e[a]) for a in range(2)] + [torch.zeros_like(f[0])]

    def zou_he(self, f):
        """Velocity inlet at x = 0 and pressure outlet (density 1) at x = nx - 1."""
        a = [v[0, 1:-1, 0] for v in f]
        ok = self.fluid[0, 1:-1, 0]
        rho = (a[0] + a[2] + a[4] + 2 * (a[3] + a[7] + a[6])) / (1 - self.inlet)
        ru, t = rho * self.inlet, (a[2] - a[4]) / 2
        for i, v in ((1, a[3] + 2 / 3 * ru), (5, a[7] + ru / 6 - t), (8, a[6] + ru / 6 + t)):
            f[i, 0, 1:-1, 0] = torch.where(ok, v, a[i])
        a = [v[0, 1:-1, -1] for v in f]
        ok = self.fluid[0, 1:-1, -1]
        ru, t = a[0] + a[2] + a[4] + 2 * (a[1] + a[5] + a[8]) - 1, (a[2] - a[4]) / 2
        for i, v in ((3, a[1] - 2 / 3 * ru), (7, a[5] - ru / 6 + t), (6, a[8] - ru / 6 - t)):
            f[i, 0, 1:-1, -1] = torch.where(ok, v, a[i])

    def step(self, last):
        """One time step; the Globals of the model on the last one."""
        f = self.pulled()
        g = None
        if last and self.q == 9 and self.model.endswith("_drag"):
            j = self.momentum(f)
            g = [2 * j[a][self.solid].sum() for a in (0, 1)]
        back = f[self.opp]
        if self.lid is not None:
            ladd = torch.stack([6 * w * e[0] * self.p["u0"] * torch.ones_like(f[0]) for e, w in zip(self.es, self.w)])
            back = torch.where(self.lid, back + ladd, back)
        fb = torch.where(self.bounce, back, f)
        if self.q == 9:
            self.zou_he(fb)
        rho = fb.sum(0)
        j = self.momentum(fb)
        if self.q == 9 and self.model.startswith("d2q9_SRT"):
            out = fb + (self.feq(rho, *j) - fb) / self.tau
        elif self.q == 9:
            # second moments relax with tau, the third and fourth orders fully
            eq = self.feq(rho, *j)
            n = fb - eq
            s2 = 1 - 1 / self.tau
            pi = [sum(e[a] * e[b] * n[i] for i, e in enumerate(self.es) if e[a] * e[b]) for a, b in ((0, 0), (1, 1), (0, 1))]
            out = eq + s2 * torch.stack([w * 4.5 * ((e[0] * e[0] - 1 / 3) * pi[0] + (e[1] * e[1] - 1 / 3) * pi[1] +
                                                    2 * e[0] * e[1] * pi[2]) for e, w in zip(self.es, self.w)])
        elif self.q == 19:
            m = (self.m @ fb.reshape(19, -1)).reshape(fb.shape)
            neq = self.gamma[:, None, None, None] * (m - self.req19(m))
            del m
            j[0] = j[0] + self.force * rho
            m = neq
            m[0], m[3], m[5], m[7] = rho, j[0], j[1], j[2]
            k = [i for i in range(19) if i not in (0, 3, 5, 7)]
            m[k] += self.req19(m)[k]
            out = (self.minv @ m.reshape(19, -1)).reshape(fb.shape)
            if last:
                g = self.globals19(rho, j, f, fb)
        elif self.model == "d3q27":
            eq = self.feq(rho, *j)
            jf = [j[0] + self.force, j[1], j[2]]
            out = self.feq(rho, *jf) + (1 - 1 / self.tau) * (fb - eq)
            if last:
                at = self.fluid
                g = [((jf[0] + self.force / 2) / rho)[at].sum(), (j[1] / rho)[at].sum(), (j[2] / rho)[at].sum()]
                solid = self.bounce
                g += [2 * j[a][solid].sum() for a in range(3)]
        else:
            out = self.cumulants(fb, rho)
            if last:
                at = self.fluid
                jh = [j[0] + self.force / 2, j[1], j[2]]
                zero = torch.zeros((), dtype=f.dtype, device=f.device)
                g = [rho[at].sum(), (jh[0] / rho)[at].sum(), zero, zero, zero, rho[at].sum()] + [v[at].sum() for v in jh]
        self.f = torch.where(self.bounce, fb, out)
        return g

    def req19(self, m):
        rho, jx, jy, jz = m[0], m[3], m[5], m[7]
        xx, yy, zz = jx * jx / rho, jy * jy / rho, jz * jz / rho
        j2 = xx + yy + zz
        z = torch.zeros_like(rho)
        a, b = 2 * xx - yy - zz, yy - zz
        return torch.stack([rho, 19 * j2 - 11 * rho, 3 * rho - 2 * j2, jx, -2 / 3 * jx, jy, -2 / 3 * jy, jz, -2 / 3 * jz, a, -a, b,
                            -b, jx * jy / rho, jy * jz / rho, jx * jz / rho, z, z, z])

    def globals19(self, rho, j, f, fb):
        # sums over the collided nodes of rho/19, J/10 and their quotients, as
        # the model defines its Globals
        at = self.fluid
        r, jj = rho[at] / 19, [v[at] / 10 for v in j]
        u = [v / r for v in jj]
        zero = torch.zeros((), dtype=f.dtype, device=f.device)
        g = [zero] * 16 + [v.sum() for v in u] + [v.sum() for v in jj] + [r.sum(), at.sum().double()]
        if self.lid is not None:
            total = torch.zeros_like(f[:3])
            nx, ny = f.shape[3], f.shape[2]
            for i, e in enumerate(self.es):
                if any(e):
                    src = torch.roll(self.fluid, (e[2], e[1], e[0]), (0, 1, 2)) & self.lid
                    mom = (f[i] + fb[self.opp[i]]) * src
                    for a in range(3):
                        if e[a]:
                            total[a] += e[a] * mom
            x = torch.arange(nx, device=f.device).double() - 0.5 * (nx - 1)
            y = (torch.arange(ny, device=f.device).double() - 0.5 * (ny - 1))[:, None]
            g += [total[0].sum(), total[1].sum(), total[2].sum(), (x * total[1] - y * total[0]).sum()]
        return g + [zero, torch.sqrt(u[0] ** 2 + u[1] ** 2 + u[2] ** 2).max()]

    def cumulants(self, f, rho):
        """The cumulant collision: moments, cumulants of f/rho by the rule for
        derivatives of a logarithm, relaxation, and back."""
        powers = sorted(((a, b, c) for a in range(3) for b in range(3) for c in range(3)), key=sum)
        m, c = {}, {}
        ex, ey, ez = ([e[a] for e in self.es] for a in range(3))
        for n in powers:
            m[n] = sum((ex[i] ** n[0] * ey[i] ** n[1] * ez[i] ** n[2]) * f[i] for i in range(27)
                       if ex[i] ** n[0] * ey[i] ** n[1] * ez[i] ** n[2])

        def rest(n, c, m):
            ax = [a for a in range(3) if n[a]][0]
            d = tuple(1 if a == ax else 0 for a in range(3))
            low = tuple(n[a] - d[a] for a in range(3))
            s = 0.0
            for k in powers:
                if k != low and all(k[a] <= low[a] for a in range(3)):
                    b = math.prod(math.comb(low[a], k[a]) for a in range(3))
                    s = s + b * c[tuple(k[a] + d[a] for a in range(3))] * m[tuple(low[a] - k[a] for a in range(3))]
            return s

        for n in powers[1:]:
            c[n] = (m[n] - rest(n, c, m)) / rho
        xx, yy, zz = (2, 0, 0), (0, 2, 0), (0, 0, 2)
        x, y, z = (1, 0, 0), (0, 1, 0), (0, 0, 1)
        w0 = 1 / self.tau
        u = [c[x] + self.force / (2 * rho), c[y], c[z]]
        dx = -w0 / 2 * (2 * c[xx] - c[yy] - c[zz]) - 0.5 * (c[xx] + c[yy] + c[zz] - 1)
        dy = dx + 1.5 * w0 * (c[xx] - c[yy])
        dz = dx + 1.5 * w0 * (c[xx] - c[zz])
        k = 3 * (1 - w0 / 2)
        a = (1 - w0) * (c[xx] - c[yy]) - k * (u[0] ** 2 * dx - u[1] ** 2 * dy)
        b = (1 - w0) * (c[xx] - c[zz]) - k * (u[0] ** 2 * dx - u[2] ** 2 * dz)
        t = 1 - 1.5 * (u[0] ** 2 * dx + u[1] ** 2 * dy + u[2] ** 2 * dz)
        c[xx], c[yy], c[zz] = (a + b + t) / 3, (t - 2 * a + b) / 3, (t - 2 * b + a) / 3
        c[x] = c[x] + self.force
        zero = torch.zeros_like(rho)
        for n in powers:
            if sum(n) == 2 and max(n) == 1:
                c[n] = c[n] * (1 - w0)
            if sum(n) >= 3:
                c[n] = zero
        new = {(0, 0, 0): rho}
        for n in powers[1:]:
            new[n] = c[n] * rho + rest(n, c, new)
        one = {0: ((0, 1.0), (2, -1.0)), 1: ((1, 0.5), (2, 0.5)), -1: ((1, -0.5), (2, 0.5))}
        return torch.stack([sum(a[1] * b[1] * d[1] * new[(a[0], b[0], d[0])] for a in one[e[0]] for b in one[e[1]] for d in one[e[2]])
                            for e in self.es])

    def fields(self):
        """Velocity and density (pressure) of the streamed populations."""
        f = self.pulled()
        rho = f.sum(0)
        if self.model == "d3q27_cumulant":
            f = torch.where(self.bounce, f[self.opp], f)
        j = self.momentum(f)
        if self.q == 27:
            j[0] = j[0] + self.force / 2
        u = torch.stack([v / rho for v in j], -1)
        still = self.bounce if self.model == "d3q27_cumulant" else self.wall if self.q == 19 else None
        if still is not None:
            u[still] = 0.0
        if self.lid is not None:
            u[self.lid] = torch.tensor([self.p["u0"], 0.0, 0.0], dtype=u.dtype, device=u.device)
        return u, (rho if self.q == 9 else (rho - 1) / 3)


def _exact_one(case, shape, p):
    L = _Exact(case["model"], shape, p)
    for i in range(case["steps"]):
        g = L.step(i == case["steps"] - 1)
    zero = torch.zeros((), dtype=torch.float64, device=L.f.device)
    if case["model"] in ("d2q9_SRT", "d2q9"):
        g = [zero] * (1 if case["model"] == "d2q9_SRT" else 4)
    elif case["model"] == "d2q9_SRT_drag":
        g = g + [zero]
    elif case["model"] == "d2q9_drag":
        g = [zero] * 3 + g + [zero]
    elif L.q == 27:
        g = g + [zero]
    u, rho = L.fields()
    return torch.stack([v.reshape(()) for v in g]).cpu().numpy(), u.cpu().numpy(), rho.cpu().numpy()


def exact(case, seed):
    shapes = _shapes(case)
    nodes = sum(a * b * c for a, b, c in shapes)
    # about 20 seconds: a step's launches, and its passes over memory
    cost = 120 if Q[case["model"]] != 27 else 60 if case["model"] == "d3q27" else 900
    seconds = case["steps"] * (len(shapes) * cost * 8e-6 + nodes * Q[case["model"]] * 8 * (40 if cost == 900 else 12) / 3e12)
    if seconds > 18:
        return None
    got = [_exact_one(case, s, _inputs(case, s, seed, k)) for k, s in enumerate(shapes)]
    if case["boxes"]:
        return {"globals": np.stack([g for g, _, _ in got]), "u": [u for _, u, _ in got]}
    g, u, rho = got[0]
    return {"globals": g, "u": u, "rho": rho}
