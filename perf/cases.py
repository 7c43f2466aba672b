"""The work whose time is watched: peridynamic simulations of one body on one GPU, called as a
user's program calls them.

Paths (`"path"` of a case):
  vv     `steps` Velocity Verlet steps and the export of displacement, velocity and damage, as
         a job does between two exports;
  dr     `steps` adaptive dynamic relaxation steps under a constant load, and the export;
  force  one force density at positions that the caller supplies, for programs that drive
         their own time loop;
  nk     one Newton-Krylov load step from the undeformed body to a tight residual;
  setup  everything between a described body and its first step: bond search, device layout,
         stable time step, force density at t = 0.

Bodies are lattices of `nx` x `ny` x `nz` points with a jitter of 0.05 spacings, clamped at one
end, moving with smooth velocities far below the critical stretch, so that a case may run any
number of passes without the body coming apart.  `horizon` is in spacings; `sets` > 1 splits
the body into layers with parameter sets of their own; `crack` opens a precrack; `precision`,
`material` (BB, OSB, CPD), `model` and `zem` (CPD), `correction` (the energy surface
correction) and `permit` (bonds may fail) are the options of the framework.

Run from anywhere: the package is found next to this folder."""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "peridynamics.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DX = 1e-3
E_MOD, NU, RHO = 70e9, 0.25, 2700.0
FIELDS = ("displacement", "velocity", "damage")  # what a run exports


def _case(name, path, material, nx, ny, nz, steps=1, precision="fp64", horizon=3.015, sets=1,
          crack=False, model="svk", zem="silling", correction=False, permit=True, drive=False):
    c = {"path": path, "material": material, "nx": nx, "ny": ny, "nz": nz, "steps": steps,
         "precision": precision, "horizon": horizon, "sets": sets, "crack": crack, "model": model,
         "zem": zem, "correction": correction, "permit": permit, "drive": drive}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a thousand points: a coupled program asks for one force density per exchange
        _case("force osb 1k", "force", "OSB", 10, 10, 10),
        # a parameter study's specimen: many steps of a small plate, latency counts
        _case("vv bb 6k", "vv", "BB", 40, 40, 4, steps=200),
        # the pre-cracked plate of the fracture studies, mixed precision
        _case("vv bb mixed plate 1M", "vv", "BB", 500, 500, 4, steps=50, precision="mixed",
              crack=True),
        # the throughput workload: the largest body, in the reference's precision
        _case("vv bb 2M", "vv", "BB", 200, 200, 50, steps=100),
        # a wide horizon on an odd block: long neighbour tables, two parameter sets
        _case("vv bb wide two sets 121k", "vv", "BB", 61, 53, 37, steps=50, horizon=5.015, sets=2),
        # the torsion bar, state-based, driven through a position-dependent condition
        _case("vv osb bar 512k", "vv", "OSB", 160, 80, 40, steps=50, drive=True, permit=False),
        # a mid-sized ragged block, state-based, mixed precision
        _case("vv osb mixed 159k", "vv", "OSB", 97, 53, 31, steps=100, precision="mixed"),
        # the torsion bar, correspondence material
        _case("vv cpd bar 512k", "vv", "CPD", 160, 80, 40, steps=50, permit=False),
        # a smaller correspondence body, the other stabilisation and a hyperelastic model
        _case("vv cpd zemwan 54k", "vv", "CPD", 60, 30, 30, steps=80, model="neohooke", zem="wan"),
        # quasi-static relaxation of a mid-sized plate under a dead load
        _case("dr bb 100k", "dr", "BB", 100, 100, 10, steps=50, permit=False),
        # an implicit load step of a small block
        _case("nk bb 14k", "nk", "BB", 40, 36, 10, permit=False),
        # every job's start: building the bonds of a half-million-point body
        _case("setup bb 576k", "setup", "BB", 120, 120, 40),
    ]


def draw(rng):
    path = rng.choices(("vv", "force", "dr", "nk", "setup"), (56, 12, 10, 7, 15))[0]
    material = "BB" if path == "nk" else rng.choices(("BB", "OSB", "CPD"), (45, 30, 25))[0]
    top = {"vv": 1e6, "force": 3e5, "dr": 4e5, "nk": 1.6e4, "setup": 6e5}[path]
    if material == "CPD":
        top = min(top, 4e5)
    n = math.exp(rng.uniform(math.log(1e3), math.log(top)))
    shape = rng.choice(("block", "plate", "bar"))
    if shape == "plate":
        nz = rng.randint(4, 8)
        nx = max(8, round(math.sqrt(n / nz) * rng.uniform(0.8, 1.25)))
        ny = max(8, round(n / nz / nx))
    elif shape == "bar":
        nz = max(5, round((n / rng.uniform(4, 9)) ** (1 / 3)))
        ny = max(5, round(nz * rng.uniform(1.0, 2.0)))
        nx = max(8, round(n / nz / ny))
    else:
        nx = max(8, round(n ** (1 / 3) * rng.uniform(0.8, 1.25)))
        ny = max(8, round(n ** (1 / 3) * rng.uniform(0.8, 1.25)))
        nz = max(5, round(n / nx / ny))
    n = nx * ny * nz
    # a step of a correspondence body costs about four bond-based ones
    per = {"BB": 1, "OSB": 2, "CPD": 4}[material]
    steps = min(200, max(10, int(3e7 / (n * per)))) if path in ("vv", "dr") else 1
    if path == "dr":
        steps = min(steps, 50 if material == "BB" else 15)
    precision = "mixed" if path in ("vv", "force") and rng.random() < 0.25 else "fp64"
    horizon = 3.015
    if path != "nk" and n < 2e5 and rng.random() < 0.25:
        horizon = rng.choice((4.015, 5.015))
    sets = 2 if path in ("vv", "force", "setup") and precision == "fp64" and rng.random() < 0.25 else 1
    correction = path in ("vv", "force") and sets == 1 and material in ("BB", "OSB") and rng.random() < 0.15
    crack = material == "BB" and path in ("vv", "setup") and rng.random() < 0.3
    return _case(None, path, material, nx, ny, nz, steps, precision, horizon, sets, crack,
                 rng.choice(("svk", "neohooke")), rng.choice(("silling", "silling", "wan")),
                 correction, path not in ("dr", "nk") and rng.random() < 0.7,
                 path == "vv" and rng.random() < 0.2)


# ------------------------------------------------------------------------------ inputs
def _inputs(case, seed):
    """The body and its motion as plain arrays: what the framework gets and what exact() uses."""
    rng = np.random.default_rng([seed, case["nx"], case["ny"], case["nz"]])
    shape = (case["nx"], case["ny"], case["nz"])
    n = shape[0] * shape[1] * shape[2]
    g = [(np.arange(m) - (m - 1) / 2) * DX for m in shape]
    pos = np.empty((3, shape[2], shape[1], shape[0]))  # x fastest
    pos[0], pos[1], pos[2] = g[0], g[1][:, None], g[2][:, None, None]
    pos = pos.reshape(3, n)
    pos += rng.uniform(-0.05 * DX, 0.05 * DX, (3, n))
    length = [m * DX for m in shape]
    x0 = -length[0] / 2
    # two smooth modes per component, zero at the clamped end: some 10 m/s, strains of about 1e-3
    amp = rng.uniform(2.0, 5.0, (3, 2)) * rng.choice((-1.0, 1.0), (3, 2))
    wave = rng.integers(1, 3, (3, 2, 3)) * (math.pi / np.array(length))
    phase = rng.uniform(0, math.pi, (3, 2))
    s = {"shape": shape, "n": n, "pos": pos, "volume": np.full(n, DX ** 3), "amp": amp,
         "wave": wave, "phase": phase, "x0": x0, "lx": length[0],
         "clamp": pos[0] < x0 + 2.5 * DX, "end": pos[0] > -x0 - 2.5 * DX,
         "E": [E_MOD * rng.uniform(0.9, 1.1), E_MOD * rng.uniform(0.4, 0.6)],
         "rho": [RHO, RHO * rng.uniform(1.1, 1.3)],
         "delta": case["horizon"] * DX, "omega": rng.uniform(100.0, 300.0), "freq": rng.uniform(2e4, 6e4),
         "load": rng.uniform(2e9, 6e9) * rng.choice((-1.0, 1.0)),
         "pull": rng.uniform(0.5, 1.0) * 2e-3 * DX * shape[1]}
    s["layer"] = (pos[1] > 0).astype(np.int64) if case["sets"] > 1 else np.zeros(n, np.int64)
    if case["crack"]:
        on = pos[0] <= x0 + 0.25 * length[0]
        near = 2 * s["delta"]
        s["crack_a"] = on & (pos[1] >= 0) & (pos[1] <= near)
        s["crack_b"] = on & (pos[1] < 0) & (pos[1] >= -near)
    return s


def _velocity(s, d, p):
    """Initial velocity component d at positions p (3 x m)."""
    ramp = (p[0] - s["x0"]) / s["lx"]
    v = 0.0
    for k in range(2):
        w = s["wave"][d, k]
        v = v + s["amp"][d, k] * np.sin(w[0] * p[0] + s["phase"][d, k]) * np.cos(w[1] * p[1]) * np.cos(w[2] * p[2])
    return v * ramp


def _initial_velocity(s):
    return np.stack([_velocity(s, d, s["pos"]) for d in range(3)], axis=1)


def _displaced(s):
    """Positions (n, 3) of a force case: strains of about 1e-3."""
    f = 2e-4 * DX * max(s["shape"])
    return s["pos"].T + _initial_velocity(s) * f


def _body(case, s):
    import peridynamics as pd
    if case["material"] == "CPD":
        mat = pd.CMaterial(model=pd.NeoHooke() if case["model"] == "neohooke" else pd.SaintVenantKirchhoff(),
                           zem=pd.ZEMWan() if case["zem"] == "wan" else pd.ZEMSilling())
    else:
        kind = pd.BBMaterial if case["material"] == "BB" else pd.OSBMaterial
        mat = kind(correction=pd.EnergySurfaceCorrection) if case["correction"] else kind()
    body = pd.Body(mat, s["pos"], s["volume"])
    for k in range(case["sets"]):
        name = f"layer{k}"
        pd.point_set(body, name, s["layer"] == k)
        kw = {"horizon": s["delta"], "rho": s["rho"][k], "E": s["E"][k]}
        if case["material"] != "BB":
            kw["nu"] = NU
        if case["permit"]:
            kw["Gc"] = 2e6
        pd.material(body, name, **kw)
    if case["crack"]:
        pd.point_set(body, "crack_a", s["crack_a"])
        pd.point_set(body, "crack_b", s["crack_b"])
        pd.precrack(body, "crack_a", "crack_b")
    pd.point_set(body, "clamp", s["clamp"])
    pd.point_set(body, "end", s["end"] & ~s["clamp"])
    if case["path"] == "nk":
        pull = s["pull"]
        for d in "xyz":
            pd.displacement_bc(lambda p: 0.0, body, "clamp", d)
        pd.displacement_bc(lambda p: pull, body, "end", "y")
        return body
    for d in "xyz":
        pd.velocity_bc(lambda t: 0.0, body, "clamp", d)
    if case["path"] == "dr":
        load = s["load"]
        pd.forcedensity_bc(lambda t: load, body, "end", "x")
        return body
    if case["drive"]:
        # the end is turned to and fro about the bar's axis
        om, fr = s["omega"], 2 * math.pi * s["freq"]
        pd.velocity_bc(lambda p, t: -om * math.cos(fr * t) * p[2], body, "end", "y")
        pd.velocity_bc(lambda p, t: om * math.cos(fr * t) * p[1], body, "end", "z")
    return body


def _newton(pd):
    return pd.NewtonKrylov(steps=1, tol=1e-30, rel_tol=1e-11, maxiter=40, gmres_restart=60,
                           gmres_maxiter=600, gmres_reltol=1e-8, gmres_abstol=1e-30, precond="two_level")


def prepare(case, seed):
    import peridynamics as pd
    s = _inputs(case, seed)
    body = _body(case, s)
    st = {"case": case, "pd": pd}
    if case["path"] == "setup":
        st["body"] = body
        return st
    dh = st["dh"] = pd.MI355XBodyDataHandler(body, precision=case["precision"])
    if case["path"] == "vv":
        st["vv"] = vv = pd.VelocityVerlet(steps=case["steps"])
        dh.set("velocity", _initial_velocity(s))
        dh.init_time_solver(vv)
        dh.initialize(vv)
        st["next"] = 1
    elif case["path"] == "dr":
        st["dr"] = pd.DynamicRelaxation(steps=case["steps"])
        dh.calc_force_density(0.0, st["dr"].dt)
    elif case["path"] == "force":
        st["x"] = _displaced(s)
    else:
        st["nk"] = _newton(pd)
        st["zero"] = np.zeros((s["n"], 3))
        st["x"] = np.ascontiguousarray(s["pos"].T)
        dh.init_newton_krylov(st["nk"])
    return st


def run(st):
    case, pd = st["case"], st["pd"]
    if case["path"] == "setup":
        dh = pd.MI355XBodyDataHandler(st["body"], precision=case["precision"])
        vv = pd.VelocityVerlet(steps=1)
        dh.init_time_solver(vv)
        dh.initialize(vv)
        out = {"bonds": dh.n_bonds, "dt": vv.dt, "active": dh.get("n_active_bonds"),
               "damage": dh.get("damage")}
        dh.close()
        return out
    dh = st["dh"]
    if case["path"] == "vv":
        vv = st["vv"]
        vv.n_steps = st["next"] + case["steps"] - 1
        dh.solve(vv, first_step=st["next"])
        st["next"] += case["steps"]
        return {f: dh.get(f) for f in FIELDS}
    if case["path"] == "dr":
        dh.solve_dr(st["dr"])
        return {f: dh.get(f) for f in FIELDS}
    if case["path"] == "force":
        dh.set("position", st["x"])
        dh.calc_force_density()
        return {"b_int": dh.get("b_int"), "damage": dh.get("damage")}
    dh.set("displacement", st["zero"])
    dh.set("position", st["x"])
    dh.nk_load_step(st["nk"], 1)
    return {"displacement": dh.get("displacement")}


# ------------------------------------------------------------------------------ compulsory work
def _offsets(horizon, slack=0.18):
    r = int(math.floor(horizon + slack))
    return [(i, j, k) for k in range(-r, r + 1) for j in range(-r, r + 1) for i in range(-r, r + 1)
            if (i or j or k) and math.sqrt(i * i + j * j + k * k) <= horizon + slack]


def _bonds(case):
    """Bonds of the lattice without the jitter."""
    m = (case["nx"], case["ny"], case["nz"])
    return sum(max(0, m[0] - abs(i)) * max(0, m[1] - abs(j)) * max(0, m[2] - abs(k))
               for i, j, k in _offsets(case["horizon"], 0.0))


def work(case):
    """Per step and bond: which neighbour (2 bytes tell it from the others of its surroundings)
    and, unless FP32 carries the stretch, the FP64 reference length; per step and point: x, u and
    v read and written, volume and reference position read.  Arithmetic: the bond sums."""
    n, nb = case["nx"] * case["ny"] * case["nz"], _bonds(case)
    bond = 2 if case["precision"] == "mixed" else 10
    if case["correction"]:
        bond += 4 if case["precision"] == "mixed" else 8
    flops = {"BB": 22, "OSB": 50, "CPD": 90}[case["material"]] * nb
    if case["path"] == "setup":
        return {"bytes": 32 * n + 12 * nb + 16 * n, "flops": 10 * nb}
    if case["path"] == "force":
        return {"bytes": bond * nb + (32 + 24 + 24 + 8) * n, "flops": flops}
    if case["path"] == "nk":
        # at the least forty products with the Jacobian, each two forces and one bond sweep
        return {"bytes": 40 * (bond * nb + 200 * n), "flops": 40 * 2 * flops}
    extra = 8 * 12 if case["path"] == "dr" else 0
    return {"bytes": case["steps"] * (bond * nb + (176 + extra) * n) + 56 * n,
            "flops": case["steps"] * (flops + 30 * n)}


# ------------------------------------------------------------------------------ 64-bit values
class _Lattice:
    """The body's bonds by lattice offset, on torch tensors in 64 bits."""

    def __init__(self, case, s):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        nx, ny, nz = s["shape"]
        self.dim = (nz, ny, nx)
        self.X = self.field(s["pos"].T)
        self.V = DX ** 3
        self.delta = s["delta"]
        layer = torch.as_tensor(s["layer"], device=self.dev).view(self.dim)
        E = [s["E"][k] for k in range(case["sets"])]
        nu = NU
        pick = lambda v: torch.tensor(v, dtype=torch.float64, device=self.dev)[layer]  # noqa: E731
        K = [e / (3 * (1 - 2 * nu)) for e in E]
        G = [e / (2 * (1 + nu)) for e in E]
        lam = [e * nu / ((1 + nu) * (1 - 2 * nu)) for e in E]
        bc = [18 * k / (math.pi * self.delta ** 4) for k in K]
        self.K, self.G, self.lam, self.bc = pick(K), pick(G), pick(lam), pick(bc)
        self.mu = self.G
        self.rho = pick([s["rho"][k] for k in range(case["sets"])])
        self.nb = torch.zeros(self.dim, dtype=torch.float64, device=self.dev)
        self.na = torch.zeros_like(self.nb)
        self.off = []
        crack = case["crack"]
        if crack:
            a = torch.as_tensor(s["crack_a"], device=self.dev).view(self.dim)
            b = torch.as_tensor(s["crack_b"], device=self.dev).view(self.dim)
        for ox, oy, oz in _offsets(case["horizon"]):
            lo = [max(0, -o) for o in (oz, oy, ox)]
            hi = [m - max(0, o) for m, o in zip(self.dim, (oz, oy, ox))]
            if any(h <= q for q, h in zip(lo, hi)):
                continue
            i = tuple(slice(q, h) for q, h in zip(lo, hi))
            j = tuple(slice(q + o, h + o) for q, h, o in zip(lo, hi, (oz, oy, ox)))
            D = [x[j] - x[i] for x in self.X]
            d2 = (D[0] * D[0] + D[1] * D[1]) + D[2] * D[2]
            inside = d2 <= self.delta * self.delta
            act = inside
            if crack:
                act = inside & ~((a[i] & b[j]) | (b[i] & a[j]))
            self.nb[i] += inside
            self.na[i] += act
            self.off.append((i, j, act.to(torch.float64), torch.sqrt(d2), inside))

    def field(self, a):
        a = torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64).to(self.dev)
        return [a[:, d].contiguous().view(self.dim) for d in range(3)]

    def zeros(self, k=3):
        return [torch.zeros(self.dim, dtype=torch.float64, device=self.dev) for _ in range(k)]

    def out(self, v):
        return torch.stack([x.reshape(-1) for x in v], dim=1)

    def damage(self):
        return (1.0 - self.na / self.nb).reshape(-1)

    def pairs(self, x):
        for i, j, act, L, _ in self.off:
            d = [c[j] - c[i] for c in x]
            l = torch.sqrt((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2])
            yield i, j, act, L, d, l

    def force(self, case, x):
        return {"BB": self._bb, "OSB": self._osb, "CPD": self._cpd}[case["material"]](case, x)

    def _bb(self, case, x):
        b = self.zeros()
        for i, j, act, L, d, l in self.pairs(x):
            f = act * (0.5 * (self.bc[i] + self.bc[j])) * ((l - L) / L) * self.V / l
            for c in range(3):
                b[c][i] += f * d[c]
        return b

    def _osb(self, case, x):
        wvol, dil = self.zeros(2)
        for i, j, act, L, d, l in self.pairs(x):
            w = act * (self.delta / L) * self.V
            wvol[i] += w * L * L
            dil[i] += w * L * (l - L)
        dil = 3.0 / wvol * dil
        b = self.zeros()
        for i, j, act, L, d, l in self.pairs(x):
            G, K = 0.5 * (self.G[i] + self.G[j]), 0.5 * (self.K[i] + self.K[j])
            f = 0.0
            for q in (i, j):
                c1 = 15.0 * G / wvol[q]
                f = f + dil[q] * (3.0 * K / wvol[q] - c1 / 3.0) * L + c1 * (l - L)
            f = act * (self.delta / L) / l * f * self.V
            for c in range(3):
                b[c][i] += f * d[c]
        return b

    def _cpd(self, case, x):
        Km, Ft = self.zeros(9), self.zeros(9)
        ref = self.X
        for i, j, act, L, d, l in self.pairs(x):
            D = [c[j] - c[i] for c in ref]
            w = act * (self.delta / L) * self.V
            for r in range(3):
                for c in range(3):
                    Km[3 * r + c][i] += w * D[r] * D[c]
                    Ft[3 * r + c][i] += w * d[r] * D[c]
        mat = lambda v: torch.stack(v, dim=-1).view(*self.dim, 3, 3)  # noqa: E731
        Ki = torch.linalg.inv(mat(Km))
        F = mat(Ft) @ Ki
        one = torch.eye(3, dtype=torch.float64, device=self.dev)
        C = F.transpose(-1, -2) @ F
        lam, mu = self.lam[..., None, None], self.mu[..., None, None]
        if case["model"] == "neohooke":
            Ci = torch.linalg.inv(C)
            J = torch.linalg.det(F)[..., None, None]
            S = mu * (one - Ci) + lam * torch.log(J) * Ci
        else:
            Eg = 0.5 * (C - one)
            tr = Eg.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
            S = lam * tr * one + 2 * mu * Eg
        PK = F @ S @ Ki
        if case["zem"] == "wan":
            trk = Ki.diagonal(dim1=-2, dim2=-1).sum(-1)[..., None, None]
            Z = lam * trk * one + mu * (Ki + Ki.transpose(-1, -2))
        else:
            beta = 0.5 * self.bc / self.delta  # ZEMSilling's default Cs
            Z = beta[..., None, None] * one
        Q = PK - Z @ F
        Q = [[Q[..., r, c].contiguous() for c in range(3)] for r in range(3)]
        Z = [[Z[..., r, c].contiguous() for c in range(3)] for r in range(3)]
        b = self.zeros()
        for i, j, act, L, d, l in self.pairs(x):
            D = [c[j] - c[i] for c in ref]
            w = act * (self.delta / L) * self.V
            for r in range(3):
                t = sum((Q[r][c][i] + Q[r][c][j]) * D[c] for c in range(3))
                cols = range(3) if case["zem"] == "wan" else (r,)
                b[r][i] += w * sum(((Z[r][c][i] + Z[r][c][j]) * d[c] for c in cols), t)
        return b

    def stable_dt(self):
        s = self.zeros(1)[0]
        for i, j, act, L, inside in self.off:
            s[i] += torch.where(inside, self.V * self.bc[i] / L, torch.zeros_like(L))
        return 0.7 * float(torch.sqrt(2.0 * self.rho / s).min())


def _too_long(case, offsets):
    n = case["nx"] * case["ny"] * case["nz"]
    ops = {"BB": 22, "OSB": 65, "CPD": 150}[case["material"]]
    return case["steps"] * offsets * ops * (n * 24 / 4e12 + 6e-6) > 14.0


def exact(case, seed):
    if case["correction"] or _too_long(case, len(_offsets(case["horizon"]))):
        return None
    s = _inputs(case, seed)
    g = _Lattice(case, s)
    if case["path"] == "setup":
        return {"bonds": None, "dt": g.stable_dt(), "active": g.na.reshape(-1), "damage": g.damage()}
    if case["path"] == "force":
        return {"b_int": g.out(g.force(case, g.field(_displaced(s)))), "damage": g.damage()}
    if case["path"] == "vv":
        return _exact_vv(case, s, g)
    if case["path"] == "dr":
        return _exact_dr(case, s, g)
    return _exact_nk(case, s, g)


def _mask(g, m):
    return torch.as_tensor(m, device=g.dev).view(g.dim)


def _exact_vv(case, s, g):
    dt = g.stable_dt()
    u, vh = g.zeros(), None
    v = g.field(_initial_velocity(s))
    a = g.zeros()
    x = [c.clone() for c in g.X]
    clamp, end = _mask(g, s["clamp"]), _mask(g, s["end"] & ~s["clamp"])
    for n in range(1, case["steps"] + 1):
        vh = [v[d] + 0.5 * dt * a[d] for d in range(3)]
        t = n * dt
        for d in range(3):
            vh[d] = torch.where(clamp, torch.zeros_like(vh[d]), vh[d])
        if case["drive"]:
            w = s["omega"] * math.cos(2 * math.pi * s["freq"] * t)
            vh[1] = torch.where(end, -w * g.X[2], vh[1])
            vh[2] = torch.where(end, w * g.X[1], vh[2])
        for d in range(3):
            u[d] = u[d] + dt * vh[d]
            x[d] = x[d] + dt * vh[d]
        b = g.force(case, x)
        a = [b[d] / g.rho for d in range(3)]
        v = [vh[d] + 0.5 * dt * a[d] for d in range(3)]
    return {"displacement": g.out(u), "velocity": g.out(v), "damage": g.damage()}


def _exact_dr(case, s, g):
    dt = 1.0
    dens = 0.25 * dt * dt * g.nb * (5 * math.pi * g.delta ** 2 * g.bc)
    u, vh, vo, bo, v = g.zeros(), g.zeros(), g.zeros(), g.zeros(), g.zeros()
    x = [c.clone() for c in g.X]
    clamp, end = _mask(g, s["clamp"]), _mask(g, s["end"] & ~s["clamp"])
    load = torch.where(end, torch.full_like(x[0], s["load"]), torch.zeros_like(x[0]))
    for n in range(1, case["steps"] + 1):
        for d in range(3):
            vh[d] = torch.where(clamp, torch.zeros_like(vh[d]), vh[d])
            u[d] = u[d] + dt * vh[d]
            x[d] = x[d] + dt * vh[d]
        b = g.force(case, x)
        tot = [b[0] + load, b[1], b[2]]
        if n == 1:
            vn = [0.5 * dt * tot[d] / dens for d in range(3)]
        else:
            c1 = sum(float(torch.where(vh[d] != 0, -u[d] * u[d] * (b[d] - bo[d]) / (dt * dens * vo[d]),
                                       torch.zeros_like(vh[d])).sum()) for d in range(3))
            c2 = sum(float((u[d] * u[d]).sum()) for d in range(3))
            cn = 2 * math.sqrt(c1 / c2) if c2 != 0 and c1 / c2 > 0 else 0.0
            cn = 1.9 if cn > 2.0 else cn
            vn = [((2 - cn * dt) * vh[d] + 2 * dt * tot[d] / dens) / (2 + cn * dt) for d in range(3)]
        v = [0.5 * (vo[d] + vn[d]) for d in range(3)]
        vh, vo, bo = vn, [c.clone() for c in vn], b
    return {"displacement": g.out(u), "velocity": g.out(v), "damage": g.damage()}


def _exact_nk(case, s, g):
    """Newton's method on the exact linearisation, conjugate gradients on its matrix."""
    n = s["n"]
    idx = torch.arange(n, device=g.dev).view(g.dim)
    free = torch.ones(n, 3, dtype=torch.bool, device=g.dev)
    clamp, end = torch.as_tensor(s["clamp"], device=g.dev), torch.as_tensor(s["end"] & ~s["clamp"], device=g.dev)
    free[clamp] = False
    free[end, 1] = False
    u = torch.zeros(n, 3, dtype=torch.float64, device=g.dev)
    u[end, 1] = s["pull"]
    X = g.out(g.X)
    ii, jj, LL, bb = [], [], [], []
    for i, j, act, L, inside in g.off:
        m = inside.reshape(-1)
        ii.append(idx[i].reshape(-1)[m])
        jj.append(idx[j].reshape(-1)[m])
        LL.append(L.reshape(-1)[m])
        bb.append((0.5 * (g.bc[i] + g.bc[j])).reshape(-1)[m])
    ii, jj, LL, bb = torch.cat(ii), torch.cat(jj), torch.cat(LL), torch.cat(bb)
    order = torch.argsort(ii, stable=True)
    ii, jj, LL, bb = ii[order], jj[order], LL[order], bb[order]
    one = torch.eye(3, dtype=torch.float64, device=g.dev)
    crow = torch.zeros(n + 1, dtype=torch.int64, device=g.dev)
    crow[1:] = torch.cumsum(torch.bincount(ii, minlength=n), 0)
    add = lambda t: torch.zeros(n, *t.shape[1:], dtype=torch.float64, device=g.dev).index_add_(0, ii, t)  # noqa: E731
    first = None
    for _ in range(12):
        d = (X + u)[jj] - (X + u)[ii]
        l = d.norm(dim=1)
        eps = (l - LL) / LL
        r = add((bb * eps * g.V / l)[:, None] * d) * g.V
        r = torch.where(free, r, torch.zeros_like(r))
        first = float(r.norm()) if first is None else first
        if float(r.norm()) < 1e-13 * first:
            break
        nn = d / l[:, None]
        C = (bb * g.V * g.V)[:, None, None] * ((1 / LL - eps / l)[:, None, None] * nn[:, :, None] * nn[:, None, :]
                                                + (eps / l)[:, None, None] * one)
        diag = add(C)
        Minv = torch.linalg.inv(diag)
        ell = torch.zeros(n, int((crow[1:] - crow[:-1]).max()), 3, 3, dtype=torch.float64, device=g.dev)
        nbr = torch.zeros(n, ell.shape[1], dtype=torch.int64, device=g.dev)
        at = torch.arange(ii.numel(), device=g.dev) - crow[ii]
        ell[ii, at], nbr[ii, at] = C, jj

        def apply(p):
            y = (diag @ p[:, :, None])[:, :, 0] - (ell * p[nbr][:, :, None, :]).sum((1, 3))
            return torch.where(free, y, torch.zeros_like(y))

        du, res = torch.zeros_like(u), r.clone()
        z = torch.where(free, (Minv @ res[:, :, None])[:, :, 0], torch.zeros_like(res))
        p, rz = z.clone(), (res * z).sum()
        for it in range(3000):
            q = apply(p)
            alpha = rz / (p * q).sum()
            du += alpha * p
            res -= alpha * q
            if it % 20 == 0 and float(res.norm()) < 1e-12 * float(r.norm()):
                break
            z = torch.where(free, (Minv @ res[:, :, None])[:, :, 0], torch.zeros_like(res))
            new = (res * z).sum()
            p, rz = z + (new / rz) * p, new
        u = u + du
    return {"displacement": u}
