"""The work a program hands this library, as timed cases.

A pass is what such a program does between two outputs: a number of time
steps, then the output.  The runs (`kind` "run") write the volume averages and
the FP64 fields on the device; `particles` and `twoway` also read the particle
records back; `batch` advances an ensemble of small lattices together;
`diagnostics` is the averages and the x, y, z rulers that a run appends to its
.dat files; `restart` loads a checkpoint, steps, and writes the next one.

Lattice sizes, Rayleigh numbers and particle loads are those of bench.py, the
tests and ch4g/workloads.py: Poiseuille 4x64x4, convection from 64x32 to
1024x512 and 512^3, channels of 64^3 to 192^3, forced turbulence with the
Smagorinsky closure, one particle per 33 nodes and fewer.

`exact` is a plain FP64 torch step of the same model (D3Q19 BGK with the Guo
force, the y walls, the forcings and the local-strain closure)."""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ch4-project_amd"))

from ch4g import Lattice, abi, step_batch  # noqa: E402

PRECISION = {"fp64": abi.FP64, "fp32dev": abi.FP32_DEV, "fp32store": abi.FP32_STORE}
UFF = 0.05  # free-fall velocity of the convection runs
NU_MIN = 5e-4  # smallest viscosity a convection run is given (ch4g/workloads.py)
# grids of the served parameter sweep (ch4g/workloads.py)
SWEEP_GRIDS = [(64, 32), (96, 48), (128, 64), (192, 96), (256, 128)]


def listed():
    def run(name, flow, nx, ny, nz, precision, steps, **more):
        return dict(name=name, kind="run", flow=flow, NX=nx, NY=ny, NZ=nz, precision=precision, steps=steps, **more)

    return [
        # the smallest run: a validation channel, every launch far below the GPU's size
        run("poiseuille-4x64x4-fp64", "channel", 4, 64, 4, "fp64", 100),
        # 2-D convection at its standard size, in both storages that production runs use
        run("rb-512x256-fp32", "rb", 512, 256, 1, "fp32dev", 400, Ra=1e8),
        run("rb-512x256-fp64", "rb", 512, 256, 1, "fp64", 400, Ra=1e8),
        # 2-D convection with rows and columns that fill no tile
        run("rb-969x487-fp32", "rb", 969, 487, 1, "fp32dev", 200, Ra=3e8),
        # a 3-D channel of the served stream, rows of 78 nodes
        run("channel-78-fp32", "channel", 78, 78, 78, "fp32dev", 200),
        # 3-D convection in the reference's own precision
        run("rb-256^3-fp64", "rb", 256, 256, 256, "fp64", 20, Ra=1e9),
        # 3-D convection at the largest size, the headline run
        run("rb-512^3-fp32", "rb", 512, 512, 512, "fp32dev", 20, Ra=1e9),
        # forced turbulence with the closure and one-way particles, records written at the end
        dict(name="hit-192-particles-fp32", kind="particles", flow="hit", NX=192, NY=192, NZ=192, precision="fp32dev",
             steps=200, les="local", particles=200_000),
        # 3-D convection coupled to heavy particles (one per 34 nodes)
        dict(name="rb-256^3-twoway-fp32", kind="twoway", flow="rb", NX=256, NY=256, NZ=256, precision="fp32dev",
             steps=32, Ra=1e8, particles=500_000),
        # an ensemble of small convection runs advanced together
        dict(name="sweep-32-runs-fp32", kind="batch", flow="rb", count=32, precision="fp32dev", steps=128),
        # the diagnostics of a run: averages and rulers
        dict(name="diagnostics-256^3-fp32", kind="diagnostics", flow="rb", NX=256, NY=256, NZ=256, precision="fp32dev",
             steps=8, Ra=1e9),
        # restart from a checkpoint and write the next
        dict(name="restart-96x80x112-fp64", kind="restart", flow="rb", NX=96, NY=80, NZ=112, precision="fp64", steps=16,
             Ra=1e7),
    ]


# ---------------------------------------------------------------------------
# more cases of the same ranges

def _size(rng, lo, hi):
    """log-uniform whole number; every second one odd or not a multiple of anything"""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.5 else max(lo, n // 8 * 8)


def draw(rng):
    r = rng.random()
    if r < 0.62:
        kind = "run"
    else:
        kind = ("particles", "twoway", "batch", "diagnostics", "restart")[int((r - 0.62) / 0.38 * 5) % 5]
    if kind == "batch":
        return dict(kind="batch", flow="rb", count=_size(rng, 4, 48), precision=rng.choice(["fp32dev", "fp32dev", "fp64"]),
                    steps=_size(rng, 32, 256))
    precision = rng.choice(["fp32dev", "fp32dev", "fp32dev", "fp64", "fp64", "fp32store"])
    c = dict(kind=kind, precision=precision)
    flow = {"particles": "hit", "twoway": "rb"}.get(kind) or rng.choice(["rb2d", "rb2d", "rb3d", "channel", "hit"])
    if flow == "rb2d":
        s = rng.uniform(0.0, 1.0)  # 64x32 to 2048x1024 at the aspect ratios of the served stream
        c.update(flow="rb", NX=_size(rng, 32, 2048) if rng.random() < 0.3 else int(round(64 * 32 ** s)),
                 NY=int(round(32 * 32 ** s)), NZ=1)
    elif flow in ("rb", "rb3d"):
        c.update(flow="rb", NX=_size(rng, 32, 320), NY=_size(rng, 24, 320), NZ=_size(rng, 16, 320))
    elif flow == "channel":
        n = _size(rng, 4, 192)
        c.update(flow="channel", NX=n, NY=max(16, n), NZ=n if rng.random() < 0.6 else _size(rng, 4, 192))
    else:
        n = _size(rng, 16, 224)
        c.update(flow="hit", NX=n, NY=n, NZ=n, les=rng.choice(["local", "local", "none", "fd"]))
    if kind == "restart":
        for a in ("NX", "NY", "NZ"):  # checkpoints pass through host arrays
            c[a] = min(c[a], 128)
    if kind == "diagnostics":
        for a in ("NX", "NY", "NZ"):
            c[a] = min(c[a], 256) if c["NZ"] > 1 else c[a]
    n = c["NX"] * c["NY"] * c["NZ"]
    if c["flow"] == "rb":
        h = c["NY"]  # what the rows resolve, up to 1e9
        lo = 1e6 if kind == "twoway" else 1e5
        c["Ra"] = float("%.3g" % min(1e9, math.exp(rng.uniform(math.log(lo), math.log(1e8))), (UFF * h / NU_MIN) ** 2))
    if kind in ("particles", "twoway"):
        c["particles"] = max(100, min(500_000, int(n * math.exp(rng.uniform(math.log(0.001), math.log(0.05))))))
        c.setdefault("les", "none")
    # enough steps that a pass is mostly steps, as between two outputs, within the largest case's cost
    c["steps"] = max(4, min({"run": 400, "restart": 32, "diagnostics": 8}.get(kind, 200), int(1.2e9 / n)))
    return c


# ---------------------------------------------------------------------------
# configurations

def _nodes(case):
    return case["NX"] * case["NY"] * case["NZ"]


def _config(case, seed):
    """abi.Config of the case; `seed` is the run's random seed (temperature noise, forcing phases)."""
    nx, ny, nz, prec, seed = case["NX"], case["NY"], case["NZ"], PRECISION[case["precision"]], 1 + seed % (2 ** 31 - 2)
    if case["flow"] == "rb":
        nu = UFF * ny * (1.0 / case["Ra"]) ** 0.5
        bg, g = UFF * UFF / ny, 1.0
        if case["kind"] == "twoway":
            g = 2e-5  # the particles' gravity; beta_t g is the fluid's
        flags = (abi.LB_FLUID | abi.LB_TEMPERATURE | abi.TEMPERATURE_BUOYANCY | abi.FLUID_BC_Y | abi.TEMPERATURE_BC_Y |
                 abi.TEMPERATURE_INITIAL_LINEAR | abi.TEMPERATURE_INITIAL_ADD_NOISE)
        return abi.make_config(nx, ny, nz, flags, precision=prec, seed=seed, tau_u=3 * nu + 0.5, tau_t=3 * nu + 0.5,
                               beta_t=bg / g, gravity_y=g, T_bot=1.0, T_top=0.0, T_ref=0.0, noise_t=1e-3)
    if case["flow"] == "channel":
        tau = 1.0 if nx <= 8 else 0.6
        nu = (tau - 0.5) / 3.0
        return abi.make_config(nx, ny, nz, abi.LB_FLUID | abi.FLUID_FORCING_POISEUILLE | abi.FLUID_BC_Y, precision=prec,
                               seed=seed, tau_u=tau, Amp_x=1e-6 * ny * ny / (8.0 * nu))
    flags = abi.LB_FLUID | abi.FLUID_FORCING_HIT
    flags |= {"none": 0, "local": abi.FLUID_LES | abi.FLUID_LES_LOCAL_STRAIN, "fd": abi.FLUID_LES}[case["les"]]
    return abi.make_config(nx, ny, nz, flags, precision=prec, seed=seed, tau_u=0.52 if case["les"] == "none" else 0.5015,
                           Amp_x=1e-5, Amp_y=1e-5, Amp_z=1e-5, les_cs=0.1)


def _channel_start(case, seed):
    """Populations [NZ][NY][NX][19] of a channel with random low modes on its velocity."""
    nz, ny, nx = case["NZ"], case["NY"], case["NX"]
    r = np.random.default_rng(seed)
    z, y, x = np.meshgrid((np.arange(nz) + 0.5) / nz, (np.arange(ny) + 0.5) / ny, (np.arange(nx) + 0.5) / nx, indexing="ij")
    shape = 4.0 * y * (1.0 - y)
    u = np.zeros((3,) + x.shape)
    u[0] = 0.03 * shape
    for _ in range(4):
        k = r.integers(1, 4, 3)
        for a in range(3):
            u[a] += 0.004 * shape * r.uniform(-1, 1) * np.sin(2 * np.pi * (k[0] * x + k[2] * z + r.random()) + np.pi * k[1] * y)
    u2 = (u * u).sum(0)
    p = np.empty((nz, ny, nx, 19))
    for q in range(19):
        cu = sum(C[q][a] * u[a] for a in range(3))
        p[..., q] = W[q] * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * u2)
    return p


def _flow_start(case, seed):
    """(p, g) of a checkpoint: a convection or turbulence state written by an earlier run."""
    if case["flow"] == "channel":
        return _channel_start(case, seed), None
    p = _channel_start(dict(case), seed)
    if case["flow"] != "rb":
        return p, None
    nz, ny, nx = case["NZ"], case["NY"], case["NX"]
    r = np.random.default_rng(seed + 1)
    y = (np.arange(ny) + 0.5) / ny
    t = (1.0 - y)[None, :, None] + 0.05 * np.sin(np.pi * y)[None, :, None] * r.standard_normal((nz, 1, nx)) / 3.0
    t = t + 1e-3 * r.uniform(-1, 1, (nz, ny, nx))
    return p, t[..., None] * np.array(W)


def _response_time(case):
    """of the heavy particles: a volume of 0.03 lattice cells each ((4/3) pi (3 nu beta tau)^(3/2)), 2 steps at least"""
    return max(2.0, 0.037 / (3.0 * 0.6 * UFF * case["NY"] * (1.0 / case["Ra"]) ** 0.5)) if case["kind"] == "twoway" else 16.0


def _particle_start(case, seed):
    """Positions and response times: half tracers, half inertial, or one heavy type when they act back."""
    n, r = case["particles"], np.random.default_rng(seed + 2)
    a = np.zeros(n, dtype=abi.particle_dtype())
    a["name"] = np.arange(n)
    for axis, m in (("x", case["NX"]), ("y", case["NY"]), ("z", case["NZ"])):
        a[axis] = r.uniform(0.0, m, n)
    if case["kind"] == "twoway":
        a["tau_drag"], a["beta_coeff"] = _response_time(case), 0.6
    else:
        a["tau_drag"][n // 2:] = r.uniform(1.0, 50.0, n - n // 2)
    return a


def _fields(n, fluid=True, thermal=True):
    new = lambda m: torch.zeros(m, dtype=torch.float64, device="cuda")  # noqa: E731
    return new(n) if fluid else None, new(3 * n) if fluid else None, new(n) if thermal else None


def _lattice(case, seed):
    lat = Lattice(_config(case, seed))
    if case["flow"] == "channel":
        lat.set_populations(_channel_start(case, seed))
    else:
        lat.initial_conditions()
    if case["kind"] in ("particles", "twoway"):
        flags = abi.LAGRANGE_WRAP
        if case["kind"] == "twoway":
            flags |= (abi.LAGRANGE_GRADIENT | abi.LAGRANGE_ADDEDMASS | abi.LAGRANGE_GRAVITY | abi.LAGRANGE_TWOWAY_MOMENTUM)
        tau = _response_time(case)
        lat.particles_init(abi.make_particle_config(flags, 1, tau_drag=(1, tau, tau), beta_coeff=(1, 0.6, 0.6)))
        lat.set_particles(_particle_start(case, seed))
    return lat


def _sweep(case, seed):
    r = np.random.default_rng(seed)
    # every grid of the sweep in turn, so that the work does not depend on the seed
    return [dict(kind="run", flow="rb", NX=g[0], NY=g[1], NZ=1, precision=case["precision"], steps=case["steps"],
                 Ra=float(math.exp(r.uniform(math.log(1e5), math.log(1e7)))), seed=int(r.integers(1, 2 ** 31 - 1)))
            for g in (SWEEP_GRIDS[i % len(SWEEP_GRIDS)] for i in range(case["count"]))]


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "batch":
        runs = _sweep(case, seed)
        lats = [Lattice(_config(c, c["seed"])) for c in runs]
        for lat in lats:
            lat.initial_conditions()
            lat.step(1)  # lattices join an ensemble after their first step
        at = np.concatenate([[0], np.cumsum([_nodes(c) for c in runs])])
        dens, u, t = _fields(int(at[-1]))
        state.update(lats=lats, fields=(dens, u, t),
                     parts=[(dens[a:b], u[3 * a:3 * b], t[a:b]) for a, b in zip(at[:-1].tolist(), at[1:].tolist())])
        return state
    if case["kind"] == "restart":
        state.update(lat=Lattice(_config(case, seed)), checkpoint=_flow_start(case, seed))
        return state
    state["lat"] = lat = _lattice(case, seed)
    if case["kind"] == "diagnostics":
        lat.step(case["steps"])
        return state
    state["fields"] = _fields(_nodes(case), True, case["flow"] == "rb")
    return state


# ---------------------------------------------------------------------------
# one pass

def _row(averages):
    """the row a run appends to its averages file: node coordinates, then the averages"""
    v = np.array(list(averages.values()))
    return v[:3], v[3:]


def _output(lat, fields):
    dens, u, t = fields
    return _row(lat.dump_averages_noalloc(dens.data_ptr(), u.data_ptr(), None if t is None else t.data_ptr()))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        step_batch(state["lats"], case["steps"])
        rows = np.stack([_output(lat, f)[1] for lat, f in zip(state["lats"], state["parts"])])
        return {"rows": rows, "dens": state["fields"][0], "u": state["fields"][1], "t": state["fields"][2]}
    lat = state["lat"]
    if kind == "diagnostics":
        row = _row(lat.dump_averages())
        rulers = [r.view(np.float64).reshape(len(r), len(abi.OUTPUT_FIELDS)) for r in lat.dump_rulers()]
        return {"row": row, "rulers": [(r[:, :3], r[:, 3:]) for r in rulers]}
    if kind == "restart":
        lat.set_populations(*state["checkpoint"])
        lat.step(case["steps"])
        p, g = lat.get_populations()
        h = lat.hydro_fields()
        return {"p": p, "g": g if case["flow"] == "rb" else None, "dens": h["dens"], "u": h["u"],
                "t": h["t"] if case["flow"] == "rb" else None}
    lat.step(case["steps"])
    row = _output(lat, state["fields"])
    out = {"row": row, "dens": state["fields"][0], "u": state["fields"][1], "t": state["fields"][2]}
    if kind in ("particles", "twoway"):
        a = lat.particles()
        a = a.view(np.float64).reshape(len(a), len(abi.PARTICLE_FIELDS))
        # members of ch4g_particle: position, velocity, the last velocity and both accelerations, fluid velocity, the rest
        out.update(x=a[:, 1:4], v=a[:, 4:7], before=a[:, 7:16], u_at=a[:, 16:19], rest=a[:, 19:])
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    if case["kind"] == "batch":
        return {k: sum(work(c)[k] for c in _sweep(case, 0)) for k in ("bytes", "flops")}
    n, r = _nodes(case), 8 if case["precision"] == "fp64" else 4
    sets = 2 if case["flow"] == "rb" else 1
    # a step: every population read and written once, and the lagged temperature or relaxation time
    step_bytes = n * r * (2 * 19 * sets + (2 if sets == 2 or case.get("les", "none") != "none" else 0))
    step_flops = n * (300 + 200 * (sets - 1))
    state, fields = n * r * 19 * sets, n * 8 * (4 + (sets - 1))
    if case["kind"] == "diagnostics":
        return {"bytes": float(state + 2 * fields), "flops": float(n * 150)}
    b, f = case["steps"] * step_bytes + state + fields, case["steps"] * step_flops + n * 60
    if case["kind"] == "restart":
        b += 2 * n * 8 * 19 * sets
    if case["kind"] in ("particles", "twoway"):
        # rows read and written and eight corners a step; with gradients 32 nodes; the records at the end
        rows = (12 + 20) * 8 + 8 * 12 if case["kind"] == "particles" else (40 + 40) * 8 + 32 * 16 + 8 * 24
        b += case["particles"] * (case["steps"] * rows + 78 * 8)
        f += case["particles"] * case["steps"] * (200 if case["kind"] == "particles" else 1500)
        if case["kind"] == "twoway":
            b += case["steps"] * n * (2 * 3 * r + 4 * 4)  # feedback written and read, fields written
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same in plain FP64 torch

C = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (1, -1, 0), (-1, 1, 0),
     (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1), (0, 1, 1), (0, 1, -1), (0, -1, 1), (0, -1, -1)]
OPP = [C.index((-a, -b, -c)) for a, b, c in C]
W = [1 / 3] + [1 / 18] * 6 + [1 / 36] * 12
MODES = [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (0, 1, 1), (1, 0, 1)]


class _Drand48:
    """drand48's sequence: one number at a time, or many at once."""
    A, INC, MASK = 0x5DEECE66D, 0xB, (1 << 48) - 1

    def __init__(self, seed):
        self.x = ((seed & 0xFFFFFFFF) << 16) | 0x330E

    def one(self):
        self.x = (self.A * self.x + self.INC) & self.MASK
        return self.x / 2.0 ** 48

    def many(self, n, device):
        out = torch.tensor([(self.A * self.x + self.INC) & self.MASK], dtype=torch.int64, device=device)
        a, c, have = self.A, self.INC, 1  # the map that jumps `have` numbers on
        while have < n:
            signed = a - (1 << 64) if a >= 1 << 63 else a
            out = torch.cat([out, (out * signed + c) & self.MASK])[:n]
            a, c, have = (a * a) & self.MASK, (a * c + c) & self.MASK, 2 * have
        self.x = int(out[-1])
        return out.double() / 2.0 ** 48

    def gauss(self):
        while True:
            u1, u2 = -1 + self.one() * 2, -1 + self.one() * 2
            w = u1 ** 2 + u2 ** 2
            if 0 < w < 1:
                return u1 * math.sqrt((-2 * math.log(w)) / w)


class _Plain:
    """One lattice: populations [19][NZ][NY][NX] in FP64."""

    def __init__(self, case, seed, start=None):
        self.case, self.cfg = case, _config(case, seed)
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        nx, ny, nz = case["NX"], case["NY"], case["NZ"]
        self.shape = (nz, ny, nx)
        full = lambda v: torch.as_tensor(v, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.w = full(W).reshape(19, 1, 1, 1)
        self.c = full(C).t().contiguous()
        self.thermal, self.hit = case["flow"] == "rb", case["flow"] == "hit"
        self.rng = _Drand48(self.cfg.seed)
        self.nu, self.kappa = (self.cfg.tau_u - 0.5) / 3.0, (self.cfg.tau_t - 0.5) / 3.0
        self.tau = None
        self.g = None
        if start is None and case["flow"] == "channel":
            start = (_channel_start(case, seed), None)
        if start is not None:
            self.f = full(start[0]).permute(3, 0, 1, 2).contiguous()
            if self.thermal:
                self.g = full(start[1]).permute(3, 0, 1, 2).contiguous()
        else:
            self.f = self.w.expand(19, nz, ny, nx).clone()
            if self.thermal:
                y = torch.arange(ny, dtype=torch.float64, device=self.dev) + 0.5
                t = (1.0 - y / ny).reshape(1, ny, 1).expand(nz, ny, nx)
                t = t + 1e-3 * (2.0 * self.rng.many(nx * ny * nz, self.dev).reshape(nz, ny, nx) - 1.0)
                self.g = self.w * t
        if self.hit:
            # a restart without initial conditions starts from phases of 0
            self.phi = [[self.rng.one() if start is None else 0.0 for _ in range(3)] for _ in MODES]
            self.walk()
        self.force_u = self.force(self.g.sum(0) if self.thermal else None)

    def walk(self):
        turnover = self.case["NX"] / 0.1
        for p in self.phi:
            for a in range(3):
                p[a] += -p[a] / turnover + self.rng.gauss() * math.sqrt(2.0 * 0.01 / turnover)

    def force(self, t):
        """the body force, broadcastable to [NZ][NY][NX], a component at a time"""
        cfg = self.cfg
        if self.thermal:
            return [0.0, cfg.beta_t * (t - 0.5) * cfg.gravity_y, 0.0]
        if self.case["flow"] == "channel":
            return [2.0 * cfg.Amp_x * 4.0 * self.nu / cfg.NY ** 2, 0.0, 0.0]
        total = [0.0, 0.0, 0.0]
        s = []
        for a, m in enumerate((cfg.NX, cfg.NY, cfg.NZ)):
            x = (torch.arange(m, dtype=torch.float64, device=self.dev) + 0.5) / m
            at = [-1 if b == 2 - a else 1 for b in range(3)]
            s.append([torch.sin(2 * 3.14159265359 * (k[a] * x + p[a])).reshape(at) for k, p in zip(MODES, self.phi)])
        for i, k in enumerate(MODES):
            amp = (k[0] ** 2 + k[1] ** 2 + k[2] ** 2) ** (-1.0 / 3.0) * cfg.Amp_x
            sx, sy, sz = s[0][i], s[1][i], s[2][i]
            total = [total[0] + amp * (sy + sz), total[1] + amp * (sx + sz), total[2] + amp * (sy + sx)]
        return total

    def moments(self):
        rho = self.f.sum(0)
        j = torch.tensordot(self.c, self.f, 1)
        return rho, torch.stack([j[a] / rho + 0.5 * self.force_u[a] for a in range(3)])

    def equilibrium(self, rho, u, cu):
        return self.w * rho * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * (u * u).sum(0))

    def closure(self, rho, u, cu):
        """relaxation time of the Smagorinsky closure"""
        cs2 = self.cfg.les_cs ** 2
        if self.case["les"] == "local":
            d = self.f - self.equilibrium(rho, u, cu)
            m = lambda a, b: torch.tensordot(self.c[a] * self.c[b], d, 1)  # noqa: E731
            # the reference's tensor has xz in the place of zz, and no zx
            xx, yy, xy, xz, yz = m(0, 0), m(1, 1), m(0, 1), m(0, 2), m(1, 2)
            ss = xx * xx + 2 * xy * xy + xz * xz + yy * yy + 2 * yz * yz + xz * xz
            last = self.cfg.tau_u if self.tau is None else self.tau
            strain = torch.sqrt(2.0 * ss) / (2.0 / 3.0 * rho * last)
        else:
            grad = lambda a, b: 0.5 * (torch.roll(u[a], -1, 2 - b) - torch.roll(u[a], 1, 2 - b))  # noqa: E731
            strain = torch.sqrt(0.5 * sum((grad(a, b) + grad(b, a)) ** 2 for a in range(3) for b in range(3)))
        return 3.0 * (strain * cs2 + self.nu) + 0.5

    def stream(self, post, wall):
        """the streamed populations; `wall`(q, row) gives those that enter at a y wall"""
        out = torch.empty_like(post)
        for q, (a, b, c) in enumerate(C):
            out[q] = torch.roll(post[q], (c, b, a), (0, 1, 2))
            if b and not self.hit:
                row = 0 if b > 0 else self.shape[1] - 1
                out[q][:, row, :] = wall(q, row)
        return out

    def step(self):
        cfg = self.cfg
        rho, u = self.moments()
        t = self.g.sum(0) if self.thermal else None
        cu = torch.tensordot(self.c.t(), u, 1)
        omega = 1.0 / cfg.tau_u
        if self.hit:
            self.walk()
            if self.case["les"] != "none":
                self.tau = self.closure(rho, u, cu)
                omega = 1.0 / self.tau
        force = self.force(t)
        post = self.f - omega * (self.f - self.equilibrium(rho, u, cu))
        uf = sum(u[a] * force[a] for a in range(3))
        for q in range(19):
            cf = sum(C[q][a] * force[a] for a in range(3) if C[q][a])
            post[q] += (1.0 - 0.5 / cfg.tau_u) * W[q] * rho * (3.0 * (cf - uf) + 9.0 * cu[q] * cf)
        self.f = self.stream(post, lambda q, row: post[OPP[q]][:, row, :])
        if self.thermal:
            post_g = self.g - (self.g - self.equilibrium(t, u, cu)) / cfg.tau_t
            self.g = self.stream(post_g, lambda q, row: post_g[q][:, row, :] +
                                 W[q] * 2.0 * ((cfg.T_bot if row == 0 else cfg.T_top) - t[:, row, :]))
        self.force_u = force

    def hydro(self):
        rho, u = self.moments()
        return rho, u, self.g.sum(0) if self.thermal else None

    def terms(self):
        """the members of the averages at every node, [26][NZ][NY][NX]"""
        rho, u, t = self.hydro()
        nz, ny, nx = self.shape
        d = torch.zeros((26,) + self.shape, dtype=torch.float64, device=self.dev)
        ar = lambda m, at: (torch.arange(m, dtype=torch.float64, device=self.dev) + 0.5).reshape(at)  # noqa: E731
        d[0], d[1], d[2] = ar(nx, (1, 1, -1)), ar(ny, (1, -1, 1)), ar(nz, (-1, 1, 1))

        def grad(v, b):
            if self.shape[2 - b] == 1:
                return torch.zeros_like(v)
            r = 0.5 * (torch.roll(v, -1, 2 - b) - torch.roll(v, 1, 2 - b))
            if b == 1 and not self.hit:
                r[:, 0] = -1.5 * v[:, 0] + 2.0 * v[:, 1] - 0.5 * v[:, 2]
                r[:, -1] = 1.5 * v[:, -1] - 2.0 * v[:, -2] + 0.5 * v[:, -3]
            return r

        d[3:6], d[6:9], d[9], d[10], d[12] = u, u * u, rho, 0.5 * (u * u).sum(0), rho * rho
        for a in range(3):
            for b in range(3):
                d[11] += 0.5 * self.nu * (grad(u[a], b) + grad(u[b], a)) ** 2
        if self.thermal:
            g = torch.stack([grad(t, b) for b in range(3)])
            d[13], d[14], d[15], d[16:19] = t, t * t, self.kappa * (g * g).sum(0), g
            d[19:22] = u * t
            d[22:25] = -self.kappa * g + u * t
        return d

    def normal(self, sums, norm, tnorm):
        """sums [...][26] as the averages files hold them (coordinates left as they are)"""
        o, cfg = sums.clone(), self.cfg
        o[..., 3:13] *= norm
        o[..., 13:22] *= tnorm
        if self.thermal:
            o[..., 22:25] *= tnorm * cfg.NY / self.kappa
            o[..., 25] = o[..., 11].pow(1.25) * o[..., 15].pow(-0.75) * (cfg.gravity_y * cfg.beta_t) ** -1.5
        return o

    def row(self):
        n = float(self.shape[0] * self.shape[1] * self.shape[2])
        v = self.normal(self.terms().sum((1, 2, 3)), 1.0 / n, 1.0 / n)
        return v[:3], v[3:]

    def rulers(self):
        d, out = self.terms(), []
        nz, ny, nx = self.shape
        for b, (norm, tnorm) in enumerate(((1 / (ny * nz), 1 / (ny * nz)), (1 / (nx * nz), 1 / (nx * nz)),
                                           (1 / (nx * ny), 1 / (ny * nz)))):
            o = self.normal(d.sum([1 + a for a in range(3) if a != 2 - b]).t(), norm, tnorm)
            x = o[:, b] * norm
            o[:, :3] = 0.0
            o[:, b] = x
            out.append((o[:, :3], o[:, 3:]))
        return out

    def fields(self):
        rho, u, t = self.hydro()
        return rho.reshape(-1), u.permute(1, 2, 3, 0).reshape(-1), t.reshape(-1) if t is not None else None


class _Points:
    """Tracers and particles with Stokes drag on the velocity of a _Plain."""

    def __init__(self, plain, case, seed):
        a = _particle_start(case, seed)
        put = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=plain.dev)  # noqa: E731
        self.plain = plain
        self.x = torch.stack([put(a[k]) for k in "xyz"])
        self.tau = put(a["tau_drag"])
        self.v, self.v_old, self.a_old, self.count = torch.zeros_like(self.x), None, None, 0

    def fluid(self):
        u = self.plain.hydro()[1]
        n = torch.tensor(self.plain.shape[::-1], dtype=torch.float64, device=u.device).reshape(3, 1)
        s = torch.remainder(self.x, n) - 0.5
        i = torch.floor(s)
        w = s - i
        total = 0.0
        for corner in range(8):
            d = torch.tensor([corner & 1, corner >> 1 & 1, corner >> 2], dtype=torch.float64, device=u.device).reshape(3, 1)
            at = torch.remainder(i + d, n).long()
            total = total + u[:, at[2], at[1], at[0]] * torch.where(d > 0, w, 1.0 - w).prod(0)
        return total

    def step(self):
        u = self.fluid()
        inertial = self.tau > 0
        first = self.count == 0
        v = torch.where(inertial, self.v, u)
        acc = torch.where(inertial, (u - v) / torch.where(inertial, self.tau, torch.ones_like(self.tau)), torch.zeros_like(u))
        self.x = self.x + (v if first else 0.5 * (3.0 * v - self.v_old))
        self.v_old = v
        self.v = torch.where(inertial, v + (acc if first else 0.5 * (3.0 * acc - self.a_old)), u)
        n = torch.tensor(self.plain.shape[::-1], dtype=torch.float64, device=u.device).reshape(3, 1)
        self.x = torch.remainder(self.x, n)
        self.a_old, self.u, self.count = acc, u, self.count + 1


def exact(case, seed):
    if case["kind"] == "twoway":
        return None
    if case["kind"] == "batch":
        if case["count"] * case["steps"] > 5000:
            return None
        rows, fields = [], []
        for c in _sweep(case, seed):
            s = _Plain(c, c["seed"])
            for _ in range(1 + case["steps"]):
                s.step()
            rows.append(s.row()[1])
            fields.append(s.fields())
        return {"rows": torch.stack(rows), "dens": torch.cat([f[0] for f in fields]), "u": torch.cat([f[1] for f in fields]),
                "t": torch.cat([f[2] for f in fields])}
    n = _nodes(case)
    if case["steps"] * (n + 1e5) > 2.4e9 or n > 3e7 or (n > 2e6 and not torch.cuda.is_available()):
        return None
    if case["kind"] == "restart":
        s = _Plain(case, seed, _flow_start(case, seed))
    else:
        s = _Plain(case, seed)
    points = None
    if case["kind"] == "particles":
        for _ in range(3):  # the one position drawn by particles_init
            s.rng.one()
        points = _Points(s, case, seed)
    for _ in range(case["steps"]):
        s.step()
        if points:
            points.step()
    if case["kind"] == "diagnostics":
        return {"row": s.row(), "rulers": s.rulers()}
    dens, u, t = s.fields()
    if case["kind"] == "restart":
        nz, ny, nx = s.shape
        aos = lambda v: v.permute(1, 2, 3, 0).contiguous()  # noqa: E731
        return {"p": aos(s.f), "g": aos(s.g) if s.thermal else None, "dens": dens.reshape(s.shape),
                "u": u.reshape(s.shape + (3,)), "t": t.reshape(s.shape) if t is not None else None}
    out = {"row": s.row(), "dens": dens, "u": u, "t": t}
    if points:
        out.update(x=points.x.t(), v=points.v.t(), u_at=points.u.t(), rest=None, before=None)
    return out
