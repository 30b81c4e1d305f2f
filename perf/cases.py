"""Measured cases of wildfires_amd: what its users have it do, each through
the public entry points, over the range of sizes, precisions and directions.

A case's `kind`:
  run       one forecast of a solver that a program keeps: the initial state
            goes in from host arrays, `steps` time steps run, the state comes
            back (Solver.set_state, Solver.step and the pinned snapshot that
            the C driver writes its files from)
  ensemble  the same for a batched ensemble of uneven grids
  train     Adam steps of the learned closure on rows the trainer holds
  eval      the closure network on rows of host features

exact() restates the method in 64 bits with torch alone (upwind RHS, SGS with
van Driest damping, immersed terrain, Fourier-tridiagonal pressure iteration,
projection), so that the outputs' own error can be measured.
"""
import ctypes
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from wildfires_amd import _abi, api, closure

CLOSURE_FILE = os.path.join(os.path.dirname(os.path.abspath(closure.__file__)), "data", "closure.npz")

# Node spacing, time step, constants and initial state per scenario (the
# spacings are those of the repository's 256x256x128 hill workload, its
# 64x64x32 flat workload and its learned-closure workload).
SETUPS = {
    # burning line over a Gaussian hill, seeded fuel load
    "hill": dict(dx=400.0 / 255, dz=50.0 / 127, dt=0.005, Y_h=0.5,
                 keys=dict(A=1e5, Y_f=10.0, T_max=1500.0)),
    # flat ground, a small hot block in a turned wind
    "flat": dict(dx=200.0 / 63, dz=20.0 / 31, dt=0.01, Y_h=0.5, keys=dict(T_inf=300.0)),
    # flat ground, a hot line segment over deep fuel (the closure's scenario)
    "thermal": dict(dx=200.0 / 255, dz=20.0 / 127, dt=0.01, Y_h=2.0,
                    keys=dict(T_inf=300.0, A=1e5, Y_f=10.0, T_max=1500.0)),
}

# Physical constants: the parameter reader's defaults (read by exact()).
CONSTANTS = dict(mu=1.802e-5, T_inf=288.15, H_C=21e6, A=1e9, Y_f=0.0, T_act=18040.8533, T_pc=523.0, c_p=1007.0,
                 k=0.02476, delta=0.1, rho_inf=1.225, g=-9.807, C_s=0.2, Pr=0.7329, T_min=288.15, T_max=2500.0,
                 T_dead=288.15, tol=1e-10, iters=50)
SIGMA, A_VD = 5.670374419e-8, 26.0

# Members of an ensemble: pairs of grids of three sizes, as an uneven
# ensemble of forecasts holds them.
ENSEMBLE_GRIDS = ((64, 64, 32), (128, 128, 64), (256, 256, 64))

TRAIN_ROWS = 100_000


def listed():
    return [
        # the smallest forecast: every launch and wait counts
        dict(name="small_fp64", kind="run", setup="hill", precision="fp64", Nx=24, Ny=20, Nz=16, steps=5),
        # the small quick-look grid, in both precisions
        dict(name="flat64_fp64", kind="run", setup="flat", precision="fp64", Nx=64, Ny=64, Nz=32, steps=20),
        dict(name="flat64_mixed", kind="run", setup="flat", precision="mixed", Nx=64, Ny=64, Nz=32, steps=40),
        # node counts as people choose them, not as transforms like them
        dict(name="odd_fp64", kind="run", setup="hill", precision="fp64", Nx=100, Ny=80, Nz=50, steps=10),
        dict(name="odd_mixed", kind="run", setup="hill", precision="mixed", Nx=201, Ny=151, Nz=81, steps=10),
        # an ordinary terrain forecast
        dict(name="mid_fp64", kind="run", setup="hill", precision="fp64", Nx=128, Ny=128, Nz=64, steps=10),
        # production size, in both precisions
        dict(name="hill256_fp64", kind="run", setup="hill", precision="fp64", Nx=256, Ny=256, Nz=128, steps=10),
        dict(name="hill256_mixed", kind="run", setup="hill", precision="mixed", Nx=256, Ny=256, Nz=128, steps=20),
        # production size with the learned closure on most nodes
        dict(name="closure256_mixed", kind="run", setup="thermal", precision="mixed", closure=True, Nx=256, Ny=256,
             Nz=128, steps=20),
        # a forecast ensemble of uneven grids
        dict(name="ensemble_mixed", kind="ensemble", per_grid=2, steps=30),
        # closure training in its own batches, and scoring of rows with it
        dict(name="train", kind="train", batch=8192, steps=60),
        dict(name="eval", kind="eval", rows=100_000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("run", "ensemble", "train", "eval"), (80, 6, 7, 7))[0]
    if kind == "ensemble":
        return dict(kind=kind, per_grid=rng.choice((1, 2)), steps=rng.randrange(4, 21))
    if kind == "train":
        return dict(kind=kind, batch=_log_int(rng, 256, 32768), steps=rng.randrange(8, 49))
    if kind == "eval":
        return dict(kind=kind, rows=_log_int(rng, 100, 100_000))
    c = dict(kind=kind, setup=rng.choice(("hill", "hill", "flat", "thermal")),
             precision=rng.choice(("fp64", "fp64", "mixed")), Nx=_log_int(rng, 16, 256), Ny=_log_int(rng, 16, 256),
             Nz=_log_int(rng, 12, 128))
    if c["precision"] == "mixed" and c["setup"] == "thermal":
        c["closure"] = rng.random() < 0.6
    if rng.random() < 0.2:
        c["method"] = "RK2"
    nodes = c["Nx"] * c["Ny"] * c["Nz"]
    c["steps"] = max(2, min(20, int(1e7 / nodes)))
    return c


# ------------------------------------------------------------- inputs ----


class Grid:
    """Grid, terrain and fuel depth of one run, and the parameter-file keys
    that give the solver the same."""

    def __init__(self, setup, Nx, Ny, Nz, steps, method="RK4"):
        s = SETUPS[setup]
        self.setup, self.Nx, self.Ny, self.Nz, self.steps, self.method = setup, Nx, Ny, Nz, steps, method
        self.Lx, self.Ly, self.Lz = s["dx"] * (Nx - 1), s["dx"] * (Ny - 1), s["dz"] * (Nz - 1)
        self.dx, self.dy, self.dz = self.Lx / (Nx - 1), self.Ly / (Ny - 1), self.Lz / (Nz - 1)
        self.t_max = s["dt"] * steps
        self.dt = self.t_max / steps
        self.x, self.y, self.z = (np.arange(n) * h for n, h in ((Nx, self.dx), (Ny, self.dy), (Nz, self.dz)))
        self.hill = dict(height=0.35 * self.Lz, x=0.5 * self.Lx, y=0.5 * self.Ly, length=0.18 * self.Lx,
                         width=0.18 * self.Ly)
        self.topo = np.zeros((Nx, Ny))
        if setup == "hill":
            h = self.hill
            ex, ey = ((self.x - h["x"]) / h["length"]) ** 2, ((self.y - h["y"]) / h["width"]) ** 2
            self.topo = h["height"] * np.exp(-ex[:, None] - ey[None, :])
        dzk = np.append(np.diff(self.z), self.z[-1] - self.z[-2])
        k = np.arange(Nz)
        inside = (self.topo[..., None] - dzk <= self.z) & (self.z <= self.topo[..., None])
        self.cut = np.where(inside, k, 0).max(-1)
        self.nzy = np.where(self.z <= self.topo[..., None] + s["Y_h"], k + 1, 0).max(-1)
        self.Nzm = int(self.nzy.max())
        self.const = dict(CONSTANTS, **s["keys"])
        self.keys = dict(Nx=Nx, Ny=Ny, Nz=Nz, Nt=steps, NT=steps, x_min=0.0, x_max=self.Lx, y_min=0.0, y_max=self.Ly,
                         z_min=0.0, z_max=self.Lz, t_min=0.0, t_max=self.t_max, z_domain=0, method=method,
                         U0_type="power_law", z_r=2.0, alpha_u=1.0 / 7.0, u_r=5.0, T0_shape="parallelepiped",
                         T_0=1000.0, p_top=0.0, time_step_log=0, Y_h=s["Y_h"], Y0_x_start=0.0, Y0_x_end=self.Lx,
                         Y0_y_start=0.0, Y0_y_end=self.Ly, Y0_xa=1.0, Y0_ya=1.0, **s["keys"])
        if setup == "hill":
            self.keys.update(topo_shape="hill", hill_center_x=h["x"], hill_center_y=h["y"], hill_length=h["length"],
                             hill_width=h["width"], hill_height=h["height"])
        else:
            self.keys["topo_shape"] = "flat"

    def params(self):
        """The Parameters structure, as a program reads it from its file."""
        d = tempfile.mkdtemp(prefix="wfp", dir="/tmp")
        path = os.path.join(d, "case.txt")
        with open(path, "w") as f:
            for key, v in self.keys.items():
                f.write("%s = %s\n" % (key, repr(float(v)) if isinstance(v, float) else v))
        p = api.read_parameters(path, output_root=os.path.join(d, "o"))
        shutil.rmtree(d, ignore_errors=True)
        return p

    def initial(self, seed):
        """u, v, w, T, Y (float64, z fastest) of a seeded initial state: a
        power-law wind with gusts, the scenario's hot gas and fuel load."""
        rng = np.random.default_rng([seed, self.Nx, self.Ny, self.Nz])
        sh = (self.Nx, self.Ny, self.Nz)
        speed = rng.uniform(4.0, 7.0)
        turn = math.radians(rng.uniform(-30.0, 30.0)) if self.setup == "flat" else 0.0
        wind = speed * (self.z / 2.0) ** (1.0 / 7.0)
        vel = [np.broadcast_to(f * wind, sh).copy() for f in (math.cos(turn), math.sin(turn), 0.0)]
        zeta = self.z / self.Lz
        for f in vel:  # gusts: a few long waves, 0.3 m/s, zero on the ground and on top
            for _ in range(3):
                m, n, q = rng.integers(1, 5), rng.integers(1, 5), rng.integers(1, 4)
                ph = 2 * np.pi * (m * self.x[:, None] / self.Lx + n * self.y[None, :] / self.Ly) + rng.uniform(0, 6.28)
                f += (0.3 * np.cos(ph))[..., None] * np.sin(np.pi * q * zeta)
        T = np.full(sh, self.const["T_inf"])
        deep = self.z[None, None, :] <= self.topo[..., None]
        if self.setup == "hill":  # a line across y
            at, half, up = rng.uniform(0.2, 0.4) * self.Lx, max(1.0, self.dx), 1.0
            hot = np.broadcast_to(np.abs(self.x - at)[:, None] <= half, sh[:2])
        elif self.setup == "flat":  # a block upwind
            at, across = rng.uniform(0.1, 0.33) * self.Lx, rng.uniform(0.2, 0.8) * self.Ly
            hot, up = (np.abs(self.x - at)[:, None] <= 4.0) & (np.abs(self.y - across)[None, :] <= 4.0), 2.0
        else:  # a line segment
            at, half, up = rng.uniform(0.15, 0.4) * self.Lx, max(1.0, self.dx), 2.0
            hot = (np.abs(self.x - at)[:, None] <= half) & (np.abs(self.y / self.Ly - 0.5)[None, :] <= 0.25)
        deep = self.z[None, None, :] <= self.topo[..., None] + up
        T[hot[..., None] & deep] = 1000.0
        Y = rng.uniform(0.8, 1.0, sh[:2] + (self.Nzm,)) if self.setup == "hill" else np.ones(sh[:2] + (self.Nzm,))
        Y[np.arange(self.Nzm) >= self.nzy[..., None]] = 0.0
        dead = np.arange(self.Nz) < self.cut[..., None]
        for f in vel:
            f[dead] = 0.0
        T[dead] = self.const["T_dead"]
        Y[dead[..., :self.Nzm]] = 0.0
        return vel + [T, Y]


def _grid(case):
    return Grid(case["setup"], case["Nx"], case["Ny"], case["Nz"], case["steps"], case.get("method", "RK4"))


def _members(case):
    return [Grid("flat", *g, case["steps"]) for g in ENSEMBLE_GRIDS for _ in range(case["per_grid"])]


def _pack(fields):
    y = np.concatenate([f.ravel() for f in fields])
    return y, np.zeros(fields[0].size)


def _rows(block, n, seed):
    """Feature rows around the closure's training data, most of them inside
    its range, with target viscosities that grow with the strain."""
    b = closure.unpack(block)
    rng = np.random.default_rng([seed, n])
    lo, hi = b["lo"].astype(np.float64), b["hi"].astype(np.float64)
    std = np.where(b["inv_std"] > 0, 1.0 / np.maximum(b["inv_std"], 1e-30), 0.0)
    f = b["mean"] + std * rng.standard_normal((n, 12))
    most = rng.random(n) < 0.95
    f[most] = np.clip(f[most], lo, hi)
    strain = np.sqrt((f[:, :9] ** 2).sum(1))
    nu = b["out_scale"] * np.minimum(1.0, 0.3 * strain / strain.mean())
    return f, nu


def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        g = _grid(case)
        y0, p0 = _pack(g.initial(seed))
        solver = api.Solver(g.params(), case["precision"])
        if case.get("closure"):
            solver.set_closure(closure.load(CLOSURE_FILE))
        # the copy a program keeps of the forecast: the mixed form's fields are single precision, and so is theirs
        kept = torch.zeros(y0.size + p0.size, dtype=torch.float32 if case["precision"] == "mixed" else torch.float64)
        return dict(kind=kind, solver=solver, y0=y0, p0=p0, steps=case["steps"], kept=kept)
    if kind == "ensemble":
        members = _members(case)
        states = [_pack(g.initial(seed + 1000 * i)) for i, g in enumerate(members)]
        return dict(kind=kind, ensemble=api.Ensemble([g.params() for g in members]), states=states, steps=case["steps"])
    block = closure.load(CLOSURE_FILE)
    if kind == "train":
        rows = max(TRAIN_ROWS, 2 * case["batch"])
        start = block.copy()
        start[48:-2] *= 0.9  # a network still to be fitted
        return dict(kind=kind, trainer=api.ClosureTrainer(start, *_rows(block, rows, seed)), steps=case["steps"],
                    batch=case["batch"])
    return dict(kind=kind, block=block, features=_rows(block, case["rows"], seed)[0])


# ---------------------------------------------------------------- runs ----


def _snapshot(solver):
    """The state and p as the C driver takes them for its files: converted
    and downloaded into the solver's pinned host buffer."""
    lib, y, p = api.lib(), _abi.DBL_P(), _abi.DBL_P()
    rc = lib.wf_solver_checkpoint_begin(solver.handle)
    rc = rc or lib.wf_solver_checkpoint_wait(solver.handle, ctypes.byref(y), ctypes.byref(p))
    if rc:
        raise RuntimeError("snapshot: %s" % lib.wf_last_error())
    # the two arrays follow one another in the one buffer
    return np.ctypeslib.as_array(y, shape=(solver.params.S + solver.params.N,))


def _fields(params, flat):
    N, S = params.N, params.S
    return dict({n: flat[q * N:(q + 1) * N] for q, n in enumerate("uvwT")}, Y=flat[4 * N:S], p=flat[S:S + N])


def run(state):
    if state["kind"] == "run":
        solver = state["solver"]
        solver.set_state(state["y0"], state["p0"])
        solver.step(1, state["steps"])
        # the pinned buffer is the solver's own and is used again: the program copies what it keeps
        return _fields(solver.params, state["kept"].copy_(torch.from_numpy(_snapshot(solver))))
    if state["kind"] == "ensemble":
        e = state["ensemble"]
        for i, (y0, p0) in enumerate(state["states"]):
            e.set_state(i, y0, p0)
        e.step(1, state["steps"])
        out = []
        for i, prm in enumerate(e.params):
            y, p = e.get_state(i)
            y, p = torch.from_numpy(y).float(), torch.from_numpy(p).float()
            out.append(dict(_fields(prm, y), p=p))
        return out
    if state["kind"] == "train":
        state["trainer"].train(state["steps"], state["batch"], 1e-3)
        return state["trainer"].params()[48:-1]
    return list(api.closure_eval(state["block"], state["features"]))


# ---------------------------------------------------------------- work ----


def _run_work(g, precision, closed):
    N, phi = g.Nx * g.Ny * g.Nz, g.Nzm / g.Nz
    size, solves = (8, 50) if precision == "fp64" else (4, 20)
    if g.setup != "hill":
        solves *= 0.4
    stages = 2 if g.method == "RK2" else 4
    # a stage reads its input, y_n and the running combination and writes two
    # of them; a solve reads f's operands, writes p and moves the half
    # spectrum in and out of its three passes; the projection reads and writes
    # the state; the state crosses the bus once each way
    per_step = size * ((20 + 5 * phi) * stages + 12 + 15 * (solves - 1))
    flops = stages * 700 + solves * (60 + 5 * math.log2((g.Nx - 1) * (g.Ny - 1))) + 60
    if closed:
        flops += stages * 2 * (12 * 64 + 64 * 64 + 64)
    return N * (per_step * g.steps + 2 * 8 * (5 + phi)), N * flops * g.steps


def work(case):
    kind = case["kind"]
    if kind == "run":
        b, f = _run_work(_grid(case), case["precision"], case.get("closure"))
    elif kind == "ensemble":
        parts = [_run_work(g, "mixed", False) for g in _members(case)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    else:
        rows = case["rows"] if kind == "eval" else case["batch"] * case["steps"]
        net = 12 * 64 + 64 * 64 + 64
        b = rows * (12 * 8 + 12) if kind == "eval" else rows * 28 + case["steps"] * 4 * 5106 * 5
        f = rows * 2 * net * (1 if kind == "eval" else 3)
    return {"bytes": b, "flops": f}


# --------------------------------------------------------------- exact ----


def _network(block, f):
    """nu_t of raw inputs f (n x 12) in the block's dtype of 64 bits."""
    b = {k: torch.as_tensor(v, dtype=torch.float64, device=f.device) for k, v in closure.unpack(block).items()}
    act = lambda h: h * torch.sigmoid(1.702 * h)  # noqa: E731
    out = torch.empty(f.shape[0], dtype=torch.float64, device=f.device)
    for at in range(0, f.shape[0], 1 << 20):
        part = f[at:at + (1 << 20)]
        h = act((part - b["mean"]) * b["inv_std"] @ b["W1"].T + b["b1"])
        h = act(h @ b["W2"].T + b["b2"])
        out[at:at + part.shape[0]] = b["out_scale"] * torch.nn.functional.softplus(h @ b["w3"] + b["b3"], threshold=50)
    inside = ((f >= b["lo"]) & (f <= b["hi"])).all(1)
    return out, inside


class Exact:
    """The time step in 64 bits on full (Nx, Ny, Nz) tensors."""

    def __init__(self, g, block=None):
        self.g, self.block = g, block
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=self.dev)  # noqa: E731
        Nz, z = g.Nz, g.z
        h = np.diff(z)
        D1, D2, F, B = (np.zeros((Nz, Nz)) for _ in range(4))
        for k in range(Nz):
            if k <= Nz - 3:
                F[k, k:k + 3] = (-(2 * h[k] + h[k + 1]) / (h[k] * (h[k] + h[k + 1])),
                                 (h[k] + h[k + 1]) / (h[k] * h[k + 1]), -h[k] / (h[k + 1] * (h[k] + h[k + 1])))
            if k >= 2:
                a, b = h[k - 2], h[k - 1]
                B[k, k - 2:k + 1] = b / (a * (a + b)), -(a + b) / (a * b), (a + 2 * b) / (b * (a + b))
        for k in range(1, Nz - 1):
            a, b = h[k - 1], h[k]
            D1[k, [k - 1, k + 1]] = -1 / (a + b), 1 / (a + b)
            D2[k, k - 1:k + 2] = 2 / (a * (a + b)), -2 / (a * b), 2 / (b * (a + b))
        D1[0], D1[-1] = F[0], B[-1]
        a, b, c = h[:3]
        D2[0, :4] = ((6 * a + 4 * b + 2 * c) / (a * (a + b) * (a + b + c)), -(4 * a + 4 * b + 2 * c) / (a * b * (b + c)),
                     (4 * a + 2 * b + 2 * c) / (b * c * (a + b)), -(4 * a + 2 * b) / (c * (b + c) * (a + b + c)))
        c, b, a = h[-3:]
        D2[-1, -4:] = (-(2 * b + 4 * a) / (c * (c + b) * (c + b + a)), (2 * c + 2 * b + 4 * a) / (c * b * (b + a)),
                       -(2 * c + 4 * b + 4 * a) / (a * b * (c + b)), (2 * c + 4 * b + 6 * a) / (a * (b + a) * (c + b + a)))
        up, down = F.copy(), B.copy()  # the difference taken for w < 0 and w > 0
        up[Nz - 2:], down[:2] = B[Nz - 2:], F[:2]
        self.D1, self.D2, self.up, self.down = t(D1), t(D2), t(up), t(down)
        self.idx = {(ax, d): torch.as_tensor((np.arange(n) + d) % (n - 1), device=self.dev)
                    for ax, n in ((0, g.Nx), (1, g.Ny)) for d in (-2, -1, 1, 2)}
        self.cut, self.nzy, self.z = t(g.cut)[..., None], t(g.nzy)[..., None], t(z)
        k = torch.arange(Nz, device=self.dev)
        self.dead, self.fuel, self.k = k < self.cut, k < self.nzy, k
        self.zibm = (self.z - t(g.topo)[..., None]).clamp_min(0)
        self.h = h
        dzk = np.append(h, h[-1])
        self.Delta = t((g.dx * g.dy * dzk) ** (1.0 / 3.0))
        # tridiagonal systems of the half spectrum (ky halved), pivots and multipliers
        nx, ny, nz = g.Nx - 1, g.Ny - 1, Nz - 1
        kx, ky = 2 * np.pi * np.fft.fftfreq(nx, 1 / nx) / g.Lx, 2 * np.pi * np.arange(ny // 2 + 1) / g.Ly
        K2 = t(kx)[:, None] ** 2 + t(ky)[None, :] ** 2
        lower = 2 / (h[:-1] * (h[:-1] + h[1:]))
        self.c = [(h[0] + h[1]) / (h[0] * h[1]) - 0.5 * h[0] * K2 - 1 / h[1]]
        self.u, self.l = [torch.full_like(K2, -1.0 / h[0])], []
        for r in range(1, nz):
            diag = -(K2 + 2 / (h[r - 1] * h[r]))
            self.l.append(lower[r - 1] / self.u[-1])
            self.u.append(diag - self.l[-1] * self.c[-1])
            self.c.append(2 / (h[r] * (h[r - 1] + h[r])))
        self.l, self.u = [[v[..., None] for v in a] for a in (self.l, self.u)]
        self.top_div = 2 / (h[-1] * (h[-2] + h[-1]))

    def at(self, f, ax, d):
        return f.index_select(ax, self.idx[ax, d])

    def dd(self, f, ax):
        return (self.at(f, ax, 1) - self.at(f, ax, -1)) / (2 * (self.g.dx, self.g.dy)[ax])

    def zz(self, f, D):
        return (f.reshape(-1, self.g.Nz) @ D.T).reshape(f.shape)

    def lap(self, f):
        g = self.g
        return ((self.at(f, 0, 1) - 2 * f + self.at(f, 0, -1)) / g.dx ** 2 +
                (self.at(f, 1, 1) - 2 * f + self.at(f, 1, -1)) / g.dy ** 2 + self.zz(f, self.D2))

    def conditions(self, s):
        """Cut, top and dead nodes, in place."""
        u, v, w, T, Y = s
        h = torch.as_tensor(self.h, device=self.dev)
        h0, h1 = h[self.cut], h[self.cut + 1]
        pick = lambda f, d: f.gather(2, self.cut + d)  # noqa: E731
        edge = lambda a, b: ((h0 + h1) ** 2 * a - h0 ** 2 * b) / (h1 * (2 * h0 + h1))  # noqa: E731
        Tc = edge(pick(T, 1), pick(T, 2))
        Yin = torch.where(self.fuel, Y, 0.0)
        Yc = torch.where(self.cut < self.nzy, edge(pick(Yin, 1), pick(Yin, 2)), pick(Y, 0))
        for f in (u, v, w):
            f.scatter_(2, self.cut, 0.0)
        T.scatter_(2, self.cut, Tc)
        Y.scatter_(2, self.cut, Yc)
        a, b = self.h[-1], self.h[-2]
        for f in (u, v, w, T):
            f[..., -1] = ((b + a) ** 2 * f[..., -2] - a ** 2 * f[..., -3]) / (b * (b + 2 * a))
        for f in (u, v, w):
            f[self.dead] = 0.0
        T[self.dead] = self.g.const["T_dead"]
        Y[self.dead & self.fuel] = 0.0

    def heat(self, T, Y):
        c = self.g.const
        K = torch.where(T > c["T_pc"], c["A"] * torch.exp(-c["T_act"] / T), 0.0)
        Yn = torch.where(self.fuel, Y, 0.0)
        return K, Yn, c["H_C"] * Yn * K / c["c_p"]

    def phi(self, s):
        g, c = self.g, self.g.const
        u, v, w, T, Y = s
        grad = [[self.dd(f, 0), self.dd(f, 1), self.zz(f, self.D1)] for f in (u, v, w, T)]
        laps = [self.lap(f) for f in (u, v, w, T)]
        rho = c["T_inf"] * c["rho_inf"] / T
        K, Yn, q = self.heat(T, Y)
        adv = []
        for f in (u, v, w, T):
            tot = 0.0
            for ax, vel, h in ((0, u, g.dx), (1, v, g.dy)):
                back = (3 * f - 4 * self.at(f, ax, -1) + self.at(f, ax, -2)) / (2 * h)
                ahead = (-3 * f + 4 * self.at(f, ax, 1) - self.at(f, ax, 2)) / (2 * h)
                tot = tot + vel.clamp_min(0) * back + vel.clamp_max(0) * ahead
            adv.append(tot + w.clamp_min(0) * self.zz(f, self.down) + w.clamp_max(0) * self.zz(f, self.up))
        gT = grad[3]
        g2 = gT[0] ** 2 + gT[1] ** 2 + gT[2] ** 2
        cond = (12 * SIGMA * c["delta"] * T ** 2 * g2 + (c["k"] + 4 * SIGMA * c["delta"] * T ** 3) * laps[3]) \
            / (rho * c["c_p"]) + q
        nu = c["mu"] / rho
        G = grad[:3]
        S = [[0.5 * (G[a][b] + G[b][a]) for b in range(3)] for a in range(3)]
        div = G[0][0] + G[1][1] + G[2][2]
        mod = 2 * (G[0][0] ** 2 + G[1][1] ** 2 + G[2][2] ** 2)
        for a, b in ((0, 1), (0, 2), (1, 2)):
            mod = mod + (G[a][b] + G[b][a]) ** 2
        for a in range(3):
            S[a][a] = G[a][a] - div / 3
        mu_t = rho * (c["C_s"] * self.Delta) ** 2 * torch.sqrt(mod)
        learned = None
        if self.block is not None:
            f = torch.stack([x.reshape(-1) for r in G for x in r] +
                            [torch.sqrt(g2).reshape(-1), self.Delta.expand_as(T).reshape(-1), Yn.reshape(-1)], 1)
            nu_t, learned = _network(self.block, f)
            del f
            learned = learned.reshape(T.shape)
            mu_t = torch.where(learned, rho * nu_t.reshape(T.shape), mu_t)
        divU = nu * cond / T
        tau = c["mu"] * torch.sqrt(G[0][2][..., 0] ** 2 + G[1][2][..., 0] ** 2)
        utau = torch.sqrt(tau / rho[..., 0])[..., None]
        yes = lambda m, d: m if learned is None else torch.where(d, 1.0, m)  # noqa: E731

        def damped(move):
            """mu_t at a neighbour, damped with the node's own viscosity."""
            fw = 1 - torch.exp(-move(self.zibm) * move(utau) / A_VD / nu)
            return move(mu_t) * yes(fw ** 2, None if learned is None else move(learned))

        def shifted(k):  # neighbour in z (the edge planes are overwritten by the conditions)
            j = (self.k + k).clamp(0, g.Nz - 1)
            return lambda f: f if f.shape[2] == 1 else f.index_select(2, j)

        hz = torch.as_tensor(np.concatenate([[1.0], self.h[:-1] + self.h[1:], [1.0]]), device=self.dev)
        m0 = damped(lambda f: f)
        gm = [(damped(lambda f: self.at(f, 0, 1)) - damped(lambda f: self.at(f, 0, -1))) / (2 * g.dx),
              (damped(lambda f: self.at(f, 1, 1)) - damped(lambda f: self.at(f, 1, -1))) / (2 * g.dy),
              (damped(shifted(1)) - damped(shifted(-1))) / hz]
        part = lambda f, ax: self.dd(f, ax) if ax < 2 else self.zz(f, self.D1)  # noqa: E731
        out = []
        for a in range(3):
            divS = part(S[0][a], 0) + part(S[1][a], 1) + part(S[2][a], 2)
            sgs = 2 * (gm[0] * S[0][a] + gm[1] * S[1][a] + gm[2] * S[2][a] + m0 * divS) / rho
            out.append(nu * laps[a] - adv[a] + sgs + part(divU, a) / 3)
        out[2] = out[2] + c["g"] * (rho - c["rho_inf"]) / rho
        out.append(cond - adv[3] + (gm[0] * gT[0] + gm[1] * gT[1] + gm[2] * gT[2] + m0 * laps[3]) / (rho * c["Pr"]))
        out.append(-c["Y_f"] * K * Yn)
        self.conditions(out)
        return out

    def solve(self, f, top):
        """p on the unique nodes from f (nz planes, plane 0 unused) and the top plane."""
        g = self.g
        d = torch.view_as_real(torch.fft.rfft2(f))
        d[0] = 0.5 * self.h[0] * d[1]
        d[-1] -= torch.view_as_real(torch.fft.rfft2(top)) / self.top_div
        for r in range(1, len(self.u)):
            d[r].addcmul_(d[r - 1], self.l[r - 1], value=-1)
        d[-1] /= self.u[-1]
        for r in range(len(self.u) - 2, -1, -1):
            if r:
                d[r].add_(d[r + 1], alpha=-float(self.c[r]))
            else:
                d[r].addcmul_(d[r + 1], self.c[0][..., None], value=-1)
            d[r] /= self.u[r]
        return torch.fft.irfft2(torch.view_as_complex(d), s=(g.Nx - 1, g.Ny - 1))

    def pressure(self, s, Tn, p):
        g, c = self.g, self.g.const
        u, v, w, T, Y = s
        rho = c["T_inf"] * c["rho_inf"] / Tn
        gT = [self.dd(T, 0), self.dd(T, 1), self.zz(T, self.D1)]
        _, _, q = self.heat(T, Y)
        divT = (12 * SIGMA * c["delta"] * T ** 2 * (gT[0] ** 2 + gT[1] ** 2 + gT[2] ** 2) +
                (c["k"] + 4 * SIGMA * c["delta"] * T ** 3) * self.lap(T)) / (c["T_inf"] * c["rho_inf"] * c["c_p"]) + q / T
        part = lambda f, ax: self.dd(f, ax) if ax < 2 else self.zz(f, self.D1)  # noqa: E731
        A = rho * (part(u, 0) + part(v, 1) + part(w, 2) - divT) / g.dt
        gr = [part(rho, a) / rho for a in range(3)]
        for _ in range(c["iters"]):
            f = A
            for a in range(3):
                f = f + gr[a] * part(p, a)
            f = f[:-1, :-1, :-1].permute(2, 0, 1).contiguous()
            new = self.solve(f, p[:-1, :-1, -1].contiguous()).permute(1, 2, 0)
            old, p = p, p.clone()
            p[:-1, :-1, :-1] = new
            p[-1] = p[0]
            p[:, -1] = p[:, 0]
            if float((p - old).abs().max()) <= c["tol"]:
                break
        return p, rho, [part(p, a) for a in range(3)]

    def run(self, fields):
        g, c = self.g, self.g.const
        y = [torch.as_tensor(f, device=self.dev) for f in fields]
        Y = torch.zeros((g.Nx, g.Ny, g.Nz), dtype=torch.float64, device=self.dev)
        Y[..., :g.Nzm] = y[4]
        y[4] = Y
        p = torch.zeros_like(y[0])
        go = lambda k, a: [f + a * d for f, d in zip(y, k)]  # noqa: E731
        for _ in range(g.steps):
            k1 = self.phi(y)
            if g.method == "RK4":
                k2 = self.phi(go(k1, g.dt / 2))
                k3 = self.phi(go(k2, g.dt / 2))
                k4 = self.phi(go(k3, g.dt))
                s = [f + g.dt / 6 * (a + 2 * b + 2 * d + e) for f, a, b, d, e in zip(y, k1, k2, k3, k4)]
            else:
                k2 = self.phi(go(k1, g.dt))
                s = [f + g.dt / 2 * (a + b) for f, a, b in zip(y, k1, k2)]
            p, rho, gp = self.pressure(s, y[3], p)
            for a in range(3):
                s[a] = s[a] - g.dt * gp[a] / rho
            self.conditions(s)
            s[3].clamp_(c["T_min"], c["T_max"])
            s[4][..., :g.Nzm].clamp_(0.0, 1.0)
            y = s
        out = {n: f.reshape(-1).cpu() for n, f in zip("uvwT", y)}
        return dict(out, Y=y[4][..., :g.Nzm].reshape(-1).cpu(), p=p.reshape(-1).cpu())


def _exact_train(case, seed):
    block = closure.load(CLOSURE_FILE)
    f, nu = _rows(block, max(TRAIN_ROWS, 2 * case["batch"]), seed)
    b = {k: torch.as_tensor(v, dtype=torch.float64) for k, v in closure.unpack(block).items()}
    x, t = (torch.as_tensor(f) - b["mean"]) * b["inv_std"], torch.as_tensor(nu) / b["out_scale"]
    names = ("W1", "b1", "W2", "b2", "w3", "b3")
    prm = [b[n] * (0.9 if n != "b3" else 1.0) for n in names]
    m, s, at = [0.0] * 6, [0.0] * 6, 0
    for step in range(1, case["steps"] + 1):
        if at + case["batch"] > x.shape[0]:
            at = 0
        prm = [q.detach().requires_grad_() for q in prm]
        h = x[at:at + case["batch"]] @ prm[0].T + prm[1]
        h = (h * torch.sigmoid(1.702 * h)) @ prm[2].T + prm[3]
        z = (h * torch.sigmoid(1.702 * h)) @ prm[4] + prm[5]
        loss = ((torch.nn.functional.softplus(z, threshold=50) - t[at:at + case["batch"]]) ** 2).mean()
        grad = torch.autograd.grad(loss, prm)
        m = [0.9 * a + 0.1 * d for a, d in zip(m, grad)]
        s = [0.999 * a + 0.001 * d * d for a, d in zip(s, grad)]
        prm = [q.detach() - 1e-3 * (a / (1 - 0.9 ** step)) / (torch.sqrt(d / (1 - 0.999 ** step)) + 1e-8)
               for q, a, d in zip(prm, m, s)]
        at += case["batch"]
    return torch.cat([q.reshape(-1) for q in prm])


def exact(case, seed):
    kind = case["kind"]
    if kind == "run":
        g = _grid(case)
        return Exact(g, closure.load(CLOSURE_FILE) if case.get("closure") else None).run(g.initial(seed))
    if kind == "ensemble":  # the largest grids' runs would take minutes
        return [Exact(g).run(g.initial(seed + 1000 * i)) if g.Nx < 128 else None for i, g in enumerate(_members(case))]
    if kind == "train":
        return _exact_train(case, seed)
    block = closure.load(CLOSURE_FILE)
    return [_network(block, torch.as_tensor(_rows(block, case["rows"], seed)[0]))[0], None]
