"""The work whose speed counts: time steps of dynamic-rupture simulations and
the fit of the learned Newton guess, through the public entry points
(``dynfd3dcuda_amd.Solver``, ``dynfd3dcuda_amd.mlp``).

listed() are the cases, draw() gives further ones of the same ranges,
prepare() makes the inputs and the solver that a program has in hand before
it steps, run() is one pass, work() what a pass cannot do without, and
exact() the 64-bit values of the cases whose mathematics fits in a page of
torch.
"""
import math
import os
import shutil
import tempfile
import weakref

import numpy as np
import torch

import dynfd3dcuda_amd as dyn
from dynfd3dcuda_amd import configs, mlp

NETWORK = os.path.join(os.path.dirname(dyn.__file__), "data", "newton_guess_4x64x64x1.f32")

# A whole volume is put in and read back through host copies: programs do
# that on grids up to about this many points (a 400 x 300 x 200 wavefield is
# 0.9 GB); larger runs start at rest and record their fault.
VOLUME_POINTS = 30_000_000

# What a run records of its fault at every output step.  The solver
# accumulates slip and state in 64 bits; a record holds them in 32, as the
# output files do.
RECORD = ("Vs1", "Vs2", "Tn", "Ts1", "Ts2", "slip", "State", "init_t0", "rup_sensor", "FW")


def listed():
    base = {"kind": "sw", "grid": "curved", "media": "layers", "metric": 0, "pml": 20, "cerjan": 0, "smooth": 0,
            "newton": 0, "steps": 8, "outputs": 0}
    return [
        # the smallest rupture grid of the test suite, one step at a time: a
        # program that looks at its fault after every step
        dict(base, name="sw_30x80x50_one_step", nx=30, ny=80, nz=50, media="halves", pml=8, steps=1),
        # waves without a fault: a given wavefield propagates through two
        # half spaces under a free surface (odd sizes)
        dict(base, name="wave_97x125x81", kind="wave", grid="flat", media="halves", nx=97, ny=125, nz=81, pml=10,
             steps=2),
        # the plain method on its small grid: flat, Cerjan sponge
        dict(base, name="sw_flat_100x200x100", grid="flat", media="halves", nx=100, ny=200, nz=100, pml=0, cerjan=20),
        # the curved slip-weakening workload
        dict(base, name="sw_curved_400x300x200", nx=400, ny=300, nz=200),
        # the curved rate-and-state workload with the learned Newton guess
        dict(base, name="rs_curved_400x300x200", kind="rs", newton=2, nx=400, ny=300, nz=200),
        # the large mixed-precision workload on half its fault-normal extent
        # (three such runs fit one card)
        dict(base, name="rs_large_800x1000x500", kind="rs", newton=2, metric=2, nx=800, ny=1000, nz=500),
        # thermal pressurization with the strongly weakening slip law, odd sizes
        dict(base, name="tp_151x211x133", kind="tp", nx=151, ny=211, nz=133, steps=4),
        # a three-dimensional velocity model with the fault tractions
        # smoothed after every step, odd sizes
        dict(base, name="sw_media3d_smooth_203x281x147", media="volume", smooth=1, nx=203, ny=281, nz=147),
        # the metric stored in plain bfloat16, the reference's Newton rule, odd sizes
        dict(base, name="rs_bf16_251x187x143", kind="rs", metric=1, nx=251, ny=187, nz=143),
        # a job of ten steps that writes one record of its output files
        dict(base, name="sw_outputs_200x160x120", nx=200, ny=160, nz=120, steps=10, outputs=1),
        # gradient and predictions of the guess network on collected samples
        {"name": "guess_60000", "kind": "guess", "samples": 60_000},
    ]


def draw(rng):
    """A case of the same ranges: grids of 0.2 to 400 million points (their
    logarithm spread evenly, most sizes odd) with every fault law, metric
    form, medium and absorbing layer; now and then a sample set."""
    if rng.random() < 0.1:
        return {"kind": "guess", "samples": int(math.exp(rng.uniform(math.log(2_000), math.log(500_000))))}
    kind = rng.choice(["wave", "sw", "sw", "rs", "rs", "tp"])
    metric = rng.choice([0, 0, 1, 2, 2])
    # memory follows the metric form (three states fit one card) and the
    # 64-bit diffusion levels of thermal pressurization their fault
    top = {0: 300e6, 1: 350e6, 2: 380e6}[metric]
    points = math.exp(rng.uniform(math.log(0.2e6), math.log(top)))
    side = points ** (1.0 / 3.0)
    nx = max(30, int(side * math.exp(rng.uniform(-0.3, 0.4))))
    ny = max(80, int(side * math.exp(rng.uniform(-0.2, 0.5))))
    nz = max(50, int(points / (nx * ny)))
    small = min(nx, ny, nz)
    layer = 20 if small >= 60 else 12 if small >= 30 else 8
    cerjan = layer if rng.random() < 0.2 else 0
    media = rng.choice(["halves", "layers", "layers", "volume"])
    if media == "volume" and points > VOLUME_POINTS:
        media = "layers"
    outputs = int(kind == "sw" and points < 8e6 and rng.random() < 0.3)
    return {"kind": kind, "grid": "flat" if kind == "wave" else rng.choice(["flat", "curved", "curved"]),
            "media": "halves" if kind == "wave" else media, "metric": metric, "pml": 0 if cerjan else layer,
            "cerjan": cerjan, "smooth": int(kind == "sw" and rng.random() < 0.3),
            "newton": rng.choice([0, 1, 2]) if kind == "rs" else 0, "nx": nx, "ny": ny, "nz": nz,
            "steps": 10 if outputs else 1 if points < 1e6 else rng.choice([2, 4, 8]), "outputs": outputs}


# ---------------------------------------------------------------- inputs

def _points(case):
    return case["nx"] * case["ny"] * case["nz"]


def _spacing(case):
    """Finer grids for larger runs, as in the workloads: 100, 50 and 25 m."""
    return 100.0 if _points(case) < 10e6 else 50.0 if _points(case) < 100e6 else 25.0


def _wavefield(nx, ny, nz, seed):
    """A smooth seeded wavefield [9][nx][nz][ny] on the padded grid (host,
    float32): waves of 12 to 60 cells, velocities of about 0.1 m/s and the
    stresses that go with them; the ghost layers are zero."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rng = np.random.default_rng(seed)
    W = torch.zeros((9, nx, nz, ny), dtype=torch.float32, device=dev)
    for c in range(9):
        f = W[c, 3:-3, 3:-3, 3:-3]
        for _ in range(3):
            x, z, y = (torch.sin(torch.arange(n, dtype=torch.float32, device=dev) * (2 * math.pi / rng.uniform(12, 60))
                                 + rng.uniform(0, 2 * math.pi)) for n in f.shape)
            f += (rng.uniform(0.5, 1.0) * (0.05 if c < 3 else 3e5)) * x[:, None, None] * (z[:, None] * y)
    return W.cpu().numpy()


def _rupture_inputs(case, seed):
    """Parameters and input arrays of one simulation."""
    NX, NY, NZ, kind = case["nx"], case["ny"], case["nz"], case["kind"]
    DH = _spacing(case)
    DT = 6e-5 * DH
    rng = np.random.default_rng(seed)
    curved = case["grid"] == "curved"
    p = configs._params(NX, NY, NZ, DH, DT, 8000, NormalRefine=int(curved), Rupture=int(kind != "wave"),
                        INPORT_GRID_TYPE=int(curved), usePML=int(case["pml"] > 0), PML_N=case["pml"] or 20,
                        useCerjan=int(case["cerjan"] > 0), DAMP_N=case["cerjan"] or 20, MetricBF16=case["metric"],
                        FaultSmooth=case["smooth"], NewtonMode=case["newton"])
    c = {"params": p}
    if case["media"] == "halves":
        p.update({"bi_vp2": 5400.0, "bi_vs2": 3120.0, "bi_rho2": 2600.0})
    elif case["media"] == "layers":
        c["media1d"] = configs.three_layer_media()
    else:
        vs = 3300.0 + 60.0 * rng.standard_normal((8, 8, 8))
        idx = [np.minimum(np.arange(n) * 8 // n, 7) for n in (NX, NZ, NY)]
        vs = vs[np.ix_(*idx)].astype(np.float32)
        c["media3d"] = (vs * np.float32(math.sqrt(3.0)), vs, np.full_like(vs, 2670.0))
    geom = configs.bent_fault_geometry(NY, NZ, DH, 20.0, rng) if curved else configs.flat_geometry(NY, NZ, DH)
    if curved:
        c["geom"] = geom
        c["topo"] = configs.sum_of_gaussians_topography(NX, NY, DH, rng, hmax=500.0)
    if kind == "wave":
        return c
    frame = configs.fault_frame(geom, DH)
    if kind == "sw":
        c["stress"] = configs._sw_stress(NY, NZ, DH, rng, 70e6, 3e6, 1e3, 3.0, frame=frame)
        return c
    L = {"rs": 0.1, "tp": 0.4}[kind]
    p.update({"Friction_type": 1 if kind == "rs" else 3, "RS_V0": 1e-6, "RS_f0": 0.6, "RS_Vini": 1e-12, "RS_L": L,
              "RS_fw": 0.2, "smooth_load_T": 0.5})
    c["stress"] = configs._rs_stress(NY, NZ, DH, rng, frame=frame, L=L)
    if case["newton"]:
        p.update({"NewtonTol": 1e-10, "NewtonFallbackIter": 20})
    if case["newton"] == 2:
        p["NewtonMLP"] = NETWORK
    if kind == "tp":
        p["TP_n"] = 21
        c["stress"]["TP_hy"] = np.full_like(c["stress"]["L"], 2.0 ** -11)
    return c


def _samples(n, seed):
    """Rate-state samples as the trials produce them: the four guess features
    and the log10 slip rate that solves e^u / 2 + u = s."""
    rng = np.random.default_rng(seed)
    s = rng.uniform(-30.0, 60.0, n)
    f = np.stack([np.where(s <= 0, s, np.log1p(np.maximum(s, 0.0))), rng.uniform(0.0, 90.0, n),
                  rng.uniform(-9.0, -2.0, n), rng.uniform(-14.0, 1.0, n)], axis=1).astype(np.float32)
    u = np.where(s <= 0, s, np.log(2.0 * np.maximum(s, 1e-3)))
    for _ in range(40):
        e = np.exp(np.minimum(u, 60.0))
        u = u - (0.5 * e + u - s) / (0.5 * e + 1.0)
    t = f[:, 2] + (u - math.log(2.0)) / math.log(10.0) + 0.02 * rng.standard_normal(n)
    return f, t.astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "guess":
        f, t = _samples(case["samples"], seed)
        return {"case": case, "feat": f, "target": t, "params": mlp.load(NETWORK)}
    c = _rupture_inputs(case, seed)
    state = {"case": case, "it": 0}
    if case["outputs"]:
        out = tempfile.mkdtemp(prefix="rupture_out_")
        c["params"]["OUT"] = out
    s = dyn.Solver(c["params"])
    if case["outputs"]:
        weakref.finalize(s, shutil.rmtree, out, True)
    try:
        configs.apply(c, s)
        if "media3d" in c:
            s.set_media3d(*c["media3d"])
        s.setup()
    except dyn.CgfdmError as e:
        s.close()
        raise MemoryError(str(e)) if "hipMalloc" in str(e) else e
    if _points(case) <= VOLUME_POINTS:
        d = s.dims()
        s.put("W", _wavefield(d["nx"], d["ny"], d["nz"], seed))
    if case["kind"] in ("rs", "tp"):  # half way up the nucleation ramp
        state["it"] = int(0.25 / c["params"]["DT"]) // 8 * 8
    state["solver"], state["out"] = s, c["params"]["OUT"] if case["outputs"] else None
    return state


# ---------------------------------------------------------------- one pass

class Fields(dict):
    """The fields of a solver by name, each read from the device when it is
    looked at: what a step leaves behind is the solver's own state, and a
    program copies the fields it wants when it wants them."""

    def __init__(self, read):
        super().__init__(dict.fromkeys(read))
        self._read = read

    def __getitem__(self, name):
        return self._read[name]()

    def get(self, name, default=None):
        return self[name] if name in self else default

    def values(self):
        return [self[k] for k in self]

    def items(self):
        return [(k, self[k]) for k in self]


def _field(solver, name):
    def read():
        a = solver.get(name)
        return a.astype(np.float32) if a.dtype == np.float64 else a
    return read


def _last_slice(path, shape):
    """Vx, Vy, Vz of the last record of a wave-slice file (its tail; netCDF
    classic files hold big-endian floats)."""
    def read():
        n = 3 * shape[0] * shape[1]
        with open(path, "rb") as f:
            f.seek(-4 * n, os.SEEK_END)
            return np.frombuffer(f.read(4 * n), ">f4").astype(np.float32).reshape(3, *shape)
    return read


def run(state):
    case = state["case"]
    if case["kind"] == "guess":
        loss, grad = mlp.grad(state["params"], state["feat"], state["target"])
        return {"loss": loss, "grad": grad, "log10_rate": mlp.forward(state["params"], state["feat"])}
    s = state["solver"]
    s.run(state["it"], case["steps"], write_outputs=bool(case["outputs"]))
    state["it"] += case["steps"]
    read = {}
    if case["kind"] != "wave":
        read.update((n, _field(s, n)) for n in RECORD)
    if case["kind"] == "tp":
        read.update((n, _field(s, n)) for n in ("TP_T", "TP_P"))
    if _points(case) <= VOLUME_POINTS:
        read["W"] = _field(s, "W")
    if case["outputs"]:
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        for plane, shape in (("xy", (nx, ny)), ("xz", (nx, nz)), ("yz", (nz, ny))):
            read["wave_" + plane] = _last_slice(os.path.join(state["out"], f"wave_{plane}_mpi000000.nc"), shape)
    return Fields(read)


def work(case):
    """Bytes and operations of one pass.  A step of the four-stage scheme
    reads the nine words of each stage's input, the step start where a stage
    needs it and the accumulator, and writes the stage value and the
    accumulator: 126 words a point, and in each stage the metric and media
    words as stored.  An absorbing point moves its auxiliary words besides
    (153 bytes a face and stage).  Each stage takes nine derivatives along
    three axes (9 operations each) and about 150 operations more."""
    if case["kind"] == "guess":
        n = case["samples"]
        net = 2 * (4 * 64 + 64 * 64 + 64)
        return {"bytes": n * (2 * 16 + 4 + 4), "flops": n * 4 * net}
    n, steps, N = _points(case), case["steps"], case["pml"]
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    coef = {0: 48, 1: 24, 2: 20 if case["media"] != "volume" else 30}[case["metric"]]
    faces = N * (2 * ny * nz + 2 * nx * nz + nx * ny)
    return {"bytes": steps * (n * (126 * 4 + 4 * coef) + 4 * 153 * faces), "flops": steps * 4 * n * (27 * 9 + 150)}


# ---------------------------------------------------------------- 64 bits

def exact(case, seed):
    if case["kind"] == "guess":
        return _exact_guess(case, seed)
    if case["kind"] == "wave" and case["metric"] == 0 and _points(case) <= 4e6:
        return {"W": _exact_wave(case, seed)}
    return None


def _bf16(x):
    """Rounded to bfloat16, the operand format of the network's middle layer,
    with the gradient of the identity."""
    return x + (x.to(torch.float32).to(torch.bfloat16).to(torch.float64) - x).detach()


def _exact_guess(case, seed):
    f, t = _samples(case["samples"], seed)
    f, t = torch.from_numpy(f).double(), torch.from_numpy(t).double()
    P = torch.from_numpy(mlp.load(NETWORK)).double().requires_grad_(True)
    o = mlp.OFF
    W1, W2 = P[o["W1"]:o["b1"]].reshape(64, 4), P[o["W2"]:o["b2"]].reshape(64, 64)
    b1, b2, w3, b3 = P[o["b1"]:o["W2"]], P[o["b2"]:o["w3"]], P[o["w3"]:o["b3"]], P[o["b3"]]
    fixed = P.detach()
    x = (f - fixed[0:4]) * fixed[4:8]
    h1 = _bf16(torch.relu(x @ W1.T + b1))
    out = torch.relu(h1 @ _bf16(W2).T + b2) @ w3 + b3
    loss = ((out - (t - fixed[8]) / fixed[9]) ** 2).mean()
    loss.backward()
    return {"loss": loss.item(), "grad": P.grad.numpy(), "log10_rate": (out * fixed[9] + fixed[8]).detach().numpy()}


def _exact_wave(case, seed):
    """The wave scheme on a Cartesian grid of two half spaces in 64 bits:
    the one-sided five-point operators whose directions cycle with the step,
    the four-stage Runge-Kutta combine, the absorbing layers with their
    auxiliary fields (or the sponge), and the free surface: velocity
    derivatives across it from its zero traction, tractions mirrored with
    the opposite sign above it."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    DH = _spacing(case)
    DT = 6e-5 * DH
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    W = torch.from_numpy(_wavefield(nx + 6, ny + 6, nz + 6, seed)).double().to(dev)
    # fields [9][x][z][y]; axis numbers of x, y, z below
    dim = (0, 2, 1)
    n = (nx, ny, nz)

    def shaped(v, a):
        return torch.as_tensor(np.asarray(v), dtype=torch.float64, device=dev).reshape([-1 if d == dim[a] else 1 for d in range(3)])

    half = np.arange(nx) + 3 < nx // 2
    vp, vs, rho = (shaped(np.where(half, a, b), 0) for a, b in ((6000.0, 5400.0), (3464.0, 3120.0), (2670.0, 2600.0)))
    mu = rho * vs ** 2
    lam = rho * vp ** 2 - 2 * mu
    l2m = lam + 2 * mu

    # absorbing profiles along each axis: alpha, beta and d / beta
    N = case["pml"]
    A, B, D = [], [], []
    for a in range(3):
        al, be, da = np.zeros(n[a]), np.ones(n[a]), np.zeros(n[a])
        if N:
            R = 10.0 ** -((math.log10(N) - 1.0) / math.log10(2.0) + 3.0)
            L0 = DH * (N - 1)
            dmax = -6000.0 / (2.0 * L0) * math.log(R) * 3.0
            depth = np.full(n[a], -1.0)
            depth[:N] = (N - 1 - np.arange(N)) * DH
            if a < 2:
                depth[n[a] - N:] = np.arange(N) * DH
            r = np.where(depth >= 0, depth / L0, 0.0)
            al = np.where(depth >= 0, math.pi * (1.0 - r), 0.0)
            be = 1.0 + 2.0 * r * r
            da = dmax * r * r / be
        A.append(shaped(al, a))
        B.append(shaped(be, a))
        D.append(shaped(da, a))
    damp = torch.ones((), dtype=torch.float64, device=dev)
    if case["cerjan"]:
        M = case["cerjan"]
        al = math.sqrt(-math.log(0.92)) / M
        for a in range(3):
            v = np.ones(n[a])
            v[:M] = np.exp(-(al * (M - np.arange(M))) ** 2)
            if a < 2:
                v[n[a] - M:] = v[:M][::-1]
            damp = torch.minimum(damp, shaped(v, a))
    bands = []  # (axis, first, last) of every absorbing face
    if N:
        for a in range(3):
            bands.append((a, 0, N))
            if a < 2:
                bands.append((a, n[a] - N, n[a]))

    C = (0.29164704779069994, 0.66674514216519998, 1.2501177132452999, 0.33341180882999999, 0.041686285540599999)

    def shift(f, a, s):  # interior view of a padded field, moved s points along axis a
        idx = [slice(3, m - 3) for m in f.shape]
        idx[dim[a]] = slice(3 + s, f.shape[dim[a]] - 3 + s)
        return f[tuple(idx)]

    def drp(f, a, s):  # s: the operator's direction
        return s * (-C[0] * shift(f, a, -s) - C[1] * shift(f, a, 0) + C[2] * shift(f, a, s) - C[3] * shift(f, a, 2 * s)
                    + C[4] * shift(f, a, 3 * s)) / DH

    top = nz - 1
    T = {(0, 0): 3, (0, 1): 6, (0, 2): 7, (1, 0): 6, (1, 1): 4, (1, 2): 8, (2, 0): 7, (2, 1): 8, (2, 2): 5}

    def axis_rhs(a, dv, dt):
        """Rates from the derivatives along axis a: velocities from the
        tractions dt[3], stresses from the velocities dv[3]."""
        h = [dt[c] / rho for c in range(3)]
        h += [(l2m if c == a else lam) * dv[a] for c in range(3)]
        zero = torch.zeros_like(dv[0])
        h += [mu * (dv[1 - a] if a < 2 else zero), mu * (dv[2 - a] if a != 1 else zero),
              mu * (dv[3 - a] if a > 0 else zero)]
        return h

    def rates(W, aux, flags):
        d = [[drp(W[c], a, flags[a]) for c in range(3)] for a in range(3)]
        t = [[drp(W[T[a, c]], a, flags[a]) for c in range(3)] for a in range(3)]
        h = [torch.zeros((nx, nz, ny), dtype=torch.float64, device=dev) for _ in range(9)]
        plain = [axis_rhs(a, d[a], t[a]) for a in range(3)]  # what drives the auxiliary fields
        # free surface, velocities: the traction-free condition on the top
        # row, narrower differences on the two rows below it
        s = flags[2]
        dz = [v.clone() for v in d[2]]
        row = slice(top, top + 1)
        x_, y_ = [(d[a][2] / B[a])[:, row] for a in (0, 1)]
        dz[0][:, row], dz[1][:, row] = -x_, -y_
        dz[2][:, row] = -lam / l2m * ((d[0][0] / B[0])[:, row] + (d[1][1] / B[1])[:, row])
        for c in range(3):
            f = W[c]
            dz[c][:, top - 1] = (s * (shift(f, 2, s) - shift(f, 2, 0)) / DH)[:, top - 1]
            dz[c][:, top - 2] = (s * (-7.0 / 6.0 * shift(f, 2, 0) + 4.0 / 3.0 * shift(f, 2, s)
                                      - 1.0 / 6.0 * shift(f, 2, 2 * s)) / DH)[:, top - 2]
        # and tractions: zero on the top row, mirrored with the opposite sign
        tz = [v.clone() for v in t[2]]
        for c in range(3):
            f = W[T[2, c]].clone()
            k = top + 3
            f[:, k] = 0.0
            for m in (1, 2, 3):
                f[:, k + m] = -f[:, k - m]
            tz[c][:, top - 2:] = drp(f, 2, s)[:, top - 2:]
        for a in range(3):
            for c, v in enumerate(axis_rhs(a, dz if a == 2 else d[a], tz if a == 2 else t[a])):
                h[c] += v / B[a]
        rate = []
        for (a, lo, hi), y in zip(bands, aux):
            at = [slice(None)] * 3
            at[dim[a]] = slice(lo, hi)
            at = tuple(at)
            src = torch.stack(plain[a])[(slice(None),) + at]
            if a < 2:  # the velocity derivatives that the free surface ties to this axis
                w = torch.zeros((9, nx, 1, ny), dtype=torch.float64, device=dev)
                zz = -lam / l2m * d[a][a][:, row]
                w[3], w[4], w[5] = lam * zz, lam * zz, l2m * zz
                w[7 + a] = -mu * d[a][2][:, row]
                src = src.clone()
                src[:, :, top:] += w[(slice(None),) + at]
            cut = y / B[a][tuple(slice(lo, hi) if q == dim[a] else slice(None) for q in range(3))]
            for c in range(9):
                h[c][at] -= cut[c]
            da, aa = (v[tuple(slice(lo, hi) if q == dim[a] else slice(None) for q in range(3))] for v in (D[a], A[a]))
            rate.append(-(aa + da) * y + da * src)
        return torch.stack(h), rate

    # directions along x, y, z of the eight steps of a cycle
    flag_rows = ((-1, -1, -1), (1, 1, -1), (1, 1, 1), (-1, -1, 1), (-1, 1, -1), (1, -1, -1), (1, -1, 1), (-1, 1, 1))
    RA, RB = (0.5, 0.5, 1.0), (1.0 / 6.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 6.0)
    aux = []
    for a, lo, hi in bands:
        shape = [9, nx, nz, ny]
        shape[1 + dim[a]] = hi - lo
        aux.append(torch.zeros(shape, dtype=torch.float64, device=dev))
    inner = (slice(None),) + (slice(3, -3),) * 3
    for it in range(case["steps"]):
        start, acc = W[inner].clone(), W[inner].clone()
        aux0, aux_acc = [y.clone() for y in aux], [y.clone() for y in aux]
        for k in range(4):
            sign = -1 if k % 2 else 1
            h, rate = rates(W, aux, [sign * f for f in flag_rows[it % 8]])
            acc += RB[k] * DT * h
            W[inner] = damp * (acc if k == 3 else start + RA[k] * DT * h)
            for q, r in enumerate(rate):
                aux_acc[q] += RB[k] * DT * r
                aux[q] = aux_acc[q].clone() if k == 3 else aux0[q] + RA[k] * DT * r
    return W.cpu().numpy().reshape(-1)
