"""The solves that this library is measured on, through its public entry points.

Every case is an ensemble of initial-value problems whose inputs lie in GPU
memory (the device entry points of include/bacon_gpu.h, called through
bacon_amd._lib as a program that holds its data in torch tensors does), except
the batched builder's, which takes and returns host arrays.  Input
distributions are those of bacon_amd.workloads.

The methods are the reference's: Runge-Kutta 4(5) and 2(3), Adams5, BDF6; with
them the path output, the shared-matrix linear systems and the discrete
adjoint.  Sizes run from a short window of a few thousand trajectories to the
million-instance ensemble.
"""
import ctypes as C
import math

import numpy as np
import torch

from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd.adjoint import solve_vjp

DEV = "cuda:0"
F64 = torch.float64

DIM = {"lorenz": 3, "lotka_volterra": 2, "two_level": 4, "robertson": 3}
METHOD = {"rk45": L.RK45, "rk23": L.RK23, "adams5": L.ADAMS5, "adams3": L.ADAMS3,
          "bdf6": L.BDF6, "bdf2": L.BDF2}


def listed():
    return [
        # a short forecast window over a few thousand trajectories, called in a
        # loop: a few hundred step attempts, so launches and latency count
        dict(name="rk45_window", kind="rk", method="rk45", rhs="lorenz", n=4096, t_end=0.1,
             tol=1e-6, mixed=False, dt_min=1e-12, dt_max=0.1),
        # the plain ensemble of a thousand trajectories over a long horizon:
        # far fewer instances than the chip has lanes
        dict(name="rk45_plain", kind="rk", method="rk45", rhs="lorenz", n=1024, t_end=10.0,
             tol=1e-6, mixed=False, dt_min=1e-6, dt_max=0.1),
        # the large ensemble: a million instances whose end times and
        # tolerances differ, handed out longest first
        dict(name="rk45_million", kind="rk", method="rk45", rhs="lorenz", n=1 << 20, t_end=20.0,
             tol=1e-10, mixed=True, dt_min=1e-12, dt_max=0.1),
        # complex state through the batched builder: host arrays in and out
        dict(name="builder_two_level", kind="builder", method="rk45", rhs="two_level", n=100003,
             t_end=10.0, tol=1e-8, dt_min=1e-12, dt_max=0.1),
        # the low-order pair on a mild tolerance
        dict(name="rk23_population", kind="rk", method="rk23", rhs="lotka_volterra", n=50000,
             t_end=5.0, tol=1e-4, mixed=False, dt_min=1e-9, dt_max=0.1),
        # dense output at shared times (t_eval of the usual solvers)
        dict(name="path_at_times", kind="path", rhs="lorenz", n=65536, t_end=10.0, tol=1e-6,
             stops=100, capacity=101, every=1, inst_major=False),
        # every accepted step into a ring of the last 64
        dict(name="path_ring", kind="path", rhs="lorenz", n=262144, t_end=10.0, tol=1e-6,
             stops=0, capacity=64, every=1, inst_major=False),
        # the predictor-corrector on the plain workload's distribution
        dict(name="adams5_ensemble", kind="adams", method="adams5", rhs="lorenz", n=262144,
             t_end=10.0, tol=1e-6, dt_min=1e-6, dt_max=0.1),
        # dense systems that share one matrix
        dict(name="linear_128", kind="linear", dim=128, n=32768, t_end=5.0, tol=1e-9),
        # gradients of a fit to 20 observations, all outputs
        dict(name="adjoint_fit", kind="adjoint", n=262144, t_end=15.0, tol=1e-8, obs=20),
        # the stiff reaction-diffusion system
        dict(name="bdf6_brusselator", kind="bdf", method="bdf6", rhs="brusselator", dim=32,
             n=32768, t_end=10.0, tol=1e-7, dt_max=0.1, lu=64),
        # stiff chemical kinetics, a small system
        dict(name="bdf6_robertson", kind="bdf", method="bdf6", rhs="robertson", dim=3, n=16384,
             t_end=0.2, tol=1e-6, dt_max=5e-4, lu=64),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["rk", "rk", "rk", "builder", "path", "path", "adams", "linear", "adjoint",
                       "bdf", "bdf"])
    if kind == "rk":
        method = rng.choice(["rk45", "rk45", "rk23"])
        rhs = rng.choice(["lorenz", "lotka_volterra", "two_level"])
        if method == "rk23":
            return dict(kind=kind, method=method, rhs=rhs, n=int(_log(rng, 256, 200000)),
                        t_end=rng.uniform(0.1, 2.0), tol=_log(rng, 1e-5, 1e-3), mixed=False,
                        dt_min=1e-9, dt_max=0.1)
        return dict(kind=kind, method=method, rhs=rhs, n=int(_log(rng, 256, 1000000)),
                    t_end=_log(rng, 0.1, 10.0), tol=_log(rng, 1e-9, 1e-4),
                    mixed=rng.random() < 0.5, dt_min=1e-12, dt_max=0.1)
    if kind == "builder":
        return dict(kind=kind, method="rk45", rhs=rng.choice(["two_level", "lotka_volterra"]),
                    n=int(_log(rng, 1000, 300000)), t_end=rng.uniform(1.0, 10.0),
                    tol=_log(rng, 1e-9, 1e-5), dt_min=1e-12, dt_max=0.1)
    if kind == "path":
        stops = rng.choice([0, rng.randint(3, 120)])
        return dict(kind=kind, rhs=rng.choice(["lorenz", "lotka_volterra"]),
                    n=int(_log(rng, 1000, 200000)), t_end=rng.uniform(1.0, 10.0),
                    tol=_log(rng, 1e-8, 1e-5), stops=stops,
                    capacity=stops + 1 if stops else rng.choice([16, 50, 64, 100]),
                    every=1 if stops else rng.choice([1, 1, 3, 10]),
                    inst_major=rng.random() < 0.3)
    if kind == "adams":
        return dict(kind=kind, method="adams5", rhs=rng.choice(["lorenz", "lotka_volterra"]),
                    n=int(_log(rng, 256, 262144)), t_end=rng.uniform(0.5, 10.0),
                    tol=_log(rng, 1e-6, 1e-4), dt_min=1e-9, dt_max=0.1)
    if kind == "linear":
        return dict(kind=kind, dim=rng.choice([32, 64, 128]), n=int(_log(rng, 100, 32768)),
                    t_end=rng.uniform(0.5, 5.0), tol=_log(rng, 1e-9, 1e-5))
    if kind == "adjoint":
        return dict(kind=kind, n=int(_log(rng, 1000, 262144)), t_end=rng.uniform(2.0, 15.0),
                    tol=_log(rng, 1e-8, 1e-5), obs=rng.randint(2, 30))
    rhs = rng.choice(["brusselator", "brusselator", "robertson", "lotka_volterra"])
    if rhs == "brusselator":
        dim = rng.choice([4, 8, 16, 32, 32])
        return dict(kind=kind, method=rng.choice(["bdf6", "bdf6", "bdf2"]), rhs=rhs, dim=dim,
                    n=int(_log(rng, 64, 8192)), t_end=rng.uniform(0.05, 1.0),
                    tol=_log(rng, 1e-7, 1e-5), dt_max=0.1,
                    lu=rng.choice([64, 32]) if dim == 32 else 64)
    if rhs == "robertson":
        return dict(kind=kind, method="bdf6", rhs=rhs, dim=3, n=int(_log(rng, 256, 16384)),
                    t_end=rng.uniform(0.02, 0.2), tol=_log(rng, 1e-7, 1e-5), dt_max=5e-4, lu=64)
    return dict(kind=kind, method="bdf6", rhs=rhs, dim=2, n=int(_log(rng, 256, 16384)),
                t_end=rng.uniform(0.5, 5.0), tol=_log(rng, 1e-7, 1e-5), dt_max=0.1, lu=64)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Draws:
    """Seeded draws on the GPU, one row per call."""

    def __init__(self, seed, n):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)
        self.n = n

    def uniform(self, a, b):
        return a + (b - a) * torch.rand(self.n, generator=self.g, device=DEV, dtype=F64)

    def log_uniform(self, a, b):
        return torch.exp(self.uniform(math.log(a), math.log(b)))

    def normal(self):
        return torch.randn(self.n, generator=self.g, device=DEV, dtype=F64)

    def full(self, v):
        return torch.full((self.n,), v, device=DEV, dtype=F64)


def _problem(rhs, d, dim):
    """(y0 [dim, n], params [P, n]) of the distributions in bacon_amd.workloads."""
    if rhs == "lorenz":
        rho = d.uniform(20.0, 40.0)
        y0 = [d.uniform(-15, 15), d.uniform(-15, 15), d.uniform(5, 40)]
        return torch.stack(y0), torch.stack([d.full(10.0), rho, d.full(8.0 / 3.0)])
    if rhs == "lotka_volterra":
        p = [d.log_uniform(0.5, 2.0) for _ in range(4)]
        return torch.stack([d.uniform(0.5, 2.0), d.uniform(0.5, 2.0)]), torch.stack(p)
    if rhs == "two_level":
        p = [d.uniform(-2.0, 2.0), d.uniform(-2.0, 2.0), d.log_uniform(0.01, 0.2)]
        y0 = torch.stack([d.normal() for _ in range(4)])
        return y0 / y0.square().sum(0).sqrt(), torch.stack(p)
    if rhs == "robertson":
        p = [0.04 * d.log_uniform(0.5, 2.0), 3e7 * d.log_uniform(0.5, 2.0),
             1e4 * d.log_uniform(0.5, 2.0)]
        return torch.stack([d.full(1.0), d.full(0.0), d.full(0.0)]), torch.stack(p)
    B = d.log_uniform(2.0, 4.0)
    cells = dim // 2
    y0 = [1.0 + 0.1 * d.normal() for _ in range(cells)] + [B + 0.1 * d.normal()
                                                            for _ in range(cells)]
    return torch.stack(y0), torch.stack([d.full(1.0), B, d.full(0.02)])


def _inputs(case, seed):
    kind, n = case["kind"], case["n"]
    d = _Draws(seed, n)
    if kind == "linear":
        N = case["dim"]
        g = np.random.default_rng(seed)
        Q, R = np.linalg.qr(g.standard_normal((N, N)))
        Q = Q * np.sign(np.diag(R))[None, :]
        D = np.exp(g.uniform(math.log(0.1), math.log(10.0), N))
        b = g.standard_normal(N)
        y0 = torch.stack([d.normal() for _ in range(N)])
        return dict(y0=y0, params=None, A=-(Q * D[None, :]) @ Q.T, b=b, Q=Q, D=D)
    if kind == "adjoint":
        y0, p = _problem("lotka_volterra", d, 2)
        obs = torch.arange(1, case["obs"] + 1, device=DEV, dtype=F64) * (case["t_end"] / case["obs"])
        obs[-1] = case["t_end"]
        # data near the trajectories: positive, of the states' own scale
        targets = torch.stack([d.log_uniform(0.3, 3.0) for _ in range(2 * case["obs"])])
        return dict(y0=y0, params=p, obs=obs, targets=targets.reshape(case["obs"], 2, n))
    rhs = case["rhs"]
    y0, p = _problem(rhs, d, case.get("dim") or DIM[rhs])
    r = dict(y0=y0, params=p)
    if case.get("mixed"):
        r["t_end"] = d.uniform(0.05 * case["t_end"], case["t_end"])
        r["tol"] = d.log_uniform(case["tol"], max(1e-4, 10 * case["tol"]))
    return r


# ---------------------------------------------------------------------------
# the calls
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    s = dict(case=case, **_inputs(case, seed))
    if kind == "adjoint":
        return s
    if kind == "builder":
        s["workload"] = dict(rhs=case["rhs"], dim=DIM[case["rhs"]], y0=s["y0"].cpu().numpy(),
                             params=s["params"].cpu().numpy(), t0=0.0,
                             t_end=np.full(n, case["t_end"]), tol=np.full(n, case["tol"]),
                             dt_min=case["dt_min"], dt_max=case["dt_max"])
        return s
    dim = s["y0"].shape[0]
    out = dict(t=torch.zeros(n, device=DEV, dtype=F64),
               y=torch.zeros((dim, n), device=DEV, dtype=F64),
               status=torch.zeros(n, device=DEV, dtype=torch.int32),
               counts=torch.zeros((n, 2), device=DEV, dtype=torch.int32))
    p = s["params"]
    d = L.EnsembleDesc(
        n=n, dim=dim, n_params=0 if p is None else p.shape[0], y0=s["y0"].data_ptr(),
        params=None if p is None else p.data_ptr(), t0_s=0.0, t_end_s=case["t_end"],
        tol_s=case["tol"], dt_min_s=case.get("dt_min", 1e-12), dt_max_s=case.get("dt_max", 0.1),
        t_out=out["t"].data_ptr(), y_out=out["y"].data_ptr(), status=out["status"].data_ptr(),
        counts=out["counts"].data_ptr())
    if case.get("mixed"):
        d.t_end, d.tol = s["t_end"].data_ptr(), s["tol"].data_ptr()
        # longest first by the cost model of workloads.cost_order
        cost = s["t_end"] * s["tol"].pow(-0.25)
        s["order"] = torch.argsort(cost, descending=True, stable=True).to(torch.int32)
        d.order = s["order"].data_ptr()
    if kind == "linear":
        s["shared"] = torch.from_numpy(np.concatenate([s["A"].reshape(-1), s["b"]])).to(DEV)
        d.shared = s["shared"].data_ptr()
    if kind == "path":
        cap = case["capacity"]
        lead = (n, cap) if case["inst_major"] else (cap, n)
        out["path_t"] = torch.zeros(lead, device=DEV, dtype=F64)
        out["path_y"] = torch.zeros((n, cap, dim) if case["inst_major"] else (cap, dim, n),
                                    device=DEV, dtype=F64)
        out["path_len"] = torch.zeros(n, device=DEV, dtype=torch.int32)
        flags = L.PATH_INSTANCE_MAJOR if case["inst_major"] else 0
        if case["stops"]:
            k = torch.arange(1, case["stops"] + 1, device=DEV, dtype=F64)
            s["stops"] = k * (case["t_end"] / (case["stops"] + 1))
            flags |= L.PATH_STOPS_ONLY
        s["path"] = L.PathDesc(capacity=cap, every=case["every"], n_stops=case["stops"],
                               flags=flags,
                               stops=s["stops"].data_ptr() if case["stops"] else None,
                               path_t=out["path_t"].data_ptr(), path_y=out["path_y"].data_ptr(),
                               path_len=out["path_len"].data_ptr())
    s["desc"], s["out"] = d, out
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "adjoint":
        return solve_vjp("lotka_volterra", s["y0"], s["params"], s["obs"], s["targets"],
                         t_end=case["t_end"], tol=case["tol"])
    if kind == "builder":
        return ivp.solve_ensemble(METHOD[case["method"]], s["workload"])
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    d = C.byref(s["desc"])
    lib = L.lib()
    if kind == "rk":
        rc = lib.bg_rk_solve_device(METHOD[case["method"]], L.RHS[case["rhs"]], L.INTENDED, d,
                                    None, stream)
    elif kind == "linear":
        rc = lib.bg_rk_solve_device(L.RK45, L.RHS["linear"], L.INTENDED, d, None, stream)
    elif kind == "path":
        rc = lib.bg_rk_solve_path_device(L.RK45, L.RHS[case["rhs"]], L.INTENDED, d,
                                         C.byref(s["path"]), stream)
    elif kind == "adams":
        rc = lib.bg_adams_solve_device(METHOD[case["method"]], L.RHS[case["rhs"]], L.INTENDED, d,
                                       stream)
    else:
        rc = lib.bg_bdf_solve_device(METHOD[case["method"]], L.RHS[case["rhs"]], L.INTENDED,
                                     case["lu"], d, stream)
    if rc != 0:
        raise RuntimeError(f"{case['kind']}: status {rc}")
    return s["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# floating-point operations of one right-hand side (fma = 2)
RHS_FLOPS = {"lorenz": 8, "lotka_volterra": 7, "two_level": 20, "robertson": 10}


def _rk_attempt(rhs, dim, method="rk45"):
    """Operations of one step attempt: stage combinations, the stages'
    right-hand sides and their scaling by dt, error norm, controller."""
    combos, stages = (24, 6) if method == "rk45" else (12, 4)
    return 2 * dim * combos + stages * (RHS_FLOPS[rhs] + dim) + 2 * dim + 8


# step attempts per unit time at tolerance 1e-6 (RK45; RK23 at 1e-4; Adams5 at
# 1e-6; BDF steps at 1e-7), as the distributions above give them
RATE = {("rk45", "lorenz"): 302.0, ("rk45", "lotka_volterra"): 11.0, ("rk45", "two_level"): 10.0,
        ("rk23", "lorenz"): 24000.0, ("rk23", "lotka_volterra"): 290.0,
        ("rk23", "two_level"): 290.0, ("adams5", "lorenz"): 730.0,
        ("adams5", "lotka_volterra"): 33.0}


def _attempts(method, rhs, t_end, tol):
    ref, power = (1e-4, -0.5) if method == "rk23" else (1e-6, -0.25)
    return max(4.0, RATE[(method, rhs)] * t_end * (tol / ref) ** power)


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "linear":
        N = case["dim"]
        a = max(8.0, 84.0 * case["t_end"] * (case["tol"] / 1e-9) ** -0.1)
        flops = n * a * (6 * (2.0 * N * N + 2 * N) + 2 * N * 24)
        return {"bytes": 8.0 * (2 * N * n + n + N * N + N) + 12 * n, "flops": flops}
    if kind == "adjoint":
        steps = 0.7 * _attempts("rk45", "lotka_volterra", case["t_end"], case["tol"])
        flops = n * steps * (_rk_attempt("lotka_volterra", 2) + 334)
        io = 2 + 4 + 2 * case["obs"] + 1 + 4 + 2 + 2 * case["obs"] + 3
        return {"bytes": n * (8.0 * io + 12), "flops": flops}
    rhs = case["rhs"]
    dim = case.get("dim") or DIM[rhs]
    n_params = 4 if rhs == "lotka_volterra" else 3
    bytes_ = n * (8.0 * (dim + n_params + 1 + dim) + 12)
    if kind == "bdf":
        frhs = {"brusselator": 9.5 * dim}.get(rhs) or RHS_FLOPS[rhs]
        resid = frhs + 15 * dim
        # two Jacobian inverses and four Broyden iterations per step
        step = 2 * ((1 + 2 * min(dim, 4)) * resid + 2 * dim ** 3 + 2 * dim ** 2) \
            + 4 * (resid + 8 * dim ** 2 + 10 * dim)
        steps = max(8.0, case["t_end"] / case["dt_max"] if rhs == "robertson" else
                    16.0 * case["t_end"])
        return {"bytes": bytes_, "flops": n * steps * step}
    if kind == "adams":
        per = 2 * (RHS_FLOPS[rhs] + 10 * dim) + 20
        return {"bytes": bytes_, "flops": n * per * _attempts("adams5", rhs, case["t_end"],
                                                              case["tol"])}
    method = case.get("method", "rk45")
    if case.get("mixed"):
        # mean over t_end ~ U[0.05, 1] t_end and log-uniform tolerances
        hi = max(1e-4, 10 * case["tol"])
        mean = 4.0 * (case["tol"] ** -0.25 - hi ** -0.25) / math.log(hi / case["tol"])
        a = _attempts(method, rhs, 0.525 * case["t_end"], mean ** -4.0)
        bytes_ += 20.0 * n
    else:
        a = _attempts(method, rhs, case["t_end"], case["tol"])
    if kind == "path":
        kept = case["stops"] + 1 if case["stops"] else min(case["capacity"], a / case["every"])
        bytes_ += n * (8.0 * kept * (1 + dim) + 4)
    return {"bytes": bytes_, "flops": n * a * _rk_attempt(rhs, dim, method)}


# ---------------------------------------------------------------------------
# exact values: the differential equation's solution in 64 bits
# ---------------------------------------------------------------------------
def _rhs(rhs, p, dim):
    if rhs == "lorenz":
        return lambda y: torch.stack([p[0] * (y[1] - y[0]), y[0] * (p[1] - y[2]) - y[1],
                                      y[0] * y[1] - p[2] * y[2]])
    if rhs == "lotka_volterra":
        return lambda y: torch.stack([p[0] * y[0] - p[1] * y[0] * y[1],
                                      p[3] * y[0] * y[1] - p[2] * y[1]])
    if rhs == "robertson":
        def f(y):
            a, b, c = p[0] * y[0], p[2] * y[1] * y[2], p[1] * y[1] * y[1]
            return torch.stack([b - a, a - b - c, c])
        return f
    cells = dim // 2

    def f(y):
        u, v = y[:cells], y[cells:]
        uuv = u * u * v
        cl = p[2] * (cells * cells)
        lap = lambda x: torch.roll(x, 1, 0) - 2.0 * x + torch.roll(x, -1, 0)  # noqa: E731
        return torch.cat([p[0] + uuv - (p[1] + 1.0) * u + cl * lap(u),
                          p[1] * u - uuv + cl * lap(v)])
    return f


def _integrate(f, y, T, steps):
    """Gragg's modified midpoint rule extrapolated over 2, 4, .. 12 substeps
    (order 12), `steps` equal steps over T."""
    H = T / steps
    for _ in range(steps):
        rows = []
        f0 = f(y)
        for m in (2, 4, 6, 8, 10, 12):
            h = H / m
            a, b = y, y + h * f0
            for _ in range(m - 1):
                a, b = b, a + 2.0 * h * f(b)
            row = [0.5 * (a + b + h * f(b))]
            for k, prev in enumerate(rows[-1] if rows else []):
                ratio = (m / (m - 2.0 * (k + 1))) ** 2 - 1.0
                row.append(row[k] + (row[k] - prev) / ratio)
            rows.append(row)
        y = rows[-1][-1]
    return y


def _two_level(p, y0, t):
    hd, ho, g = p
    c0, c1 = torch.complex(y0[0], y0[1]), torch.complex(y0[2], y0[3])
    w = torch.hypot(hd, ho)
    co, si, d = torch.cos(w * t), torch.sin(w * t) / w, torch.exp(-g * t)
    r0 = d * (co * c0 - 1j * si * (hd * c0 + ho * c1))
    r1 = d * (co * c1 - 1j * si * (ho * c0 - hd * c1))
    return torch.stack([r0.real, r0.imag, r1.real, r1.imag])


def _fit_gradient(case, s):
    """Loss and gradients of the fit from the variational equations: the state
    with its derivatives by the four parameters and the two initial values."""
    n, p, m = case["n"], s["params"], case["obs"]
    z = torch.zeros((14, n), device=DEV, dtype=F64)
    z[:2] = s["y0"]
    z[10] = 1.0  # d x / d x0
    z[13] = 1.0  # d w / d w0

    def f(z):
        x, w = z[0], z[1]
        xw = x * w
        a11, a12 = p[0] - p[1] * w, -p[1] * x
        a21, a22 = p[3] * w, p[3] * x - p[2]
        sx, sw = z[2::2], z[3::2]
        dx, dw = a11 * sx + a12 * sw, a21 * sx + a22 * sw
        dx[0] += x
        dx[1] -= xw
        dw[2] -= w
        dw[3] += xw
        return torch.cat([torch.stack([p[0] * x - p[1] * xw, p[3] * xw - p[2] * w]),
                          torch.stack([dx, dw], 1).reshape(12, n)])

    loss = torch.zeros(n, device=DEV, dtype=F64)
    grad = torch.zeros((6, n), device=DEV, dtype=F64)
    obs_y, t = [], 0.0
    for k in range(m):
        tk = float(s["obs"][k])
        z = _integrate(f, z, tk - t, max(1, math.ceil((tk - t) / 0.15)))
        t = tk
        r = z[:2] - s["targets"][k]
        loss += r.square().sum(0)
        grad += 2.0 * (z[2::2] * r[0] + z[3::2] * r[1])
        obs_y.append(z[:2].clone())
    return dict(loss=loss, grad_params=grad[:4], grad_y0=grad[4:], obs_y=torch.stack(obs_y),
                t=torch.full((n,), case["t_end"], device=DEV, dtype=F64), y=z[:2], status=None,
                counts=None)


def exact(case, seed):
    kind, n, T = case["kind"], case["n"], case["t_end"]
    if case.get("mixed") and case["rhs"] == "lorenz" and T > 12.0:
        return None  # past that horizon the system's chaos makes any last bit an answer of its own
    s = _inputs(case, seed)
    if kind == "adjoint":
        return _fit_gradient(case, s)
    end = s.get("t_end", torch.full((n,), T, device=DEV, dtype=F64))
    out = dict(t=end, y=None, status=None, counts=None)
    if kind == "linear":
        Q, D = torch.from_numpy(s["Q"]).to(DEV), torch.from_numpy(s["D"]).to(DEV)
        x = torch.from_numpy(np.linalg.solve(s["A"], -s["b"])).to(DEV)[:, None]
        out["y"] = x + Q @ (torch.exp(-D * T)[:, None] * (Q.T @ (s["y0"] - x)))
        return out
    rhs, p = case["rhs"], s["params"]
    if kind == "builder":
        out = dict(t=end, y=None, status=None, n_accepted=None, n_rejected=None)
    if kind == "path":
        out.update(path_t=None, path_y=None, path_len=None)
    if rhs == "two_level":
        out["y"] = _two_level(p, s["y0"], end)
        return out
    f = _rhs(rhs, p, s["y0"].shape[0])
    # step lengths that resolve the systems' fastest scales
    h = {"lorenz": 0.02, "lotka_volterra": 0.1, "robertson": 4e-4, "brusselator": 0.02}[rhs]
    steps = lambda span: max(1, math.ceil(span / h))  # noqa: E731
    if kind == "path" and case["stops"]:
        k = case["stops"]
        y, at = s["y0"], []
        for _ in range(k + 1):
            y = _integrate(f, y, T / (k + 1), steps(T / (k + 1)))
            at.append(y)
        pt = torch.arange(1, k + 2, device=DEV, dtype=F64) * (T / (k + 1))
        py = torch.stack(at)  # [k + 1, dim, n]
        out["y"] = y
        out["path_t"] = pt[:, None].expand(k + 1, n).contiguous()
        out["path_y"] = py
        if case["inst_major"]:
            out["path_t"] = out["path_t"].T.contiguous()
            out["path_y"] = py.permute(2, 0, 1).contiguous()
        return out
    out["y"] = _integrate(f, s["y0"], end, steps(T))
    return out
