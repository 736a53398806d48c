"""The work that users of this library have it do, as cases that can be timed and checked.

Each case is one call of a gopf program: a solver (or a batch, a transform, an adjoint) that
the program holds, a run of steps through the public entry points, and the read-back of what
it computed, as an epoch of pf.Solver.Solve with a callback does.  Kinds:

  euler     Cahn-Hilliard, semi-implicit Euler, one field in 2D or 3D (examples/cahnHilliard);
            with "series" the free energy is recorded before every step
  precip    the two-field strain precipitate with its Khachaturyan term
            (examples/strain_single_precipitate), Euler or RK4
  implicit  Cahn-Hilliard under ImplicitEuler with the default Newton-Krylov settings
  adjoint   dJ/dc0 and dJ/d(scalar) of a run of Euler steps
  sweep     a batch of sims of three sizes, each with its own scalars
  fourier   the FourierTransform drop-in on host arrays, forward and back

A solver carries its fields from one pass to the next, as a program's epochs do; the passes
whose cost depends on the field (implicit) or that need its start (adjoint) set it first.
"""
import math

import numpy as np
import torch

import gopf_amd as G
from gopf_amd import workloads as W

DT2, DT3 = 0.1, 0.05          # the time steps of the 2D and 3D Cahn-Hilliard workloads
BULK = [0.0, 0.0, 1.0, -2.0, 1.0]   # f(c) = c^2 (1 - c)^2

# transform lengths with a compiled schedule that a 2D side may take; any side up to 64 is
# taken too (by direct transforms where it has no schedule), odd ones among them
SIDES = [64, 80, 96, 100, 112, 128, 160, 192, 200, 224, 250, 256, 320, 384, 400, 448, 500, 512, 640, 768, 800, 896,
         1000, 1024]
SMALL = [9, 12, 15, 16, 20, 24, 27, 30, 32, 33, 40, 45, 48, 50, 56, 60, 63]


def listed():
    return [
        # the smallest call: a test-sized grid, a few steps, the field read back
        {"name": "euler2d_32_fp64", "kind": "euler", "d0": 32, "d1": 32, "d2": 0, "prec": "fp64", "steps": 50,
         "series": False},
        # a two-dimensional study with its energy curve, in plain FP64
        {"name": "euler2d_128_fp64_series", "kind": "euler", "d0": 128, "d1": 128, "d2": 0, "prec": "fp64",
         "steps": 1000, "series": True},
        # a rectangular domain whose sides are no powers of two
        {"name": "euler2d_400x250_fp64", "kind": "euler", "d0": 400, "d1": 250, "d2": 0, "prec": "fp64", "steps": 500,
         "series": False},
        # a large two-dimensional domain in FP32-bulk
        {"name": "euler2d_1024_fp32", "kind": "euler", "d0": 1024, "d1": 1024, "d2": 0, "prec": "fp32", "steps": 1000,
         "series": False},
        # an ordinary three-dimensional domain, radix-5 sides, plain FP64
        {"name": "euler3d_100_fp64", "kind": "euler", "d0": 100, "d1": 100, "d2": 100, "prec": "fp64", "steps": 500,
         "series": False},
        # the headline workload
        {"name": "euler3d_256_fp32", "kind": "euler", "d0": 256, "d1": 256, "d2": 256, "prec": "fp32", "steps": 1000,
         "series": False},
        # the elastic precipitate at its configured size, and a smaller one in plain FP64
        {"name": "precip_rk4_192_fp32", "kind": "precip", "d0": 192, "prec": "fp32", "stepper": "rk4", "steps": 100},
        {"name": "precip_rk4_96_fp64", "kind": "precip", "d0": 96, "prec": "fp64", "stepper": "rk4", "steps": 100},
        # unconditionally stable stepping: Newton-Krylov in every step
        {"name": "implicit_128", "kind": "implicit", "d0": 128, "d1": 128, "d2": 0, "dt": 0.1, "steps": 10},
        # gradients for fitting an initial field and a scalar
        {"name": "adjoint_512_fp64", "kind": "adjoint", "d0": 512, "d1": 512, "prec": "fp64", "steps": 400,
         "every": 100},
        # a parameter sweep of uneven sims
        {"name": "sweep_96_fp32", "kind": "sweep", "side": 128, "count": 32, "prec": "fp32", "steps": 300},
        # the transform behind gopf's own steppers, on the program's host array
        {"name": "fourier_128", "kind": "fourier", "d0": 128, "d1": 128, "d2": 128, "prec": "fp64"},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _near(sides, v):
    return min(sides, key=lambda s: abs(math.log(s / v)))


def draw(rng):
    """One more case: the kind by weight, sizes over the logarithm of their range."""
    top = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["euler", "euler", "euler", "precip", "precip", "implicit", "adjoint", "sweep", "fourier"])
        prec = rng.choice(["fp32", "fp64"])
        if kind == "euler" and rng.random() < 0.55:
            a, b = (_near(SMALL + SIDES, _log(rng, 9, 1024)) for _ in range(2))
            c = {"kind": kind, "d0": a, "d1": b, "d2": 0, "prec": prec, "steps": int(_log(rng, 20, 1000)),
                 "series": rng.random() < 0.3}
        elif kind == "euler":
            a = _near(SMALL + [s for s in SIDES if s <= 256], _log(rng, 12, 256))
            c = {"kind": kind, "d0": a, "d1": a, "d2": a, "prec": prec, "steps": int(_log(rng, 20, 600)),
                 "series": rng.random() < 0.2}
        elif kind == "precip":
            a = _near([s for s in SMALL if s >= 15] + [s for s in SIDES if s <= 192], _log(rng, 15, 192))
            c = {"kind": kind, "d0": a, "prec": prec, "stepper": rng.choice(["euler", "rk4", "rk4"]),
                 "steps": int(_log(rng, 10, 100))}
        elif kind == "implicit":
            if rng.random() < 0.7:
                a, b = (_near(SMALL + [s for s in SIDES if s <= 320], _log(rng, 12, 320)) for _ in range(2))
                d = 0
            else:
                a = b = d = _near(SMALL, _log(rng, 9, 48))
            c = {"kind": kind, "d0": a, "d1": b, "d2": d, "dt": round(_log(rng, 0.02, 0.2), 3),
                 "steps": rng.randint(2, 10)}
        elif kind == "adjoint":
            a, b = (_near(SMALL + [s for s in SIDES if s <= 512], _log(rng, 24, 512)) for _ in range(2))
            c = {"kind": kind, "d0": a, "d1": b, "prec": prec, "steps": int(_log(rng, 40, 400)),
                 "every": rng.choice([25, 50, 100])}
        elif kind == "sweep":
            c = {"kind": kind, "side": rng.choice([48, 64, 80, 96, 128, 160]), "count": int(_log(rng, 3, 32)),
                 "prec": prec, "steps": int(_log(rng, 30, 300))}
        else:
            a, b, d = (rng.choice([rng.randint(5, 64), _near(SIDES, _log(rng, 64, 200)), rng.randint(65, 160)])
                       for _ in range(3))
            c = {"kind": kind, "d0": a, "d1": b, "d2": d, "prec": prec}
            if rng.random() < 0.3:
                c["d2"], c["d0"], c["d1"] = 0, a * 3, b * 3
        if _cost(c) <= top:
            return c


def _dims(case):
    d = [case[k] for k in ("d0", "d1", "d2") if case.get(k)]
    return [case["d0"]] * 3 if case["kind"] == "precip" else d


def _classes(case):
    s, k = case["side"], case["count"]
    return [((s, s), k), ((2 * s, 2 * s), k + k // 2), ((4 * s, 4 * s), max(1, k // 2))]


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _fft(n):
    return 5.0 * n * math.log2(max(n, 2))


def work(case):
    """Per step, the state once in and once out and the transforms that a step has (a real
    transform is half a complex one); the host arrays of the read-back are not counted."""
    kind = case["kind"]
    s = 4 if case.get("prec") == "fp32" else 8
    if kind == "sweep":
        n = sum(a * b * k for (a, b), k in _classes(case))
        one = sum(k * _fft(a * b) for (a, b), k in _classes(case))
        return {"bytes": 2.0 * n * s * case["steps"], "flops": case["steps"] * (one + 20.0 * n)}
    n = math.prod(_dims(case))
    if kind == "euler":
        return {"bytes": 2.0 * n * s * case["steps"], "flops": case["steps"] * (_fft(n) + 20.0 * n)}
    if kind == "precip":
        # two fields and the lagged one; per stage two transforms each way, three elastic ones
        stages = 4 if case["stepper"] == "rk4" else 1
        return {"bytes": 5.0 * n * s * case["steps"],
                "flops": case["steps"] * ((2 * stages + 1.5) * _fft(n) + 60.0 * n * stages)}
    if kind == "implicit":
        # about 36 residuals a step (Newton checks and six points per Krylov vector)
        return {"bytes": 36 * 2.0 * n * s * case["steps"], "flops": 36 * case["steps"] * (1.5 * _fft(n) + 40.0 * n)}
    if kind == "adjoint":
        # forward, recompute and reverse
        return {"bytes": 3 * 2.0 * n * s * case["steps"], "flops": 3 * case["steps"] * (_fft(n) + 20.0 * n)}
    return {"bytes": 4 * 16.0 * n, "flops": 2 * _fft(n)}


def tolerance(case):
    """About four times what FP32-bulk is off the plain FP64 path after two passes; interfaces
    amplify rounding locally, so the largest difference is far above the mean one."""
    kind, fp32 = case["kind"], case.get("prec") == "fp32"
    if kind == "implicit":
        # each step's root is found to 1e-7 in the residual's largest value
        return {"rel": 2e-7, "max": 2e-6}
    if kind == "fourier":
        return {"rel": 2e-6, "max": 2e-5} if fp32 else {"rel": 2e-15, "max": 1e-13}
    if not fp32:
        return {"rel": 4e-12, "max": 1e-9}
    if kind == "precip":
        return {"rel": 1.6e-5, "max": 1.2e-4}
    if kind == "adjoint":
        return {"rel": 1.6e-4, "max": 1.2e-3}
    if kind == "sweep":
        return {"rel": 4e-4, "max": 0.18}
    if case["d2"]:
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 1.6e-4, "max": 0.04} if case["steps"] > 300 else {"rel": 4e-5, "max": 4e-3}


# ---------------------------------------------------------------------------
# inputs, the same for the library and for exact()
# ---------------------------------------------------------------------------
def _ch_field(seed, n):
    return 0.5 + 0.1 * (np.random.default_rng(seed).random(n) - 0.5)


def _precip_fields(seed, N):
    """1 inside a centred sphere and 0 outside, plus U(-0.01, 0.01)."""
    rng = np.random.default_rng(seed)
    x = (np.arange(N) - N / 2) ** 2
    r2 = x[:, None, None] + x[None, :, None] + x[None, None, :]
    ball = (r2 < (20.0 * N / 192.0) ** 2).astype(np.float64).reshape(-1)
    return [ball + rng.uniform(-0.01, 0.01, N ** 3) for _ in range(2)]


def _sweep_scalars(seed, sims):
    """(M, kappa) of each sim, between 0.1 and 10."""
    return np.exp(np.random.default_rng(seed + 1).uniform(math.log(0.1), math.log(10.0), (sims, 2)))


def _ch_model(dims, data=None):
    m = G.Model()
    m.AddField("conc", data, n=math.prod(dims))
    for k, v in W.ch_scalars(1.0, 1.0).items():
        m.AddScalar(k, v)
    m.AddEquation(W.CH_EQUATION)
    m.Init()
    return m


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "euler":
        dims = _dims(case)
        m = _ch_model(dims, _ch_field(seed, math.prod(dims)))
        st["solver"] = G.Solver(m, dims, DT3 if case["d2"] else DT2, precision=case["prec"])
    elif kind == "precip":
        N = case["d0"]
        conc, phase = _precip_fields(seed, N)
        m = G.Model()
        m.AddField("conc", conc)
        m.AddField("phase", phase)
        for k, v in W.PRECIPITATE_SCALARS.items():
            m.AddScalar(k, v)
        for name, poly in W.precipitate_polynomials().items():
            m.RegisterPolynomial(name, poly)
        m.RegisterExplicitTerm("LIN_ELAST", G.HomogeneousModulusLinElast("phase", G.CubicMaterial(110.0, 60.0, 30.0),
                                                                         0.01 * np.eye(3)))
        for e in W.PRECIPITATE_EQUATIONS:
            m.AddEquation(e)
        m.Init()
        st["solver"] = G.Solver(m, [N, N, N], 0.01, stepper=case["stepper"], precision=case["prec"])
    elif kind == "implicit":
        dims = _dims(case)
        st["c0"] = _ch_field(seed, math.prod(dims))
        st["solver"] = G.Solver(_ch_model(dims, st["c0"]), dims, case["dt"], stepper="implicitEuler")
    elif kind == "adjoint":
        dims = _dims(case)
        n = math.prod(dims)
        st["c0"] = _ch_field(seed, n)
        st["target"] = _ch_field(seed + 1, n)
        st["solver"] = G.Solver(_ch_model(dims, st["c0"]), dims, DT2, precision=case["prec"])
    elif kind == "sweep":
        classes = _classes(case)
        m = _ch_model((4, 4))
        b = G.Batch(m, classes, DT2, precision=case["prec"])
        for s, (M, kappa) in enumerate(_sweep_scalars(seed, len(b))):
            for k, v in W.ch_scalars(M, kappa).items():
                b.SetScalar(s, k, v)
            b.SetField(s, _ch_field(seed + 2 + s, math.prod(b.shapes[s])))
        st["batch"] = b
    else:
        dims = _dims(case)
        rng = np.random.default_rng(seed)
        n = math.prod(dims)
        st["data"] = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        st["ft"] = G.FourierTransform(dims, precision=case["prec"])
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "euler":
        s = st["solver"]
        if not case["series"]:
            s.Propagate(case["steps"])
            return s.Field("conc").real
        s.MonitorEnergy(BULK, 1.0)
        s.Propagate(case["steps"])
        energy, mass = s.EnergySeries()
        return {"conc": s.Field("conc").real, "energy": energy, "mass": mass}
    if kind == "precip":
        s = st["solver"]
        s.Propagate(case["steps"])
        return {f: s.Field(f).real for f in ("conc", "phase")}
    if kind == "implicit":
        s = st["solver"]
        s.SetField("conc", st["c0"])
        s.Propagate(case["steps"])
        return s.Field("conc").real
    if kind == "adjoint":
        s = st["solver"]
        s.SetField("conc", st["c0"])
        loss, grad, scal = s.Adjoint(case["steps"], st["target"], ["mk"], checkpoint_every=case["every"])
        return {"loss": loss, "grad": grad, "mk": scal["mk"]}
    if kind == "sweep":
        b = st["batch"]
        b.Propagate(case["steps"])
        out, s = [], 0
        for _, k in _classes(case):
            out.append(np.stack([b.Field(i).real for i in range(s, s + k)]))
            s += k
        return out
    ft = st["ft"]
    spectrum = ft.FFT(st["data"].copy())
    return {"spectrum": spectrum, "back": ft.IFFT(spectrum.copy())}


# ---------------------------------------------------------------------------
# the same results in 64 bits, from the equations
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _freqs(dims, dev):
    """Frequencies of the half spectrum, the Nyquist ones +1/2, per axis."""
    out = []
    for a, n in enumerate(dims):
        k = torch.arange(n // 2 + 1 if a == len(dims) - 1 else n, dtype=torch.float64, device=dev) / n
        k = torch.where(k > 0.5, k - 1.0, k)
        out.append(k.reshape([-1 if i == a else 1 for i in range(len(dims))]))
    return out


def _lap(dims, dev):
    return -4.0 * math.pi ** 2 * sum(f * f for f in _freqs(dims, dev))


def _weights(dims, dev):
    """How often each value of the half spectrum stands in the whole one."""
    nx = dims[-1]
    w = torch.full((nx // 2 + 1,), 2.0, dtype=torch.float64, device=dev)
    w[0] = 1.0
    if nx % 2 == 0:
        w[-1] = 1.0
    return w


def _ch_exact(case, seed):
    dev, dims = _device(), _dims(case)
    dt = DT3 if case["d2"] else DT2
    c = torch.from_numpy(_ch_field(seed, math.prod(dims))).to(dev).reshape(dims)
    L, w = _lap(dims, dev), _weights(dims, dev)
    den = 1.0 / (1.0 - dt * (2.0 * L - L * L))
    energy, mass = [], []
    for _ in range(case["steps"]):
        ch = torch.fft.rfftn(c)
        if case["series"]:
            grad = (w * -L * (ch.real ** 2 + ch.imag ** 2)).sum() / c.numel()
            energy.append((c * c * (1.0 - c) ** 2).sum() + 0.5 * grad)
            mass.append(c.sum())
        c = torch.fft.irfftn((ch + dt * L * torch.fft.rfftn(4.0 * c ** 3 - 6.0 * c ** 2)) * den, s=dims)
    conc = c.reshape(-1).cpu().numpy()
    if not case["series"]:
        return conc
    return {"conc": conc, "energy": torch.stack(energy).cpu().numpy(), "mass": torch.stack(mass).cpu().numpy()}


def _elastic_kernel(f, nyquist_free):
    """K(k) with sigma* : strain(k) = K(k) H(k): the equilibrium displacement of the cubic
    material (110, 60, 30) under the misfit 0.01 I, by the adjugate of its 3 x 3 matrix."""
    c11, c12, c44, eps = 110.0, 60.0, 30.0, 0.01
    sig = (c11 + 2.0 * c12) * eps
    # the material's entries: C_iiii, C_iijj and C_ijij
    def entry(i, j, k, l):
        if i == j == k == l:
            return c11
        if i == j and k == l:
            return c12
        return c44 if (i == k and j == l) else 0.0
    A = [[sum(entry(a, j, b, l) * f[j] * f[l] for j in range(3) for l in range(3) if entry(a, j, b, l))
          for b in range(3)] for a in range(3)]
    rhs = [sig * f[a] for a in range(3)]
    minor = lambda i, j: (A[(i + 1) % 3][(j + 1) % 3] * A[(i + 2) % 3][(j + 2) % 3]  # noqa: E731
                          - A[(i + 1) % 3][(j + 2) % 3] * A[(i + 2) % 3][(j + 1) % 3])
    det = sum(A[0][j] * minor(0, j) for j in range(3))
    zero = det == 0.0
    det = torch.where(zero, torch.ones_like(det), det)
    K = 0.0
    for a in range(3):
        wa = sum(minor(b, a) * rhs[b] for b in range(3)) / det
        K = K + sig * nyquist_free[a] * torch.where(zero, torch.zeros_like(wa), wa)
    return K, 0.5 * 3.0 * sig * eps


def _precip_exact(case, seed):
    dev, N, dt = _device(), case["d0"], 0.01
    dims = [N, N, N]
    y = [torch.from_numpy(v).to(dev).reshape(dims) for v in _precip_fields(seed, N)]
    # gopf's frequencies of an index are (row, column, depth)
    fz, fy, fx = _freqs(dims, dev)
    f = [fy + 0.0 * (fx + fz), fx + 0.0 * (fy + fz), fz + 0.0 * (fx + fy)]
    K, estar = _elastic_kernel(f, [torch.where(v.abs() == 0.5, torch.zeros_like(v), v) for v in f])
    D = 0.1 * _lap(dims, dev)

    def sources(c, p):
        H, dH = 3 * p ** 2 - 2 * p ** 3, 6 * p - 6 * p ** 2
        chem = -(0.1 * c * (1 - H) - 0.1 * (1 - c) * H)
        phase = -(-0.05 * c ** 2 * dH + 0.05 * (1 - c) ** 2 * dH + 0.1 * (2 * p - 6 * p ** 2 + 4 * p ** 3))
        return [torch.fft.rfftn(chem), torch.fft.rfftn(phase)]

    lag = torch.zeros_like(y[1])
    for _ in range(case["steps"]):
        H, dH = 3 * lag ** 2 - 2 * lag ** 3, 6 * lag - 6 * lag ** 2
        stress = torch.fft.irfftn(K * torch.fft.rfftn(H), s=dims)
        el = torch.fft.rfftn(dH * (stress - 2.0 * estar * H))
        start = [torch.fft.rfftn(v) for v in y]
        r = sources(*y)
        r[1] = r[1] + el
        if case["stepper"] == "euler":
            new = [(s + dt * k) / (1.0 - dt * D) for s, k in zip(start, r)]
        else:
            new = [s + dt / 6.0 * k for s, k in zip(start, r)]
            for corr, prep in ((0.5, 1.0 / 3.0), (0.5, 1.0 / 3.0), (1.0, 1.0 / 6.0)):
                mid = [torch.fft.irfftn((s + corr * dt * k) / (1.0 - corr * dt * D), s=dims) for s, k in zip(start, r)]
                r = sources(*mid)
                r[1] = r[1] + el
                new = [s + prep * dt * k for s, k in zip(new, r)]
            new = [s / (1.0 - dt * D) for s in new]
        y = [torch.fft.irfftn(s, s=dims) for s in new]
        lag = y[1]
    return {"conc": y[0].reshape(-1).cpu().numpy(), "phase": y[1].reshape(-1).cpu().numpy()}


def _implicit_exact(case, seed):
    """Each step's root by fixed-point iteration of the exponential-integrator update."""
    dev, dims, dt = _device(), _dims(case), case["dt"]
    c = torch.from_numpy(_ch_field(seed, math.prod(dims))).to(dev).reshape(dims)
    L = _lap(dims, dev)
    D = 2.0 * L - L * L
    ex, small = torch.exp(D * dt), D.abs() < 1e-5
    S = torch.where(small, torch.ones_like(D), D)
    source = lambda v: L * torch.fft.rfftn(4.0 * v ** 3 - 6.0 * v ** 2)  # noqa: E731
    for _ in range(case["steps"]):
        orig, prev = torch.fft.rfftn(c) * ex, source(c)
        x = c
        for it in range(200):
            r = source(x)
            upd = prev * (ex - 1.0) / S + (r - prev) / dt * (ex - S * dt - 1.0) / (S * S)
            upd = torch.where(small, 0.5 * dt * (r + prev * ex), upd)
            nxt = torch.fft.irfftn(orig + upd, s=dims)
            off = float((nxt - x).abs().max())
            x = nxt
            if off < 1e-14:
                break
        c = x
    return c.reshape(-1).cpu().numpy()


def _adjoint_exact(case, seed):
    dev, dims = _device(), _dims(case)
    n = math.prod(dims)
    c0 = torch.from_numpy(_ch_field(seed, n)).to(dev).reshape(dims)
    target = torch.from_numpy(_ch_field(seed + 1, n)).to(dev).reshape(dims)
    L, w = _lap(dims, dev), _weights(dims, dev)
    A = 1.0 / (1.0 - DT2 * (2.0 * L - L * L))
    states = [c0]
    for _ in range(case["steps"]):
        c = states[-1]
        new = (torch.fft.rfftn(c) + DT2 * L * torch.fft.rfftn(4.0 * c ** 3 - 6.0 * c ** 2)) * A
        states.append(torch.fft.irfftn(new, s=dims))
    r = states[-1] - target
    loss, lam, mk = float((r * r).sum()), 2.0 * r, 0.0
    for k in range(case["steps"], 0, -1):
        c, lh = states[k - 1], torch.fft.rfftn(lam) * A
        # d c_k / d mk = -dt L^2 A c_k in k-space
        mk += float((w * (-DT2 * L * L) * (lh * torch.fft.rfftn(states[k]).conj()).real).sum()) / n
        lam = torch.fft.irfftn(lh, s=dims) + (12.0 * c ** 2 - 12.0 * c) * torch.fft.irfftn(DT2 * L * lh, s=dims)
    return {"loss": loss, "grad": lam.reshape(-1).cpu().numpy(), "mk": mk}


def _sweep_exact(case, seed):
    dev = _device()
    out, s = [], 0
    classes = _classes(case)
    scal = _sweep_scalars(seed, sum(k for _, k in classes))
    for dims, k in classes:
        n = math.prod(dims)
        c = torch.from_numpy(np.stack([_ch_field(seed + 2 + i, n) for i in range(s, s + k)])).to(dev)
        c = c.reshape((k,) + tuple(dims))
        M, kappa = (torch.from_numpy(scal[s:s + k, j].copy()).to(dev).reshape(k, 1, 1) for j in (0, 1))
        L = _lap(dims, dev)
        A = 1.0 / (1.0 - DT2 * (2.0 * M * L - M * kappa * L * L))
        B = DT2 * M * L * A
        for _ in range(case["steps"]):
            g = torch.fft.rfft2(4.0 * c ** 3 - 6.0 * c ** 2)
            c = torch.fft.irfft2(torch.fft.rfft2(c) * A + g * B, s=dims)
        out.append(c.reshape(k, -1).cpu().numpy())
        s += k
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "euler":
        return _ch_exact(case, seed)
    if kind == "precip":
        return _precip_exact(case, seed)
    if kind == "implicit":
        return _implicit_exact(case, seed)
    if kind == "adjoint":
        return _adjoint_exact(case, seed)
    if kind == "sweep":
        return _sweep_exact(case, seed)
    dims = _dims(case)
    rng = np.random.default_rng(seed)
    n = math.prod(dims)
    x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    return {"spectrum": np.fft.fftn(x.reshape(dims)).reshape(-1), "back": x * n}
