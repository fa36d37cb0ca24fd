"""The work that programs have this library do, as cases that can be timed and compared.

``listed()`` names the cases, ``draw(rng)`` gives one more of the same ranges, ``prepare(case, seed)``
makes what a program holds before the call (states in device memory, a context, the step's
scalars), ``run(state)`` is one pass through the public entry points, ``work(case)`` the bytes and
operations the pass cannot do without, and ``exact(case, seed)`` the same results from plain torch
operations in 64 bits.

Kinds of cases (a program's inner loop in each):
  ot        run_ot's loop body: CFL time step of the state, then one unforced step
  turb      run_turb's loop body: one forced step, then the CFL speed folded into it
  bridge    the MarchBridge scheme's step at a fixed dt/dx, with or without passive species
  ct        the constrained-transport driver's body: one forced CT step, then its CFL speed
  hydro     one step of the 5-variable march, with or without passive scalars
  diag      the diagnostics of a state
  adjoint   the reverse of one forced step, and the derivative along the forcing amplitude
  ensemble  a batch of boxes restarted from given states and advanced some sweeps
"""
import math

import numpy as np
import torch

from glmmhdturb_amd import (BoxSpec, Ensemble, Params, Solver, dxof, hydro_args, march_args, step_args)

GAMMA = 5.0 / 3.0
F = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # a two-dimensional Orszag-Tang run (the test suite's 128 x 128 x 1): launch and latency bound
        dict(name="ot_128x128x1_f64", kind="ot", nx=128, ny=128, nz=1, precision="f64", riemann="hlld", recon="plm"),
        # one small box of driven turbulence, the middle of the ensemble's size range
        dict(name="turb_64_f64", kind="turb", nx=64, ny=64, nz=64, precision="f64", riemann="hlld", recon="ppm"),
        # the benchmark's headline step
        dict(name="turb_256_f64", kind="turb", nx=256, ny=256, nz=256, precision="f64", riemann="hlld", recon="ppm"),
        # run_turb's default reconstruction on a ragged grid in single precision
        dict(name="turb_200x150x121_f32", kind="turb", nx=200, ny=150, nz=121, precision="f32", riemann="hlld", recon="plm"),
        # the bridge libraries' march on the reference's benchmark grid
        dict(name="bridge_480_f32", kind="bridge", nx=480, ny=480, nz=480, precision="f32", recon="plm", nsp=0),
        # constrained transport, forced, in both precisions
        dict(name="ct_256_f64", kind="ct", nx=256, ny=256, nz=256, precision="f64", riemann="hlld", recon="plm"),
        dict(name="ct_180x130x99_f32", kind="ct", nx=180, ny=130, nz=99, precision="f32", riemann="hlld", recon="plm"),
        # the hydro march on the reference's benchmark grid, and a small ragged one with passive scalars
        dict(name="hydro_480_f32", kind="hydro", nx=480, ny=480, nz=480, precision="f32", nsp=0),
        dict(name="hydro_100x75x61_f64_scalars", kind="hydro", nx=100, ny=75, nz=61, precision="f64", nsp=2),
        # diagnostics of the headline grid, printed every few hundred steps of a run
        dict(name="diag_256_f64", kind="diag", nx=256, ny=256, nz=256, precision="f64"),
        # one reverse step at the adjoint benchmark's size
        dict(name="adjoint_128_f64", kind="adjoint", nx=128, ny=128, nz=128, precision="f64", riemann="hlld", recon="ppm"),
        # a batch of small forced boxes of uneven size
        dict(name="ensemble_16_f64", kind="ensemble", nbox=16, small=32, large=64, sweeps=8, precision="f64"),
    ]


def _grid(rng, lo, hi):
    """A cubic or mildly uneven grid whose edges are spread over [lo, hi] by their logarithm."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if rng.random() < 0.3:
        n = max(lo, int(n) // 8 * 8)
        return dict(nx=n, ny=n, nz=n)
    e = [min(hi, max(lo, int(round(n * math.exp(rng.uniform(-0.3, 0.3)))))) for _ in range(3)]
    return dict(nx=e[0], ny=e[1], nz=e[2])


def draw(rng):
    kind = rng.choice(["ot", "turb", "turb", "bridge", "ct", "hydro", "diag", "adjoint", "ensemble"])
    prec = rng.choice(["f64", "f32"])
    if kind == "ot":
        n = rng.randrange(48, 400)
        return dict(kind=kind, nx=n, ny=max(32, int(n * rng.uniform(0.5, 1.0))), nz=rng.choice([1, 1, 2, 5]), precision=prec,
                    riemann=rng.choice(["hlld", "hll", "llf"]), recon=rng.choice(["plm", "ppm"]))
    if kind == "turb":
        return dict(kind=kind, **_grid(rng, 24, 256), precision=prec, riemann=rng.choice(["hlld", "hlld", "hll"]),
                    recon=rng.choice(["plm", "ppm"]))
    if kind == "bridge":
        return dict(kind=kind, **_grid(rng, 32, 320), precision=rng.choice(["f32", "f32", "f64"]),
                    recon=rng.choice(["plm", "ppm_spike"]), nsp=rng.choice([0, 2]))
    if kind == "ct":
        return dict(kind=kind, **_grid(rng, 24, 256), precision=prec, riemann=rng.choice(["hlld", "hll"]),
                    recon=rng.choice(["plm", "plm", "ppm_spike"]))
    if kind == "hydro":
        return dict(kind=kind, **_grid(rng, 32, 360), precision=prec, nsp=rng.choice([0, 2]))
    if kind == "diag":
        return dict(kind=kind, **_grid(rng, 24, 256), precision=prec)
    if kind == "adjoint":
        return dict(kind=kind, **_grid(rng, 24, 120), precision="f64", riemann=rng.choice(["hlld", "hll"]),
                    recon=rng.choice(["plm", "ppm"]))
    return dict(kind="ensemble", nbox=rng.randrange(4, 13), small=rng.randrange(24, 41), large=rng.randrange(48, 73),
                sweeps=8, precision=prec)


# ---------------------------------------------------------------------------------------------
# inputs: fields of random Fourier modes with a falling spectrum, plus grid-scale noise
# ---------------------------------------------------------------------------------------------
class _Modes:
    """Random real fields sum_m a_m cos(2 pi k_m.x + phi_m) of unit variance on a periodic grid; all
    fields of one object share their wave vectors."""

    def __init__(self, rng, shape, kmax=6, count=40, slope=1.8, dev="cuda"):
        nx, ny, nz = shape
        k = rng.integers(-kmax, kmax + 1, size=(count, 3))
        k[(k == 0).all(axis=1)] = (1, 1, 0)
        k[:, 0] *= nx > 1
        k[:, 1] *= ny > 1
        k[:, 2] *= nz > 1
        self.k = k.astype(np.float64)
        self.kk = np.maximum(np.sqrt((self.k ** 2).sum(1)), 1.0)
        self.amp = self.kk ** -slope
        self.amp *= math.sqrt(2.0 / (self.amp ** 2).sum())
        self.shape, self.rng, self.dev = shape, rng, dev
        self.basis = [np.exp(2j * np.pi * self.k[:, d, None] * ((np.arange(n) + 0.5) / n)) for d, n in enumerate(shape)]

    def field(self, weight=None, phase=None):
        """(nz, ny, nx) float64 tensor."""
        nx, ny, nz = self.shape
        a = self.amp if weight is None else self.amp * weight
        ph = self.rng.uniform(0, 2 * np.pi, len(a)) if phase is None else phase
        cx, cy, cz = (torch.from_numpy(b).to(self.dev) for b in (self.basis[0], self.basis[1],
                                                                  self.basis[2] * (a * np.exp(1j * ph))[:, None]))
        zy = (cz[:, :, None] * cy[:, None, :]).reshape(len(a), nz * ny)
        left = torch.cat([zy.real, -zy.imag]).T.contiguous()
        return (left @ torch.cat([cx.real, cx.imag])).reshape(nz, ny, nx)

    def solenoidal(self):
        """Three fields with k.a = 0, of unit variance together."""
        d = self.rng.standard_normal((len(self.amp), 3))
        u = self.k / self.kk[:, None]
        d -= u * (d * u).sum(1, keepdims=True)
        d /= np.maximum(np.sqrt((d ** 2).sum(1, keepdims=True)), 1e-3)
        ph = self.rng.uniform(0, 2 * np.pi, len(self.amp))
        return [self.field(d[:, c], ph) for c in range(3)]


def _rng(seed, salt):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, salt])


def _noise(shape, seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return torch.randn(tuple(reversed(shape)), generator=g, device="cuda", dtype=torch.float64)


def _gas(shape, seed):
    """Density, three velocities and pressure of transonic turbulence."""
    m = _Modes(_rng(seed, 1), shape)
    rho = torch.exp(0.35 * m.field() + 0.01 * _noise(shape, seed, 11))
    v = [0.7 * x + 0.005 * _noise(shape, seed, 12 + c) for c, x in enumerate(m.solenoidal())]
    p = rho ** GAMMA * torch.exp(0.1 * m.field())
    return rho, v, p


def _glm_state(shape, seed, dtype, nsp=0):
    rho, v, p = _gas(shape, seed)
    m = _Modes(_rng(seed, 2), shape)
    b = [0.4 * x for x in m.solenoidal()]
    b[0] += 0.5
    u = torch.empty((9 + nsp,) + rho.shape, dtype=dtype, device="cuda")
    u[0] = rho
    for c in range(3):
        u[1 + c] = rho * v[c]
        u[5 + c] = b[c]
    u[4] = (p / (GAMMA - 1.0) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
            + 0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2))
    u[8] = 0.02 * m.field()
    if nsp:
        x = 1.0 / (1.0 + torch.exp(-3.0 * m.field()))
        u[9], u[10] = rho * x, rho * (1.0 - x)
    return u


def _ct_state(shape, seed, dtype):
    """Face fields from the discrete curl of a vector potential: div B = 0 to rounding."""
    rho, v, p = _gas(shape, seed)
    m = _Modes(_rng(seed, 3), shape)
    a = [m.field(1.0 / m.kk) for _ in range(3)]
    up = lambda f, d: torch.roll(f, -1, 2 - d)  # noqa: E731
    bf = [(up(a[2], 1) - a[2]) - (up(a[1], 2) - a[1]), (up(a[0], 2) - a[0]) - (up(a[2], 0) - a[2]),
          (up(a[1], 0) - a[1]) - (up(a[0], 1) - a[0])]
    s = 0.25 / math.sqrt(sum(float((x * x).mean()) for x in bf) / 3.0)
    bf = [x * s for x in bf]
    bf[2] += 0.2
    u = torch.empty((8,) + rho.shape, dtype=dtype, device="cuda")
    for c in range(3):
        u[5 + c] = bf[c]
        u[1 + c] = rho * v[c]
    bc = [0.5 * (u[5 + c].double() + up(u[5 + c].double(), c)) for c in range(3)]
    u[0] = rho
    u[4] = (p / (GAMMA - 1.0) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
            + 0.5 * (bc[0] ** 2 + bc[1] ** 2 + bc[2] ** 2))
    return u


def _hydro_state(shape, seed, dtype, nsp):
    rho, v, p = _gas(shape, seed)
    u = torch.empty((5 + nsp,) + rho.shape, dtype=dtype, device="cuda")
    u[0] = rho
    for c in range(3):
        u[1 + c] = rho * v[c]
    u[4] = p / 0.4 + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
    if nsp:
        x = 1.0 / (1.0 + torch.exp(-3.0 * _Modes(_rng(seed, 4), shape).field()))
        u[5], u[6] = rho * x, rho * (1.0 - x)
    return u


def _afield(seed, g, dtype):
    """A solenoidal acceleration field of order one in the shells 1-3, as the OU forcing gives."""
    m = _Modes(_rng(seed, 5), (g, g, g), kmax=2, count=24, slope=1.0)
    return torch.stack(m.solenoidal()).to(dtype).contiguous()


def _ot_state(shape, seed, dtype):
    """The Orszag-Tang vortex, displaced by a seeded shift, with small seeded perturbations."""
    nx, ny, nz = shape
    r = _rng(seed, 6)
    sx, sy = r.uniform(0, 1, 2)
    x = 2 * math.pi * ((torch.arange(nx, device="cuda", dtype=torch.float64) + 0.5) / nx + sx)[None, None, :]
    y = 2 * math.pi * ((torch.arange(ny, device="cuda", dtype=torch.float64) + 0.5) / ny + sy)[None, :, None]
    one = torch.ones((nz, ny, nx), device="cuda", dtype=torch.float64)
    m = _Modes(r, shape, kmax=4, count=12)
    rho = 25.0 / (36.0 * math.pi) * torch.exp(0.05 * m.field())
    p = 5.0 / (12.0 * math.pi) * torch.exp(0.05 * m.field())
    sb = 1.0 / math.sqrt(4.0 * math.pi)
    v = [-torch.sin(y) * one, torch.sin(x) * one, 0.02 * m.field()]
    b = [-sb * torch.sin(y) * one, sb * torch.sin(2 * x) * one, 0.02 * m.field()]
    u = torch.empty((9, nz, ny, nx), dtype=dtype, device="cuda")
    u[0] = rho
    for c in range(3):
        u[1 + c] = rho * v[c]
        u[5 + c] = b[c]
    u[4] = p / (GAMMA - 1.0) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + 0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
    u[8] = 0.0
    return u


def _params(case):
    shape = (case["nx"], case["ny"], case["nz"])
    return Params(N=case["nx"], nx=shape[0], ny=shape[1], nz=shape[2], gamma=GAMMA, courant=0.3 if case["kind"] != "ot" else 0.4,
                  cs0=math.sqrt(GAMMA), turb_T=0.5, turb_Ndt=100, comp_frac=0.0, turb_seed=1, turb_gs=64, turb_kmin=1.0,
                  turb_kmax=3.0)


T_NOW = 0.4       # time of the step: the forcing ramp is T_NOW / turb_T
DTDX = 0.05       # dt/dx of the bridge and hydro steps


def _inputs(case, seed):
    """The pass's inputs as tensors and numbers (without a context)."""
    kind, dtype = case["kind"], F[case["precision"]]
    shape = (case["nx"], case["ny"], case["nz"])
    d = {"shape": shape, "p": _params(case)}
    if kind == "ot":
        d["u"] = _ot_state(shape, seed, dtype)
    elif kind == "ct":
        d["u"] = _ct_state(shape, seed, dtype)
    elif kind == "hydro":
        d["u"] = _hydro_state(shape, seed, dtype, case["nsp"])
    else:
        d["u"] = _glm_state(shape, seed, dtype, case.get("nsp", 0))
    if kind in ("turb", "ct", "adjoint"):
        d["afield"] = _afield(seed, 64, dtype)
        q = _ct_prim(d["u"].double(), _P(d["p"])) if kind == "ct" else _c2p(d["u"].double().unbind(0), _P(d["p"]))
        d["dt"] = d["p"].courant * dxof(d["p"]) / float(_cfl(q, _P(d["p"])))
    if kind == "adjoint":
        m = _Modes(_rng(seed, 7), shape)
        d["lam1"] = torch.stack([m.field() + 0.05 * _noise(shape, seed, 70 + v) for v in range(9)])
    return d


def _ens_boxes(case, seed):
    r = _rng(seed, 8)
    sizes = sorted({case["small"], (case["small"] + case["large"]) // 2, case["large"]})
    out = []
    for b in range(case["nbox"]):
        n = sizes[b % len(sizes)]
        out.append(BoxSpec(N=n, amp=1.8e5 * float(r.uniform(0.3, 2.0)) * (min(64, n) / 64.0) ** 3, seed=1000 + b,
                           turb_gs=min(64, n)))
    return out


# ---------------------------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        boxes = _ens_boxes(case, seed)
        ens = Ensemble(boxes, Params(gamma=GAMMA), case["precision"])
        init = [_glm_state(b.shape, int(seed) + 17 * k, F[case["precision"]]) for k, b in enumerate(boxes)]
        ens.graph(True)
        return {"kind": kind, "ens": ens, "init": init, "sweeps": case["sweeps"]}
    d = _inputs(case, seed)
    s = Solver(d["p"], case["precision"])
    st = {"kind": kind, "case": case, "s": s, "p": d["p"], "u": d["u"], "out": s.new_state(d["u"].shape[0])}
    if "afield" in d:
        s.setup_forcing(d["p"], 1.0)
        s.set_afield(d["afield"])
        st["dt"] = d["dt"]
    if kind == "bridge":
        st["args"] = march_args(DTDX, GAMMA, ch=1.0, glm_fac=0.98, recon=case["recon"])
    elif kind == "hydro":
        st["args"] = hydro_args(DTDX)
    elif kind == "ct":
        st["args"] = step_args(d["p"], d["dt"], T_NOW, do_turb=True, riemann=case["riemann"], recon=case["recon"],
                               predictor="oned")
    elif kind == "adjoint":
        st["afield"], st["lam1"] = d["afield"], d["lam1"]
        st["args"] = step_args(d["p"], d["dt"], T_NOW, do_turb=True, riemann=case["riemann"], recon=case["recon"])
    return st


def run(state):
    kind = state["kind"]
    if kind == "ensemble":
        ens = state["ens"]
        for dst, src in zip(ens.u0, state["init"]):
            dst.copy_(src)
        torch.cuda.current_stream().synchronize()   # the ensemble runs on its own stream
        ens.reset()
        ens.step(state["sweeps"])
        ens.sync()
        return [ens.current(b) for b in range(ens.nbox)]
    s, u, out = state["s"], state["u"], state["out"]
    if kind == "ot":
        dt = s.compute_dt(u)
        s.step_plm(u, out, state["p"], dt, 0.0, riemann=state["case"]["riemann"], recon=state["case"]["recon"],
                   scheme="multi", want_cfl=False)
        return out, dt
    if kind == "turb":
        s.step_plm(u, out, state["p"], state["dt"], T_NOW, do_turb=True, riemann=state["case"]["riemann"],
                   recon=state["case"]["recon"])
        return out, s.cfl_max()
    if kind == "bridge":
        if state["case"]["nsp"]:
            s.step_species(u, out, state["args"], state["case"]["nsp"])
        else:
            s.step(u, out, state["args"])
        return out
    if kind == "ct":
        s.ct_step(u, out, state["args"])
        return out, s.cfl_max()
    if kind == "hydro":
        s.hydro_step(u, out, state["args"], nsp=state["case"]["nsp"], cma=state["case"]["nsp"] > 0)
        return out
    if kind == "diag":
        d = s.diagnostics(u)
        return {k: float(v) for k, v in d.items()}
    s.step_adjoint(u, state["lam1"], out, state["args"], state["afield"])
    return out, s.adjoint_force_dot(reset=True)


# planes read and written per cell, and operations per cell (an FMA is two) of the scheme's formulas
PLANES = {"ot": 27, "turb": 18, "bridge": 18, "ct": 24, "hydro": 10, "diag": 9, "adjoint": 27}
FLOPS = {"ot": 2300, "turb": 3000, "bridge": 1500, "ct": 2200, "hydro": 700, "diag": 90, "adjoint": 9000}


def work(case):
    size = 8 if case["precision"] == "f64" else 4
    if case["kind"] == "ensemble":
        cells = sum(b.cells() for b in _ens_boxes(case, 0)) * case["sweeps"]
        return {"bytes": 18 * size * cells, "flops": FLOPS["turb"] * cells}
    cells = case["nx"] * case["ny"] * case["nz"]
    return {"bytes": (PLANES[case["kind"]] + 2 * case.get("nsp", 0)) * size * cells, "flops": FLOPS[case["kind"]] * cells}


# ---------------------------------------------------------------------------------------------
# the same steps in plain torch operations, 64 bits.  Fields are lists of (nz, ny, nx) tensors;
# direction d is tensor axis 2 - d.
# ---------------------------------------------------------------------------------------------
class _P:
    """Scalars of the point functions."""

    def __init__(self, p, ch=1.0, fac=1.0, pfl=None, gamma=None):
        self.g = p.gamma if gamma is None else gamma
        self.smallr, self.smallc = p.smallr, p.smallc
        self.pfl = p.smallr * p.smallc ** 2 / self.g if pfl is None else pfl
        self.ch, self.fac = ch, fac


def _max(a, c):
    return torch.clamp(a, min=c)


def _sq(v):
    return v[0] * v[0] + v[1] * v[1] + v[2] * v[2]


def _c2p(c, P):
    rho = _max(c[0], P.smallr)
    v = [c[1] / rho, c[2] / rho, c[3] / rho]
    pr = _max((P.g - 1.0) * (c[4] - 0.5 * _sq(c[1:4]) / rho - 0.5 * _sq(c[5:8])), P.pfl)
    return [rho, *v, pr, *c[5:9], *[x / rho for x in c[9:]]]


def _p2c(q, P):
    e = q[4] / (P.g - 1.0) + 0.5 * q[0] * _sq(q[1:4]) + 0.5 * _sq(q[5:8])
    return [q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], e, *q[5:9]]


def _fast(q, bn, P):
    c2, b2 = P.g * q[4] / q[0], _sq(q[5:8]) / q[0]
    h = 0.5 * (b2 + c2)
    return torch.sqrt(h + torch.sqrt(_max(h * h - c2 * bn * bn / q[0], 0.0)))


def _cfl(q, P):
    return (((q[1].abs() + _fast(q, q[5], P)) + (q[2].abs() + _fast(q, q[6], P))) + (q[3].abs() + _fast(q, q[7], P))).max()


def _flux(q, d, P):
    """Ideal-MHD flux along d (no normal field and psi components)."""
    un, bn, vb = q[1 + d], q[5 + d], q[1] * q[5] + q[2] * q[6] + q[3] * q[7]
    b2 = _sq(q[5:8])
    pt = q[4] + 0.5 * b2
    e = q[4] / (P.g - 1.0) + 0.5 * q[0] * _sq(q[1:4]) + 0.5 * b2
    f = [q[0] * un]
    f += [q[0] * un * q[1 + c] - bn * q[5 + c] + (pt if c == d else 0.0) for c in range(3)]
    f += [(e + pt) * un - bn * vb]
    f += [torch.zeros_like(un) if c == d else un * q[5 + c] - q[1 + c] * bn for c in range(3)]
    return f + [torch.zeros_like(un)]


def _lo(f, d):
    return torch.roll(f, 1, 2 - d)


def _hi(f, d):
    return torch.roll(f, -1, 2 - d)


def _moncen(l, m, r):
    dl, dr = m - l, r - m
    dc = 0.5 * (dl + dr)
    s = torch.minimum(2.0 * torch.minimum(dl.abs(), dr.abs()), dc.abs())
    return torch.where(dl * dr <= 0.0, torch.zeros_like(s), torch.copysign(s, dc.detach()))


def _half(q, d):
    return [0.5 * _moncen(_lo(x, d), x, _hi(x, d)) for x in q]


def _parabola(l, m, r, c):
    """Monotonised three-point parabola edges with curvature weight c."""
    sl, cu = 0.25 * (r - l), (l - 2.0 * m + r) * c
    a, b = m - sl + cu, m + sl + cu
    dq = b - a
    diff, lim = (m - 0.5 * (a + b)) * dq, dq * dq / 6.0
    flat = (b - m) * (m - a) <= 0.0
    lo = torch.where(flat, m, torch.where(diff > lim, 3.0 * m - 2.0 * b, a))
    hi = torch.where(flat, m, torch.where(diff < -lim, 3.0 * m - 2.0 * a, b))
    return lo, hi


def _jump(p):
    """No neighbouring pressures differ by more than a factor of two."""
    ok = None
    for d in range(3):
        l, r = _lo(p, d), _hi(p, d)
        hi = torch.maximum(p, torch.maximum(l, r))
        lo = _max(torch.minimum(p, torch.minimum(l, r)), 1e-20)
        x = hi / lo <= 2.0
        ok = x if ok is None else ok & x
    return ok


def _select(cond, a, b):
    return [torch.where(cond, x, y) for x, y in zip(a, b)]


def _hlld(L, R, P):
    """Miyoshi & Kusano (2005) in the x-normal frame; L, R share their normal field."""
    bn = L[5]

    def side(q):
        b2 = _sq(q[5:8])
        return q[4] + 0.5 * b2, q[4] / (P.g - 1.0) + 0.5 * q[0] * _sq(q[1:4]) + 0.5 * b2

    (ptL, EL), (ptR, ER) = side(L), side(R)
    cf = torch.maximum(_fast(L, bn, P), _fast(R, bn, P))
    SL = torch.clamp(torch.minimum(L[1], R[1]) - cf, max=0.0)
    SR = _max(torch.maximum(L[1], R[1]) + cf, 0.0)
    aL, aR = SL - L[1], SR - R[1]
    den = aR * R[0] - aL * L[0]
    SM = (aR * R[0] * R[1] - aL * L[0] * L[1] - ptR + ptL) / den
    pts = (aR * R[0] * ptL - aL * L[0] * ptR + L[0] * R[0] * aR * aL * (R[1] - L[1])) / den

    def star(q, S, a, pt, E):
        ds = _max(q[0] * a / (S - SM), 1e-12)
        dk = q[0] * a * (S - SM) - bn * bn
        sm = dk.abs() < 1e-12
        dk = torch.where(sm, torch.ones_like(dk), dk)
        fac = torch.where(sm, torch.zeros_like(dk), bn * (SM - q[1]) / dk)
        gb = torch.where(sm, torch.ones_like(dk), (q[0] * a * a - bn * bn) / dk)
        vy, vz, by, bz = q[2] - q[6] * fac, q[3] - q[7] * fac, q[6] * gb, q[7] * gb
        vb, vbs = q[1] * bn + q[2] * q[6] + q[3] * q[7], SM * bn + vy * by + vz * bz
        Es = (a * E - pt * q[1] + pts * SM + bn * (vb - vbs)) / (S - SM)
        return ds, vy, vz, by, bz, Es, vbs

    dLs, vyL, vzL, byL, bzL, EsL, vbL = star(L, SL, aL, ptL, EL)
    dRs, vyR, vzR, byR, bzR, EsR, vbR = star(R, SR, aR, ptR, ER)
    rL, rR = torch.sqrt(dLs), torch.sqrt(dRs)
    SLs, SRs = SM - bn.abs() / rL, SM + bn.abs() / rR
    sg = torch.where(bn >= 0.0, torch.ones_like(bn), -torch.ones_like(bn))
    den = rL + rR
    vy = (rL * vyL + rR * vyR + (byR - byL) * sg) / den
    vz = (rL * vzL + rR * vzR + (bzR - bzL) * sg) / den
    by = (rL * byR + rR * byL + rL * rR * (vyR - vyL) * sg) / den
    bz = (rL * bzR + rR * bzL + rL * rR * (vzR - vzL) * sg) / den
    vb = SM * bn + vy * by + vz * bz
    z = torch.zeros_like(bn)

    def fan(q, S, Ss, E, ds, vys, vzs, bys, bzs, Es, Ess, outer):
        f = _flux(q, 0, P)
        u = [q[0], q[0] * q[1], q[0] * q[2], q[0] * q[3], E, bn, q[6], q[7], z]
        us = [ds, ds * SM, ds * vys, ds * vzs, Es, bn, bys, bzs, z]
        uss = [ds, ds * SM, ds * vy, ds * vz, Ess, bn, by, bz, z]
        f1 = [a + S * (b - c) for a, b, c in zip(f, us, u)]
        f2 = [a + Ss * b - (Ss - S) * c - S * e for a, b, c, e in zip(f, uss, us, u)]
        return _select(outer, f1, f2)

    left = fan(L, SL, SLs, EL, dLs, vyL, vzL, byL, bzL, EsL, EsL - rL * (vbL - vb) * sg, SLs >= 0.0)
    right = fan(R, SR, SRs, ER, dRs, vyR, vzR, byR, bzR, EsR, EsR + rR * (vbR - vb) * sg, SRs < 0.0)
    return _select(SM >= 0.0, left, right)


def _two_wave(L, R, P, riemann, ch):
    """HLL or LLF in the x-normal frame."""
    cL, cR = _fast(L, L[5], P), _fast(R, R[5], P)
    fL, fR, uL, uR = _flux(L, 0, P), _flux(R, 0, P), _p2c(L, P), _p2c(R, P)
    if riemann == "llf":
        s = _max(torch.maximum(L[1].abs() + cL, R[1].abs() + cR), ch)
        return [0.5 * (a + b) - 0.5 * s * (y - x) for a, b, x, y in zip(fL, fR, uL, uR)]
    SL = torch.clamp(torch.minimum(L[1] - cL, R[1] - cR), max=0.0)
    SR = _max(torch.maximum(L[1] + cL, R[1] + cR), 0.0)
    return [(SR * a - SL * b + SL * SR * (y - x)) / (SR - SL) for a, b, x, y in zip(fL, fR, uL, uR)]


def _rot(q, d):
    i = [d, (d + 1) % 3, (d + 2) % 3]
    return [q[0], *[q[1 + k] for k in i], q[4], *[q[5 + k] for k in i], *q[8:9]]


def _unrot(f, d):
    out = list(f)
    for c in range(3):
        out[1 + (d + c) % 3], out[5 + (d + c) % 3] = f[1 + c], f[5 + c]
    return out


def _riemann(Lq, Rq, d, P, riemann):
    """GLM flux through a d face: floors, the (Bn, psi) pair, the solver."""
    L, R = _rot(Lq, d), _rot(Rq, d)
    for q in (L, R):
        q[0], q[4] = _max(q[0], P.smallr), _max(q[4], P.pfl)
    bn = 0.5 * (L[5] + R[5]) - (R[8] - L[8]) * (0.5 / P.ch)
    psi = 0.5 * (L[8] + R[8]) - 0.5 * P.ch * (R[5] - L[5])
    L[5], R[5] = bn, bn
    f = _hlld(L, R, P) if riemann == "hlld" else _two_wave(L, R, P, riemann, P.ch)
    f = list(f)
    f[5], f[8] = psi, P.ch * P.ch * bn
    f = _unrot(f, d)
    return f[:9] + [f[0] * torch.where(f[0] >= 0.0, a, b) for a, b in zip(Lq[9:], Rq[9:])]


def _kick(af, shape, p):
    """ramp times the trilinear interpolation of the (3, g, g, g) forcing field to the cell centres."""
    g = af.shape[-1]
    out = af
    for d in range(3):
        n = shape[d]
        c = (torch.arange(n, device=af.device, dtype=torch.float64) + 0.5) / n * g
        i = torch.floor(c)
        w = (c - i).reshape([-1] + [1] * d)
        i = i.long()
        out = out.index_select(3 - d, i % g) * (1.0 - w) + out.index_select(3 - d, (i + 1) % g) * w
    return min(T_NOW / p.turb_T, 1.0) * out


def _force(r, acc, dt, P, min_rho=1e-5):
    """Momentum kick with the energy bookkeeping of the OU forcing."""
    rho = _max(r[0], P.smallr)
    fl = r[0] * P.smallc ** 2
    e, m = r[4], []
    for c in range(3):
        e = torch.maximum(e - 0.5 * r[1 + c] ** 2 / rho, fl)
    for c in range(3):
        m.append(r[1 + c] + rho * acc[c] * dt)
        e = torch.maximum(e + 0.5 * m[c] ** 2 / rho, fl)
    on = r[0] >= min_rho
    return [r[0], *[torch.where(on, a, b) for a, b in zip(m, r[1:4])], torch.where(on, e, r[4]), *r[5:]]


def _glm_step(u, P, dtdx, *, riemann, recon, predictor, guard, revert, floor, kick=None, dt=0.0):
    """One step of the conserved fields u (9, or 11 with species); returns the new fields."""
    q = _c2p(u, P)
    nv = len(u)
    up = _jump(q[4]) if recon == "ppm" else None
    mh = None
    if predictor == "full":
        acc = [0.0] * 9
        for d in range(3):
            hs = _half(q[:9], d)
            fp, fm = _flux([a + b for a, b in zip(q, hs)], d, P), _flux([a - b for a, b in zip(q, hs)], d, P)
            acc = [a + b - c for a, b, c in zip(acc, fp, fm)]
        mh = _c2p([a - 0.5 * dtdx * b for a, b in zip(_p2c(q, P), acc)], P)
    tot = [0.0] * nv
    for d in range(3):
        hs = _half(q, d)
        m = mh
        if predictor != "full":
            fp, fm = _flux([a + b for a, b in zip(q, hs)], d, P), _flux([a - b for a, b in zip(q, hs)], d, P)
            m = _c2p([a - 0.5 * dtdx * (b - c) for a, b, c in zip(_p2c(q, P), fp, fm)], P)
            m += [q[v] - dtdx * q[1 + d] * hs[v] for v in range(9, nv)]
        if revert:
            m = _select((m[0] <= P.smallr) | (m[4] <= P.pfl), q, m)
        if recon == "plm":
            lo, hi = [a - b for a, b in zip(m, hs)], [a + b for a, b in zip(m, hs)]
        else:
            e = [_parabola(_lo(x, d), x, _hi(x, d), 1.0 / 12.0 if recon == "ppm" else 1.0 / 6.0) for x in q]
            if recon == "ppm_spike":
                for v, least in ((0, P.smallr), (4, P.pfl)):
                    e[v] = (_max(e[v][0], least), _max(e[v][1], least))
            lo, hi = [a + (x[0] - b) for a, x, b in zip(m, e, q)], [a + (x[1] - b) for a, x, b in zip(m, e, q)]
            if recon == "ppm":
                lo = _select(up, lo, [a - b for a, b in zip(m, hs)])
                hi = _select(up, hi, [a + b for a, b in zip(m, hs)])
        if guard == "iflo":
            lo = _select((lo[0] < P.smallr) | (lo[4] < P.pfl), q, lo)
            hi = _select((hi[0] < P.smallr) | (hi[4] < P.pfl), q, hi)
        elif guard == "clamp":
            for s in (lo, hi):
                s[0], s[4] = _max(s[0], P.smallr), _max(s[4], P.pfl)
        f = _riemann([_lo(x, d) for x in hi], lo, d, P, riemann)
        tot = [a + (b - _hi(b, d)) for a, b in zip(tot, f)]
        del lo, hi, f, hs
    r = [a + dtdx * b for a, b in zip(u, tot)]
    if floor:
        e = P.pfl / (P.g - 1.0) + 0.5 * _sq(r[5:8])
        low = r[0] < P.smallr
        z = torch.zeros_like(e)
        r[0], r[4] = torch.where(low, z + P.smallr, r[0]), torch.where(low, e, r[4])
        r[1:4] = [torch.where(low, z, x) for x in r[1:4]]
    r[8] = r[8] * P.fac
    return r if kick is None else _force(r, kick, dt, P)


def _cube(p, dt):
    """P of a step of the cube scheme: cleaning speed and psi decay."""
    dx = dxof(p)
    ch = p.courant * dx / dt / 3.0 * p.glm_ch_scale
    return _P(p, ch, math.exp(-(ch * ch / (p.glm_cp_coef * p.boxlen * ch)) * dt))


def _ct_prim(u, P):
    bc = [0.5 * (u[5 + c] + _hi(u[5 + c], c)) for c in range(3)]
    return _c2p([*[u[v] for v in range(5)], *bc], P)


def _ct_step(u, P, dtdx, riemann, recon, kick, dt):
    q = _ct_prim(u, P)
    flx = []
    for d in range(3):
        hs = _half(q, d)
        fp, fm = _flux([a + b for a, b in zip(q, hs)], d, P), _flux([a - b for a, b in zip(q, hs)], d, P)
        m = _c2p([a - 0.5 * dtdx * (b - c) for a, b, c in zip(_p2c(q, P), fp, fm)], P)
        if recon == "plm":
            lo, hi = [a - b for a, b in zip(m, hs)], [a + b for a, b in zip(m, hs)]
        else:
            e = [_parabola(_lo(x, d), x, _hi(x, d), 1.0 / 6.0) for x in q]
            lo, hi = [a + (x[0] - b) for a, x, b in zip(m, e, q)], [a + (x[1] - b) for a, x, b in zip(m, e, q)]
        for s in (lo, hi):
            s[0], s[4] = _max(s[0], P.smallr), _max(s[4], P.pfl)
        L, R = _rot([_lo(x, d) for x in hi], d), _rot(lo, d)
        L[5], R[5] = u[5 + d], u[5 + d]
        f = _hlld(L, R, P) if riemann == "hlld" else _two_wave(L, R, P, riemann, 0.0)
        f = list(f)
        f[5] = torch.zeros_like(f[0])
        flx.append(_unrot(f, d))
    X, Y, Z = flx
    ez = 0.25 * (Y[5] + _lo(Y[5], 0) - X[6] - _lo(X[6], 1))
    ex = 0.25 * (Z[6] + _lo(Z[6], 1) - Y[7] - _lo(Y[7], 2))
    ey = 0.25 * (X[7] + _lo(X[7], 2) - Z[5] - _lo(Z[5], 0))
    r = [u[v] + dtdx * ((X[v] - _hi(X[v], 0)) + (Y[v] - _hi(Y[v], 1)) + (Z[v] - _hi(Z[v], 2))) for v in range(5)]
    b = [u[5] - dtdx * ((_hi(ez, 1) - ez) - (_hi(ey, 2) - ey)), u[6] - dtdx * ((_hi(ex, 2) - ex) - (_hi(ez, 0) - ez)),
         u[7] - dtdx * ((_hi(ey, 0) - ey) - (_hi(ex, 1) - ex))]
    low = r[0] < P.smallr
    z = torch.zeros_like(r[0])
    e = P.pfl / (P.g - 1.0) + 0.5 * _sq(q[5:8])
    r = [torch.where(low, z + P.smallr, r[0]), *[torch.where(low, z, x) for x in r[1:4]], torch.where(low, e, r[4])]
    return _force(r, kick, dt, P) + b


def _hydro_step(u, dtdx, nsp, g=1.4, least=1e-6):
    rho = _max(u[0], least)
    v = [u[1] / rho, u[2] / rho, u[3] / rho]
    q = [rho, *v, _max((g - 1.0) * (u[4] - 0.5 * rho * _sq(v)), least), *[x / rho for x in u[5:]]]

    def cons(q):
        return [q[0], *[q[0] * x for x in q[1:4]], q[4] / (g - 1.0) + 0.5 * q[0] * _sq(q[1:4]), *[q[0] * x for x in q[5:]]]

    def flux(q, U, d):
        f = [x * q[1 + d] for x in U]
        f[1 + d] = f[1 + d] + q[4]
        f[4] = (U[4] + q[4]) * q[1 + d]
        return f

    out = cons(q)
    for d in range(3):
        s = [_moncen(_lo(x, d), x, _hi(x, d)) for x in q]
        un, sn, h = q[1 + d], s[1 + d], 0.5 * dtdx
        m = [x - h * un * y for x, y in zip(q, s)]
        m[0] = m[0] - h * q[0] * sn
        m[1 + d] = m[1 + d] - h * s[4] / q[0]
        m[4] = m[4] - h * g * q[4] * sn
        lo, hi = [a - 0.5 * b for a, b in zip(m, s)], [a + 0.5 * b for a, b in zip(m, s)]
        for e in (lo, hi):
            e[0], e[4] = _max(e[0], least), _max(e[4], least)
        L, R = [_lo(x, d) for x in hi], lo
        UL, UR = cons(L), cons(R)
        FL, FR = flux(L, UL, d), flux(R, UR, d)
        aL, aR = torch.sqrt(g * L[4] / L[0]), torch.sqrt(g * R[4] / R[0])
        sL, sR = torch.minimum(L[1 + d] - aL, R[1 + d] - aR), torch.maximum(L[1 + d] + aL, R[1 + d] + aR)
        f = [(sR * a - sL * b + sL * sR * (y - x)) / (sR - sL) for a, b, x, y in zip(FL, FR, UL, UR)]
        f[5:] = [f[0] * torch.where(f[0] >= 0.0, a, b) for a, b in zip(L[5:], R[5:])]
        f = _select(sL >= 0.0, FL, _select(sR <= 0.0, FR, f))
        out = [a - dtdx * (_hi(b, d) - b) for a, b in zip(out, f)]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return None        # the forcing realisation is the library's own random stream
    d = _inputs(case, seed)
    p, shape = d["p"], d["shape"]
    u = d["u"].double().unbind(0)
    dx = dxof(p)
    if kind == "ot":
        dt = p.courant * dx / float(_cfl(_c2p(u, _P(p)), _P(p)))
        r = _glm_step(u, _cube(p, dt), dt / dx, riemann=case["riemann"], recon=case["recon"], predictor="full", guard="none",
                      revert=True, floor=True)
        return torch.stack(r), dt
    if kind == "bridge":
        r = _glm_step(u, _P(p, 1.0, 0.98, pfl=1e-6), DTDX, riemann="hll", recon=case["recon"], predictor="oned",
                      guard="clamp", revert=False, floor=False)
        return torch.stack(r)
    if kind == "hydro":
        return torch.stack(_hydro_step(u, DTDX, case["nsp"]))
    if kind == "diag":
        m2, b2 = _sq(u[1:4]), _sq(u[5:8])
        db = sum(_hi(u[5 + c], c) - _lo(u[5 + c], c) for c in range(3)).abs() / (2.0 * dx)
        mass, ke2 = float(u[0].sum()), float((m2 / _max(u[0], p.smallr)).sum())
        vrms = math.sqrt(ke2 / mass)
        xh = float(((u[1] * u[5] + u[2] * u[6] + u[3] * u[7]) / u[0]).sum())
        vals = [mass, ke2, float(db.max()), float(u[0].min()), 1.0, float((0.5 * m2 / u[0]).sum()), float((0.5 * b2).sum()),
                xh, float(u[4].sum()), float((u[8] * u[8]).sum())]
        keys = ("mass", "ke2", "divbmax", "rhomin", "finite", "ekin", "emag", "cross_helicity", "etot", "psi2")
        return dict(zip(keys, vals), vrms=vrms, mach=vrms / p.cs0)
    kick = _kick(d["afield"].double(), shape, p).unbind(0)
    if kind == "ct":
        r = _ct_step(u, _P(p), d["dt"] / dx, case["riemann"], case["recon"], kick, d["dt"])
        out = torch.stack(r)
        return out, float(_cfl(_ct_prim(out, _P(p)), _P(p)))
    opt = dict(riemann=case["riemann"], recon=case["recon"], predictor="full", guard="iflo", revert=True, floor=True, dt=d["dt"])
    if kind == "turb":
        P = _cube(p, d["dt"])
        r = _glm_step(u, P, d["dt"] / dx, kick=kick, **opt)
        return torch.stack(r), float(_cfl(_c2p(r, P), P))
    x = [t.clone().requires_grad_(True) for t in u]
    s = torch.ones((), dtype=torch.float64, device="cuda", requires_grad=True)
    r = _glm_step(x, _cube(p, d["dt"]), d["dt"] / dx, kick=[a * s for a in kick], **opt)
    g = torch.autograd.grad(sum((a * b).sum() for a, b in zip(r, d["lam1"])), [*x, s])
    return torch.stack(g[:9]), float(g[9])
