"""Timed workloads of the library: operator applies, whole sweeps and a gradient step.

A case is a dict of plain values.  ``prepare`` builds what a program holds before the call
(operator, solver, device tensors), ``run`` makes one pass through the public entry points,
``work`` states what a pass cannot do without, ``tolerance`` how far another correct
implementation may be, and ``exact`` computes the same outputs in float64 with plain torch,
from the formulas and without the library.

Lengths are in units of the smallest radius unless a case's solver takes physical units.
"""
import ctypes
import math

import numpy as np
import torch

import cumpm_amd
from cumpm_amd import _capi as C
from cumpm_amd import autograd as A

A.load_with_torch()

# Ewald splitting parameter of every case but the large random one (the library's default)
XI = 0.5


def listed():
    return [
        # one right-hand side on a small lattice: a program that solves one system at a time;
        # launches and latency are all there is (simple cubic 8^3, spacing 3, grid 32^3, support 8)
        dict(name="apply-cubic512-fp64-b1", kind="apply", shape="cubic", n=512, spacing=3.0, tol=1e-8, grid=32,
             support=8, rhs=1, prec="double"),
        # the monolayer sweep's inner apply: 10 frequencies x 3 polarisations in one batch
        dict(name="apply-hex4000-mixed-b30", kind="apply", shape="hex", cols=80, rows=50, tol=1e-6, rhs=30, prec="mixed"),
        # the same monolayer in FP64, one frequency with three polarisations
        dict(name="apply-hex4000-fp64-b3", kind="apply", shape="hex", cols=80, rows=50, tol=1e-6, rhs=3, prec="double"),
        # a three-dimensional assembly on a grid of odd lengths with a Bloch wave vector
        dict(name="apply-random7001-bloch-mixed-b5", kind="apply", shape="random", n=7001, tol=1e-4, rhs=5, prec="mixed",
             kx=0.05, ky=-0.03),
        # the largest assembly: 100,000 spheres on 256^3, 4 frequencies x 3 polarisations
        dict(name="apply-random100k-mixed-b12", kind="apply", shape="random", n=100000, tol=1e-6, xi=0.9292, grid=256,
             support=8, rhs=12, prec="mixed"),
        # the monolayer with quadrupoles on every particle, a batch of 15
        dict(name="apply-quads-hex4000-mixed-b15", kind="apply", shape="hex", cols=80, rows=50, tol=1e-6, rhs=15,
             prec="mixed", quads="all"),
        # quadrupoles on part of a three-dimensional assembly, FP64, one frequency
        dict(name="apply-quads-random1500-fp64-b3", kind="apply", shape="random", n=1500, tol=1e-4, rhs=3, prec="double",
             quads="half"),
        # spheres of many radii (each its own), 20 frequencies of one polarisation
        dict(name="apply-poly1000-mixed-b20", kind="poly", n=1000, tol=1e-6, rhs=20, prec="mixed"),
        # an isolated assembly (open boundaries, as for electron energy loss) with quadrupoles
        dict(name="apply-direct3000-quads-mixed-b6", kind="direct", n=3000, rhs=6, prec="mixed", quads="all"),
        # the headline sweep over a trajectory of two frames: batched, FP32 inner iterations
        # with FP64 residuals, 10 frequencies x 3 polarisations per frame
        dict(name="sweep-hex4000-refined-2frames", kind="sweep", shape="hex", cols=80, rows=50, tol=1e-6, freqs=10,
             frames=2, method="gmres", prec="refined", batched=True),
        # the reference's order on a three-dimensional lattice: one system after the other with
        # guesses from the previous frequencies, BiCGSTAB, mixed precision, tolerance 1e-3
        dict(name="sweep-cubic4096-bicgstab-auto", kind="sweep", shape="cubic", n=4096, spacing=2.4, tol=1e-3, freqs=4,
             frames=1, method="bicgstab", prec="auto", batched=False),
        # a step of parameter fitting: forward solve, loss, adjoint solve, gradients (FP64)
        dict(name="grad-hex120-quads-fp64", kind="grad", cols=12, rows=10, tol=1e-6, freqs=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: sizes spread over their logarithm, odd ones among them."""
    kind = rng.choice(["apply", "apply", "apply", "apply", "quads", "quads", "poly", "direct", "sweep", "sweep", "grad"])
    prec = rng.choice(["mixed", "mixed", "double"])
    tol = rng.choice([1e-3, 1e-4, 1e-6])
    if kind in ("apply", "quads"):
        quads = rng.choice(["all", "half"]) if kind == "quads" else "none"
        shape = rng.choice(["hex", "random", "random", "cubic"])
        if shape == "hex":
            c = dict(kind="apply", shape="hex", cols=_log(rng, 12, 90), rows=2 * _log(rng, 6, 28))
            n = c["cols"] * c["rows"]
        else:
            n = _log(rng, 400, 3000 if quads != "none" else 30000)
            c = dict(kind="apply", shape=shape, n=n)
            if shape == "cubic":
                c["n"] = n = max(8, round(n ** (1 / 3))) ** 3
                c["spacing"] = round(rng.uniform(2.3, 3.0), 3)
        c.update(tol=tol, rhs=max(1, min(_log(rng, 1, 48), 300000 // n)), prec=prec, quads=quads)
        if rng.random() < 0.25:
            c.update(kx=round(rng.uniform(-0.1, 0.1), 4), ky=round(rng.uniform(-0.1, 0.1), 4))
        return c
    if kind == "poly":
        return dict(kind="poly", n=_log(rng, 100, 1300), tol=tol, rhs=_log(rng, 1, 60), prec=prec)
    if kind == "direct":
        return dict(kind="direct", n=_log(rng, 50, 5000), rhs=_log(rng, 1, 20), prec=prec,
                    quads=rng.choice(["none", "half", "all"]))
    if kind == "sweep":
        method = rng.choice(["gmres", "bicgstab"])
        if rng.random() < 0.5:
            return dict(kind="sweep", shape="hex", cols=_log(rng, 12, 80), rows=2 * _log(rng, 6, 25), tol=1e-6,
                        freqs=rng.randint(3, 10), frames=rng.randint(1, 2), method=method, prec="refined", batched=True)
        return dict(kind="sweep", shape="cubic", n=_log(rng, 8, 16) ** 3, spacing=round(rng.uniform(2.3, 3.0), 3),
                    tol=1e-3, freqs=rng.randint(2, 5), frames=1, method=method, prec="auto", batched=rng.random() < 0.5)
    return dict(kind="grad", cols=_log(rng, 9, 16), rows=2 * _log(rng, 4, 7), tol=rng.choice([1e-4, 1e-6]),
                freqs=rng.randint(1, 5))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _rng(seed):
    return np.random.default_rng([int(seed), 20])


def _geometry(case, rng):
    """(positions (N, 3), box) in units of the radius; at most a few pairs of the displaced
    lattices overlap, and slightly."""
    if case["shape"] == "hex":
        cols, rows, s = case["cols"], case["rows"], 2.2
        j, i = np.meshgrid(np.arange(rows), np.arange(cols), indexing="ij")
        pos = np.stack([((i + 0.5 * (j % 2)) * s).ravel(), (j * s * math.sqrt(3) / 2).ravel(), np.zeros(i.size)], 1)
        return pos + rng.normal(0.0, 0.04, pos.shape), np.array([cols * s, rows * s * math.sqrt(3) / 2, 50.0])
    if case["shape"] == "cubic":
        m = round(case["n"] ** (1 / 3))
        s = case["spacing"]
        g = (np.arange(m) + 0.5) * s
        pos = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
        return pos + rng.uniform(-0.05, 0.05, pos.shape), np.full(3, m * s)
    # a random subset of lattice sites, each displaced: volume fraction about 0.3
    s = np.array([2.33, 2.378, 2.43])
    m = math.ceil(case["n"] ** (1 / 3))
    g = np.arange(m) + 0.5
    sites = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3) * s
    pos = sites[rng.permutation(len(sites))[:case["n"]]]
    return pos + rng.uniform(-0.18, 0.18, pos.shape), m * s


def _poly_geometry(case, rng):
    """Radii uniform in 1 to 4, placed one after the other where they overlap none (periodic),
    at a volume fraction of about 0.2."""
    n = case["n"]
    L, rad, pos, k = 7.635 * n ** (1 / 3), rng.uniform(1.0, 4.0, n), np.zeros((n, 3)), 0
    while k < n:
        c = rng.uniform(0.0, L, 3)
        d = pos[:k] - c
        d -= L * np.round(d / L)
        if np.all(np.einsum("ij,ij->i", d, d) >= (rad[:k] + rad[k]) ** 2):
            pos[k] = c
            k += 1
    return pos, np.full(3, L), rad


def _quad_particles(case, N):
    q = case.get("quads", "none")
    return np.arange(N) if q == "all" else np.arange(0, N, 2) if q == "half" else np.zeros(0, int)


def _drude(omega):
    return 4.0 - 1.7 ** 2 / (omega ** 2 + 1j * omega * 0.08)


def _self_coef(eps):
    return -3.0 / (4.0 * np.pi * (1.0 - eps))


def _apply_inputs(case, seed):
    """Positions, box, radii, quadrupole particles, self coefficients [B][N] and x [B][n]."""
    rng = _rng(seed)
    radii = None
    if case["kind"] == "poly":
        pos, box, radii = _poly_geometry(case, rng)
    elif case["kind"] == "direct":
        pos, box = _geometry(dict(shape="random", n=case["n"]), rng)
    else:
        pos, box = _geometry(case, rng)
    N, B = len(pos), case["rhs"]
    q = _quad_particles(case, N)
    eps = _drude(np.linspace(0.2, 0.8, B) if B > 1 else np.array([0.45]))
    sc = np.repeat(_self_coef(eps)[:, None], N, 1)
    x = rng.standard_normal((B, 3 * N + 5 * len(q), 2)).view(np.complex128)[..., 0]
    return pos, box, radii, q, np.ascontiguousarray(sc), x


def _frames(case, seed):
    rng = _rng(seed)
    got = [_geometry(case, rng) for _ in range(case["frames"])]
    return np.stack([p for p, _ in got]), got[0][1]


def _sweep_eps(case, seed):
    return _drude(np.linspace(0.2, 0.8, case["freqs"]) + _rng(seed + 7).uniform(-0.01, 0.01, case["freqs"]))


def _grad_inputs(case, seed):
    rng = _rng(seed)
    pos, box = _geometry(dict(shape="hex", cols=case["cols"], rows=case["rows"]), rng)
    N = len(pos)
    spread = 1.0 + rng.uniform(-0.05, 0.05, (3, N))
    par = [4.0 * spread[0], 1.7 * spread[1], 0.08 * spread[2]]  # eps_inf, wp, gamma
    return pos, box, np.linspace(0.25, 0.75, case["freqs"] + 2)[1:-1], par


# ---------------------------------------------------------------------------
# The library's side
# ---------------------------------------------------------------------------

_PREC = {"double": C.PREC_DOUBLE, "mixed": C.PREC_MIXED}


class _Op:
    """An operator handle of the C API with its input and output on the GPU."""

    def __init__(self, case, seed):
        lib = C.load()
        pos, box, radii, q, sc, x = _apply_inputs(case, seed)
        self.h = ctypes.c_void_p()
        if case["kind"] == "direct":
            one = np.ones(1)
            C.check(lib.mpm_op_create_direct(C.dptr(one), 1, ctypes.byref(self.h)))
        else:
            d = C.OpDesc()
            d.box[:] = [float(v) for v in box]
            d.errortol = case["tol"]
            d.xi = case.get("xi", XI)
            if case.get("grid"):
                d.grid[:] = [case["grid"]] * 3
            d.support = case.get("support", 0)
            if radii is None:
                C.check(lib.mpm_op_create(ctypes.byref(d), ctypes.byref(self.h)))
            else:
                C.check(lib.mpm_op_create_poly(ctypes.byref(d), C.dptr(radii), radii.size, ctypes.byref(self.h)))
        if len(q):
            C.check(lib.mpm_op_set_quads(self.h, (ctypes.c_int * len(q))(*[int(v) for v in q]), len(q)))
        xyz = np.ascontiguousarray(pos)
        C.check(lib.mpm_op_set_positions(self.h, C.dptr(xyz), len(pos)))
        if case.get("kx") or case.get("ky"):
            C.check(lib.mpm_op_set_bloch(self.h, case.get("kx", 0.0), case.get("ky", 0.0)))
        C.check(lib.mpm_op_set_self_coef(self.h, C.dptr(sc.view(np.float64)), sc.shape[0]))
        self.x = torch.from_numpy(x).cuda()
        self.y = torch.zeros_like(self.x)
        self.B = case["rhs"]
        self.prec = _PREC[case["prec"]]
        self.parts = C.PART_REAL if case["kind"] == "direct" else C.PART_ALL

    def __del__(self):
        if self.h and C._lib is not None:
            C._lib.mpm_op_destroy(self.h)

    def run(self):
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        C.check(C.load().mpm_op_apply(self.h, ctypes.c_void_p(self.x.data_ptr()), ctypes.c_void_p(self.y.data_ptr()),
                                      self.B, self.prec, self.parts, stream))
        return self.y


class _Sweep:
    """A dipole solver and the frames of a trajectory."""

    def __init__(self, case, seed):
        self.frames, box = _frames(case, seed)
        self.solver = cumpm_amd.dipole_solver(box, _sweep_eps(case, seed), radius=1.0, tol=case["tol"], quiet=True,
                                              solver_type=case["method"], field_type="monodisperse",
                                              precision=case["prec"], batched=case["batched"])

    def run(self):
        self.solver.reset()
        self.solver.compute(self.frames)
        return self.solver.get_dipoles(physical=False)


class _Grad:
    """Drude parameters of every particle and the operator of a differentiable solve."""

    def __init__(self, case, seed):
        pos, box, self.omega, par = _grad_inputs(case, seed)
        self.op = A.Operator(box, pos, quadrupoles=True, ewald_tol=case["tol"], tol=1e-10)
        self.par = [torch.from_numpy(p).cuda() for p in par]
        self.b = A.uniform_rhs(self.op, np.eye(3), len(self.omega))

    def run(self):
        W, op = len(self.omega), self.op
        par = [p.clone().requires_grad_(True) for p in self.par]
        sc = A.self_coefficient(A.drude(self.omega, *par))
        x = op.solve(self.b, sc.repeat_interleave(3, 0))
        loss = A.extinction(op.dipoles(x).reshape(W, 3, op.N, 3), np.eye(3), self.omega)
        loss = loss + op.quadrupoles(x).abs().square().sum()
        loss.backward()
        op.reports.clear()
        return {"x": x.detach(), "eps_inf": par[0].grad, "wp": par[1].grad, "gamma": par[2].grad}


def prepare(case, seed):
    return {"sweep": _Sweep, "grad": _Grad}.get(case["kind"], _Op)(case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------------------
# What a pass needs, and how exact it is
# ---------------------------------------------------------------------------

def _sizes(case):
    """(N, Q, grid lengths, stencil points, cutoff) of a periodic case."""
    if case["kind"] == "poly":
        N, Q, amax = case["n"], 0, 4.0
        box = np.full(3, 7.635 * N ** (1 / 3))
    else:
        c = dict(case, shape="hex") if case["kind"] == "grad" else case
        pos, box = _geometry(c, _rng(0))
        N, amax = len(pos), 1.0
        Q = N if case["kind"] == "grad" else len(_quad_particles(case, N))
    n, _, P, rc, _, _ = _sizing(case, box, amax)
    w = P if case["kind"] == "poly" else 2 * (P // 2) + 1
    return N, Q, n, w ** 3, rc, box


def _apply_work(case, B):
    N, Q, n, stencil, rc, box = _sizes(case)
    V = n[0] * n[1] * n[2]
    comps = 1 if case["kind"] == "poly" else 8 if Q else 3
    per = 3 if case["kind"] == "poly" else 0  # the poly stencil carries a vector weight
    used = (3 * N + 5 * Q) * 4 * stencil * (1 + per / 3)
    pairs = N * min(N, N / np.prod(box) * 4.19 * rc ** 3)
    flops = B * (2 * used + 2 * comps * 5 * V * math.log2(V) + 12 * comps * V + 30 * pairs)
    return {"bytes": 32.0 * B * (3 * N + 5 * Q) + 24.0 * N, "flops": float(flops)}


def work(case):
    if case["kind"] == "direct":
        N, Q = case["n"], len(_quad_particles(case, case["n"]))
        B = case["rhs"]
        return {"bytes": 32.0 * B * (3 * N + 5 * Q), "flops": float(N) * N * (30 + B * (28 + 150 * Q / N))}
    if case["kind"] in ("apply", "poly"):
        return _apply_work(case, case["rhs"])
    # applies per system: what GMRES / BiCGSTAB take here at these tolerances on average
    systems = 3 * case["freqs"] * case.get("frames", 1)
    applies = {"grad": 60}.get(case["kind"], 27 if case["tol"] < 1e-4 else 10)
    w = _apply_work(case, systems)
    w["flops"] *= applies
    return w


def tolerance(case):
    if case["kind"] == "grad":
        return {"rel": 1e-8, "max": 1e-6}  # solves converged to 1e-10
    if case["kind"] == "sweep":
        # converged to tol (a result is within half of it): two solves differ by less than this
        return {"rel": 3 * case["tol"], "max": 100 * case["tol"]}
    if case["prec"] == "double":
        return {"rel": 1e-13, "max": 1e-11}
    # FP32 grid or FP32 pair sums: 0.5 to 1.4e-7 and 5e-7 from float64 are measured
    return {"rel": 2e-6, "max": 1e-4} if case["kind"] == "direct" else {"rel": 6e-7, "max": 4e-5}


# ---------------------------------------------------------------------------
# The same outputs in float64 with plain torch
# ---------------------------------------------------------------------------

PI = math.pi


def _sizing(case, box, amax=1.0):
    """Grid lengths, spacings, support P, cutoff, spectral split per axis, xi."""
    tol, xi = case["tol"], case.get("xi", XI)
    rc = max(math.sqrt(-math.log(tol)) / xi, 2.0 * amax)
    n = [case["grid"]] * 3 if case.get("grid") else [math.ceil(1.0 + L * 2 * xi * xi * rc / PI) for L in box]
    h = [L / m for L, m in zip(box, n)]
    if case["kind"] == "poly":
        hm = sum(h) / 3
        P = math.ceil(2.0 / hm - 2.0 * math.log(tol) / PI)
        return n, h, P, rc, [P * (hm * xi) ** 2 / PI] * 3, xi
    P = case.get("support") or math.ceil(-2.0 * math.log(tol) / PI)
    return n, h, P, rc, [P * (d * xi) ** 2 / PI for d in h], xi


def _images(r, x, even_p, odd_p, even_b, odd_b, a, b, A0, B0, reg):
    """a (odd +- even) e^{-(r +- 2)^2 x^2} + b (even +- odd) erfc((r +- 2) x) + A0 e^{-r^2 x^2}
    + B0 erfc(r x), plus reg where the spheres overlap (r < 2)."""
    f = A0 * torch.exp(-r * r * x * x) + B0 * torch.erfc(r * x)
    for s in (1.0, -1.0):
        f = f + a * (odd_p + s * even_p) * torch.exp(-(r + 2 * s) ** 2 * x * x)
        f = f + b * (even_b + s * odd_b) * torch.erfc((r + 2 * s) * x)
    return torch.where(r < 2.0, f + reg, f)


def _dipole_tables(r, x):
    """Perpendicular and parallel pair functions of two unit spheres (screened part)."""
    s15, c1, c0 = PI ** 1.5, 3 - 12 * x ** 2 + 32 * x ** 4, 2 * (3 + 4 * x ** 2 - 32 * x ** 4)
    q4 = 36 * x ** 4 * (1 - 4 * x ** 2)
    be = -8 * x ** 6 * r ** 6 - q4 * r ** 4 - 18 * x ** 2 * (1 - 8 * x ** 2) * r ** 2 + 3 - 36 * x ** 2
    perp = _images(
        r, x, -8 * x ** 4 * r ** 4 - 8 * x ** 2 * (3 + 2 * x ** 2) * r ** 2 + c0,
        4 * x ** 4 * r ** 5 + 8 * x ** 2 * (2 - 7 * x ** 2) * r ** 3 + c1 * r,
        be + 256 * x ** 6, 256 * x ** 6 * r ** 3, 1 / (1024 * s15 * x ** 5 * r ** 3), 1 / (2048 * PI * x ** 6 * r ** 3),
        (-4 * x ** 4 * r ** 4 - 8 * x ** 2 * (2 - 9 * x ** 2) * r ** 2 - 3 + 36 * x ** 2) / (512 * s15 * x ** 5 * r ** 2),
        -be / (1024 * PI * x ** 6 * r ** 3), -1 / (4 * PI * r ** 3) + (1 - 9 * r / 16 + r ** 3 / 32) / (4 * PI))
    be = -16 * x ** 6 * r ** 6 - q4 * r ** 4 - 3 + 36 * x ** 2
    para = _images(
        r, x, -16 * x ** 4 * r ** 4 - 4 * x ** 2 * (3 - 4 * x ** 2) * r ** 2 - c0,
        8 * x ** 4 * r ** 5 + 2 * x ** 2 * (7 - 20 * x ** 2) * r ** 3 - c1 * r,
        be - 256 * x ** 6, 128 * x ** 6 * r ** 3, 1 / (512 * s15 * x ** 5 * r ** 3), 1 / (1024 * PI * x ** 6 * r ** 3),
        (-8 * x ** 4 * r ** 4 - 2 * x ** 2 * (7 - 36 * x ** 2) * r ** 2 + 3 - 36 * x ** 2) / (256 * s15 * x ** 5 * r ** 2),
        -be / (512 * PI * x ** 6 * r ** 3), 1 / (2 * PI * r ** 3) + (1 - 9 * r / 8 + r ** 3 / 8) / (4 * PI))
    return [perp, para]


def _quad_tables(r, x):
    """Field of a quadrupole (three functions), then the gradient couplings (four)."""
    s15 = PI ** 1.5
    out = []
    be = (48 * x ** 8 * r ** 8 + 32 * x ** 6 * (3 - 8 * x ** 2) * r ** 6 - 24 * x ** 4 * (3 - 16 * x ** 2) * r ** 4
          + 72 * x ** 2 * (1 - 8 * x ** 2) * r ** 2 - 45 + 480 * x ** 2)
    out.append(_images(
        r, x, 48 * x ** 6 * r ** 6 + 8 * x ** 4 * (3 - 8 * x ** 2) * r ** 4 - 4 * x ** 2 * (3 - 8 * x ** 2) ** 2 * r ** 2
        - 2 * (45 + 24 * x ** 2 - 64 * x ** 4 + 512 * x ** 6),
        -24 * x ** 6 * r ** 7 - 4 * x ** 4 * (9 - 8 * x ** 2) * r ** 5 + 2 * x ** 2 * (21 - 80 * x ** 2 + 64 * x ** 4) * r ** 3
        - (45 - 120 * x ** 2 + 192 * x ** 4 - 512 * x ** 6) * r,
        be + 4096 * x ** 8, 0.0, 15 / (16384 * s15 * x ** 7 * r ** 4), 15 / (32768 * PI * x ** 8 * r ** 4),
        15 / (8192 * s15 * x ** 7 * r ** 3) * (24 * x ** 6 * r ** 6 + 4 * x ** 4 * (9 - 32 * x ** 2) * r ** 4
                                               - 2 * x ** 2 * (21 - 128 * x ** 2) * r ** 2 + 45 - 480 * x ** 2),
        -15 / (16384 * PI * x ** 8 * r ** 4) * be,
        -15 / (4 * PI * r ** 4) + 15 * r ** 2 / (64 * PI) * (1 - 3 * r ** 2 / 16)))
    be = (80 * x ** 8 * r ** 8 + 160 * x ** 6 * (3 - 8 * x ** 2) * r ** 6 + 120 * x ** 4 * (3 - 16 * x ** 2) * r ** 4
          - 120 * x ** 2 * (1 - 8 * x ** 2) * r ** 2 + 45 - 480 * x ** 2)
    out.append(_images(
        r, x, 80 * x ** 6 * r ** 6 + 8 * x ** 4 * (45 + 8 * x ** 2) * r ** 4
        - 4 * x ** 2 * (15 + 48 * x ** 2 - 64 * x ** 4) * r ** 2 + 2 * (45 + 24 * x ** 2 - 64 * x ** 4 + 512 * x ** 6),
        -40 * x ** 6 * r ** 7 - 20 * x ** 4 * (11 - 24 * x ** 2) * r ** 5 - 2 * x ** 2 * (45 - 80 * x ** 2 + 64 * x ** 4) * r ** 3
        + (45 - 120 * x ** 2 + 192 * x ** 4 - 512 * x ** 6) * r,
        be - 4096 * x ** 8, -2048 * x ** 8 * r ** 5, 3 / (16384 * s15 * x ** 7 * r ** 4), 3 / (32768 * PI * x ** 8 * r ** 4),
        15 / (8192 * s15 * x ** 7 * r ** 3) * (8 * x ** 6 * r ** 6 + 4 * x ** 4 * (11 - 32 * x ** 2) * r ** 4
                                               + 2 * x ** 2 * (9 - 64 * x ** 2) * r ** 2 - 9 + 96 * x ** 2),
        -3 / (16384 * PI * x ** 8 * r ** 4) * be,
        3 / (4 * PI * r ** 4) - 3 * r / (8 * PI) * (1 - 5 * r / 8 + 5 * r ** 3 / 128)))
    be = (-8 * x ** 6 * r ** 6 - 12 * x ** 4 * (3 - 8 * x ** 2) * r ** 4 - 6 * x ** 2 * (3 - 16 * x ** 2) * r ** 2
          + 3 - 24 * x ** 2)
    out.append(_images(
        r, x, -8 * x ** 4 * r ** 4 - 24 * x ** 2 * r ** 2 + 6, 4 * x ** 4 * r ** 5 + 16 * x ** 2 * (1 - 2 * x ** 2) * r ** 3 + 3 * r,
        be, 128 * x ** 6 * r ** 3, 5 / (1024 * s15 * x ** 5 * r ** 2), 5 / (2048 * PI * x ** 6 * r ** 2),
        5 / (512 * s15 * x ** 5 * r) * (-4 * x ** 4 * r ** 4 - 16 * x ** 2 * (1 - 3 * x ** 2) * r ** 2 - 3 + 24 * x ** 2),
        -5 / (1024 * PI * x ** 6 * r ** 2) * be, 5 * r / (8 * PI) * (1 - 3 * r / 4 + r ** 3 / 16)))
    be = (16 * x ** 8 * r ** 8 + (96 * x ** 6 - 128 * x ** 8) * r ** 6 + (72 * x ** 4 - 192 * x ** 6 + 256 * x ** 8) * r ** 4
          - (24 * x ** 2 - 96 * x ** 4 + 256 * x ** 6) * r ** 2 + 9 - 48 * x ** 2 + 192 * x ** 4)
    out.append(_images(
        r, x, -16 * x ** 6 * r ** 6 - (72 * x ** 4 - 64 * x ** 6) * r ** 4 + (12 * x ** 2 - 64 * x ** 4) * r ** 2
        - (18 - 48 * x ** 2),
        8 * x ** 6 * r ** 7 + (44 * x ** 4 - 32 * x ** 6) * r ** 5 + (18 * x ** 2 + 32 * x ** 4) * r ** 3
        - (9 + 24 * x ** 2) * r,
        be, 0.0, 75 / (16384 * s15 * x ** 7 * r ** 3), -75 / (32768 * PI * x ** 8 * r ** 3),
        -75 / (8192 * s15 * x ** 7 * r ** 2) * (8 * x ** 6 * r ** 6 + (44 * x ** 4 - 64 * x ** 6) * r ** 4
                                                + (18 * x ** 2 - 64 * x ** 4 + 128 * x ** 6) * r ** 2
                                                - 9 + 48 * x ** 2 - 192 * x ** 4),
        75 / (16384 * PI * x ** 8 * r ** 3) * be, 75 * r * (4 - r ** 2) ** 2 / (1024 * PI)))
    be = (288 * x ** 10 * r ** 10 + (3600 * x ** 8 - 4800 * x ** 10) * r ** 8
          + (10800 * x ** 6 - 28800 * x ** 8 + 38400 * x ** 10) * r ** 6
          + (5400 * x ** 4 - 21600 * x ** 6 + 57600 * x ** 8) * r ** 4
          - (1350 * x ** 2 - 7200 * x ** 4 + 28800 * x ** 6) * r ** 2 + 405 - 2700 * x ** 2 + 14400 * x ** 4)
    out.append(_images(
        r, x, 96 * x ** 8 * r ** 8 + (1056 * x ** 6 - 1216 * x ** 8) * r ** 6
        + (2160 * x ** 4 - 4320 * x ** 6 - 256 * x ** 8) * r ** 4
        - (360 * x ** 2 - 1680 * x ** 4 - 768 * x ** 6 + 1024 * x ** 8) * r ** 2
        + 270 - 1080 * x ** 2 - 192 * x ** 4 + 512 * x ** 6 - 4096 * x ** 8,
        -48 * x ** 8 * r ** 9 - (576 * x ** 6 - 608 * x ** 8) * r ** 7 - (1536 * x ** 4 - 2576 * x ** 6 + 3968 * x ** 8) * r ** 5
        - (360 * x ** 2 + 360 * x ** 4 + 640 * x ** 6 - 512 * x ** 8) * r ** 3
        + (135 + 180 * x ** 2 + 480 * x ** 4 - 768 * x ** 6 + 2048 * x ** 8) * r,
        be + 49152 * x ** 10, 49152 * x ** 10 * r ** 5, 3 / (32768 * s15 * x ** 9 * r ** 5), 1 / (65536 * PI * x ** 10 * r ** 5),
        1 / (16384 * s15 * x ** 9 * r ** 4) * (
            144 * x ** 8 * r ** 8 + (1728 * x ** 6 - 2400 * x ** 8) * r ** 6
            + (4608 * x ** 4 - 13200 * x ** 6 + 19200 * x ** 8) * r ** 4
            + (1080 * x ** 2 - 5400 * x ** 4 + 19200 * x ** 6) * r ** 2 - 405 + 2700 * x ** 2 - 14400 * x ** 4),
        -1 / (32768 * PI * x ** 10 * r ** 5) * be,
        -3 / (2 * PI) * (1 / r ** 5 - 1 + 25 * r / 32 - 25 * r ** 3 / 256 + 3 * r ** 5 / 512)))
    be = (-96 * x ** 10 * r ** 10 + (-720 * x ** 8 + 960 * x ** 10) * r ** 8
          - (720 * x ** 6 - 1920 * x ** 8 + 2560 * x ** 10) * r ** 6 + (360 * x ** 4 - 1440 * x ** 6 + 3840 * x ** 8) * r ** 4
          - (270 * x ** 2 - 1440 * x ** 4 + 5760 * x ** 6) * r ** 2 + 135 - 900 * x ** 2 + 4800 * x ** 4)
    out.append(_images(
        r, x, -96 * x ** 8 * r ** 8 - 576 * (x ** 6 - x ** 8) * r ** 6 - (480 * x ** 6 + 256 * x ** 8) * r ** 4
        + (720 * x ** 4 + 768 * x ** 6 - 1024 * x ** 8) * r ** 2
        + 270 - 1080 * x ** 2 - 192 * x ** 4 + 512 * x ** 6 - 4096 * x ** 8,
        48 * x ** 8 * r ** 9 + (336 * x ** 6 - 288 * x ** 8) * r ** 7 + (216 * x ** 4 + 144 * x ** 6 + 128 * x ** 8) * r ** 5
        - (180 * x ** 2 - 120 * x ** 4 + 640 * x ** 6 - 512 * x ** 8) * r ** 3
        + (135 + 180 * x ** 2 + 480 * x ** 4 - 768 * x ** 6 + 2048 * x ** 8) * r,
        be + 16384 * x ** 10, 0.0, -15 / (65536 * s15 * x ** 9 * r ** 5), -15 / (131072 * PI * x ** 10 * r ** 5),
        15 / (32768 * s15 * x ** 9 * r ** 4) * (
            48 * x ** 8 * r ** 8 + (336 * x ** 6 - 480 * x ** 8) * r ** 6
            + (216 * x ** 4 - 720 * x ** 6 + 1280 * x ** 8) * r ** 4
            - (180 * x ** 2 - 840 * x ** 4 + 2560 * x ** 6) * r ** 2 + 135 - 900 * x ** 2 + 4800 * x ** 4),
        15 / (65536 * PI * x ** 10 * r ** 5) * be,
        -15 * (r ** 2 - 4) ** 3 * (3 * r ** 4 + 6 * r ** 2 + 8) / (2048 * PI * r ** 5)))
    be = (288 * x ** 10 * r ** 10 + (720 * x ** 8 - 960 * x ** 10) * r ** 8
          - (720 * x ** 6 - 1920 * x ** 8 + 2560 * x ** 10) * r ** 6
          + (1080 * x ** 4 - 4320 * x ** 6 + 11520 * x ** 8) * r ** 4
          - (1350 * x ** 2 - 7200 * x ** 4 + 28800 * x ** 6) * r ** 2 + 945 - 6300 * x ** 2 + 33600 * x ** 4)
    out.append(_images(
        r, x, -288 * x ** 8 * r ** 8 - (288 * x ** 6 + 192 * x ** 8) * r ** 6
        + (720 * x ** 4 - 480 * x ** 6 + 1792 * x ** 8) * r ** 4
        - (1080 * x ** 2 + 2160 * x ** 4 + 5376 * x ** 6 - 7168 * x ** 8) * r ** 2
        - (1890 - 7560 * x ** 2 - 1344 * x ** 4 + 3584 * x ** 6 - 28672 * x ** 8),
        144 * x ** 8 * r ** 9 + (288 * x ** 6 + 96 * x ** 8) * r ** 7 - (432 * x ** 4 - 912 * x ** 6 + 896 * x ** 8) * r ** 5
        + (720 * x ** 2 - 2280 * x ** 4 + 4480 * x ** 6 - 3584 * x ** 8) * r ** 3
        - (945 + 1260 * x ** 2 + 3360 * x ** 4 - 5376 * x ** 6 + 14336 * x ** 8) * r,
        be + 114688 * x ** 10, 0.0, -15 / (65536 * s15 * x ** 9 * r ** 5), 15 / (131072 * PI * x ** 10 * r ** 5),
        15 / (32768 * s15 * x ** 9 * r ** 4) * (
            144 * x ** 8 * r ** 8 + (288 * x ** 6 - 480 * x ** 8) * r ** 6
            - (432 * x ** 4 - 1200 * x ** 6 + 1280 * x ** 8) * r ** 4
            + (720 * x ** 2 - 3000 * x ** 4 + 6400 * x ** 6) * r ** 2 - 945 + 6300 * x ** 2 - 33600 * x ** 4),
        -15 / (65536 * PI * x ** 10 * r ** 5) * be,
        -15 * (3584 - 80 * r ** 6 - 30 * r ** 8 + 9 * r ** 10) / (2048 * PI * r ** 5)))
    return out


def _poly_pair(r, a, b, x):
    """Pair functions of spheres of radii a, b that do not overlap (screened part)."""
    fp, fa = torch.zeros_like(r), torch.zeros_like(r)
    for sa in (-1.0, 1.0):
        for sb in (-1.0, 1.0):
            p, q = sa * a, sb * b
            s, m, t = p + q, p * p - 4 * p * q + q * q, p * p + q * q
            c3, e3 = 4 * p ** 3 - 3 * p * q * s + 4 * q ** 3, p ** 3 - 3 * p * q * s + q ** 3
            m2, d2 = t - p * q, (p * p - q * q) ** 2
            E = torch.exp(-(r + s) ** 2 * x * x) / (PI ** 1.5 * (p * q * r) ** 3 * x ** 5)
            F = torch.erfc((r + s) * x) / (PI * (p * q * r) ** 3 * x ** 6)
            tail = 4 * s * s * m * x ** 4
            fp = fp + E / 1024 * (4 * x ** 4 * r ** 5 - 4 * s * x ** 4 * r ** 4
                                  + (16 * x ** 2 + 8 * (p * q - 4 * t) * x ** 4) * r ** 3
                                  - (12 * s * x ** 2 + 8 * c3 * x ** 4) * r ** 2 + (3 - 12 * m2 * x ** 2 - tail) * r
                                  + 3 * s + 4 * c3 * x ** 2 + tail * s)
            fp = fp + F / 2048 * (-8 * x ** 6 * r ** 6 + 36 * x ** 4 * (2 * t * x ** 2 - 1) * r ** 4
                                  + 128 * (p ** 3 + q ** 3) * x ** 6 * r ** 3
                                  + (-18 * x ** 2 + 72 * t * x ** 4 + 72 * d2 * x ** 6) * r ** 2 + 3 - 18 * t * x ** 2
                                  - 36 * d2 * x ** 4 - 2 * tail * s * s * x ** 2)
            fa = fa + E / 512 * (8 * x ** 4 * r ** 5 - 8 * s * x ** 4 * r ** 4
                                 + (14 * x ** 2 - 4 * (7 * t - 4 * p * q) * x ** 4) * r ** 3
                                 - (6 * s * x ** 2 + 4 * e3 * x ** 4) * r ** 2 + (-3 + 12 * m2 * x ** 2 + tail) * r
                                 - 3 * s - 4 * c3 * x ** 2 - tail * s)
            fa = fa + F / 1024 * (-16 * x ** 6 * r ** 6 + 36 * x ** 4 * (2 * t * x ** 2 - 1) * r ** 4
                                  + 64 * (p ** 3 + q ** 3) * x ** 6 * r ** 3 - 3 + 18 * t * x ** 2 + 36 * d2 * x ** 4
                                  + 2 * tail * s * s * x ** 2)
    return fp, fa


def _poly_self(a, x):
    """Real-space self value of a sphere of radius a."""
    e = (1 - 2 * a * a * x * x) * torch.exp(-4 * a * a * x * x) - 1 + 6 * a * a * x * x
    return e / (16 * PI ** 1.5 * a ** 6 * x ** 3) + (1 - torch.erf(2 * a * x)) / (4 * PI * a ** 3)


class _Plain:
    """The periodic operator A at fixed positions: y = A x for x [B][3N + 5Q], float64 torch."""

    def __init__(self, case, pos, box, radii=None, quads=()):
        dev = torch.device("cuda")
        f = lambda v: torch.as_tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)  # noqa: E731
        self.poly = radii is not None
        amax = 1.0 if radii is None else float(np.max(radii))
        self.n, h, self.P, self.rc, eta, xi = _sizing(case, box, amax)
        self.N, self.Q = len(pos), len(quads)
        self.qi = torch.as_tensor(np.asarray(quads, np.int64), device=dev)
        p, L = f(pos), f(box)
        self.xi, self.h3 = xi, h[0] * h[1] * h[2]
        kb = (case.get("kx", 0.0), case.get("ky", 0.0), 0.0)
        n = self.n
        V = n[0] * n[1] * n[2]
        # stencils: nearest grid point and the weights of the points around it
        half = (self.P - 1) // 2 if self.poly else self.P // 2
        off = range(-half, self.P - half) if self.poly else range(-half, half + 1)
        g = torch.floor(p / f(h) + 0.5)
        d0 = g * f(h) - p
        self.ax = [[(g[:, d].long() + o) % n[d] for o in off] for d in range(3)]
        self.gd = [[d0[:, d] + o * h[d] for o in off] for d in range(3)]
        if self.poly:
            self.rad, self.eta = f(radii), eta[0]
        else:
            cs = (2 * xi * xi / PI) ** 1.5 / math.sqrt(eta[0] * eta[1] * eta[2])
            self.w = [[torch.exp(-2 * xi * xi * v * v / eta[d]) * (cs if d == 0 else 1.0) for v in self.gd[d]]
                      for d in range(3)]
        # k space
        G = [torch.fft.fftfreq(m, 1.0 / m, dtype=torch.float64, device=dev) * (2 * PI / L[d]) for d, m in enumerate(n)]
        for d, m in enumerate(n):
            G[d] = G[d].reshape([-1 if e == d else 1 for e in range(3)])
        k = [G[d] - kb[d] for d in range(3)]
        k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
        zero = k2 < (1e-12 if self.poly else 1e-24)
        k2 = torch.where(zero, torch.ones_like(k2), k2)
        km = torch.sqrt(k2)
        off0 = lambda t: torch.where(zero, torch.zeros_like(k2), t)  # noqa: E731
        if self.poly:
            self.scale = off0(torch.exp(-(1 - self.eta) * k2 / (4 * xi * xi)) / k2 / V)
        else:
            ek = torch.exp(-(k2 - sum(G[d] ** 2 * eta[d] for d in range(3))) / (4 * xi * xi)) / V
            j1 = (torch.sin(km) / km - torch.cos(km)) / km
            j2 = (3 / k2 - 1) * torch.sin(km) / km - 3 * torch.cos(km) / k2
            self.kh = [off0(v / km) for v in k]
            self.c = [off0(9 * j1 ** 2 * ek / k2), off0(-22.5 * j1 * j2 * ek / k2), off0(45 * j1 * j2 * ek / k2),
                      off0(112.5 * j2 ** 2 * ek / k2)]
        # real-space pairs and their functions at max(r, 1), linear in tables sampled at 0.001
        self._pairs(p, L)
        u = self.r
        dist = torch.linalg.vector_norm(u, dim=1)
        self.u = u / (dist.clamp_min(1e-6) if self.poly else dist.clamp_min(1.0))[:, None]
        self.phase = torch.exp(-1j * (kb[0] * u[:, 0] + kb[1] * u[:, 1]))
        if self.poly:
            self.f = _poly_pair(dist.clamp_min(1e-6), self.rad[self.i], self.rad[self.j], xi)
            self.self_d, self.self_q = _poly_self(self.rad, xi)[:, None], 0.0
            return
        t = (dist.clamp(1.0, 9.999) - 1.0) / 0.001
        e = t.long().clamp_max(8998)
        t = (dist.clamp(1.0, 9.999) - (1.0 + e.double() * 0.001)) / 0.001
        r = 1.0 + torch.arange(9000, dtype=torch.float64) * 0.001
        tabs = [v.to(dev) for v in _dipole_tables(r, xi) + (_quad_tables(r, xi) if self.Q else [])]
        self.f = [v[e] * (1 - t) + v[e + 1] * t for v in tabs]
        x2 = xi * xi
        self.self_d = ((-1 + 6 * x2 + (1 - 2 * x2) * math.exp(-4 * x2)) / (16 * PI ** 1.5 * xi ** 3)
                       + math.erfc(2 * xi) / (4 * PI))
        sp = math.sqrt(PI)
        self.self_q = 0.25 / PI * (3 * (3 - 10 * x2 + 20 * x2 ** 2) / (8 * sp * xi ** 5)
                                   - 3 * (3 + 2 * x2 + 4 * x2 ** 2) * math.exp(-4 * x2) / (8 * sp * xi ** 5)
                                   + 3 * math.erfc(2 * xi))

    def _pairs(self, p, L):
        step = max(1, 20_000_000 // self.N)
        ii, jj, rr = [], [], []
        for a in range(0, self.N, step):
            r = p[None, :, :] - p[a:a + step, None, :]
            r = r - L * torch.round(r / L)
            d2 = r.square().sum(-1)
            d2[torch.arange(r.shape[0], device=p.device), torch.arange(a, a + r.shape[0], device=p.device)] = math.inf
            i, j = torch.nonzero(torch.sqrt(d2) < self.rc, as_tuple=True)
            ii.append(i + a)
            jj.append(j)
            rr.append(r[i, j])
        self.i, self.j, self.r = torch.cat(ii), torch.cat(jj), torch.cat(rr)

    def _points(self):
        """(voxel of every particle, weight) for each stencil point: the weight [N], or [3][N]."""
        for a, ga in enumerate(self.ax[0]):
            for b, gb in enumerate(self.ax[1]):
                for c, gc in enumerate(self.ax[2]):
                    vox = (ga * self.n[1] + gb) * self.n[2] + gc
                    if not self.poly:
                        yield vox, self.w[0][a] * self.w[1][b] * self.w[2][c]
                        continue
                    gd = torch.stack([self.gd[0][a], self.gd[1][b], self.gd[2][c]])
                    d, x2, eta, r = torch.linalg.vector_norm(gd, dim=0), self.xi ** 2, self.eta, self.rad
                    k = 3 / (8 * math.sqrt(2) * PI ** 1.5 * r ** 3 * math.sqrt(eta) * self.xi * d ** 3)
                    far = k * ((eta + 4 * r * x2 * d) * torch.exp(-2 * (d + r) ** 2 * x2 / eta)
                               - (eta - 4 * r * x2 * d) * torch.exp(-2 * (d - r) ** 2 * x2 / eta))
                    near = 8 * math.sqrt(2) * self.xi ** 5 * torch.exp(-2 * r * x2 / eta) / (PI ** 1.5 * eta ** 2.5)
                    yield vox, torch.where(d >= 1e-6, far, near) * gd

    def _reciprocal(self, p, q):
        """Field (and gradient) of dipoles p [B][3][N] and quadrupoles q [B][5][N] on the grid and back."""
        B, N, V = p.shape[0], self.N, self.n[0] * self.n[1] * self.n[2]
        src = p if q is None else torch.cat([p, q], 1)
        comps = 1 if self.poly else src.shape[1]
        grid = torch.zeros((B * comps, V, 2), dtype=torch.float64, device=p.device)
        pts = list(self._points()) if self.poly else None
        for vox, w in pts or self._points():
            v = (src * w).sum(1, keepdim=True) if self.poly else src * w
            grid.index_add_(1, vox, torch.view_as_real(v.reshape(B * comps, N).contiguous()))
        F = torch.fft.fftn(torch.view_as_complex(grid).reshape(B, comps, *self.n), dim=(2, 3, 4))
        del grid
        if self.poly:
            F = F * self.scale
        else:
            kh = self.kh
            e = sum(F[:, c] * kh[c] for c in range(3))
            s, t = self.c[0] * e, None
            if q is not None:
                dots = [kh[0] ** 2 - kh[2] ** 2, 2 * kh[0] * kh[1], 2 * kh[0] * kh[2], kh[1] ** 2 - kh[2] ** 2,
                        2 * kh[1] * kh[2]]
                gq = sum(F[:, 3 + c] * dots[c] for c in range(5))
                s, t = s + 1j * self.c[1] * gq, 1j * self.c[2] * e + self.c[3] * gq
                fac = [kh[0] ** 2 - 1 / 3, kh[0] * kh[1], kh[0] * kh[2], kh[1] ** 2 - 1 / 3, kh[1] * kh[2]]
                for c in range(5):
                    F[:, 3 + c] = t * fac[c]
            for c in range(3):
                F[:, c] = s * kh[c]
        F = (torch.fft.ifftn(F, dim=(2, 3, 4)) * V).reshape(B, comps, V)
        out = torch.zeros((B, src.shape[1], N), dtype=torch.complex128, device=p.device)
        for vox, w in pts or self._points():
            out += F[:, :, vox] * w
        return out * self.h3

    def _real(self, p, q):
        """Screened pair sums, as [B][3 (+ 5)][N]."""
        i, u = self.i, self.u.T
        out = torch.zeros((p.shape[0], 3 if q is None else 8, self.N), dtype=torch.complex128, device=p.device)
        for b in range(p.shape[0]):
            pj = p[b][:, self.j]
            pu = (pj * u).sum(0)
            v = self.f[0] * pj + (self.f[1] - self.f[0]) * pu * u
            if q is not None:
                t0, t1, t2, g1, g2, g3, g4 = self.f[2:]
                Q = q[b][:, self.j]
                Qr = torch.stack([Q[0] * u[0] + Q[1] * u[1] + Q[2] * u[2], Q[1] * u[0] + Q[3] * u[1] + Q[4] * u[2],
                                  Q[2] * u[0] + Q[4] * u[1] - (Q[0] + Q[3]) * u[2]])
                Qrr = (Qr * u).sum(0)
                v = v + 0.5 * Qrr * t0 * u + t1 * Qr
                one = torch.tensor([1.0, 0, 0, 1.0, 0], dtype=torch.float64, device=p.device)[:, None]
                at = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2)]
                uu = torch.stack([u[a] * u[c] for a, c in at])
                pp = torch.stack([pj[a] * u[c] + pj[c] * u[a] for a, c in at])
                # (the diagonal of the quadrupole term is 2 Qr_a u_a, as the sum over both orders)
                qq = torch.stack([Qr[a] * u[c] + Qr[c] * u[a] for a, c in at])
                grad = -(pu * (t0 * uu + (t1 + t2) * one) + t1 * pp)
                grad = grad + 0.5 * (Qrr * ((g1 + g3) * one + g4 * uu) + Q * g2 + 2 * g3 * qq)
                v = torch.cat([v, grad])
            out[b].index_add_(1, i, v * self.phase)
        return out

    def __call__(self, x, sc):
        """A x with self coefficients sc [B or 1][N]."""
        B, N, Q = x.shape[0], self.N, self.Q
        p = x[:, :3 * N].reshape(B, N, 3).transpose(1, 2)
        q = None
        if Q:
            q = torch.zeros((B, 5, N), dtype=x.dtype, device=x.device)
            q[:, :, self.qi] = x[:, 3 * N:].reshape(B, Q, 5).transpose(1, 2)
        step = max(1, int(1e9 // (self.n[0] * self.n[1] * self.n[2] * 16 * (8 if Q else 3))))
        y = torch.cat([self._reciprocal(p[b:b + step], None if q is None else q[b:b + step]) for b in range(0, B, step)])
        y = (y + self._real(p, q)).transpose(1, 2)
        f = (y[..., :3] + (sc[..., None] + self.self_d) * p.transpose(1, 2)).reshape(B, 3 * N)
        if not Q:
            return f
        g = y[..., 3:] + (2.5 * sc[..., None] + self.self_q) * q.transpose(1, 2)
        return torch.cat([f, g[:, self.qi].reshape(B, 5 * Q)], 1)


def _direct(pos, q, sc, x):
    """The open-boundary operator for unit spheres: point dipoles and quadrupoles, pair by pair."""
    N, Q, B = len(pos), len(q), x.shape[0]
    dev = x.device
    p = torch.as_tensor(pos, device=dev)
    dip = x[:, :3 * N].reshape(B, N, 3)
    qi = torch.as_tensor(q, device=dev)
    qd = torch.zeros((B, N, 3, 3), dtype=x.dtype, device=dev)
    if Q:
        v = x[:, 3 * N:].reshape(B, Q, 5)
        m = torch.stack([v[..., 0], v[..., 1], v[..., 2], v[..., 1], v[..., 3], v[..., 4], v[..., 2], v[..., 4],
                         -v[..., 0] - v[..., 3]], -1)
        qd[:, qi] = -m.reshape(B, Q, 3, 3)
    E = torch.zeros((B, N, 3), dtype=x.dtype, device=dev)
    G = torch.zeros((B, N, 3, 3), dtype=x.dtype, device=dev)
    one = torch.eye(3, dtype=torch.float64, device=dev)
    step = max(1, 400_000 // N)
    for a in range(0, N, step):
        r = p[None, :, :] - p[a:a + step, None, :]
        d = torch.linalg.vector_norm(r, dim=-1)
        own = torch.arange(r.shape[0], device=dev)
        d[own, own + a] = 1.0
        assert bool((d >= 1.0).all())
        u = r / d[..., None]
        c = (-1 / (4 * PI)) * torch.ones_like(d)
        c[own, own + a] = 0.0
        for b in range(B):
            pu = (dip[b] * u).sum(-1)
            E[b, a:a + step] = ((c / d ** 3)[..., None] * (3 * pu[..., None] * u - dip[b])).sum(1)
            if not Q:
                continue
            v = (qd[b][None] * u[:, :, None, :]).sum(-1)
            s = (u * v).sum(-1)
            E[b, a:a + step] += ((3 * c / d ** 4)[..., None] * (2.5 * s[..., None] * u - v)).sum(1)
            uu = u[..., :, None] * u[..., None, :]
            up = u[..., :, None] * dip[b][None, :, None, :]
            uv = u[..., :, None] * v[..., None, :]
            g = (-3 * c / d ** 4)[..., None, None] * (pu[..., None, None] * (one - 5 * uu) + up + up.transpose(-1, -2))
            g = g + (-3 * c / d ** 5)[..., None, None] * (5 * (uv + uv.transpose(-1, -2)) + 2.5 * s[..., None, None] * one
                                                         - 17.5 * s[..., None, None] * uu - qd[b][None])
            G[b, a:a + step] = g.sum(1)
    E = E + (sc[..., None] + 1 / (4 * PI)) * dip
    if not Q:
        return E.reshape(B, 3 * N)
    g = torch.stack([G[..., a, c] for a, c in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2))], -1)[:, qi]
    g = g + (2.5 * sc[:, qi, None] + 3 / (4 * PI)) * x[:, 3 * N:].reshape(B, Q, 5)
    return torch.cat([E.reshape(B, 3 * N), g.reshape(B, 5 * Q)], 1)


def _plain_solve(apply, b, cycle=70, tol=1e-12, most=8):
    """Restarted GMRES on all systems at once (least squares at the end of a cycle)."""
    B, n = b.shape
    x = torch.zeros_like(b)
    for _ in range(most):
        r = b - apply(x) if bool(x.any()) else b.clone()
        beta = torch.linalg.vector_norm(r, dim=1)
        if bool((beta <= tol * torch.linalg.vector_norm(b, dim=1)).all()):
            break
        Vb = torch.zeros((B, cycle + 1, n), dtype=b.dtype, device=b.device)
        H = torch.zeros((B, cycle + 1, cycle), dtype=b.dtype, device=b.device)
        Vb[:, 0] = r / beta[:, None].clamp_min(1e-300)
        m = cycle
        for k in range(cycle):
            w = apply(Vb[:, k].contiguous())
            for _ in range(2):
                h = (Vb[:, :k + 1].conj() * w[:, None, :]).sum(-1)
                w = w - (h[:, :, None] * Vb[:, :k + 1]).sum(1)
                H[:, :k + 1, k] += h
            hn = torch.linalg.vector_norm(w, dim=1)
            H[:, k + 1, k] = hn
            Vb[:, k + 1] = w / hn[:, None].clamp_min(1e-300)
        rhs = torch.zeros((B, m + 1, 1), dtype=b.dtype)
        rhs[:, 0, 0] = beta.cpu()
        y = torch.linalg.lstsq(H.cpu(), rhs, driver="gelsd").solution[..., 0].to(b.device)
        x = x + (y[:, :, None] * Vb[:, :m]).sum(1)
    return x


def exact(case, seed):
    if case["kind"] in ("apply", "poly", "direct"):
        pos, box, radii, q, sc, x = _apply_inputs(case, seed)
        x, sc = torch.from_numpy(x).cuda(), torch.from_numpy(sc).cuda()
        if case["kind"] == "direct":
            return _direct(pos, q, sc, x)
        return _Plain(case, pos, box, radii, q)(x, sc)
    if case["kind"] == "sweep":
        frames, box = _frames(case, seed)
        eps = _sweep_eps(case, seed)
        out = []
        for pos in frames:
            op, N, W = _Plain(case, pos, box), len(pos), len(eps)
            sc = torch.from_numpy(np.repeat(_self_coef(eps)[:, None], N, 1)).cuda().repeat_interleave(3, 0)
            b = torch.eye(3, dtype=torch.complex128, device="cuda").repeat(W, N)
            x = _plain_solve(lambda v: op(v, sc), b)
            out.append(x.reshape(W, 3, N, 3).transpose(1, 2))
        return torch.stack(out).squeeze().cpu().numpy()
    pos, box, omega, par = _grad_inputs(case, seed)
    N, W = len(pos), len(omega)
    op = _Plain(case, pos, box, None, np.arange(N))
    n = 8 * N
    zero = torch.zeros((1, N), dtype=torch.complex128, device="cuda")
    eye = torch.eye(n, dtype=torch.complex128, device="cuda")
    dense = torch.cat([op(eye[a:a + 128], zero) for a in range(0, n, 128)]).T
    par = [torch.from_numpy(p).cuda().requires_grad_(True) for p in par]
    w = torch.as_tensor(omega, device="cuda")
    eps = par[0] - par[1] ** 2 / ((w * w)[:, None] + 1j * w[:, None] * par[2])
    sc = -3.0 / (4.0 * PI * (1.0 - eps))
    diag = torch.cat([sc.repeat_interleave(3, 1), 2.5 * sc.repeat_interleave(5, 1)], 1)
    b = torch.zeros((n, 3), dtype=torch.complex128, device="cuda")
    b[:3 * N] = torch.eye(3, dtype=torch.complex128, device="cuda").repeat(N, 1)
    x = torch.stack([torch.linalg.solve(dense + torch.diag(diag[a]), b) for a in range(W)])  # [W][n][3]
    ext = torch.stack([x[:, c:3 * N:3, c].sum(1) for c in range(3)]).imag  # [3][W]
    loss = (4 * PI * 2 * PI * w * ext).sum() + x[:, 3 * N:].abs().square().sum()
    loss.backward()
    return {"x": x.detach().transpose(1, 2).reshape(3 * W, n), "eps_inf": par[0].grad, "wp": par[1].grad,
            "gamma": par[2].grad}
