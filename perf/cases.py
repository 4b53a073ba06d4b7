"""Timing cases of the linear-solve path: what a finite-volume program calls, from one
A·x on a small mesh to pressure solves on two million cells and whole time steps.

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges. ``prepare``
builds what the program holds before the call (mesh and matrix handles, device buffers),
``run`` makes one pass through the package's entry points, ``exact`` restates the result
in 64 bits with torch alone, ``work`` counts what a pass cannot do without.

Kinds:

* ``amul``: one product y = A·x, device vectors (symmetric pressure or nonsymmetric
  momentum coefficients);
* ``gamg``: a pressure solve, PCG with GAMG (damped Jacobi), matrix resident, x from 0;
* ``mixed``: the same in mixed precision to a tight tolerance;
* ``dropin``: what a program linked against the solver replacement does per pressure
  solve: new coefficients and right-hand side from host memory, PCG with GAMG smoothed by
  Gauss–Seidel (that program's default), x back to host memory;
* ``gs``: the same solver with matrix and vectors resident, as in pressure correctors;
* ``momentum``: a time step's momentum predictor: per velocity component the matrix
  ddt + div − laplacian assembled on the device, then PBiCGStab with DILU;
* ``krylov``: PCG with DIC or diagonal preconditioning, plain or reproducible sums;
* ``batch``: many small pressure systems solved together;
* ``piso``: one whole PISO time step with the default solver settings;
* ``corrector``: the explicit operators between momentum and pressure solve.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import voluma_amd as va
from voluma_amd import mesh as meshes
from voluma_amd import workloads
from voluma_amd.piso import PisoFlow

D = va.VOL_DEVICE


def listed():
    return [
        # the smallest call: a residual check on a coarse test mesh, all latency
        {"name": "amul_box_small", "kind": "amul", "mesh": "box", "nx": 13, "ny": 12, "nz": 11, "nonsym": False},
        # pressure solve of a tutorial-size case with the library's default GAMG
        {"name": "gamg_box_small", "kind": "gamg", "mesh": "box", "nx": 21, "ny": 19, "nz": 17, "pre": 2, "post": 2,
         "omega": 0.8, "tol": 1e-6},
        # the benchmark's pressure solve: 2.06M jittered tetrahedra
        {"name": "gamg_tet70", "kind": "gamg", "mesh": "tet", "nx": 70, "ny": 70, "nz": 70, "pre": 1, "post": 1,
         "omega": 0.9, "tol": 1e-6},
        # a tightly converged pressure solve in mixed precision
        {"name": "mixed_tet47", "kind": "mixed", "mesh": "tet", "nx": 52, "ny": 47, "nz": 45, "pre": 1, "post": 1,
         "omega": 0.9, "tol": 1e-10},
        # a linked program's pressure solve on the 64³ box (the reference's own solver settings)
        {"name": "dropin_box64", "kind": "dropin", "mesh": "box", "nx": 64, "ny": 64, "nz": 64, "tol": 1e-6},
        # repeated pressure correctors with the same settings on tetrahedra, everything resident
        {"name": "gs_tet40", "kind": "gs", "mesh": "tet", "nx": 41, "ny": 38, "nz": 40, "tol": 1e-6},
        # the momentum predictor of a mid-size case
        {"name": "momentum_tet52", "kind": "momentum", "mesh": "tet", "nx": 56, "ny": 51, "nz": 49, "tol": 1e-10},
        # symmetric solves without a hierarchy: scalar transport, wall distance, potential start-up
        {"name": "dic_box28", "kind": "krylov", "mesh": "box", "nx": 31, "ny": 27, "nz": 29, "precond": "DIC",
         "repro": False, "tol": 1e-8},
        # a reproducible run: exact sums, results independent of the partition
        {"name": "repro_tet16", "kind": "krylov", "mesh": "tet", "nx": 17, "ny": 15, "nz": 16, "precond": "diagonal",
         "repro": True, "tol": 1e-8},
        # a parameter study: 48 independent systems of 5k to 200k cells
        {"name": "batch_48", "kind": "batch", "systems": 48, "specs_seed": 4, "n_max": 200000, "tol": 1e-6},
        # a whole time step of a small cavity with the default solvers
        {"name": "piso_tet19", "kind": "piso", "mesh": "tet", "nx": 20, "ny": 18, "nz": 19},
        # explicit corrector operators on the large mesh
        {"name": "corrector_tet70", "kind": "corrector", "mesh": "tet", "nx": 70, "ny": 70, "nz": 70},
    ]


# cells: smallest and largest of each kind; tets and boxes are drawn alike
_RANGE = {"amul": (1500, 2000000), "gamg": (4000, 2000000), "mixed": (30000, 650000), "dropin": (8000, 260000),
          "gs": (8000, 370000), "momentum": (5000, 830000), "krylov": (3000, 60000), "piso": (1500, 40000),
          "corrector": (5000, 2000000)}


def _dims(rng, lo, hi, per):
    """nx, ny, nz with about exp(uniform) cells and sides up to 2.5 : 1 apart."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi))) / per
    f = [rng.uniform(1.0, 2.5) for _ in range(3)]
    base = (n / (f[0] * f[1] * f[2])) ** (1.0 / 3.0)
    d = [max(3, int(round(base * v))) for v in f]
    while d[0] * d[1] * d[2] * per > hi and max(d) > 3:
        d[d.index(max(d))] -= 1
    return d


def draw(rng):
    kind = rng.choice(["amul", "gamg", "mixed", "dropin", "gs", "momentum", "krylov", "batch", "piso", "corrector"])
    if kind == "batch":
        return {"kind": kind, "systems": rng.randint(3, 40), "specs_seed": rng.randint(5, 10 ** 6),
                "n_max": rng.randint(20000, 150000), "tol": 1e-6}
    # momentum, time steps and corrector operators need the skewed meshes; the others take both
    mesh = "tet" if kind in ("momentum", "piso", "corrector") else rng.choice(["box", "tet"])
    lo, hi = _RANGE[kind]
    nx, ny, nz = _dims(rng, lo, hi, 6 if mesh == "tet" else 1)
    c = {"kind": kind, "mesh": mesh, "nx": nx, "ny": ny, "nz": nz}
    if kind == "amul":
        c["nonsym"] = rng.random() < 0.5
    elif kind == "gamg":
        c["pre"] = c["post"] = rng.choice([1, 2])
        c["omega"] = 0.9 if c["pre"] == 1 else 0.8
        c["tol"] = 1e-6
    elif kind == "mixed":
        c["pre"] = c["post"] = 1
        c["omega"] = 0.9
        c["tol"] = 1e-10
    elif kind in ("dropin", "gs"):
        c["tol"] = 1e-6
    elif kind == "momentum":
        c["tol"] = 1e-10
    elif kind == "krylov":
        c["precond"] = rng.choice(["DIC", "diagonal"])
        c["repro"] = c["precond"] == "diagonal" and rng.random() < 0.6
        c["tol"] = 1e-8
    return c


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=4)
def _mesh(kind, nx, ny, nz):
    m = meshes.tet(nx, ny, nz, 0.2, 1) if kind == "tet" else meshes.box(nx, ny, nz)
    m.geometry()
    return m


def _case_mesh(case):
    return _mesh(case["mesh"], case["nx"], case["ny"], case["nz"])


@functools.lru_cache(maxsize=2)
def _batch_inputs(systems, specs_seed, n_max):
    """(meshes, xMax-like Dirichlet masks) of the batch's systems."""
    specs = workloads.batch_specs(systems, specs_seed, n_max=n_max)
    out = []
    for sp in specs:
        m = workloads.batch_mesh(sp)
        bc = np.zeros(m.n_boundary, np.int32)
        s = int(m.patch_start[sp["patch"]]) - m.n_internal
        bc[s: s + int(m.patch_size[sp["patch"]])] = 1
        out.append((m, bc))
    return out


def _case_batch(case):
    return _batch_inputs(case["systems"], case["specs_seed"], case["n_max"])


def _context():
    return va.Context(0)


class _Buffer(va.DeviceArray):
    """A device array over a torch tensor's memory (any device allocation may be passed)."""

    def __init__(self, ctx, t):
        self.ctx, self.n, self.dtype, self._ctxh = ctx, t.numel(), np.dtype(np.float64), ctx._h
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())

    def free(self):
        pass


def _dev(a, dtype=np.float64):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=dtype).reshape(-1)).cuda()


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _u(n, seed):
    return 2.0 * workloads.splitmix_uniform(n, seed) - 1.0


def _rhs(n, seed):
    b = _u(n, seed)
    return b - b.mean()


def _pressure_coeffs(m, bc):
    """diag (folded), upper of laplacian(1, p) with fixedValue 0 where bc, numpy."""
    g, ni = m.geometry(), m.n_internal
    u = g["magSf"][:ni] * g["ndc"][:ni]
    d = -(np.bincount(m.owner[:ni], u, m.n_cells) + np.bincount(m.neighbour, u, m.n_cells))
    ub = np.where(bc != 0, g["magSf"][ni:] * g["ndc"][ni:], 0.0)
    return d - np.bincount(m.owner[ni:], ub, m.n_cells), u


def _momentum_inputs(m, seed):
    return workloads.momentum_inputs(m, seed, exact=False)


class State:
    pass


def _ldu(m, ctx, gamg):
    ni = m.n_internal
    lm = va.LduMesh(ctx, m.n_cells, m.owner[:ni], m.neighbour, m.agglomeration_weights() if gamg else None)
    lm.set_boundary(m.owner[ni:])
    return lm


def _set_geometry(lm, g):
    lm.set_geometry(g["V"], g["Sf"], g["magSf"], g["w"], g["d"], g["skew"], g["skewed"])


def _controls(case):
    k = case["kind"]
    if k in ("gamg", "mixed", "batch"):
        return va.SolverControls("PCG", "GAMG", case["tol"], precision=va.MIXED if k == "mixed" else va.FP64,
                                 gamgPreSweeps=case.get("pre", 1), gamgPostSweeps=case.get("post", 1),
                                 gamgOmega=case.get("omega", 0.9), sums=va.SUMS_FAST)
    if k in ("dropin", "gs"):
        return va.SolverControls("PCG", "GAMG", case["tol"], gamgSmoother=va.GAMG_GAUSS_SEIDEL, sums=va.SUMS_FAST)
    if k == "momentum":
        return va.SolverControls("PBiCGStab", "DILU", case["tol"], sums=va.SUMS_FAST)
    return va.SolverControls("PCG", case["precond"], case["tol"], maxIter=5000,
                             sums=va.SUMS_REPRODUCIBLE if case["repro"] else va.SUMS_FAST)


def _host_inputs(case, seed):
    """What the case's inputs hold, on the host, from the seed alone."""
    kind = case["kind"]
    if kind == "batch":
        return {"b": np.concatenate([_rhs(m.n_cells, 7919 * seed + 31 * k) for k, (m, _) in enumerate(_case_batch(case))])}
    m = _case_mesh(case)
    n, nb = m.n_cells, m.n_boundary
    if kind == "amul" and case["nonsym"]:
        # upwind convection and diffusion: upper and lower differ, the diagonal dominates
        d, u = _pressure_coeffs(m, workloads.bc_fixed_xmax(m))
        s = 0.5 * np.abs(u) * _u(u.size, 7919 * seed + 11)
        return {"d": d, "u": u + s, "l": u - s, "x": _u(n, 7919 * seed + 1)}
    if kind == "amul":
        d, u = _pressure_coeffs(m, workloads.bc_fixed_xmax(m))
        return {"d": d, "u": u, "l": None, "x": _u(n, 7919 * seed + 1)}
    if kind in ("gamg", "mixed", "dropin", "gs", "krylov"):
        d, u = _pressure_coeffs(m, workloads.bc_fixed_xmax(m))
        return {"d": d, "u": u, "b": _rhs(n, 7919 * seed + 1)}
    if kind in ("momentum", "piso"):
        return _momentum_inputs(m, 1 + seed % 100003)
    return {"c": _u(n, 7919 * seed + 1), "p": _u(n, 7919 * seed + 2), "U": _u(3 * n, 7919 * seed + 3),
            "Ub": _u(3 * nb, 7919 * seed + 4), "pb": _u(nb, 7919 * seed + 5)}


def prepare(case, seed):
    s = State()
    s.kind, s.ctx = case["kind"], _context()
    h = _host_inputs(case, seed)
    if s.kind == "batch":
        ms = _case_batch(case)
        s.B = va.LduBatch(s.ctx, [(m.n_cells, m.owner[: m.n_internal], m.neighbour, m.agglomeration_weights())
                                  for m, _ in ms])
        co = [_pressure_coeffs(m, bc) for m, bc in ms]
        s.B.set(np.concatenate([c[0] for c in co]), np.concatenate([c[1] for c in co]))
        s.b, s.zero = _Buffer(s.ctx, _dev(h["b"])), _Buffer(s.ctx, _dev(np.zeros(h["b"].size)))
        s.x, s.controls = _Buffer(s.ctx, torch.zeros_like(s.b.t)), _controls(case)
        return s
    m = _case_mesh(case)
    n = m.n_cells
    if s.kind == "piso":
        s.flow = PisoFlow(s.ctx, m, h["nu"], [(0, 0, 0)] * 5 + [(1, 0, 0)], [None] * 6, ddt="Euler")
        s.dt = h["dt"]
        s.U0, s.p0, s.phi0 = _dev(h["U0"]), _dev(np.zeros(n)), _dev(h["phi"])
        s.U, s.p, s.phi = (torch.zeros_like(t) for t in (s.U0, s.p0, s.phi0))
        return s
    s.lm = _ldu(m, s.ctx, s.kind in ("gamg", "mixed", "dropin", "gs"))
    if s.kind == "corrector":
        g = m.geometry()
        _set_geometry(s.lm, g)
        nF = m.n_faces
        s.c, s.p, s.Uc, s.Ub, s.pb = (_dev(h[k]) for k in ("c", "p", "U", "Ub", "pb"))
        s.fix = _dev(np.ones(m.n_boundary), np.int32)
        s.free = _dev(np.zeros(m.n_boundary), np.int32)
        s.zero = _dev(np.zeros(m.n_boundary))
        z = lambda k: torch.zeros(k, dtype=torch.float64, device="cuda")  # noqa: E731
        s.gc, s.cf, s.gU, s.phi, s.div, s.gp = z(3 * n), z(nF), z(9 * n), z(nF), z(n), z(3 * n)
        return s
    s.A = va.LduMatrix(s.lm)
    if s.kind == "momentum":
        g = m.geometry()
        s.dt, s.nu = h["dt"], h["nu"]
        s.V, s.phi, s.magSf, s.ndc, s.w = (_dev(a) for a in (g["V"], h["phi"], g["magSf"], g["ndc"], g["w"]))
        s.Sf, s.corr = _dev(g["Sf"]), _dev(g["corr"])
        s.fix = _dev(np.ones(m.n_boundary), np.int32)
        s.U0 = [_Buffer(s.ctx, _dev(h["U0"][:, k])) for k in range(3)]
        s.Ub = [_dev(h["Ub"][:, k]) for k in range(3)]
        s.b = [_Buffer(s.ctx, torch.zeros_like(s.V)) for _ in range(3)]
        s.x = [_Buffer(s.ctx, torch.zeros_like(s.V)) for _ in range(3)]
        s.controls = _controls(case)
        return s
    if s.kind == "dropin":
        s.d, s.u, s.b, s.x, s.controls = h["d"], h["u"], h["b"], np.zeros(n), _controls(case)
        return s
    s.A.set(h["d"], h["u"], h.get("l"))
    if s.kind == "amul":
        s.x = _Buffer(s.ctx, _dev(h["x"]))
        s.y = _Buffer(s.ctx, torch.zeros_like(s.x.t))
        return s
    s.b, s.zero = _Buffer(s.ctx, _dev(h["b"])), _Buffer(s.ctx, _dev(np.zeros(n)))
    s.x, s.controls = _Buffer(s.ctx, torch.zeros_like(s.b.t)), _controls(case)
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    L, check = va.lib(), va._check
    if s.kind == "amul":
        va.amul(s.A, s.x, s.y)
        return s.y.t
    if s.kind == "dropin":
        s.A.set(s.d, s.u)
        s.x[:] = 0.0
        va.solve_ldu(s.A, s.b, s.x, s.controls)
        return s.x
    if s.kind == "batch":
        s.x.copy_from(s.zero)
        s.B.solve(s.b, s.x, s.controls)
        return s.x.t
    if s.kind == "momentum":
        h = s.A._h
        for k in range(3):
            no = va._NonOrth(s.U0[k].t.data_ptr(), s.w.data_ptr(), s.Sf.data_ptr(), s.corr.data_ptr(), s.V.data_ptr())
            check(L.vol_fvm_reset(h))
            check(L.vol_fvm_ddt_euler(h, 1, s.dt, _ptr(s.V), s.U0[k].ptr, D))
            check(L.vol_fvm_div_upwind(h, 1, _ptr(s.phi), _ptr(s.fix), _ptr(s.Ub[k]), D))
            check(L.vol_fvm_laplacian(h, -1, s.nu, None, _ptr(s.magSf), _ptr(s.ndc), _ptr(s.fix), _ptr(s.Ub[k]),
                                      ctypes.byref(no), D))
            check(L.vol_fvm_finish(h, s.b[k].ptr, D))
            s.x[k].copy_from(s.U0[k])
            va.solve_ldu(s.A, s.b[k], s.x[k], s.controls)
        return [b.t for b in s.b] + [x.t for x in s.x]
    if s.kind == "piso":
        f = s.flow
        check(L.vol_flow_set_fields(f._h, _ptr(s.U0), _ptr(s.p0), _ptr(s.phi0), D))
        f.step(s.dt)
        check(L.vol_flow_get_fields(f._h, _ptr(s.U), _ptr(s.p), _ptr(s.phi), D))
        return [s.U, s.p, s.phi]
    if s.kind == "corrector":
        h, LS = s.lm._h, va.GRAD_LEAST_SQUARES
        check(L.vol_fvc_grad(h, LS, 1, _ptr(s.c), _ptr(s.free), _ptr(s.zero), _ptr(s.gc), D))
        check(L.vol_fvc_interpolate(h, 1, _ptr(s.c), _ptr(s.gc), None, _ptr(s.cf), D))
        check(L.vol_fvc_grad(h, LS, 3, _ptr(s.Uc), _ptr(s.fix), _ptr(s.Ub), _ptr(s.gU), D))
        check(L.vol_fvc_flux(h, _ptr(s.Uc), _ptr(s.gU), _ptr(s.fix), _ptr(s.Ub), _ptr(s.phi), D))
        check(L.vol_fvc_div(h, _ptr(s.phi), _ptr(s.div), D))
        check(L.vol_fvc_grad(h, va.GRAD_GAUSS_SKEW, 1, _ptr(s.p), _ptr(s.fix), _ptr(s.pb), _ptr(s.gp), D))
        return [s.gc, s.cf, s.gU, s.phi, s.div, s.gp]
    s.x.copy_from(s.zero)
    va.solve_ldu(s.A, s.b, s.x, s.controls)
    return s.x.t


# ------------------------------------------------------------------ what a pass cannot do without
def _sizes(case):
    """cells, internal faces, boundary faces (closed forms of the generated meshes)."""
    if case["kind"] == "batch":
        ms = _case_batch(case)
        return tuple(sum(v) for v in zip(*((m.n_cells, m.n_internal, m.n_boundary) for m, _ in ms)))
    x, y, z = case["nx"], case["ny"], case["nz"]
    inner = (x - 1) * y * z + x * (y - 1) * z + x * y * (z - 1)
    outer = 2 * (x * y + y * z + x * z)
    if case["mesh"] == "tet":  # two triangles per hex face, six faces inside each hex
        return 6 * x * y * z, 2 * inner + 6 * x * y * z, 2 * outer
    return x * y * z, inner, outer


def work(case):
    """Each input and output once; for a solve also one iteration's products and vectors
    (the iteration count is the method's, so a pass's floor is counted per iteration in
    the log that goes with the timings)."""
    n, nf, nb = _sizes(case)
    kind, nF = case["kind"], nf + nb
    if kind == "amul":
        return {"bytes": 24 * n + (16 + (8 if case["nonsym"] else 0)) * nf, "flops": 2 * n + 4 * nf}
    if kind == "corrector":
        # gradLS(c), interpolate, gradLS(U), flux, div, grad(p): fields, geometry and addressing once
        by = 8 * (n + 3 * n + nF + 3 * n + 9 * n + nF + n + n + 3 * n + n) + 8 * nF * (3 + 3 + 1 + 1 + 3) + 8 * nf
        return {"bytes": by, "flops": 60 * n + 250 * nf}
    if kind == "momentum":
        return {"bytes": 3 * (8 * (n * 5 + nF * 10) + 24 * n + 24 * nf), "flops": 3 * (60 * nF + 30 * n)}
    if kind == "piso":
        return {"bytes": 16 * (4 * n + nF) + 8 * (n + 12 * nF), "flops": 400 * nF}
    return {"bytes": 24 * n + 16 * nf, "flops": 2 * n + 4 * nf}


# All sums are 64-bit. Plain tree sums against exact sums of the same solve (another
# summation order) differ by 5e-16 to 2e-15, the single operators from exact() by 1e-16 to
# 3.4e-16. Another order inside the smoothers' rows travels through every iteration as
# well, hence 1e-11 for the solves; in mixed precision 32-bit inner solves leave each
# implementation its own 3e-10 from the exact solution.
_TOL = {"amul": 5e-16, "gamg": 1e-11, "mixed": 1.5e-9, "dropin": 1e-11, "gs": 1e-11, "momentum": 1e-13,
        "krylov": 1e-11, "batch": 1e-11, "piso": 1e-10, "corrector": 2e-15}


def tolerance(case):
    if case["kind"] == "krylov" and case["repro"]:
        return "exact"
    return {"rel": _TOL[case["kind"]]}


# ------------------------------------------------------------------ the same in plain torch
def _spmv(d, u, l, own, nei):
    def mul(x):
        y = d * x
        y.index_add_(0, own, u * x[nei])
        y.index_add_(0, nei, l * x[own])
        return y

    return mul


def _cg(mul, d, b, rtol=1e-13, most=6000):
    x, r = torch.zeros_like(b), b.clone()
    z = r / d
    p, rz, stop = z.clone(), torch.dot(r, z), rtol * float(b.norm())
    for k in range(most):
        q = mul(p)
        a = rz / torch.dot(p, q)
        x += a * p
        r -= a * q
        if k % 25 == 24 and float(r.norm()) <= stop:
            break
        z = r / d
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return x


def _jacobi_bicg(mul, d, b, x, rtol=1e-15, most=400):
    r = b - mul(x)
    r0, stop = r.clone(), rtol * float(b.norm())
    p, v = torch.zeros_like(b), torch.zeros_like(b)
    rho = al = om = 1.0
    for _ in range(most):
        if float(r.norm()) <= stop:
            break
        new = float(torch.dot(r0, r))
        if new == 0.0:
            break
        p = r + (new / rho) * (al / om) * (p - om * v)
        rho = new
        y = p / d
        v = mul(y)
        al = rho / float(torch.dot(r0, v))
        s = r - al * v
        z = s / d
        t = mul(z)
        tt = float(torch.dot(t, t))
        om = float(torch.dot(t, s)) / tt if tt > 0 else 0.0
        x = x + al * y + om * z
        r = s - om * t
        if om == 0.0:
            break
    return x


def _lsgrad(g, own, nei, ni, c, de, dphi):
    """Least-squares gradient of c (n × k) with boundary constraints de, dphi."""
    n, k, dv = c.shape[0], c.shape[1], g["d"][:ni]
    w = 1.0 / (dv * dv).sum(1)
    T = (dv[:, :, None] * dv[:, None, :]) * w[:, None, None]
    wb = 1.0 / (de * de).sum(1)
    Tb = (de[:, :, None] * de[:, None, :]) * wb[:, None, None]
    M = torch.zeros(n, 3, 3, dtype=torch.float64, device=c.device)
    ob = g["own_b"]
    M.index_add_(0, own, T).index_add_(0, nei, T).index_add_(0, ob, Tb)
    r = torch.zeros(n, 3, k, dtype=torch.float64, device=c.device)
    e = (dv * w[:, None])[:, :, None] * (c[nei] - c[own])[:, None, :]
    r.index_add_(0, own, e).index_add_(0, nei, e)
    r.index_add_(0, ob, (de * wb[:, None])[:, :, None] * dphi[:, None, :])
    a = M.reshape(n, 9).unbind(1)  # adjugate inverse: small systems, written out
    det = (a[0] * (a[4] * a[8] - a[5] * a[7]) - a[1] * (a[3] * a[8] - a[5] * a[6]) + a[2] * (a[3] * a[7] - a[4] * a[6]))
    inv = torch.stack([a[4] * a[8] - a[5] * a[7], a[2] * a[7] - a[1] * a[8], a[1] * a[5] - a[2] * a[4],
                       a[5] * a[6] - a[3] * a[8], a[0] * a[8] - a[2] * a[6], a[2] * a[3] - a[0] * a[5],
                       a[3] * a[7] - a[4] * a[6], a[1] * a[6] - a[0] * a[7], a[0] * a[4] - a[1] * a[3]],
                      1).reshape(n, 3, 3) / det[:, None, None]
    return (inv[:, :, :, None] * r[:, None, :, :]).sum(2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "piso":
        return None  # a chain of solves stopped by their tolerances: no value of its own
    h = _host_inputs(case, seed)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    if kind == "batch":
        ms = _case_batch(case)
        off = np.cumsum([0] + [m.n_cells for m, _ in ms])
        co = [_pressure_coeffs(m, bc) for m, bc in ms]
        xs = []
        for k, (m, _) in enumerate(ms):
            own, nei = T(m.owner[: m.n_internal].astype(np.int64)), T(m.neighbour.astype(np.int64))
            d, u = T(co[k][0]), T(co[k][1])
            xs.append(_cg(_spmv(d, u, u, own, nei), d, T(h["b"][off[k]: off[k + 1]])))
        return torch.cat(xs).cpu().numpy()
    m = _case_mesh(case)
    g, n, ni = m.geometry(), m.n_cells, m.n_internal
    own, nei = T(m.owner[:ni].astype(np.int64)), T(m.neighbour.astype(np.int64))
    if kind == "amul":
        d, u = T(h["d"]), T(h["u"])
        return _spmv(d, u, u if h["l"] is None else T(h["l"]), own, nei)(T(h["x"])).cpu().numpy()
    if kind in ("gamg", "mixed", "dropin", "gs", "krylov"):
        d, u = T(h["d"]), T(h["u"])
        return _cg(_spmv(d, u, u, own, nei), d, T(h["b"])).cpu().numpy()
    G = {k: T(g[k]) for k in ("V", "Sf", "magSf", "w", "ndc", "corr", "d", "skew")}
    G["own_b"] = ob = T(m.owner[ni:].astype(np.int64))
    w, Sf, V = G["w"][:ni], G["Sf"], G["V"]
    if kind == "momentum":
        phi, rdt, nu = T(h["phi"]), 1.0 / h["dt"], h["nu"]
        lo = -torch.where(phi[:ni] >= 0, phi[:ni], torch.zeros_like(phi[:ni]))
        up = lo + phi[:ni]
        lap = nu * G["magSf"] * G["ndc"]
        d = rdt * V
        d.index_add_(0, own, lap[:ni] - lo).index_add_(0, nei, lap[:ni] - up).index_add_(0, ob, lap[ni:])
        up, lo = up - lap[:ni], lo - lap[:ni]
        mul, bs, xs = _spmv(d, up, lo, own, nei), [], []
        for k in range(3):
            U, Ub = T(np.ascontiguousarray(h["U0"][:, k])), T(np.ascontiguousarray(h["Ub"][:, k]))
            gr = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
            e = Sf[:ni] * (w * U[own] + (1.0 - w) * U[nei])[:, None]
            gr.index_add_(0, own, e).index_add_(0, nei, -e).index_add_(0, ob, Sf[ni:] * Ub[:, None])
            gr = gr / V[:, None]
            gf = w[:, None] * gr[own] + (1.0 - w)[:, None] * gr[nei]
            fc = nu * G["magSf"][:ni] * (G["corr"][:ni] * gf).sum(1)
            b = V * (rdt * U)
            b.index_add_(0, own, fc).index_add_(0, nei, -fc)
            b.index_add_(0, ob, Ub * (lap[ni:] - phi[ni:]))
            bs.append(b.cpu().numpy())
            xs.append(_jacobi_bicg(mul, d, b, U.clone()).cpu().numpy())
        return bs + xs
    # corrector
    c, p, U, Ub, pb = (T(h[k]) for k in ("c", "p", "U", "Ub", "pb"))
    U, Ub, sk = U.reshape(n, 3), Ub.reshape(-1, 3), G["skew"][:ni]
    nv = Sf[ni:] / G["magSf"][ni:, None]
    db = G["d"][ni:]
    nd = torch.maximum((nv * db).sum(1), 0.05 * (db * db).sum(1).sqrt())
    gc = _lsgrad(G, own, nei, ni, c[:, None], nv * nd[:, None], torch.zeros(len(pb), 1, dtype=torch.float64, device="cuda"))
    gc = gc[:, :, 0]
    mix = lambda a: w.reshape(-1, *[1] * (a.dim() - 1)) * a[own] + (1.0 - w).reshape(-1, *[1] * (a.dim() - 1)) * a[nei]  # noqa: E731
    skewed = bool(g["skewed"])
    cf = mix(c) + ((sk * mix(gc)).sum(1) if skewed else 0.0)
    cf = torch.cat([cf, c[ob]])
    gU = _lsgrad(G, own, nei, ni, U, db, Ub - U[ob])
    Uf = mix(U) + ((sk[:, :, None] * mix(gU)).sum(1) if skewed else 0.0)
    phi = torch.cat([(Uf * Sf[:ni]).sum(1), (Ub * Sf[ni:]).sum(1)])
    div = torch.zeros(n, dtype=torch.float64, device="cuda")
    div.index_add_(0, own, phi[:ni]).index_add_(0, nei, -phi[:ni]).index_add_(0, ob, phi[ni:])
    gl = _lsgrad(G, own, nei, ni, p[:, None], db, (pb - p[ob])[:, None])[:, :, 0]
    pf = mix(p) + ((sk * mix(gl)).sum(1) if skewed else 0.0)
    gp = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
    e = Sf[:ni] * pf[:, None]
    gp.index_add_(0, own, e).index_add_(0, nei, -e).index_add_(0, ob, Sf[ni:] * pb[:, None])
    gp = gp / V[:, None]
    return [v.reshape(-1).cpu().numpy() for v in (gc, cf, gU, phi, div / V, gp)]
