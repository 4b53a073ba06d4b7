"""Shared test helpers: golden fixture loading and system construction."""
import hashlib
import json
import os

import numpy as np

from voluma_amd import mesh as M
from voluma_amd import workloads as W

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")

SMALL_MESHES = {
    "box8x6x5": lambda: M.box(8, 6, 5),
    "tet5x4x3": lambda: M.tet(5, 4, 3, 0.2, 7),
    "box12": lambda: M.box(12),
}


def band(n, deg, width, seed):
    """Faces between cells at most width apart, deg / 2 per cell; what would lie past the last
    cell ends at it (a long row)."""
    rng = np.random.default_rng(seed)
    a = rng.integers(0, n - 1, n * deg // 2)
    b = np.minimum(a + 1 + rng.integers(0, width, a.size), n - 1)
    return a, b


def sweep_graph(name):
    """(cells, owner, neighbour) of graphs at the edges of the sweep plans: the largest
    one-chunk size and its neighbour, a chain (one row per level), rows of every length the
    kernels treat apart (up to 8, 12 and 20 entries, longer ones, a hub of hundreds), and
    neighbours anywhere: ``far`` has large halos (16 chunks, 12,993 of 20,400 slots forward;
    backward over 10,000 values lie past them), in ``scattered`` both directions run over."""
    rng = np.random.default_rng(5)
    if name == "chain":
        n = 8193
        a, b = np.arange(n - 1), np.arange(1, n)
    elif name == "one":
        n, (a, b) = 8192, band(8192, 6, 300, 1)
    elif name == "two":
        n, (a, b) = 8193, band(8193, 6, 300, 2)
    elif name == "wide":
        n, (a, b) = 12345, band(12345, 14, 900, 3)
    elif name == "far":
        n, (a, b) = 30000, band(30000, 16, 30000, 4)
    elif name == "scattered":
        n, (a, b) = 100_003, band(100_003, 16, 100_003, 8)
    elif name == "hub":
        n, (a, b) = 9001, band(9001, 5, 200, 6)
        a = np.concatenate([a, np.full(400, 4500), rng.integers(0, 4500, 400)])
        b = np.concatenate([b, 4501 + rng.permutation(4500)[:400], np.full(400, 4500)])
    else:
        m = M.box(23, 21, 19)
        return m.n_cells, m.owner[: m.n_internal], m.neighbour
    keep = a < b
    e = np.unique(a[keep].astype(np.int64) * n + b[keep])
    rng.shuffle(e)  # face order unrelated to cell order
    flip = rng.random(e.size) < 0.3  # faces owned by the higher cell too
    l, u = (e // n).astype(np.int32), (e % n).astype(np.int32)
    return n, np.where(flip, u, l), np.where(flip, l, u)


def sha(a):
    return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()


def mesh_hash(m):
    h = hashlib.sha256()
    for a in (m.points, m.face_off, m.face_pts, m.owner, m.neighbour, m.patch_start, m.patch_size):
        h.update(np.ascontiguousarray(a).tobytes())
    return h.hexdigest()


def load_small(name):
    with np.load(os.path.join(GOLDEN, f"small_{name}.npz"), allow_pickle=False) as z:
        return {k: z[k] for k in z.files}


def load_json(name):
    with open(os.path.join(GOLDEN, name)) as fh:
        return json.load(fh)


def solve_cases(g):
    out = []
    for i, s in enumerate(g["solve_cases"]):
        solver, pre, repro, sym = str(s).split("|")
        out.append((i, solver, pre, bool(int(repro)), bool(int(sym))))
    return out


def load_post(name):
    """Reference relax / A / H / flux / setReference fixtures of one small mesh."""
    with np.load(os.path.join(GOLDEN, f"post_{name}.npz"), allow_pickle=False) as z:
        return {k: z[k] for k in z.files}


POST_CASES = ("ms", "mv", "p")  # momentum scalar, momentum vector, pressure


def post_inputs(g, tag):
    s = g[f"{tag}_in_scalars"]
    return {"psi0": g[f"{tag}_in_psi0"], "F": g[f"{tag}_in_F"], "fv": g[f"{tag}_in_fv"],
            "bcfixed": g[f"{tag}_in_bcfixed"], "dt": float(s[0]), "nu": float(s[1]), "alpha": float(s[2]),
            "ref_cell": int(s[3]), "ref_value": float(s[4]), "pressure": bool(s[5])}


FVC_MESHES = {
    "box8x6x5": lambda: M.box(8, 6, 5),
    "tet5x4x3": lambda: M.tet(5, 4, 3, 0.2, 7),
    "tet6x5x4": lambda: M.tet(6, 5, 4, 0.24, 11),
}


def load_fvc(name):
    """Reference explicit corrector operators (Fvc.h) on one small mesh."""
    with np.load(os.path.join(GOLDEN, f"fvc_{name}.npz"), allow_pickle=False) as z:
        return {k: z[k] for k in z.files}


def fvc_bfix(m, fixed):
    """Per boundary face: 1 on the faces of the given patches."""
    ni = m.n_internal
    out = np.zeros(m.n_faces - ni, np.int32)
    for p in fixed:
        s = int(m.patch_start[p]) - ni
        out[s: s + int(m.patch_size[p])] = 1
    return out


class CompView:
    """The faces the reference's Mesh keeps of a read mesh (cyclic pairs merged into
    internal faces, empty patches dropped): the attributes the oracle's corrector
    functions read, with the geometry of those faces, and the 2-D empty direction."""

    def __init__(self, m):
        c = m.computational()
        self.n_cells, self.n_internal = m.n_cells, c["n_internal"]
        self.n_faces = len(c["faces"])
        self.n_boundary = self.n_faces - self.n_internal
        self.owner = c["owner"]
        self.neighbour = c["neighbour"]
        self._g = c["geometry"]
        self.empty_dir = c["empty_dir"]
        self.comp = c

    def geometry(self):
        return self._g


def periodic_channel():
    """An 8×5×4 unit box periodic in x (xMin/xMax a cyclic pair) with its interior points
    moved by up to ±0.025 (a fifth of a cell in x, seeded): skewed internal and cyclic
    faces; the boundary points stay, so the periodicity is a pure translation."""
    m = M.box(8, 5, 4, periodic=(True, False, False))
    pts = m.points.copy()
    inner = np.all((pts > 1e-12) & (pts < 1 - 1e-12), axis=1)
    rng = np.random.default_rng(3)
    pts[inner] += rng.uniform(-0.025, 0.025, (int(inner.sum()), 3))
    m.set_points(pts)
    return m


# ---------------------------------------------------------------- PISO step cases
# name → (mesh maker, options, number of steps, dt, reproducible sums). u_bc / p_bc are
# per kept patch; the initial fields come from piso_inputs.
PISO_CASES = {
    "box8_lid_repro": (lambda: M.box(8, 8, 8),
                       {"nu": 0.01, "u_bc": [(0, 0, 0)] * 5 + [(1, 0, 0)], "p_bc": [None] * 6}, 2, 0.005, True),
    "tet5x4x3_channel_repro": (lambda: M.tet(5, 4, 3, 0.2, 7),
                               {"nu": 0.02, "u_bc": [(1, 0, 0), None, (0, 0, 0), (0, 0, 0), (0, 0, 0), (0, 0, 0)],
                                "p_bc": [None, 0.0, None, None, None, None], "ddt": "backward",
                                "ddt_phi_coeff": -1.0, "grad_p": 2, "n_non_orth": 1}, 3, 0.01, True),
    "channel_periodic_repro": (periodic_channel,
                               {"nu": 0.02, "u_bc": [(0, 0, 0)] * 4, "p_bc": [None] * 4, "ddt": "backward",
                                "grad_p": 1, "n_non_orth": 1}, 2, 0.01, True),
    "box8_lid_default": (lambda: M.box(8, 8, 8),
                         {"nu": 0.01, "u_bc": [(0, 0, 0)] * 5 + [(1, 0, 0)], "p_bc": [None] * 6}, 2, 0.005, False),
}


def piso_inputs(m):
    """Initial U (a smooth swirl about the cell centres, zero normal component in 2-D),
    p (a linear ramp) and the face flux φ⁰ = U_f·S_f of that U (the oracle's phiHbyA
    flux with zero-gradient boundaries), on the faces the reference's Mesh keeps."""
    from oracle import oracle as O
    C = m.geometry()["C"]
    x, y, z = C[:, 0], C[:, 1], C[:, 2]
    c = m.computational()
    U0 = np.stack([np.sin(np.pi * y) * 0.5, -np.sin(np.pi * x) * 0.5, 0.0 * z if c["two_d"] else 0.2 * np.cos(x)],
                  axis=1)
    p0 = 0.1 * x - 0.05 * y
    cv = CompView(m)
    nb = cv.n_boundary
    phi0 = O.fvc_flux(cv, U0, None, np.zeros(nb, np.int32), np.zeros((nb, 3)))
    return np.ascontiguousarray(U0), np.ascontiguousarray(p0), phi0
