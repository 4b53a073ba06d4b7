"""GPU tests of the FvMatrix algebra (vol_fvm_*): the momentum matrix of
IncompressibleFlow.cpp:183-185, ddt(Euler) + div(φ, upwind) − laplacian(ν) with the
non-orthogonal correction, assembled on the GPU. Bar: every FvMatrix part, the fold
and b bit-identical to the reference's (small fixtures and full-size hashes), and the
reference's reproducible PBiCGStab solve of it reproduced bit for bit.
"""
import numpy as np
import pytest

import voluma_amd as va
from helpers import SMALL_MESHES, load_json, load_small, sha
from voluma_amd import mesh as M
from voluma_amd import workloads as W

pytestmark = pytest.mark.gpu
NAMES = list(SMALL_MESHES)
MOM_DT, MOM_NU, MOM_BC = 0.05, 0.01, 0.7  # as tests/golden/make_golden.py


@pytest.fixture(scope="module")
def ctx():
    c = va.Context(0)
    yield c
    c.close()


def _matrix(ctx, m):
    ni = m.n_internal
    lm = va.LduMesh(ctx, m.n_cells, m.owner[:ni], m.neighbour, None)
    lm.set_boundary(m.owner[ni:])
    return lm, va.LduMatrix(lm)


@pytest.mark.parametrize("name", NAMES)
def test_momentum_parts_bit_exact(ctx, name):
    g = load_small(name)
    m = SMALL_MESHES[name]()
    geo = m.geometry()
    lm, A = _matrix(ctx, m)
    bc = W.bc_fixed_xmax(m)
    bv = np.where(bc != 0, MOM_BC, 0.0)
    psi = g["mom_psi0"]
    A.fvm_reset()
    A.fvm_ddt_euler(+1, MOM_DT, geo["V"], psi)
    A.fvm_div_upwind(+1, g["div_flux"], bc, bv)
    A.fvm_laplacian(-1, geo["magSf"], geo["ndc"], bc, bv, gamma=MOM_NU,
                    nonorth={"psi": psi, "w": geo["w"], "Sf": geo["Sf"], "corr": geo["corr"], "V": geo["V"]})
    parts = A.fvm_get()
    for k in ("diag", "source", "ic", "bs", "ffc"):
        assert np.array_equal(parts[k], g["mom_" + k]), k
    b = A.fvm_finish()
    d, u, lo = A.get()
    assert np.array_equal(d, g["mom_dF"]) and np.array_equal(b, g["mom_bF"])
    assert np.array_equal(u, g["mom_upper"]) and np.array_equal(lo, g["mom_lower"])
    assert not A.symmetric


@pytest.mark.parametrize("name", NAMES)
def test_pressure_terms_and_source(ctx, name):
    """laplacian alone stays symmetric and equals vol_assemble_laplacian; the
    FvMatrix −= su source term adds su·V (FvMatrix.h:93-97)."""
    g = load_small(name)
    m = SMALL_MESHES[name]()
    geo = m.geometry()
    lm, A = _matrix(ctx, m)
    bc = W.bc_fixed_xmax(m)
    su = 2.0 * W.splitmix_uniform(m.n_cells, 77) - 1.0
    A.fvm_reset()
    A.fvm_laplacian(+1, geo["magSf"], geo["ndc"], bc)
    A.fvm_source(su, geo["V"])
    b = A.fvm_finish()
    assert A.symmetric
    d, u, lo = A.get()
    assert np.array_equal(d, g["sym_diag"]) and np.array_equal(u, g["lap_upper"]) and np.array_equal(lo, u)
    bref = 0.0 + su * geo["V"]
    np.add.at(bref, m.owner[m.n_internal:], g["lap_bs"])
    assert np.array_equal(b, bref)


def test_fvm_errors(ctx):
    m = SMALL_MESHES["box8x6x5"]()
    geo = m.geometry()
    lm, A = _matrix(ctx, m)
    with pytest.raises(va.VolumaError) as e:
        A.fvm_ddt_euler(+1, 0.1, geo["V"], np.zeros(m.n_cells))
    assert e.value.code == -1
    A.fvm_reset()
    for bad in (lambda: A.fvm_ddt_euler(2, 0.1, geo["V"], np.zeros(m.n_cells)),
                lambda: A.fvm_ddt_euler(+1, 0.0, geo["V"], np.zeros(m.n_cells))):
        with pytest.raises(va.VolumaError) as e:
            bad()
        assert e.value.code == -1
    # an unfinished matrix cannot be solved
    with pytest.raises(va.VolumaError):
        va.solve_ldu(A, np.zeros(m.n_cells), np.zeros(m.n_cells), va.SolverControls("PBiCGStab"))


def test_full_size_momentum_tet70(ctx):
    """2.06M-cell tet momentum matrices (3 components) equal the reference's by
    hash; the reference's reproducible PBiCGStab from x = U⁰ to 1e-6 is reproduced
    bit for bit; a default-mode and a mixed-precision solve converge."""
    f = load_json("cfg2_tet70_momentum.json")
    m = W.make_mesh("tet70")
    inp = W.momentum_inputs(m, 1)
    assert sha(inp["phi"]) == f["phi_sha256"] and sha(inp["U0"]) == f["U0_sha256"]
    assert inp["dt"] == f["dt"]
    lm, A = _matrix(ctx, m)
    for comp, fc in enumerate(f["components"]):
        b = W.momentum_assemble(A, m, inp, comp)
        d, u, lo = A.get()
        assert sha(d) == fc["diag_sha256"] and sha(u) == fc["upper_sha256"] and sha(lo) == fc["lower_sha256"]
        assert sha(b) == fc["b_sha256"] and sha(A.fvm_get()["ffc"]) == fc["ffc_sha256"]
        x = np.ascontiguousarray(inp["U0"][:, comp])
        p = va.solve_ldu(A, b, x, va.SolverControls("PBiCGStab", "DILU", 1e-6, 0.0, 1000, sums=va.SUMS_REPRODUCIBLE))
        r = fc["repro_pbicgstab_1e-6"]
        assert p.iterations == r["iterations"] and p.finalResidual == r["finalResidual"]
        assert sha(x) == r["x"]["sha256"]
        for prec in (va.FP64, va.MIXED):
            x2 = np.ascontiguousarray(inp["U0"][:, comp])
            p2 = va.solve_ldu(A, b, x2, va.SolverControls("PBiCGStab", "diagonal", 1e-6, 0.0, 1000, precision=prec))
            assert p2.converged
            assert np.linalg.norm(x2 - x) <= 1e-5 * np.linalg.norm(x)


@pytest.mark.parametrize("face", [None, 0, 262143, 262144, -1])
def test_single_non_orthogonal_face_is_found(ctx, face):
    """The correction is switched on by any one corrected face, wherever the scan of the
    faces (1024 blocks of 256, then on) meets it, and only that face's flux is corrected:
    γ|S| corr·∇ψ with ∇ψ = (1, 0, 0) of ψ = x on a uniform box."""
    m = M.box(50)
    geo = m.geometry()
    lm, A = _matrix(ctx, m)
    ni = m.n_internal
    corr = np.zeros_like(geo["corr"])
    f = None if face is None else face % ni
    if f is not None:
        corr[f] = (1e-3, 0.0, 0.0)
    bc = np.ones(m.n_boundary, np.int32)  # boundary values of ψ, so that the gradient is exact
    psi, bv = geo["C"][:, 0].copy(), geo["Cf"][ni:, 0].copy()
    A.fvm_reset()
    A.fvm_laplacian(+1, geo["magSf"], geo["ndc"], bc, bv, gamma=2.0,
                    nonorth={"psi": psi, "w": geo["w"], "Sf": geo["Sf"], "corr": corr, "V": geo["V"]})
    ffc = A.fvm_get()["ffc"]
    want = np.zeros(m.n_faces)
    if f is not None:
        want[f] = 2.0 * geo["magSf"][f] * 1e-3
    assert np.allclose(ffc, want, rtol=1e-9, atol=0.0)  # 64-bit sums of six terms: ~1e-13
    A.close()
    lm.close()
