"""Device solve of the assembled system (slx_plan_solve) against a direct
solve of the same system.

sl::solve(A, b) (src/expression/operation/sl.cpp:1565-1627) eliminates the
Dirichlet DOFs (mat::eliminate, src/formulation/mat.cpp:78-103), factorizes A
and merges the free and constrained values (mat::xbmerge).  The checker here
is scipy's sparse LU on the CSR the device assembled, so the comparison
isolates the solve; the reference examples' validation lines pin the whole
assemble + solve chain.
"""
import math

import numpy as np
import pytest

import sparselizard_amd as sa
from test_golden_examples import _FREE, LINE_MSH, QUAD_MSH, register_free, solve_full

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("precision", ["fp64", "f16split", "fp32"])
def test_solve_electrostatics_1d_golden(ctx, precision):
    # examples/electrostatics-1d/main.cpp:44: 21.5962 < ||x||_2 < 21.5964
    print("case solve electrostatics1d", precision, flush=True)
    p = sa.Problem(ctx, "electrostatics1d", "file=" + LINE_MSH)
    info = register_free(p)
    plan = p.generate(precision)
    x, it = plan.solve(info["ndofs"], rel_tol=1e-12)
    assert it["rel_residual"] <= 1e-12, it
    nrm = float(np.linalg.norm(x))
    assert 21.5962 < nrm < 21.5964, nrm


@pytest.mark.parametrize("kind,spec,precision", [("poisson2d", "n=40", "fp64"), ("poisson2d", "n=12;order=3", "fp64"),
                                                 ("elasticity3d", "n=4", "fp64"), ("elasticity3d", "n=4", "f16split"),
                                                 ("hppoisson3d", "n=3", "fp64")])
def test_solve_matches_direct(ctx, kind, spec, precision):
    print("case solve", kind, spec, precision, flush=True)
    p = sa.Problem(ctx, kind, spec)
    info = register_free(p)
    plan = p.generate(precision)
    ref, A, bA = solve_full(plan.csr(info["ndofs"]), info["ndofs"], info["nfree"])
    x, it = plan.solve(info["ndofs"], rel_tol=1e-12)
    print("solve", it, flush=True)
    assert it["rel_residual"] <= 1e-12, it
    assert it["outer"] >= 1 and it["inner"] >= 1
    assert it["method"] == "cg"  # symmetric systems (the symmetry check tolerates rounding)
    # residual bound 1e-12 times the condition number of these small systems
    assert relerr(x, ref) <= 1e-8, relerr(x, ref)
    # constrained entries are the Dirichlet values, exactly
    cons = np.ones(info["ndofs"], bool)
    cons[_FREE[(info["ndofs"], info["nfree"])]] = False
    rhs = plan.csr(info["ndofs"]).rhs
    assert np.array_equal(x[cons], rhs[cons])


def test_solve_projection_no_constraints(ctx):
    # order-5 projection on quads (mass matrix, no Dirichlet DOFs):
    # examples/high-order-interpolations-2d/main.cpp:68, relative L2 error < 1e-5
    print("case solve hoprojection2d", flush=True)
    p = sa.Problem(ctx, "hoprojection2d", "file=%s;order=5" % QUAD_MSH)
    info = register_free(p)
    plan = p.generate("fp64")
    v, it = plan.solve(info["ndofs"], rel_tol=1e-13, max_outer=30)
    print("solve", it, flush=True)
    assert it["method"] == "cg"
    assert it["rel_residual"] <= 1e-13, it
    b = plan.csr(info["ndofs"]).rhs
    f2 = (0.5 - math.sin(20.0) / 40.0) * (0.5 - math.sin(26.0) / 52.0)
    err = math.sqrt(max(f2 - float(b @ v), 0.0) / f2)
    assert err < 1e-5, err


def test_solve_deterministic(ctx):
    print("case solve deterministic", flush=True)
    p = sa.Problem(ctx, "elasticity3d", "n=4")
    info = register_free(p)
    plan = p.generate("fp64")
    x1, i1 = plan.solve(info["ndofs"], rel_tol=1e-11)
    x2, i2 = plan.solve(info["ndofs"], rel_tol=1e-11)
    assert i1 == i2 and np.array_equal(x1, x2)


def test_solve_argument_errors(ctx):
    p = sa.Problem(ctx, "poisson2d", "n=4")
    info = p.info()
    plan = p.plan()
    with pytest.raises(sa.SlxError, match="no assembly"):
        plan.solve(info["ndofs"])
    p.generate("fp64")
    with pytest.raises(sa.SlxError, match="must be positive"):
        plan.solve(info["ndofs"], rel_tol=0.0)


def _random_csr(rng, lens):
    n = len(lens)
    rowp = np.zeros(n + 1, np.int64)
    rowp[1:] = np.cumsum(lens)
    # repeated columns in a row are allowed (the product sums them, as scipy does)
    col = rng.integers(0, n, int(rowp[-1])).astype(np.int32)
    val = rng.standard_normal(int(rowp[-1]))
    return rowp, col, val


@pytest.mark.parametrize("case", ["short", "mixed_long", "edges", "rows4", "rows7", "rows10", "rows25", "rows50", "rows100", "rows200",
                                  "skewed", "many_short"])
def test_spmv_stream_matches_numpy(ctx, case):
    # the inner-iteration product.  Streaming: row blocks of at most 4096 nonzeros
    # and 256 rows, long rows by a whole block, more than 131072 short rows.  By rows:
    # one to 32 lanes, six and eight nonzeros each, rows much shorter and longer than
    # the mean, a last workgroup that is not full
    from sparselizard_amd import _lib as L
    print("case spmv_stream", case, flush=True)
    rng = np.random.default_rng(7)
    n = 20000
    if case == "short":
        lens = rng.integers(0, 12, n)
    elif case == "mixed_long":
        lens = rng.integers(20, 120, n)
        lens[[5, 777, n - 1]] = [4097, 9000, 12001]
    elif case.startswith("rows"):
        n, mean = 20003, int(case[4:])
        lens = rng.integers(0, 2 * mean + 1, n)
        lens[[0, 1, 9, n - 1]] = [0, min(1024, 4 * mean), 1, 3 * mean]
    elif case == "skewed":
        lens = rng.integers(2, 7, n)
        lens[rng.choice(n, 50, replace=False)] = 700
    elif case == "many_short":
        n = 140001
        lens = rng.integers(3, 9, n)
    else:
        lens = np.zeros(n, np.int64)
        lens[:300] = 1                 # more than 256 rows in one block's nonzero budget
        lens[300] = 4096               # exactly one block's budget
        lens[301] = 4095
        lens[302:] = rng.integers(0, 7, n - 302)
        lens[-1] = 3                   # nnz not a multiple of 4 at the very end
    lens = np.asarray(lens, np.int64)
    rowp, col, val = _random_csr(rng, lens)
    x = rng.standard_normal(n)
    y, xy = L.spmv_stream_probe(ctx, rowp, col, val, x)
    v32 = val.astype(np.float32).astype(np.float64)
    x32 = x.astype(np.float32).astype(np.float64)
    import scipy.sparse as sp
    A = sp.csr_matrix((v32, col, rowp), shape=(n, n))
    ref = A @ x32
    mag = abs(A) @ abs(x32)
    assert np.all(np.abs(y - ref) <= 2e-6 * np.maximum(mag, 1e-30) + 1e-30), float(np.max(np.abs(y - ref) / np.maximum(mag, 1e-30)))
    assert abs(xy - float(x32 @ y)) <= 1e-10 * float(abs(x32) @ abs(y))


@pytest.mark.parametrize("kind,spec", [("poisson2d", "n=20"), ("elasticity3d", "n=3")])
def test_matvec_and_eliminate(ctx, kind, spec):
    import scipy.sparse as sp
    print("case matvec/eliminate", kind, spec, flush=True)
    p = sa.Problem(ctx, kind, spec)
    info = register_free(p)
    plan = p.generate("fp64")
    nd, nf = info["ndofs"], info["nfree"]
    csr = plan.csr(nd)
    A = sp.csr_matrix((csr.Aval, csr.Acol, csr.Arow), shape=(nf, nf))
    D = sp.csr_matrix((csr.Dval, csr.Dcol, csr.Drow), shape=(nf, nd - nf))
    free = _FREE[(nd, nf)]
    cons = np.ones(nd, bool)
    cons[free] = False
    rng = np.random.default_rng(3)
    x = rng.standard_normal(nd)
    # mat * vec (mat.cpp:182-205)
    y = plan.matvec(x)
    yA = A @ x[free] + D @ x[cons]
    assert relerr(y[free], yA) <= 1e-13
    assert np.array_equal(y[cons], x[cons])
    # mat::eliminate (mat.cpp:78-103), of a given vector and of the assembled rhs
    e = plan.eliminate(nf, x)
    assert relerr(e, x[free] - D @ x[cons]) <= 1e-13
    e0 = plan.eliminate(nf)
    assert relerr(e0, csr.rhs[free] - D @ csr.rhs[cons]) <= 1e-13


@pytest.mark.parametrize("spec,precision", [("n=24", "fp64"), ("n=16;order=2", "fp64"), ("n=24", "f16split"),
                                            ("n=24;bx=200;by=-80", "fp64"),
                                            ("n=190;bx=4000;by=-2000", "fp64")])  # over 32768 rows: dots in more than eight parts
def test_gmres_convection_diffusion_matches_direct(ctx, spec, precision):
    # non-symmetric A: the automatic choice is GMRES; the result matches a
    # direct solve of the same assembled system
    print("case solve convdiff2d", spec, precision, flush=True)
    p = sa.Problem(ctx, "convdiff2d", spec)
    info = register_free(p)
    plan = p.generate(precision)
    ref, A, bA = solve_full(plan.csr(info["ndofs"]), info["ndofs"], info["nfree"])
    assert abs(A - A.T).max() > 1e-3 * abs(A).max()
    x, it = plan.solve(info["ndofs"], rel_tol=1e-12, max_outer=40, max_inner=100)
    print("solve", it, flush=True)
    assert it["method"] == "gmres"
    assert it["rel_residual"] <= 1e-12, it
    assert relerr(x, ref) <= 1e-8, relerr(x, ref)


def test_solve_method_choice(ctx):
    p = sa.Problem(ctx, "poisson2d", "n=12")
    info = register_free(p)
    plan = p.generate("fp64")
    x_cg, i_cg = plan.solve(info["ndofs"], rel_tol=1e-12)
    assert i_cg["method"] == "cg"
    # GMRES on the symmetric system gives the same solution
    x_gm, i_gm = plan.solve(info["ndofs"], rel_tol=1e-12, method="gmres", max_outer=40, max_inner=60)
    assert i_gm["method"] == "gmres" and i_gm["rel_residual"] <= 1e-12
    assert relerr(x_gm, x_cg) <= 1e-9
    with pytest.raises(KeyError):
        plan.solve(info["ndofs"], method="lu")


def test_solve_long_rows(ctx):
    # rows of more than 1024 nonzeros and more than 1024 row blocks: the streaming
    # product, whose partial sums are more than any other kernel's
    import scipy.sparse as sp
    print("case solve long rows", flush=True)
    p = sa.Problem(ctx, "hppoisson3d", "n=7;pmin=5;pmax=5")
    info = register_free(p)
    plan = p.generate("fp64")
    x, it = plan.solve(info["ndofs"], rel_tol=1e-11)
    print("solve", it, flush=True)
    csr, nd, nf = plan.csr(info["ndofs"]), info["ndofs"], info["nfree"]
    assert np.diff(csr.Arow).max() > 1024 and csr.Arow[-1] > 1024 * 4096
    free = _FREE[(nd, nf)]
    cons = np.ones(nd, bool)
    cons[free] = False
    b = csr.rhs[free] - sp.csr_matrix((csr.Dval, csr.Dcol, csr.Drow), shape=(nf, nd - nf)) @ csr.rhs[cons]
    r = b - sp.csr_matrix((csr.Aval, csr.Acol, csr.Arow), shape=(nf, nf)) @ x[free]
    assert it["method"] == "cg" and it["rel_residual"] <= 1e-11
    assert np.linalg.norm(r) <= 2e-11 * np.linalg.norm(b)
    assert np.array_equal(x[cons], csr.rhs[cons])
