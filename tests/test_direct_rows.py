"""Row-wise assembly (kernels/direct.hip) against the oracle: the workloads that
take it, one to many elements, compiled and interpreted coefficients, the element
kernels that SLX_TUNE_DIRECT=0 keeps, absent columns, and on synthetic descriptions
the other shapes of the kernel (two dof fields, 12 derivative pairs, two and five
columns per lane, rows of 255 columns and more, right-hand sides in the matrix
bucket) and the plans that fall back.

Gates: FP64 1e-12; the reduced modes run this kernel in FP32, whose entries are
sums of at most 12 products of rounded factors (below 14 * 6e-8 of the sum of
magnitudes), so 1e-6.
"""
import numpy as np
import pytest

import sparselizard_amd as sa
from _synthetic import Synthetic, addresses
from oracle import py_oracle

pytestmark = pytest.mark.gpu

CASES = [
    ("poisson2d", "n=2"),               # one free row
    ("poisson2d", "n=9"),               # 3 x 3, 4 pairs, three columns per lane
    ("poisson2d", "n=70"),              # compiled coefficients, several workgroups
    ("poisson2d", "n=7;order=2"),       # 6 x 6, two lanes per row
    ("convdiff2d", "n=8"),              # 6 pairs
    ("convdiff2d", "n=6;order=2"),
    ("elasticity3d", "n=2;order=1"),    # 4 x 4, three fields, 9 pairs
    ("elasticity3d", "n=3"),            # 10 x 10, four lanes per row
    ("elasticity3d", "n=10"),           # compiled records, three row classes in one launch
    ("elasticity3d", "n=11"),           # the longest rows by themselves, the others in one launch
    ("elasticity3d", "n=2;clamp=0"),    # no constrained column
]


def relerr(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def check(prob, plan, tol):
    info = prob.info()
    got = plan.csr(info["ndofs"])
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), info["ndofs"], info["nfree"])
    for name in ("Arow", "Acol", "Drow", "Dcol"):
        assert np.array_equal(getattr(got, name), getattr(ref, name)), name
    for name in ("Aval", "Dval", "rhs"):
        assert relerr(getattr(got, name), getattr(ref, name)) <= tol, name
    return got


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("f16split", 1e-6), ("bf16split", 1e-6), ("fp32mfma", 1e-6), ("fp32", 1e-6)])
@pytest.mark.parametrize("kind,spec", CASES)
def test_rows_match_oracle(ctx, kind, spec, precision, tol):
    print("case direct", kind, spec, precision, flush=True)
    prob = sa.Problem(ctx, kind, spec)
    plan = prob.generate(precision)
    assert plan.routes(precision)["row_wise"]
    a = check(prob, plan, tol)
    b = prob.generate(precision).csr(prob.info()["ndofs"])
    assert np.array_equal(a.Aval, b.Aval) and np.array_equal(a.Dval, b.Dval) and np.array_equal(a.rhs, b.rhs)


@pytest.mark.parametrize("precision", ["f16split", "fp32"])
@pytest.mark.parametrize("spec", ["n=6", "n=25"])
def test_rhs_rounds_only_its_coefficients(ctx, spec, precision):
    """The reduced modes' right-hand side sums FP64 products of FP32 coefficients: an entry of a row is off
    by 2^-24 / sqrt(3) (root mean square) at most, and rows have six of them or more: 1.4e-8."""
    prob = sa.Problem(ctx, "poisson2d", spec)
    ref = prob.generate("fp64").csr(prob.info()["ndofs"]).rhs
    got = prob.generate(precision).csr(prob.info()["ndofs"]).rhs
    assert relerr(got, ref) <= 1.5e-8


@pytest.mark.parametrize("kind,spec", [("poisson2d", "n=9"), ("elasticity3d", "n=3")])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_compiled_records(ctx, kind, spec, precision, tol):
    prob = sa.Problem(ctx, kind, spec)
    plan = prob.plan()
    assert plan.coef_mode("compiled") > 0
    check(prob, prob.generate(precision), tol)


@pytest.mark.parametrize("kind,spec", [("poisson2d", "n=9"), ("convdiff2d", "n=8"), ("elasticity3d", "n=3")])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-6)])
def test_element_kernels_agree(ctx, kind, spec, precision, tol, monkeypatch):
    """Element matrices, coefficients and system equal those of the element kernels."""
    prob = sa.Problem(ctx, kind, spec)
    plan = prob.generate(precision)
    ke, co, got = plan.element_matrices(), plan.coefficients(), plan.csr(prob.info()["ndofs"])
    monkeypatch.setenv("SLX_TUNE_DIRECT", "0")
    prob2 = sa.Problem(ctx, kind, spec)
    plan2 = prob2.generate(precision)
    assert plan.routes(precision)["row_wise"] and not plan2.routes(precision)["row_wise"]
    kb, kl = plan2.ke_layout()
    d, sel, k = prob2.desc(), [], 0
    for b in range(d.n_buckets):
        for s in range(d.buckets[b].n_slices):
            sd = d.buckets[b].slices[s]
            e, i, j = np.meshgrid(np.arange(d.buckets[b].n_elem), np.arange(sd.n_tf), np.arange(1 if sd.is_rhs else sd.n_dof), indexing="ij")
            sel.append((kb[k] + (e * sd.n_tf + i) * kl[k] + j).ravel())
            k += 1
    sel = np.concatenate(sel)
    assert relerr(ke[sel], plan2.element_matrices()[sel]) <= tol
    assert np.array_equal(co, plan2.coefficients())
    assert relerr(got.Aval, plan2.csr(prob2.info()["ndofs"]).Aval) <= tol


def drop_columns(prob, rng):
    """Later elements lose ever more of their columns (address -1, as next to a region of lower order),
    so that the rows of one class differ in length."""
    d = prob.desc()
    for b in range(d.n_buckets):
        bd = d.buckets[b]
        for s in range(bd.n_slices):
            sd = bd.slices[s]
            if sd.is_rhs:
                continue
            addr = np.ctypeslib.as_array(sd.dof_addr, shape=(sd.n_dof, bd.n_elem))
            gone = np.random.default_rng(rng).random((sd.n_dof, bd.n_elem)) < np.linspace(0.0, 0.9, bd.n_elem)
            gone[:4] = False  # the vertex functions stay
            addr[gone] = -1


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
@pytest.mark.parametrize("kind,spec", [("elasticity3d", "n=3"), ("elasticity3d", "n=23"), ("poisson2d", "n=60;order=2")])
def test_absent_columns(ctx, kind, spec, precision, tol):
    """Columns without a degree of freedom go to a row's spare accumulator, which
    the next row of the accumulator must find empty: at 23^3 cells the rows of the
    first class have 98 to 195 columns, more of them than the waves in flight hold."""
    print("case absent", kind, spec, precision, flush=True)
    prob = sa.Problem(ctx, kind, spec)
    drop_columns(prob, 7)
    plan = sa.Plan.create(ctx, prob)
    assert plan.routes(precision)["row_wise"]
    plan.assemble(prob.numeric(), precision)
    plan.sync()
    info = prob.info()
    got = plan.csr(info["ndofs"])
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), info["ndofs"], info["nfree"], nthreads=8)
    if spec == "n=23":
        lens = np.diff(got.Arow) + np.diff(got.Drow)
        assert (lens >= 128).sum() > 16 * 6 * 256 and len(np.unique(lens[lens >= 128])) > 20
    for name in ("Arow", "Acol", "Drow", "Dcol"):
        assert np.array_equal(getattr(got, name), getattr(ref, name)), name
    # entry by entry too: a leftover is one wrong entry of many
    for name in ("Aval", "Dval", "rhs"):
        a, b = getattr(got, name), getattr(ref, name)
        assert relerr(a, b) <= tol, name
        assert np.abs(a - b).max() <= 100 * tol * np.abs(b).max(), name


ALL = [(r, c) for r in range(4) for c in range(4)]
# fields of rows and columns, derivative pairs, row and column functions, elements, dofs per field, right-hand side
SHAPES = [
    (2, 1, 12, 3, 3, 50, 40, "other"),       # one lane a row
    (1, 1, 11, 5, 5, 60, 40, "same"),        # two lanes, three columns each
    (2, 2, 3, 4, 4, 70, 60, "other"),        # two lanes, two columns each
    (3, 2, 9, 10, 10, 40, 50, "same"),       # two dof fields, 9 pairs
    (1, 2, 7, 6, 6, 65, 50, "none"),
    (3, 3, 12, 10, 10, 40, 60, "other"),     # 36 coefficients a segment
    (3, 3, 9, 20, 20, 25, 60, "same"),       # five columns a lane
    (2, 1, 6, 15, 13, 33, 70, "other"),      # a last lane without columns
    (1, 1, 4, 4, 10, 64, 80, "other"),       # more columns than rows
    (3, 3, 9, 10, 10, 700, 300, "other"),    # 16-bit slots
    (2, 2, 9, 10, 10, 700, 300, "same"),
    (1, 1, 9, 20, 20, 12000, 2500, "none"),  # rows of 1300 columns: fewer than 16 of them a wave
    (1, 1, 12, 12, 12, 900, 400, "same"),
    (2, 2, 9, 10, 10, 90, 80, "apart"),      # a right-hand side that keeps its kernels, on the side stream
]


def synthetic(na, nb, n_pairs, n_tf, n_dof, n_elem, per_field, rhs, seed=3):
    rng = np.random.default_rng(seed)
    nf = max(na, nb)
    tf = [addresses(rng, n_tf, n_elem, a * per_field, (a + 1) * per_field, 0.03) for a in range(na)]
    dof = [addresses(rng, n_dof, n_elem, b * per_field, (b + 1) * per_field, 0.03) for b in range(nb)]
    mat = [dict(tf=t, dof=u, pairs=ALL[:n_pairs]) for t in tf for u in dof]
    rows = [dict(tf=t, pairs=[(a % 4, 0), (3, 0)][:2 if rhs == "apart" else 1]) for a, t in enumerate(tf)]
    buckets = [mat + rows] if rhs == "same" else [mat] if rhs == "none" else [mat, rows]
    return Synthetic(buckets, nf * per_field, rng.random(nf * per_field) < 0.1, seed)


def check_synthetic(ctx, prob, precision, tol, row_wise):
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), prob.ndofs, prob.nfree, nthreads=8)
    plan = sa.Plan.create(ctx, prob)
    assert plan.routes(precision)["row_wise"] == row_wise
    for mode in ("interpreter", "compiled"):
        plan.coef_mode(mode)
        plan.assemble(prob.numeric(), precision)
        plan.sync()
        got = plan.csr(prob.ndofs)
        for name in ("Arow", "Acol", "Drow", "Dcol"):
            assert np.array_equal(getattr(got, name), getattr(ref, name)), name
        for name in ("Aval", "Dval", "rhs"):
            a, b = getattr(got, name), getattr(ref, name)
            assert relerr(a, b) <= tol, (name, mode)
            assert np.abs(a - b).max(initial=0.0) <= 100 * tol * np.abs(b).max(initial=0.0), (name, mode)
    return ref


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("f16split", 1e-6)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_synthetic_shapes(ctx, shape, precision, tol):
    print("case synthetic", shape, precision, flush=True)
    ref = check_synthetic(ctx, synthetic(*shape), precision, tol, True)
    if shape[5] >= 700:
        assert (np.diff(ref.Arow) + np.diff(ref.Drow)).max() >= (1200 if shape[5] == 12000 else 255)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("f16split", 1e-6)])
@pytest.mark.parametrize("shape", [(1, 2, 10, 6, 6, 60, 50, "other"),       # two dof fields with more than 9 pairs
                                   (1, 3, 4, 6, 6, 2000, 300, "other"),     # two lanes a row: none of more than 254 columns
                                   (1, 1, 4, 24, 24, 30, 60, "same")],      # more than 20 columns
                         ids=lambda s: "-".join(map(str, s)))
def test_element_kernels_take_the_rest(ctx, shape, precision, tol):
    print("case synthetic", shape, precision, flush=True)
    check_synthetic(ctx, synthetic(*shape), precision, tol, False)
