"""Launches shared by the orientation buckets of one element type (24 tetrahedra
orientations at most) against the oracle: interpreted and compiled programs
(512 elements and more over all buckets), every kernel of the family (one-tile,
VALU element kernel, FP64, right-hand sides)."""
import numpy as np
import pytest

import sparselizard_amd as sa
from _synthetic import Synthetic, addresses
from oracle import py_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("f16split", 1e-6), ("bf16split", 1e-6), ("fp32", 1e-6)])
@pytest.mark.parametrize("spec,tile,compiled", [("elem=tet;term=maxwell;n=3;order=2", "1", False), ("elem=tet;term=maxwell;n=9;order=2", "1", True),
                                                ("elem=tet;term=maxwell;n=3;order=2", "0", False), ("elem=tet;term=maxwell;n=5;order=1", "1", True)])
def test_orientation_buckets(ctx, spec, tile, compiled, precision, tol, monkeypatch):
    print("case families", spec, tile, precision, flush=True)
    monkeypatch.setenv("SLX_TUNE_TILE", tile)
    prob = sa.Problem(ctx, "hcurlprojection", spec)
    info = prob.info()
    plan = prob.generate(precision)
    split = precision in ("f16split", "bf16split")
    assert plan.tile_count(precision) == (2 * sum(prob.desc().buckets[b].n_elem > 0 for b in range(prob.desc().n_buckets))
                                          if split and tile == "1" else 0)
    assert plan.routes(precision)["tile_compiled"] == (plan.tile_count(precision) if compiled else 0)
    got = plan.csr(info["ndofs"])
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), info["ndofs"], info["nfree"], nthreads=8)
    assert np.array_equal(got.Arow, ref.Arow) and np.array_equal(got.Acol, ref.Acol)
    for a, b in ((got.Aval, ref.Aval), (got.rhs, ref.rhs)):
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
def test_buckets_with_other_row_layouts(ctx, precision, tol):
    """One launch over two buckets: the two slices of the first have rows of their
    own, those of the second share theirs, so that the second slice's columns
    start at another alignment there."""
    print("case family layouts", precision, flush=True)
    rng = np.random.default_rng(5)
    pairs = [(1, 1), (2, 2), (3, 0)]
    cols = [addresses(rng, 3, 300, 0, 90), addresses(rng, 3, 300, 90, 180)]
    rows = [addresses(rng, 4, 300, 0, 90), addresses(rng, 4, 300, 90, 180)]
    buckets = [[dict(tf=rows[0], dof=cols[0], pairs=pairs), dict(tf=rows[1], dof=cols[1], pairs=pairs)],
               [dict(tf=rows[0][:, :90], dof=cols[0][:, :90], pairs=pairs), dict(tf=rows[0][:, :90], dof=cols[1][:, :90], pairs=pairs)]]
    prob = Synthetic(buckets, 180, rng.random(180) < 0.1, q_invariant=0)
    plan = sa.Plan.create(ctx, prob)
    plan.coef_mode("compiled")
    assert plan.routes(precision)["elem_fused"] == 2
    plan.assemble(prob.numeric(), precision)
    plan.sync()
    got = plan.csr(prob.ndofs)
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), prob.ndofs, prob.nfree)
    assert np.array_equal(got.Arow, ref.Arow) and np.array_equal(got.Acol, ref.Acol)
    for a, b in ((got.Aval, ref.Aval), (got.Dval, ref.Dval)):
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
