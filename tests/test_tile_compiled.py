"""The one-tile-per-element kernel compiled for its slice (kernels/tile_jit.h)
against the oracle and against the general kernel it replaces: tables in
registers (16 x 16, 6 x 6) and in LDS (the others), one to four tiles a side, a
last column tile of 2 to 11 columns (18, 25, 27, 30, 40), one and two passes over
the Gauss points, batches of one and of four elements with ragged ends, launches
over several buckets with different element counts, no more elements than one
workgroup takes.

Gates: the splits' 1e-6 and FP32's 2e-5 against the FP64 oracle, as for the
general kernel; 5e-7 against the general kernel (the same products; the sums over
the coefficients of an entry may be contracted differently, a few FP32 roundings
of at most 2 * 6e-8 each).
"""
import numpy as np
import pytest

import sparselizard_amd as sa
from oracle import py_oracle

pytestmark = pytest.mark.gpu

CASES = [("quadbatch", "instances=1;nmin=1;nmax=1"), ("quadbatch", "instances=3;nmin=2;nmax=11"), ("quadbatch", "instances=2;nmin=5;nmax=9;order=4"),
         ("newton2d", "n=9"), ("prism3d", "n=3;order=2"), ("prism3d", "n=3;order=3"), ("hcurlprojection", "elem=tet;n=3;order=1;term=maxwell"),
         ("hcurlprojection", "elem=tet;n=3;order=2;term=maxwell"), ("hppoisson3d", "n=3;pmin=2;pmax=2"), ("hppoisson3d", "n=2;pmin=3;pmax=3")]


def relerr(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("precision,tol", [("f16split", 1e-6), ("bf16split", 1e-6), ("fp32mfma", 2e-5)])
@pytest.mark.parametrize("kind,spec", CASES)
def test_matches_oracle_and_general_kernel(ctx, kind, spec, precision, tol, monkeypatch, capfd):
    print("case tile compiled", kind, spec, precision, flush=True)
    monkeypatch.setenv("SLX_TUNE_TILE_MIN", "0")
    monkeypatch.setenv("SLX_TUNE_TABLE", "none")
    got = {}
    for compiled in ("1", "0"):
        monkeypatch.setenv("SLX_TUNE_TILE_JIT", compiled)
        prob = sa.Problem(ctx, kind, spec)
        info = prob.info()
        plan = prob.plan()
        plan.coef_mode("compiled")
        n_tile = plan.tile_count(precision)
        assert n_tile >= 1
        # order-3 hexahedra in the BF16 split: the tables exceed the LDS, the general kernel runs
        fits = (spec, precision) != ("n=2;pmin=3;pmax=3", "bf16split")
        assert plan.routes(precision)["tile_compiled"] == (n_tile if compiled == "1" and fits else 0)
        plan = prob.generate(precision)
        got[compiled] = plan.csr(info["ndofs"])
    assert "not compiled" not in capfd.readouterr().err
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), info["ndofs"], info["nfree"])
    for name in ("Aval", "Dval", "rhs"):
        a, b, r = getattr(got["1"], name), getattr(got["0"], name), getattr(ref, name)
        assert relerr(a, r) <= tol, name
        assert relerr(a, b) <= 5e-7, name
