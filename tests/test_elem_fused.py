"""Element kernels compiled with their coefficient program against the oracle
and against the separate program and element kernels: triangles of order 2 with
a field in the coefficients (matrix and right-hand side in one bucket), order-1
hexahedra and prisms (Gauss-point-varying Jacobians, two matrix slices), a
constant right-hand side, order-1 quadrangles; one element over the workgroup
size and a few.  Right-hand sides of more than 16 functions (order-2 hexahedra
and prisms) keep the tiled kernel.

Gates as for the element kernels: FP64 1e-12; FP32 modes 1e-6 (sums of at most 36
rounded products per entry).
"""
import numpy as np
import pytest

import sparselizard_amd as sa
from oracle import py_oracle

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("f16split", 1e-6), ("fp32", 1e-6)])
@pytest.mark.parametrize("kind,spec,n_fused", [("newton2d", "n=2", 2), ("newton2d", "n=12", 2), ("newton2d", "n=46", 2),
                                               ("hppoisson3d", "n=3;pmin=1;pmax=1", 2), ("hppoisson3d", "n=3;pmin=1;pmax=2", 2),
                                               ("prism3d", "n=4", 3), ("prism3d", "n=3;order=2", 0), ("quadbatch", "instances=2;nmin=3;nmax=5;order=1", 1)])
def test_matches_oracle_and_separate_kernels(ctx, kind, spec, n_fused, precision, tol, monkeypatch):
    print("case elem fused", kind, spec, precision, flush=True)
    got = {}
    for fused in ("1", "0"):
        monkeypatch.setenv("SLX_TUNE_ELEM_FUSED", fused)
        prob = sa.Problem(ctx, kind, spec)
        info = prob.info()
        if kind == "newton2d":
            x = np.sin(0.37 * np.arange(info["ndofs"]))
            prob.setdata_vec(0.1 * x)
        plan = prob.plan()
        assert plan.coef_mode("compiled") > 0
        assert plan.routes(precision)["elem_fused"] == (n_fused if fused == "1" else 0)
        plan = prob.generate(precision)
        got[fused] = plan.csr(info["ndofs"]), plan.coefficients()
    ref = py_oracle.assemble(prob.desc_ptr(), prob.numeric(), info["ndofs"], info["nfree"])
    for name in ("Aval", "Dval", "rhs"):
        assert relerr(getattr(got["1"][0], name), getattr(ref, name)) <= tol, name
        assert relerr(getattr(got["1"][0], name), getattr(got["0"][0], name)) <= tol, name
    assert relerr(got["1"][1], got["0"][1]) <= tol
