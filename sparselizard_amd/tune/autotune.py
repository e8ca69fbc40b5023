"""Autotuner of the element-kernel choice and tile shape per bucket class.

A bucket class is (element type, n_tf, n_dof, coefficients constant over the
Gauss points).  For every class of every representative workload below it
times the split-precision assembly (HIP events per launch, slx_plan_profile)
with each candidate for that class alone -- the batched MFMA kernel with one
or two M tiles per wave (16 elements per workgroup tile), the factorized MFMA
kernel with each tile shape that covers the matrix ((2, 1), (4, 2) or (7, 2)
16x16 tiles per wave in rows and columns), the one-tile kernel (one element per
wave, up to 4 x 4 tiles; Gauss-point-varying classes up to 64 x 64), or the FP32
VALU element kernel --
while the workload's other classes keep the built-in choice.  Candidates whose
global-matrix error against the FP64 assembly exceeds 1e-6 are dropped, and
the fastest per class goes to kernel_table.txt (next to this script), which
the library reads at plan creation.  Every (class, candidate) runs in a fresh
process with SLX_TUNE_TABLE pointing at a one-line table.  Needs one GPU.

usage: python3 sparselizard_amd/tune/autotune.py [--out FILE] [--iters N]
"""
import argparse
import json
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

# (kind, spec): mid-size versions of the benchmark workloads and a few classes around them
WORKLOADS = [
    ("elasticity3d", "n=20;order=2"),
    ("elasticity3d", "n=24;order=1"),
    ("poisson2d", "n=400"),
    ("poisson2d", "n=200;order=2"),
    ("quadbatch", "instances=48"),
    ("newton2d", "n=300"),
    ("hppoisson3d", "n=16"),
    # isolates the order-1 hexahedra of the hp workload (a later workload's choice wins)
    ("hppoisson3d", "n=40;pmin=1;pmax=1"),
    ("prism3d", "n=40"),
    ("prism3d", "n=20;order=2"),
    ("prism3d", "n=16;order=3"),
]
# factorized tile shapes (row tiles, column tiles per wave), the variant index of the table
FACTOR_SHAPES = [(2, 1), (4, 2), (7, 2)]


def candidates(c):
    """(kernel, mtw, variant) candidates for class c = (type, n_tf, n_dof, q_inv): the
    batched kernel holds at most 16 M tiles of 16 rows, the factorized one is for
    larger element matrices (a shape must cover the rows with its 2 row waves), the
    VALU kernel takes everything.  The first is the reference of the 3 % rule."""
    m = c[1] * c[2]
    tile = [("tile", 1, -1)] if c[3] == 0 and c[1] <= 64 and c[2] <= 64 else []
    if m <= 256:
        return [("mfma", 1, -1), ("mfma", 2, -1)] + tile + [("valu", 1, -1)]
    mt = (c[1] + 15) // 16
    out = [("factor", 1, v) for v, (bm, bn) in enumerate(FACTOR_SHAPES) if 2 * bm >= mt]
    return out + tile + [("valu", 1, -1)]


def classes_of(kind, spec):
    sys.path.insert(0, ROOT)
    import sparselizard_amd as sa
    p = sa.Problem(None, kind, spec)
    d = p.desc()
    out = set()
    for b in range(d.n_buckets):
        bd = d.buckets[b]
        for s in range(bd.n_slices):
            sd = bd.slices[s]
            if not sd.is_rhs:
                out.add((bd.elem_type, sd.n_tf, sd.n_dof, 1 if bd.q_invariant else 0))
    return sorted(out)


def child(kind, spec, iters):
    """Runs in the tuning subprocess: ms per split assembly and its error."""
    sys.path.insert(0, ROOT)
    import ctypes as C
    import numpy as np
    import torch
    import sparselizard_amd as sa
    torch.cuda.init()
    ctx = sa.Context(0)
    prob = sa.Problem(ctx, kind, spec)
    info = prob.info()
    nd = prob.numeric()
    xyz = torch.from_numpy(np.ctypeslib.as_array(nd.node_xyz, shape=(3 * prob.n_nodes(),)).copy()).to("cuda:0")
    par = torch.from_numpy(np.ctypeslib.as_array(nd.params, shape=(nd.n_params * nd.param_len,)).copy()
                           if nd.n_params > 0 and nd.param_len > 0 else np.zeros(1)).to("cuda:0")
    fdata = [torch.from_numpy(f.copy()).to("cuda:0") for f in prob.field_data()]
    fptr = (C.c_void_p * len(fdata))(*[f.data_ptr() for f in fdata]) if fdata else None
    plan = prob.generate("fp64")
    ref = plan.csr(info["ndofs"])
    prob.generate("f16split")
    got = plan.csr(info["ndofs"])
    num = np.sqrt(np.sum((got.Aval - ref.Aval) ** 2) + np.sum((got.Dval - ref.Dval) ** 2))
    den = np.sqrt(np.sum(ref.Aval ** 2) + np.sum(ref.Dval ** 2))
    ms = plan.profile(C.c_void_p(xyz.data_ptr()), C.c_void_p(par.data_ptr()), nd.param_len, fptr, "f16split", iters=iters)
    print(json.dumps({"ms": sum(ms.values()), "kernels": ms, "err": float(num / max(den, 1e-300)),
                      "kernels_used": plan.kernels()}))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--out", default=os.path.join(HERE, "kernel_table.txt"))
    ap.add_argument("--iters", type=int, default=5)
    ap.add_argument("--child", nargs=2)
    ap.add_argument("--only", default="", help="tune only the workloads of this kind")
    args = ap.parse_args()
    if args.child:
        child(args.child[0], args.child[1], args.iters)
        return
    best = {}
    log = []
    for kind, spec in WORKLOADS:
        if args.only and kind != args.only:
            continue
        for c in classes_of(kind, spec):
            results = []
            for kern, mtw, var in candidates(c):
                # this class alone in the table: the workload's other classes keep the built-in choice
                with tempfile.NamedTemporaryFile("w", suffix=".txt", delete=False) as f:
                    f.write("%d %d %d %d %s %d %d\n" % (c + (kern, mtw, var)))
                    tab = f.name
                # the kernels that the table chooses between, without those that take the bucket before it is read
                env = dict(os.environ, SLX_TUNE_TABLE=tab, SLX_TUNE_DIRECT="0", SLX_TUNE_ELEM_FUSED="0")
                print("tuning %s %s class %s: %s mtw %d variant %d" % (kind, spec, c, kern, mtw, var), flush=True)
                r = subprocess.run([sys.executable, __file__, "--child", kind, spec, "--iters", str(args.iters)],
                                   env=env, capture_output=True, text=True, timeout=600)
                os.unlink(tab)
                if r.returncode != 0:
                    # a candidate the kernels reject (launch limits) is skipped
                    print("   failed: %s" % (r.stderr.strip().splitlines() or ["?"])[-1][:300], flush=True)
                    continue
                res = json.loads(r.stdout.strip().splitlines()[-1])
                print("   %.3f ms, error %.2e" % (res["ms"], res["err"]), flush=True)
                results.append((kern, mtw, var, res))
            ok = [x for x in results if x[3]["err"] <= 1e-6]
            if not ok:
                continue
            # the first candidate unless another is at least 3 % faster
            best_x = ok[0]
            for x in ok[1:]:
                if x[3]["ms"] < 0.97 * best_x[3]["ms"]:
                    best_x = x
            best[c] = best_x[:3]  # a later workload's choice for the same class wins
            log.append("# %s %s class %s: %s" % (kind, spec, c, ", ".join(
                "%s/%d%s %.3f ms" % (k, m, "/v%d" % v if v >= 0 else "", x["ms"]) for k, m, v, x in results)))
    with open(args.out, "w") as f:
        f.write("# Kernel choice and tile shape per bucket class, written by autotune.py on one MI355X\n")
        f.write("# (split precision, HIP-event time of one assembly with the class on the candidate and the\n")
        f.write("# workload's other classes on the built-in choice; candidates above 1e-6 global error\n")
        f.write("# excluded; a candidate replaces the first one only when at least 3 % faster).\n")
        f.write("# columns: elem_type n_tf n_dof q_invariant kernel mtw variant\n")
        f.write("# (mtw: M tiles per wave of the batched kernel; variant: tile shape of the factorized\n")
        f.write("# kernel, 0 = (2, 1), 1 = (4, 2), 2 = (7, 2) row and column tiles per wave)\n")
        for line in log:
            f.write(line + "\n")
        for c in sorted(best):
            f.write("%d %d %d %d %s %d %d\n" % (c + best[c]))
    print("wrote", args.out)


if __name__ == "__main__":
    main()
