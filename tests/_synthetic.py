"""Plan descriptions with random tables and addresses: shapes that no workload of
the library produces (row-wise kernel, launches shared by buckets).  Every element
is a tetrahedron with nodes of its own; the coefficients of slot k are the element
parameter k times the entry (k % 3, k // 3 % 3) of the inverse Jacobian."""
import ctypes as C

import numpy as np

from sparselizard_amd import _lib as L


class Synthetic:
    """buckets: a list of lists of slices, each a dict with tf (address array
    [n_tf][n_elem]), optional dof (address array; a right-hand side without), pairs
    (list of (tf derivative, dof derivative)) and optional table numbers."""

    def __init__(self, buckets, n_dofs, constrained, seed=0, n_gp=4, q_invariant=1):
        rng = np.random.default_rng(seed)
        self.keep = []
        d = self.d = L.PlanDesc()
        ne = [b[0]["tf"].shape[1] for b in buckets]
        d.mesh_dim, d.n_dofs, d.n_buckets = 3, n_dofs, len(buckets)
        d.n_nodes = 4 * sum(ne)
        corners = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], float)
        self.xyz = (corners + rng.uniform(-0.15, 0.15, (sum(ne), 4, 3)) + rng.uniform(0, 4, (sum(ne), 1, 3))).reshape(-1)
        d.constrained = self._arr(constrained, np.uint8, C.c_uint8)
        d.dirichlet = self._arr(rng.standard_normal(n_dofs), np.float64, C.c_double)
        d.n_consts, d.consts = 1, self._arr([1.0], np.float64, C.c_double)
        d.has_matrix = int(any("dof" in s for b in buckets for s in b))
        d.has_rhs = int(any("dof" not in s for b in buckets for s in b))
        n_params, first, rank = 0, 0, 0
        bds = (L.BucketDesc * len(buckets))()
        gp = rng.dirichlet(np.ones(4), n_gp)[:, 1:]
        gw = rng.uniform(0.5, 1.5, n_gp) / n_gp
        for b, slices in enumerate(buckets):
            bd = bds[b]
            bd.elem_type, bd.n_elem, bd.n_geo, bd.n_gp = 4, ne[b], 4, n_gp
            bd.geo_nodes = self._arr(4 * first + np.arange(4 * ne[b]), np.int32, C.c_int32)
            bd.elem_ids = self._arr(first + np.arange(ne[b]), np.int32, C.c_int32)
            bd.gp_coords, bd.gp_weights = self._arr(gp, np.float64, C.c_double), self._arr(gw, np.float64, C.c_double)
            sizes, sds, prog, k = [], (L.SliceDesc * len(slices))(), [], 0
            for s, sl in enumerate(slices):
                sd = sds[s]
                sd.frag_rank, sd.is_rhs = rank, int("dof" not in sl)
                rank += 1
                sd.n_tf, sd.n_dof = sl["tf"].shape[0], sl["dof"].shape[0] if "dof" in sl else 1
                sd.tf_addr = self._arr(sl["tf"], np.int32, C.c_int32)
                if "dof" in sl:
                    sd.dof_addr = self._arr(sl["dof"], np.int32, C.c_int32)
                terms = (L.Term * len(sl["pairs"]))()
                for t, (r, c) in enumerate(sl["pairs"]):
                    terms[t] = L.Term(r, c, k)
                    prog += [L.Instr(1, 0, 0, 0, k), L.Instr(3, 1, k % 3, k // 3 % 3, 0), L.Instr(8, 2, 0, 1, 0), L.Instr(18, 0, 2, 0, k)]
                    k += 1
                self.keep.append(terms)
                sd.n_terms, sd.terms = len(terms), terms
                for n in (sd.n_tf, sd.n_dof):  # one table per size, shared by the slices
                    if n not in sizes:
                        sizes.append(n)
                sd.tf_table, sd.dof_table = sizes.index(sd.n_tf), sizes.index(sd.n_dof)
            n_params = max(n_params, k)
            tabs = (C.POINTER(C.c_double) * len(sizes))()
            for t, n in enumerate(sizes):
                tabs[t] = self._arr(np.random.default_rng(100 * n + seed).standard_normal((4, n, n_gp)), np.float64, C.c_double)
            pr = (L.Instr * len(prog))(*prog)
            self.keep += [sds, tabs, pr]
            bd.n_tables, bd.table_nff, bd.tables = len(sizes), self._arr(sizes, np.int32, C.c_int32), tabs
            bd.n_slices, bd.slices, bd.n_instr, bd.prog = len(slices), sds, len(prog), pr
            bd.n_regs, bd.n_coefs, bd.q_invariant = 3, k, q_invariant
            first += ne[b]
        d.buckets = bds
        self.params = rng.uniform(0.5, 2.0, n_params * first)
        self.keep.append(bds)
        self.ndofs, self.nfree = n_dofs, int((np.asarray(constrained) == 0).sum())
        self.nd = L.NumericDesc()
        pd = C.POINTER(C.c_double)
        self.nd.node_xyz, self.nd.params = self.xyz.ctypes.data_as(pd), self.params.ctypes.data_as(pd)
        self.nd.n_params, self.nd.param_len = n_params, first

    def _arr(self, a, dtype, ctype):
        a = np.ascontiguousarray(a, dtype)
        self.keep.append(a)
        return a.ctypes.data_as(C.POINTER(ctype))

    def desc_ptr(self):
        return C.cast(C.pointer(self.d), C.c_void_p)

    def numeric(self):
        return self.nd


def addresses(rng, n_fun, n_elem, lo, hi, absent=0.0):
    """n_fun different numbers of lo .. hi - 1 per element, a share of them -1."""
    a = np.stack([rng.choice(hi - lo, n_fun, replace=False) for _ in range(n_elem)], 1) + lo
    a[rng.random(a.shape) < absent] = -1
    return a.astype(np.int32)
