"""Row sums of the sliced matrix copies (dev::Slices): y = A x against numpy
over row counts around a slice's 64 rows, row lengths around the limits of one
and several lanes a row, rows of unequal length, and columns that need a third
base (read from the CSR's indices).

Short rows (means up to 24 entries) keep the column order of the reference's
loops: FP64 products equal the sequential sum bit for bit.  Otherwise the sum's
order is free and |y - A x| <= (m + 1) eps sum |a_ij x_j| with m entries a row
(any order of m - 1 additions of rounded products)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_of(n, mean, spread, seed):
    """CSR with about `mean` sorted columns a row (spread: up to twice that in some rows)"""
    rng = np.random.default_rng(seed)
    lens = np.full(n, min(mean, n))
    if spread:
        lens = np.clip(rng.integers(max(1, mean // 2), 2 * mean, n), 1, n)
    cols = []
    for i in range(n):
        m = int(lens[i])
        if 4 * m >= n:
            cols.append(np.sort(rng.permutation(n)[:m]))
        else:
            cols.append(np.unique(np.concatenate([[i], rng.integers(0, n, m - 1)])))
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    return rp, np.concatenate(cols).astype(np.int32)


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 255, 257, 1000, 70001])
@pytest.mark.parametrize("mean,spread", [(1, False), (7, False), (14, True), (24, False), (25, False), (60, True),
                                         (130, False), (300, True)])
def test_products_with_sliced_rows(gpu, n, mean, spread):
    if n > 1000 and mean > 60:
        pytest.skip("the long rows are covered by the smaller matrices")
    print("slices", n, mean, spread, flush=True)
    rp, ci = rows_of(n, mean, spread, 1000 * mean + n)
    rng = np.random.default_rng(7)
    v, x = rng.standard_normal(len(ci)), rng.standard_normal(n)
    A = gpu.Matrix(rp, ci, v)
    y, y32 = A.spmv(x), A.spmv(x, precision="mixed")
    A.close()
    prod = v * x[ci]
    m = np.diff(rp)
    ref = np.array([np.sum(prod[rp[i]:rp[i + 1]].astype(np.longdouble)) for i in range(n)]).astype(np.float64)
    bound = np.array([np.sum(np.abs(prod[rp[i]:rp[i + 1]])) for i in range(n)])
    assert np.all(np.abs(y - ref) <= (m + 1) * 2.0 ** -53 * bound)
    # FP32: values, x and products rounded once each besides the additions
    assert np.all(np.abs(y32 - ref) <= (m + 4) * 2.0 ** -24 * bound)
    if len(ci) / n <= 24:
        seq = np.zeros(n)
        for j in range(int(m.max())):
            has = m > j
            seq[has] += prod[rp[:-1][has] + j]
        assert np.array_equal(y, seq)


def test_values_follow_an_update(gpu):
    """a hierarchy's sliced copies follow new values (recompute), FP64 and mixed"""
    from fem_amd import problems as P
    s1, s2 = P.damage_system(65), P.damage_system(65, seed_h=99)
    for prec in ("fp64", "mixed"):
        prm = gpu.params("vcycle", 1, 4, precision=prec)
        a, b = gpu.AMG(s1[0].rowptr, s1[0].col, s1[0].val, prm), gpu.AMG(s1[0].rowptr, s1[0].col, s1[0].val, prm)
        d = gpu.DeviceVector(len(s2[0].val))
        d.upload(s2[0].val)
        a.recompute(s2[0].val)
        b.recompute_device(d.ptr)
        ra, rb = (h.pcg(s2[0].b, tol=1e-11, max_iter=500, stop="relres") for h in (a, b))
        r = s2[0].b - s2[0].scipy() @ ra["x"]
        assert np.linalg.norm(r) <= 1e-10 * np.linalg.norm(s2[0].b)
        assert ra["iters"] == rb["iters"] and np.array_equal(ra["x"], rb["x"])
        a.close()
        b.close()


@pytest.mark.parametrize("dense", [0, 18])
def test_finest_copies_with_unequal_row_blocks(gpu, dense):
    """an aggressive hierarchy's finest matrix whose FP64 copy is cut by row
    block and whose FP32 copy is cut every 64 rows: as many slices, other rows"""
    import scipy.sparse as sp
    from fem_amd import problems as P
    s = P.damage_system(783)[0]
    A, n = s.scipy().tocsr(), s.n
    for c in (20_000, 333_333):  # a patch of `dense` rows coupled to 16 far ones each
        i = np.repeat(c - c % 256 + 60 + np.arange(dense), 16)
        j = 1000 + (c + 2039 * np.arange(len(i))) % (n - 2000)
        w = sp.coo_matrix((np.full(len(j), 1e-3), (i, j)), shape=(n, n)).tocsr()
        w = w + w.T
        A = A + sp.diags(np.asarray(w.sum(axis=1)).ravel()) - w
    A = A.tocsr()
    A.sort_indices()
    rp, ci = A.indptr, A.indices
    rows = [gpu.slice_layout(rp, ci, False, True, p)[0] for p in ("fp64", "mixed")]
    unequal = len(rows[0]) == len(rows[1]) and not np.array_equal(rows[0], rows[1])
    assert unequal == (dense > 0)
    print("finest copies", dense, len(rows[0]), flush=True)
    amg = gpu.AMG(rp, ci, A.data, gpu.params("vcycle", 1, 6, precision="mixed"))
    x = np.random.default_rng(5).standard_normal(n)
    ref, bound = A @ x, abs(A) @ np.abs(x)
    m = np.diff(rp)
    assert np.all(np.abs(amg.spmv(x) - ref) <= 2 * (m + 1) * 2.0 ** -53 * bound)
    assert np.all(np.abs(amg.spmv(x, precision="mixed") - ref) <= (m + 4) * 2.0 ** -24 * bound)
    b = np.random.default_rng(6).standard_normal(n)
    got = amg.pcg(b, tol=1e-9, max_iter=400, stop="relres")
    amg.close()
    assert np.linalg.norm(A @ got["x"] - b) <= 1e-8 * np.linalg.norm(b)


@pytest.mark.parametrize("irregular", [False, True])
def test_operator_with_longer_rows_than_the_hierarchy(gpu, irregular):
    """pcg on an operator of 49 entries a row (more sliced workgroups than the
    hierarchy's matrices have; irregular: in row blocks) under a P1 hierarchy"""
    import scipy.sparse as sp
    from fem_amd import problems as P
    s = P.poisson(408)
    n = s.n
    i = np.arange(n)
    if irregular:
        i = i[i % 50 == 0]
    j = (i[:, None] + 37 * np.arange(1, 23 if not irregular else 400)) % n
    w = sp.coo_matrix((np.full(j.size, 1e-4), (np.repeat(i, j.shape[1]), j.ravel())), shape=(n, n)).tocsr()
    w = w + w.T
    A = (s.scipy() + sp.diags(np.asarray(w.sum(axis=1)).ravel()) - w).tocsr()
    A.sort_indices()
    amg = gpu.AMG(s.rowptr, s.col, s.val, gpu.params("vcycle", 1, 5))
    op = gpu.Matrix(A.indptr, A.indices, A.data)
    assert (len(gpu.slice_layout(A.indptr, A.indices, True, True)[0]) == 0) == irregular
    b = np.random.default_rng(8).standard_normal(n)
    got = amg.pcg_operator(op, b, tol=1e-9, max_iter=500)
    op.close()
    amg.close()
    assert np.linalg.norm(A @ got["x"] - b) <= 1e-8 * np.linalg.norm(b)


@pytest.mark.parametrize("kind,coarsening", [("damage", 1), ("damage", 2), ("elastic", 1), ("elastic", 2)])
@pytest.mark.parametrize("smoother,coarse", [("mc_ssor", "l1_jacobi"), ("jacobi", "mc_sor"), ("l1_jacobi", "mc_ssor")])
def test_recomputed_copies_are_those_of_a_fresh_upload(gpu, kind, coarsening, smoother, coarse):
    """every copy that a device recompute rewrites (both precisions' values,
    slices, colour order, l1 norms) against a hierarchy that reaches the same
    values through full uploads (its pattern changes on the way)"""
    from fem_amd import problems as P
    s = P.damage_system(129)[0] if kind == "damage" else P.degraded_elasticity(65)
    row = np.repeat(np.arange(s.n), np.diff(s.rowptr))
    scale = 1.0 + 0.1 * np.random.default_rng(3).random(s.n)
    new = s.val * scale[row] * scale[s.col]
    mid = new.copy()
    mid[np.flatnonzero(s.col != row)[::3]] = 0.0
    kw = dict(smoother=smoother, coarse_smoother=coarse, coarsening=coarsening)
    prm = {p: gpu.params("vcycle", s.dof, 4, precision=p, **kw) for p in ("fp64", "mixed")}
    a, b = (gpu.AMG(s.rowptr, s.col, s.val, prm["fp64"]) for _ in range(2))
    a.recompute(new)
    b.recompute(mid)
    b.recompute(new)
    rng = np.random.default_rng(4)
    for l in range(a.depth):
        assert np.array_equal(a.level(l)["A"][2], b.level(l)["A"][2])
        x = rng.standard_normal(a.level_sizes(l)["fine"])
        for p in prm:
            assert np.array_equal(a.spmv(x, l, p), b.spmv(x, l, p)), (l, p)
    for p in ("fp64", "mixed", "fp64"):
        for h in (a, b):
            h.set_params(prm[p])
        u, v = (h.pcg(s.b, tol=1e-300, max_iter=5, stop="relres") for h in (a, b))
        assert np.array_equal(u["x"], v["x"]), p
    a.close()
    b.close()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_autotuned_forms(gpu, prec):
    """autotune times the lanes of sliced copies too: on coarse levels with a few
    hundred long rows others than the rule's (8 or 16) are twice as fast.  What it
    chooses multiplies, smooths and follows a recompute like any other form."""
    from fem_amd import problems as P
    s = P.degraded_elasticity(129)
    prm = gpu.params("vcycle", 2, 5, precision=prec, autotune=1)
    amg = gpu.AMG(s.rowptr, s.col, s.val, prm)
    tuned = amg.tuned()
    print("tuned", prec, tuned, flush=True)
    assert len(tuned) == 4 * amg.depth - 3 and all(t[2] in (1, 4, 8, 16, 32) and t[3] in (1, 4, 8, 16, 32) for t in tuned)
    rng = np.random.default_rng(12)
    other = 0
    for l in range(amg.depth):
        rp, ci, v = amg.level(l)["A"]
        m = np.diff(rp)
        rule = [1, 4, 8, 16, 32][int(np.searchsorted([24, 48, 96, 192], m.mean()))]
        other += sum(t[3] != rule for t in tuned if t[0] == l and t[1] in "AC")
        x = rng.standard_normal(len(m))
        prod = v * x[ci]
        ref, bound = np.add.reduceat(prod, rp[:-1]), np.add.reduceat(np.abs(prod), rp[:-1])
        assert np.all(np.abs(amg.spmv(x, l) - ref) <= 2 * (m + 1) * 2.0 ** -53 * bound)
        assert np.all(np.abs(amg.spmv(x, l, "mixed") - ref) <= (m + 4) * 2.0 ** -24 * bound)
    assert other > 0
    b = rng.standard_normal(s.n)
    A = s.scipy().tocsr()
    for scale in (1.0, 1.7):
        got = amg.pcg(b, tol=1e-9, max_iter=3000, stop="relres")
        assert np.linalg.norm(scale * (A @ got["x"]) - b) <= 1e-7 * np.linalg.norm(b)
        assert amg.tuned() == tuned
        amg.recompute(1.7 * s.val)
    amg.close()


def spd(n, per_row, seed):
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    i, j = rng.integers(0, n, n * per_row // 2), rng.integers(0, n, n * per_row // 2)
    A = sp.coo_matrix((-rng.uniform(0.1, 1.0, len(i)), (i, j)), shape=(n, n)).tocsr()
    A = (A + A.T).tolil()
    A.setdiag(0)
    A = A.tocsr()
    A = (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.5)).tocsr()
    A.sort_indices()
    return A


def sweep(A, colours, smoother, x, f, backward):
    d = A.diagonal()
    if smoother == "jacobi":
        return (f - (A @ x - d * x)) / d
    if smoother == "l1_jacobi":
        return x + (f - A @ x) / np.asarray(abs(A).sum(axis=1)).ravel()
    x = x.copy()
    order = range(colours.max() + 1)
    for c in reversed(order) if backward else order:
        r = np.flatnonzero(colours == c)
        x[r] = (f[r] - (A[r] @ x - d[r] * x[r])) / d[r]
    return x


@pytest.mark.parametrize("system", [("damage", 8), ("damage", 9), ("damage", 16), ("damage", 17), ("damage", 129),
                                    ("spd", 63, 10), ("spd", 65, 30), ("spd", 257, 40), ("spd", 700, 130),
                                    ("spd", 1500, 260)])
@pytest.mark.parametrize("smoother", ["jacobi", "l1_jacobi", "mc_sor", "mc_ssor"])
def test_sliced_sweeps_match_numpy(gpu, system, smoother):
    """a two-level V(1,1) cycle whose finest level is swept by slices of one and of
    several lanes a row, against the same cycle in numpy on the hierarchy's own
    matrices.  About 4 (m + 2) roundings an entry (m the longest row) in either
    precision; the coarse solve multiplies them by its condition, below 1e3 here."""
    import scipy.sparse as sp
    from fem_amd import problems as P
    print("sweeps", system, smoother, flush=True)
    A = spd(*system[1:], seed=system[1]) if system[0] == "spd" else P.damage_system(system[1])[0].scipy().tocsr()
    A.sort_indices()
    n = A.shape[0]
    amg = gpu.AMG(A.indptr, A.indices, A.data, gpu.params("vcycle", 1, 2))
    lev, top = amg.level(0), amg.level(1)
    csr = lambda m, shape: sp.csr_matrix((m[2], m[1], m[0]), shape=shape)
    nc = lev["fine"]
    keep = top["P"][1] < nc  # zero seeds of rows the reference leaves empty
    Pm = sp.csr_matrix((top["P"][2] * keep, np.where(keep, top["P"][1], 0), top["P"][0]), shape=(n, nc))
    Rm, Ac = csr(top["R"], (nc, n)), csr(lev["A"], (nc, nc)).toarray()
    f = np.random.default_rng(1).standard_normal(n)
    x = sweep(A, top["colours"], smoother, np.zeros(n), f, False)
    x = x + Pm @ np.linalg.solve(Ac, Rm @ (f - A @ x))
    x = sweep(A, top["colours"], smoother, x, f, smoother == "mc_ssor")
    m = int(np.diff(A.indptr).max())
    for prec, eps in (("fp64", 2.0 ** -53), ("mixed", 2.0 ** -24)):
        amg.set_params(gpu.params("vcycle", 1, 2, smoother=smoother, coarse_smoother=-1, precision=prec))
        it, got = amg.amg_solve(f, np.zeros(n))
        assert it == 1
        assert np.linalg.norm(got - x) <= 4e3 * (m + 2) * eps * np.linalg.norm(x), prec
    amg.close()
