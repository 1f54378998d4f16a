"""The ILU(0) Krylov loops whose scalars stay on the device: triangular levels
of a launch each (rows of few and of many entries), pcg at given iteration
limits, and GMRES whose work vectors start from memory holding NaN.

pcg is compared with the same recurrence in numpy on the library's own factors:
after k steps the iterates differ by the rounding of k dot products and
triangular solves, amplified by the system's condition (at most about 1e3 for
these diagonally dominant matrices): 1e-12 relative."""
import numpy as np
import pytest
import scipy.sparse as sp
from scipy.sparse.linalg import spsolve_triangular

pytestmark = pytest.mark.gpu


def spd(n, per_row, seed):
    """symmetric diagonally dominant, about `per_row` off-diagonals a row"""
    rng = np.random.default_rng(seed)
    m = n * per_row // 2
    i, j = rng.integers(0, n, m), rng.integers(0, n, m)
    keep = i != j
    A = sp.coo_matrix((-rng.uniform(0.1, 1.0, keep.sum()), (i[keep], j[keep])), shape=(n, n)).tocsr()
    A = A + A.T
    A = (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.5)).tocsr()
    A.sort_indices()
    return A


def numpy_pcg(A, solve, b, steps):
    h = np.linalg.norm(b)
    x, r, p, s = np.zeros_like(b), b / h, None, None
    for _ in range(steps):
        z = solve(r)
        s0, s = s, r @ z
        p = z if p is None else s / s0 * p + z
        q = A @ p
        a = s / (p @ q)
        x, r = x + a * p, r - a * q
    return x * h, np.linalg.norm(r)


@pytest.mark.parametrize("n,per_row", [(4096, 2), (4097, 6), (9001, 20)])
@pytest.mark.parametrize("ordering", ["multicolour", "natural"])
def test_pcg_steps_match_numpy(gpu, n, per_row, ordering):
    print("ilu pcg", n, per_row, ordering, flush=True)
    A = spd(n, per_row, 5 * n + per_row)
    f = gpu.ILU(A.indptr, A.indices, A.data, ordering=ordering)
    perm = f.permutation()
    L, U = (sp.csr_matrix((v, c, r), shape=(n, n)) for r, c, v in (f.factor("L"), f.factor("U")))

    def solve(r):
        w = np.empty_like(r)
        w[perm] = spsolve_triangular(U, spsolve_triangular(L, r[perm], lower=True), lower=False)
        return w

    b = np.random.default_rng(3).standard_normal(n)
    z = f.apply(b)
    assert np.linalg.norm(z - solve(b)) <= 1e-13 * np.linalg.norm(z)
    for steps in (1, 2, 3, 7):
        got = f.pcg(b, tol=1e-300, max_iter=steps, stop="relres")
        x, _ = numpy_pcg(A, solve, b, steps)
        assert got["iters"] == steps
        assert np.linalg.norm(got["x"] - x) <= 1e-12 * np.linalg.norm(x)
    # the stop: the first step at which the recurrence's residual is at most tol
    got = f.pcg(b, tol=1e-9, max_iter=500, stop="relres")
    assert numpy_pcg(A, solve, b, got["iters"])[1] <= 1.01e-9 < numpy_pcg(A, solve, b, got["iters"] - 1)[1] * 1.01
    assert np.linalg.norm(A @ got["x"] - b) <= 1e-8 * np.linalg.norm(b)
    f.close()


def test_gmres_does_not_read_its_work_vectors(gpu):
    """work vectors in memory that held NaN (freed vectors of the same size)"""
    A = spd(2000, 6, 11)
    b = np.random.default_rng(4).standard_normal(2000)
    held = [gpu.DeviceVector(2000) for _ in range(64)]
    for v in held:
        v.fill(float("nan"))
    for v in held:
        v.free()
    f = gpu.ILU(A.indptr, A.indices, A.data)
    got = f.gmres(b, m=20, tol=1e-10, max_iter=400)
    f.close()
    assert np.linalg.norm(A @ got["x"] - b) <= 1e-8 * np.linalg.norm(b)


@pytest.mark.parametrize("n,hub", [(4099, 300), (30000, 9000)])
def test_long_rows_in_wide_levels(gpu, n, hub):
    """rows past a level's slots: their other entries come from the factor's CSR"""
    print("long rows", n, hub, flush=True)
    A = spd(n, 4, n)
    for c in (n // 3, n - 5):
        j = (c + 1 + 3 * np.arange(hub)) % n
        w = sp.coo_matrix((np.full(hub, 0.01), (np.full(hub, c), j)), shape=(n, n)).tocsr()
        w = w + w.T
        A = A + sp.diags(np.asarray(w.sum(axis=1)).ravel()) - w
    A = A.tocsr()
    A.sort_indices()
    f = gpu.ILU(A.indptr, A.indices, A.data, ordering="multicolour")
    perm = f.permutation()
    L, U = (sp.csr_matrix((v, c, r), shape=(n, n)) for r, c, v in (f.factor("L"), f.factor("U")))
    assert max(f.level_entries(w) for w in "LU") < 3 * (L.nnz + U.nnz)
    b = np.random.default_rng(9).standard_normal(n)
    w = f.apply(b)[perm]
    m = int(max(np.diff(L.indptr).max(), np.diff(U.indptr).max()))
    # each sweep solves a system perturbed by at most (m + 1) eps, and the check rounds as much again
    bound = abs(L) @ (abs(U) @ np.abs(w))
    assert np.all(np.abs(L @ (U @ w) - b[perm]) <= 4 * (m + 1) * 2.0 ** -53 * bound)
    got = f.pcg(b, tol=1e-10, max_iter=300, stop="relres")
    f.close()
    assert np.linalg.norm(A @ got["x"] - b) <= 1e-9 * np.linalg.norm(b)
