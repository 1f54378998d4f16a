"""The one-workgroup triangular sweeps over level widths around their thread
counts (64, 256, 512, 1,024 and two rows a thread), record widths (3 and 4
off-diagonals) and forms the straight-line kernel does not take (longer rows,
sources outside the ring).

w = U^-1 L^-1 z satisfies |L U w - z| <= c eps |L| |U| |w| componentwise: each
sweep solves a system perturbed by at most (m + 1) eps relative (m <= 12
entries a row), their product by twice that, plus the check's own rounding."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

STENCIL = {5: [(0, 1), (1, 0)], 7: [(0, 1), (1, 0), (1, 1)], 9: [(0, 1), (1, 0), (1, 1), (1, -1)],
           25: [(0, 1), (0, 2)] + [(a, b) for a in (1, 2) for b in range(-2, 3)]}


def grid(nx, ny, points, seed):
    rng = np.random.default_rng(seed)
    r, c = np.divmod(np.arange(nx * ny), nx)
    i, j = [], []
    for dr, dc in STENCIL[points]:
        ok = (r + dr < ny) & (c + dc >= 0) & (c + dc < nx)
        i.append(np.flatnonzero(ok))
        j.append(np.flatnonzero(ok) + dr * nx + dc)
    i, j = np.concatenate(i), np.concatenate(j)
    A = sp.coo_matrix((-rng.uniform(0.1, 1.0, len(i)), (i, j)), shape=(nx * ny, nx * ny)).tocsr()
    A = A + A.T
    A = (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() + 0.1)).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("nx,ny,points", [(1, 1, 5), (2, 3, 7), (33, 50, 7), (64, 64, 5), (65, 70, 7), (300, 17, 7),
                                          (256, 256, 5), (257, 300, 7), (90, 90, 9), (513, 520, 7), (1025, 1030, 7),
                                          (40, 300, 25), (3000, 5, 9)])
def test_sweeps_by_level_width(gpu, nx, ny, points):
    print("tri sweeps", nx, ny, points, flush=True)
    A = grid(nx, ny, points, nx + ny)
    n = A.shape[0]
    f = gpu.ILU(A.indptr, A.indices, A.data)
    L, U = (sp.csr_matrix((v, c, r), shape=(n, n)) for r, c, v in (f.factor("L"), f.factor("U")))
    z = np.random.default_rng(1).standard_normal(n)
    w = f.apply(z)
    again = f.apply(z)
    f.close()
    assert np.array_equal(w, again)
    bound = abs(L) @ (abs(U) @ np.abs(w))
    assert np.all(np.abs(L @ (U @ w) - z) <= 48 * 2.0 ** -53 * bound)
