"""The LinA drop-in on the GPU against the compiled reference: the same
caller code (a C program compiled once against include/linalg and linked
against either library, and ctypes calls through the LinA names) gives the
same iteration counts and iterates."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from fem_amd import problems as P
from tests.dropin_bind import DROPIN_SO, LinA, ROOT, dptr

pytestmark = pytest.mark.gpu

from oracle.bind import REF_SO  # noqa: E402


def say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def libs(gpu, ref):
    return LinA(DROPIN_SO), LinA(ref.L)


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def test_c_caller_links_against_either_library(tmp_path):
    obj = tmp_path / "example.o"
    inc = os.path.join(ROOT, "include", "linalg")
    subprocess.run(["gcc", "-std=c99", "-O2", "-c", "-I", inc, "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "dropin_example.c"), "-o", str(obj)], check=True)
    out = {}
    for name, lib in (("dropin", DROPIN_SO), ("reference", REF_SO)):
        if not os.path.exists(lib):
            continue  # a missing drop-in fails below
        exe = tmp_path / f"example_{name}"
        d = os.path.dirname(lib)
        subprocess.run(["gcc", str(obj), "-o", str(exe), lib, f"-Wl,-rpath,{d}", "-lm", "-fopenmp"], check=True)
        r = subprocess.run([str(exe), "65"], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr
        line = [l for l in r.stdout.splitlines() if l.startswith("iterations")][-1]
        out[name] = dict(zip(line.split()[0::2], map(float, line.split()[1::2])))
        say(name, out[name])
    assert out["dropin"]["iterations"] > 1 and out["dropin"]["relres"] < 1e-8
    if "reference" not in out:
        pytest.skip("the drop-in linked and solved; oracle/_ref/libreflina.so not built (needs /root/reference at build time)")
    assert abs(out["dropin"]["iterations"] - out["reference"]["iterations"]) <= 1
    assert abs(out["dropin"]["relres"] / out["reference"]["relres"] - 1) < 1e-6
    assert abs(out["dropin"]["residuum"] / out["reference"]["residuum"] - 1) < 1e-9
    assert abs(out["dropin"]["x0"] / out["reference"]["x0"] - 1) < 1e-12


def _solve_both(libs, build, solve):
    res = []
    for lib in libs:
        ctx = build(lib)
        res.append(solve(lib, ctx))
    return res


def test_pcg_amg_matches_reference(libs):
    s = P.degraded_elasticity(17)

    def run(lib):
        A = lib.from_csr(s.rowptr, s.col, s.val)
        lib.L.PCG_default(A, None, None)
        lib.L.PCG_set_AMG_preconditioner(A, 2, 4)
        x = np.zeros(s.n)
        b = s.b.copy()
        it = lib.L.pcg(dptr(x), dptr(b), s.n, 1e-10, 1000)
        return it, x, lib.L.get_pcg_residuum()

    (i1, x1, r1), (i2, x2, r2) = run(libs[0]), run(libs[1])
    say("pcg amg iters", i1, i2, "rel", rel(x1, x2))
    assert abs(i1 - i2) <= 1 and rel(x1, x2) < 1e-12 and abs(r1 / r2 - 1) < 1e-6


def test_pcg_ilu_matches_reference(libs):
    s = P.damage_system(33)[0]

    def run(lib):
        A = lib.from_csr(s.rowptr, s.col, s.val)
        L = lib.L.sparse_zero(s.n)
        U = lib.L.sparse_zero(s.n)
        lib.L.incomplete_LU_factorization(A, L, U)
        lib.L.PCG_default(A, L, U)
        x = np.zeros(s.n)
        b = s.b.copy()
        it = lib.L.pcg(dptr(x), dptr(b), s.n, 1e-10, 1000)
        return it, x

    (i1, x1), (i2, x2) = run(libs[0]), run(libs[1])
    say("pcg ilu iters", i1, i2, "rel", rel(x1, x2))
    assert abs(i1 - i2) <= 1 and rel(x1, x2) < 1e-12


def test_pcg_host_callback_preconditioner(libs):
    """a caller-defined preconditioner (Jacobi) registered with PCG_set_precon"""
    s = P.poisson(33)
    d = s.scipy().diagonal().copy()
    PREC = C.CFUNCTYPE(C.c_int, C.c_int, C.POINTER(C.c_double), C.POINTER(C.c_double))

    @PREC
    def jacobi(n, r, z):
        for i in range(n):
            z[i] = r[i] / d[i]
        return 1

    def run(lib):
        A = lib.from_csr(s.rowptr, s.col, s.val)
        lib.L.PCG_default(A, None, None)
        lib.PCG_set_precon(C.cast(jacobi, C.c_void_p))
        x = np.zeros(s.n)
        b = s.b.copy()
        return lib.L.pcg(dptr(x), dptr(b), s.n, 1e-10, 2000), x

    (i1, x1), (i2, x2) = run(libs[0]), run(libs[1])
    say("pcg callback iters", i1, i2, "rel", rel(x1, x2))
    assert abs(i1 - i2) <= 1 and rel(x1, x2) < 1e-11


def test_amg_solve_full_multigrid_matches_reference(libs):
    """AMG_setup with FULL_AMG (Multigrid.h:38) and AMG_solve: one
    full-multigrid pass in both libraries, the same result to 1e-12."""
    s = P.degraded_elasticity(17)

    def run(lib):
        A = lib.from_csr(s.rowptr, s.col, s.val)
        lib.L.AMG_print_info(0)
        # the smoother and AMG_solve's controls are library globals: set them
        lib.L.AMG_set_smoother.argtypes = [C.c_void_p]
        lib.L.AMG_set_smoother(C.cast(lib.L.AMG_SOR_smoother, C.c_void_p))
        lib.L.AMG_set_SOR_relaxation_coeff(1.3)
        lib.L.AMG_set_eps(1e-2)
        lib.L.AMG_set_max_iter(100)
        I = lib.L.AMG_setup(A, 2, 4, 2, 3, 1, 2, 1, None, None)
        x = np.sin(np.arange(s.n) * 0.1)
        f = s.b.copy()
        it = lib.L.AMG_solve(I, dptr(f), dptr(x), None)
        lib.L.AMG_free_data(I)
        lib.free(A)
        return it, x

    (i1, x1), (i2, x2) = run(libs[0]), run(libs[1])
    say("full multigrid iters", i1, i2, "rel", rel(x1, x2))
    assert i1 == i2 == 1 and rel(x1, x2) < 1e-12


def test_bicgstab_amg_matches_reference(libs):
    s = P.poisson(33)

    def run(lib):
        A = lib.from_csr(s.rowptr, s.col, s.val)
        lib.L.RN_set_default_matrix(A)
        lib.BI_set_mat_mult(C.cast(lib.RN_default_mat_mult, C.c_void_p))
        lib.L.AMG_set_SOR_relaxation_coeff(1.0)
        lib.L.BI_set_AMG_preconditioner(A, 1, 4)
        lib.L.BI_print_info(0)
        lib.L.BI_set_eps(1e-13)
        lib.L.BI_set_max_iter(200)
        x = np.zeros(s.n)
        b = s.b.copy()
        return lib.L.BiCGStab_solve(dptr(x), dptr(b), s.n), x

    (i1, x1), (i2, x2) = run(libs[0]), run(libs[1])
    say("bicgstab iters", i1, i2, "rel", rel(x1, x2))
    assert abs(i1 - i2) <= 1 and rel(x1, x2) < 1e-10


def test_reflective_newton_matches_reference(libs):
    """set_RN_Hesse / set_RN_linear / set_RN_constraints / RN_set_params /
    RN_set_solver(RN_PCG) / reflective_newton through the LinA names"""
    s, dold, ones = P.damage_system(33, h_scale=100.0)
    n = s.n
    idx = np.arange(n, dtype=np.int32)

    def run(lib):
        L = lib.L
        H = lib.from_csr(s.rowptr, s.col, s.val)
        b = s.b.copy()
        lo, up = dold.copy(), ones.copy()
        L.RN_print_info(0)
        L.set_RN_Hesse.argtypes = [C.c_void_p]
        L.set_RN_Hesse(C.cast(H, C.c_void_p))
        L.set_RN_linear.argtypes = [C.POINTER(C.c_double)]
        L.set_RN_linear(dptr(b))
        L.set_RN_functional.argtypes = [C.c_void_p]
        L.set_RN_functional(None)
        L.RN_set_gradient.argtypes = [C.c_void_p]
        L.RN_set_gradient(None)
        L.set_RN_constraints.argtypes = [C.POINTER(C.c_int), C.POINTER(C.c_double), C.POINTER(C.c_double), C.c_int]
        L.set_RN_constraints(idx.ctypes.data_as(C.POINTER(C.c_int)), dptr(lo), dptr(up), n)
        L.RN_set_params.argtypes = [C.c_int] + [C.c_double] * 10
        L.RN_set_params(50, 1e-8, 0.1, 0.9, 0.1, float(np.sqrt(n) / 2), 1.0, 0.6, 1.1, 1e-3, 1000.0)
        L.RN_set_local_solver.argtypes = [C.c_void_p]
        L.RN_set_local_solver(None)
        L.RN_set_solver(3)
        x = dold.copy()
        L.reflective_newton.argtypes = [C.POINTER(C.c_double)]
        it = L.reflective_newton(dptr(x))
        return it, x

    (i1, x1), (i2, x2) = run(libs[0]), run(libs[1])
    say("reflective newton iters", i1, i2, "rel", rel(x1, x2))
    assert i1 == i2 and rel(x1, x2) < 1e-9


def test_eigenvalue_searches_match_reference(libs):
    """power_method, get_most_negative_eigenvector and
    get_neg_curvature_direction (linear_algebra.c:4802-4865), which Crack
    calls directly (crack.c:8995, 10528, 10648): power_method from the same
    start vector in both libraries (iterations within the rounding of the
    stopping test, estimate and iterate to 1e-9); the two-stage searches
    (start vectors drawn from the time, as in the reference) reach scipy's
    smallest eigenvalue, of a positive definite and of an indefinite matrix,
    in both libraries; matrix_norm bit-identical."""
    import scipy.sparse as sp
    from scipy.sparse.linalg import eigsh
    s = P.damage_system(17, h_scale=1.0)[0]
    A0 = s.scipy().tocsr()
    lmax = eigsh(A0, k=1, which="LA", return_eigenvectors=False)[0]
    lmin = eigsh(A0, k=1, which="SA", return_eigenvectors=False)[0]
    c = 0.5 * (lmin + eigsh(A0, k=2, which="SA", return_eigenvectors=False).max())
    Ai = (A0 - c * sp.identity(s.n, format="csr")).tocsr()
    Ai.sort_indices()
    v0 = np.random.default_rng(7).random(s.n)
    v0 /= np.linalg.norm(v0)
    out = []
    for lib in libs:
        M = lib.from_csr(A0.indptr.astype(np.int32), A0.indices.astype(np.int32), A0.data)
        Mi = lib.from_csr(Ai.indptr.astype(np.int32), Ai.indices.astype(np.int32), Ai.data)
        v = v0.copy()
        e = np.zeros(1)
        it = lib.L.power_method(M, dptr(e), dptr(v), 1000, 1e-8, None, 0.0)
        d = np.zeros(s.n)
        lo = np.zeros(1)
        lib.L.get_most_negative_eigenvector(M, dptr(lo), dptr(d), 100000, 1e-12)
        cu = np.zeros(1)
        lib.L.get_neg_curvature_direction(Mi, dptr(cu), dptr(d), 100000, 1e-12, 1e-10)
        out.append((it, e[0], v, lo[0], cu[0], lib.L.matrix_norm(M)))
        lib.free(M)
        lib.free(Mi)
    (i1, e1, v1, lo1, cu1, q1), (i2, e2, v2, lo2, cu2, q2) = out
    say("power iters", i1, i2, "eig", e1, e2, "lowest", lo1, lo2, lmin, "curvature", cu1, cu2, lmin - c)
    assert q1 == q2
    assert i1 > 0 and abs(i1 - i2) <= 1 and abs(e1 - e2) <= 1e-9 * abs(e2)
    if i1 == i2:
        assert np.linalg.norm(v1 - v2) <= 1e-9
    for lo in (lo1, lo2):
        assert abs(lo - lmin) <= 1e-6 * lmax
    for cu in (cu1, cu2):
        assert cu < 0 and abs(cu - (lmin - c)) <= 1e-6 * lmax


def test_power_method_with_empty_rows_matches_reference(libs):
    """A row list with empty rows (Len[i] == 0, as read_sparse produces from
    a file that holds such rows) is a valid operand of the reference's
    power_method: the rows act as zero rows.  The drop-in's device copy
    gives them the explicit (i, 0.0) entry, so the iteration count, the
    estimate and the iterate agree with the reference's."""
    s = P.damage_system(17, h_scale=1.0)[0]
    empty = [0, 5, s.n // 2, s.n - 1]
    v0 = np.random.default_rng(11).random(s.n)
    v0 /= np.linalg.norm(v0)
    out = []
    for lib in libs:
        M = lib.from_csr(s.rowptr, s.col, s.val)
        for i in empty:
            M.contents.Len[i] = 0     # rows emptied in place (their arrays stay allocated)
        v = v0.copy()
        e = np.zeros(1)
        it = lib.L.power_method(M, dptr(e), dptr(v), 1000, 1e-8, None, 0.0)
        for i in empty:
            M.contents.Len[i] = 1
        lib.free(M)
        out.append((it, e[0], v))
    (i1, e1, v1), (i2, e2, v2) = out
    say("power iters (empty rows)", i1, i2, "eig", e1, e2)
    assert i1 > 0 and abs(i1 - i2) <= 1 and abs(e1 - e2) <= 1e-9 * abs(e2)
    if i1 == i2:
        assert np.linalg.norm(v1 - v2) <= 1e-9
    assert all(abs(v1[i]) <= 1e-300 for i in empty)


class ItlinOpt(C.Structure):
    """struct ITLIN_OPT (LinA/itlin.h:67-78; include/linalg/itlin.h)"""
    _fields_ = [("tol", C.c_double), ("rho", C.c_double), ("i_max", C.c_int), ("maxiter", C.c_int),
                ("termcheck", C.c_int), ("convcheck", C.c_int), ("rescale", C.c_int), ("errorlevel", C.c_int),
                ("monitorlevel", C.c_int), ("datalevel", C.c_int)] + \
               [(f, C.c_void_p) for f in ("errorfile", "monitorfile", "datafile", "iterfile", "resfile", "miscfile")] + \
               [("scale", C.c_void_p)]


class ItlinInfo(C.Structure):
    _fields_ = [("precision", C.c_double), ("normdx", C.c_double), ("residuum", C.c_double)] + \
               [(f, C.c_int) for f in ("iter", "rcode", "subcode", "nomatvec", "noprecon", "noprecl", "noprecr")]


_MATVEC = C.CFUNCTYPE(None, C.c_int, C.POINTER(C.c_double), C.POINTER(C.c_double))


def _nonsymmetric(m=17):
    """the damage system plus a skew part on its own pattern (GMRES's case)"""
    s = P.damage_system(m)[0]
    A = s.scipy().tocsr()
    r = np.repeat(np.arange(s.n), np.diff(A.indptr))
    skew = np.where(A.indices > r, 0.3, np.where(A.indices < r, -0.3, 0.0)) * np.abs(A.data)
    A.data = A.data + skew
    return A, s.b


@pytest.mark.parametrize("termcheck", [0, 1])
@pytest.mark.parametrize("callbacks", ["library", "host"])
def test_gmres_matches_reference(libs, termcheck, callbacks):
    """gmres (gmres.c:308-501) as FEM.c drives it (FEM.c:531-541, 737-744):
    ILU(0) factors of PCG_default, PCG_mult as the operator, PCG_preconlr as
    the right preconditioner, restart 30, then x = M^-1 y.  Either the
    library's own callbacks (which the drop-in runs on the device) or host
    callbacks (scipy products and triangular solves, staged through host
    copies); CheckOnRestart and CheckEachIter.  Iteration counts equal, the
    solutions to 1e-9, rcode 0 in both libraries, and the solution solves the
    system."""
    from scipy.sparse.linalg import spsolve_triangular
    A, b = _nonsymmetric()
    n = A.shape[0]
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    out = []
    for lib in libs:
        M = lib.from_csr(rp, ci, A.data)
        L = lib.L.sparse_zero(n)
        U = lib.L.sparse_zero(n)
        assert lib.L.incomplete_LU_factorization(M, L, U) == 1
        lib.L.PCG_default.argtypes = [C.c_void_p] * 3
        lib.L.PCG_default(M, L, U)
        keep = []
        if callbacks == "library":
            mv, pr = C.cast(lib.L.PCG_mult, C.c_void_p), C.cast(lib.L.PCG_preconlr, C.c_void_p)
        else:
            Ld = LinA.to_lists(L)
            Ud = LinA.to_lists(U)
            import scipy.sparse as sps

            def tocsr(rows):
                r = np.repeat(np.arange(n), [len(c) for c, _ in rows])
                return sps.csr_matrix((np.concatenate([v for _, v in rows]), (r, np.concatenate([c for c, _ in rows]))),
                                      shape=(n, n))
            Ls, Us = tocsr(Ld), tocsr(Ud)

            def host_mv(nn, x, y):
                xv = np.ctypeslib.as_array(x, shape=(nn,))
                np.ctypeslib.as_array(y, shape=(nn,))[:] = A @ xv

            def host_pr(nn, z, w):
                zv = np.ctypeslib.as_array(z, shape=(nn,))
                t = spsolve_triangular(Ls, zv, lower=True)
                np.ctypeslib.as_array(w, shape=(nn,))[:] = spsolve_triangular(Us, t, lower=False)
            keep = [_MATVEC(host_mv), _MATVEC(host_pr)]
            mv, pr = C.cast(keep[0], C.c_void_p), C.cast(keep[1], C.c_void_p)
        opt = ItlinOpt(tol=1e-10, i_max=30, maxiter=600, termcheck=termcheck)
        info = ItlinInfo()
        y = np.zeros(n)
        bb = b.copy()
        lib.L.gmres.argtypes = [C.c_int, C.POINTER(C.c_double), C.c_void_p, C.c_void_p, C.c_void_p,
                                C.POINTER(C.c_double), C.POINTER(ItlinOpt), C.POINTER(ItlinInfo)]
        lib.L.gmres.restype = None
        lib.L.gmres(n, dptr(y), mv, pr, None, dptr(bb), C.byref(opt), C.byref(info))
        x = np.zeros(n)
        lib.L.PCG_preconlr(n, dptr(y), dptr(x))
        out.append((info.iter, info.rcode, info.precision, info.nomatvec, x))
        for T in (M, L, U):
            lib.free(T)
    (i1, rc1, e1, nm1, x1), (i2, rc2, e2, nm2, x2) = out
    say("gmres", callbacks, "termcheck", termcheck, "iters", i1, i2, "eta", e1, e2, "rel", rel(x1, x2))
    assert rc1 == rc2 == 0 and i1 == i2 and nm1 == nm2
    assert rel(x1, x2) < 1e-9
    assert np.linalg.norm(b - A @ x1) <= 1e-8 * np.linalg.norm(b)


def test_gmres_argument_checks_match_reference(libs):
    """gmres's option checks (utils.c:330-420): n <= 0 -> rcode 20, tol <= 0
    -> 21; i_max beyond n reset to min(10, n); tol clamped into
    [1e-15, 1e-1]."""
    A, b = _nonsymmetric(5)
    n = A.shape[0]
    out = []
    for lib in libs:
        M = lib.from_csr(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data)
        lib.L.PCG_default.argtypes = [C.c_void_p] * 3
        lib.L.PCG_default(M, None, None)
        mv = C.cast(lib.L.PCG_mult, C.c_void_p)
        res = []
        for nn, tol, imax in ((0, 1e-8, 5), (n, 0.0, 5), (n, 0.5, 10 * n), (n, 1e-30, 3)):
            opt = ItlinOpt(tol=tol, i_max=imax, maxiter=50, termcheck=0)
            info = ItlinInfo()
            y = np.zeros(max(n, 1))
            bb = b.copy()
            lib.L.gmres.argtypes = [C.c_int, C.POINTER(C.c_double), C.c_void_p, C.c_void_p, C.c_void_p,
                                    C.POINTER(C.c_double), C.POINTER(ItlinOpt), C.POINTER(ItlinInfo)]
            lib.L.gmres(nn, dptr(y), mv, None, None, dptr(bb), C.byref(opt), C.byref(info))
            res.append((info.rcode, opt.i_max if info.rcode == 0 else None, opt.tol if info.rcode == 0 else None))
        lib.free(M)
        out.append(res)
    say("gmres checks", out)
    assert out[0] == out[1]


def _amg_info_type():
    from tests.dropin_bind import SparseMatrix
    SMP = C.POINTER(C.POINTER(SparseMatrix))

    class AmgInfo(C.Structure):
        """the leading members of amg_system_info (Multigrid.h:45-60), common
        to both libraries"""
        _fields_ = [("Coarse_A", SMP), ("Prolongation", SMP), ("Restriction", SMP), ("L", SMP), ("U", SMP),
                    ("Signs", C.POINTER(SparseMatrix)), ("Coarsening", C.POINTER(C.POINTER(C.c_int))),
                    ("Fine_sizes", C.POINTER(C.c_int)), ("Coarse_sizes", C.POINTER(C.c_int)), ("depth", C.c_int)]
    return AmgInfo


@pytest.mark.parametrize("kind", ["poisson", "elasticity"])
def test_amg_setup_fills_the_level_fields(libs, kind):
    """AMG_setup's amg_system_info holds the hierarchy as the reference's
    does (Multigrid.c:1613-1754): every level's Coarse_A, Prolongation,
    Restriction and Coarsening labels, the finest row signs, the ILU(0)
    factors L/U of every level above the coarsest and the coarsest dense LU
    -- all identical to the reference's row lists, value for value; after
    AMG_recompute_coarse_matrices with new finest values the coarse matrices
    and factors are the reference's again."""
    s = P.poisson(33) if kind == "poisson" else P.degraded_elasticity(17)
    Info = _amg_info_type()
    out = []
    for lib in libs:
        M = lib.from_csr(s.rowptr, s.col, s.val)
        lib.L.AMG_print_info(0)
        I = C.cast(lib.L.AMG_setup(M, s.dof, 4, 2, 3, 1, 0, 1, None, None), C.POINTER(Info)).contents
        d = I.depth
        r = {"depth": d, "fine": [I.Fine_sizes[l] for l in range(d)], "coarse": [I.Coarse_sizes[l] for l in range(d)]}
        for l in range(d):
            r[f"A{l}"] = LinA.to_lists(I.Coarse_A[l])
            r[f"L{l}"] = LinA.to_lists(I.L[l])
            r[f"U{l}"] = LinA.to_lists(I.U[l])
            if l > 0:
                r[f"P{l}"] = LinA.to_lists(I.Prolongation[l])
                r[f"R{l}"] = LinA.to_lists(I.Restriction[l])
                r[f"C{l}"] = [I.Coarsening[l][i] for i in range(I.Fine_sizes[l])]
        r["signs"] = LinA.to_lists(I.Signs)
        M2 = lib.from_csr(s.rowptr, s.col, s.val * (1.0 + 0.25 * np.cos(np.arange(len(s.val)))))
        lib.L.AMG_recompute_coarse_matrices.argtypes = [C.c_void_p, C.c_void_p]
        lib.L.AMG_recompute_coarse_matrices(C.addressof(I), M2)
        for l in range(d - 1):
            r[f"A{l}_new"] = LinA.to_lists(I.Coarse_A[l])
            r[f"L{l}_new"] = LinA.to_lists(I.L[l])
            r[f"U{l}_new"] = LinA.to_lists(I.U[l])
        lib.L.AMG_free_data(C.addressof(I))
        lib.free(M)
        lib.free(M2)
        out.append(r)
    say(kind, "levels", out[0]["fine"], out[1]["fine"])
    for key in out[1]:
        assert out[0][key] == out[1][key], key


@pytest.mark.parametrize("local", [False, True])
def test_reflective_newton_with_callbacks_matches_reference(libs, local):
    """The functional, gradient and Hessian given as callbacks (set_RN_functional,
    RN_set_gradient, RN_set_Hesse_function: Crack's damage step,
    crack.c:9218-9220) for a quadratic with a constant term and two unit
    rows (gradient x_i there, as Crack's Dirichlet rows); the drop-in
    recognises the quadratic and runs the device method, the reference calls
    the callbacks -- same iterations, iterates to 1e-9.  local=True: the
    local solver slot (RN_set_local_solver, the RN_UMF path) with a host
    dense solver, called on host copies by the drop-in."""
    s, dold, ones = P.damage_system(33, h_scale=100.0)
    n = s.n
    unit = np.array([5, 600])
    A = s.scipy().tolil()
    for u in unit:
        A.rows[u] = [int(u)]
        A.data[u] = [1.0]
    A = A.tocsr()
    A.sort_indices()
    b = s.b.copy()
    b[unit] = 0.0
    c0 = 3.7
    rp, ci, va = A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.copy()
    lo, up = dold.copy(), ones.copy()
    lo[unit], up[unit] = 0.0, 1.0
    idx = np.arange(n, dtype=np.int32)
    libc = C.CDLL(None)
    libc.malloc.restype = C.c_void_p
    libc.malloc.argtypes = [C.c_size_t]
    from tests.dropin_bind import SparseMatrix
    SM = C.POINTER(SparseMatrix)
    FUNC = C.CFUNCTYPE(C.c_double, C.POINTER(C.c_double), C.c_int)
    GRAD = C.CFUNCTYPE(C.c_void_p, C.POINTER(C.c_double))
    HESS = C.CFUNCTYPE(C.c_void_p, C.POINTER(C.c_double))
    SOLV = C.CFUNCTYPE(C.c_int, SM, C.POINTER(C.c_double), C.POINTER(C.c_double))
    calls = {}

    def run(lib, tag):
        L = lib.L

        def f(x, m):
            xv = np.ctypeslib.as_array(x, shape=(n,))
            return float(0.5 * xv @ (A @ xv) + b @ xv + c0)

        def g(x):
            xv = np.ctypeslib.as_array(x, shape=(n,))
            gv = A @ xv + b
            p = libc.malloc(8 * n)
            C.memmove(p, gv.ctypes.data, 8 * n)
            return p

        def h(x):
            calls[tag] = calls.get(tag, 0) + 1
            return C.cast(lib.from_csr(rp, ci, va), C.c_void_p).value

        def solve(M, x, rhs):
            m = M.contents
            D = np.zeros((m.size, m.size))
            for i in range(m.size):
                for j in range(m.Len[i]):
                    D[i, m.Indices[i][j]] += m.Values[i][j]
            xv = np.linalg.solve(D, np.ctypeslib.as_array(rhs, shape=(m.size,)))
            np.ctypeslib.as_array(x, shape=(m.size,))[:] = xv
            return 1
        cbs = (FUNC(f), GRAD(g), HESS(h), SOLV(solve))
        L.RN_print_info(0)
        L.set_RN_functional.argtypes = [C.c_void_p]
        L.RN_set_gradient.argtypes = [C.c_void_p]
        L.RN_set_Hesse_function.argtypes = [C.c_void_p, C.c_int]
        L.set_RN_functional(C.cast(cbs[0], C.c_void_p))
        L.RN_set_gradient(C.cast(cbs[1], C.c_void_p))
        L.RN_set_Hesse_function(C.cast(cbs[2], C.c_void_p), n)
        L.set_RN_constraints.argtypes = [C.POINTER(C.c_int), C.POINTER(C.c_double), C.POINTER(C.c_double), C.c_int]
        L.set_RN_constraints(idx.ctypes.data_as(C.POINTER(C.c_int)), dptr(lo), dptr(up), n)
        L.RN_set_params.argtypes = [C.c_int] + [C.c_double] * 10
        L.RN_set_params(50, 1e-8, 0.1, 0.9, 0.1, float(np.sqrt(n) / 2), 1.0, 0.6, 1.1, 1e-3, 1000.0)
        L.RN_set_local_solver.argtypes = [C.c_void_p]
        if local:
            L.RN_set_local_solver(C.cast(cbs[3], C.c_void_p))
        else:
            L.RN_set_local_solver(None)
            L.RN_set_solver(3)
        x = np.clip(dold.copy(), lo, up)
        L.reflective_newton.argtypes = [C.POINTER(C.c_double)]
        it = L.reflective_newton(dptr(x))
        # leave the globals as the other tests expect them
        L.set_RN_functional(None)
        L.RN_set_gradient(None)
        L.RN_set_Hesse_function(None, n)
        L.RN_set_local_solver(None)
        return it, x

    (i1, x1), (i2, x2) = run(libs[0], "ours"), run(libs[1], "ref")
    say("RN with callbacks", "local" if local else "pcg", "iters", i1, i2, "rel", rel(x1, x2), "hessian calls", calls)
    assert i1 > 0 and i1 == i2 and rel(x1, x2) < 1e-9
    assert np.all(x1 >= lo - 1e-12) and np.all(x1 <= up + 1e-12)
