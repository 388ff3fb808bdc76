"""The product's shape where none was tuned or set: one run of columns per
lane from a million stored values on.

Bar: a row of <= 300 terms summed in any order is within 300 * 1.1e-16 of the
host's sum relative to sum |a||x|; 1e-13 of max|y| has been the entry's bar."""
import numpy as np
import pytest

from poromec_amd import problem as P

pytestmark = pytest.mark.gpu


def _system(nen, n):
    import scipy.sparse as sp
    from poromec_amd.solver import MefSolver
    d = P.heterogeneous_box_deck(n, seed=4, sigma_lnk=0.5, corr_len=2.0, nen=nen)
    s = MefSolver(d)
    s.pform(2, True, False, d.dt, d.dt)
    ia, ja, ad, al = s.export_csrc()
    rows = np.repeat(np.arange(s.neq), np.diff(ia))
    L = sp.csr_matrix((al, (rows, ja - 1)), shape=(s.neq, s.neq))
    return s, (ia, ja, ad, al, rows), L


# below the rule's line; 32 lanes a block; 64 lanes a block
@pytest.mark.parametrize("nen,n,least", [(20, 6, 0), (8, 14, 1_000_000), (20, 8, 1_000_000),
                                         (20, 30, 64_000_000)])
def test_default_shape(nen, n, least):
    s, (_, _, ad, _, _), L = _system(nen, n)
    assert s.matrix_info()["nnz"] >= least
    x = np.random.default_rng(8).standard_normal(s.neq)
    y0 = ad * x + L @ x + L.T @ x
    y = s.spmv(x)
    assert np.abs(y - y0).max() <= 1e-13 * np.abs(y0).max()
    s.close()


@pytest.mark.parametrize("nen,n", [(8, 14), (20, 8)])
def test_infinite_value_stays_in_its_rows(nen, n):
    from poromec_amd.solver import CsrcSolver
    s, (ia, ja, ad, al, rows), L = _system(nen, n)
    x = 1.0 + np.random.default_rng(5).random(s.neq)
    y0 = ad * x + L @ x + L.T @ x
    for k in (0, len(al) // 2, len(al) - 1):
        bad = al.copy()
        bad[k] = np.inf
        cs = CsrcSolver(ia, ja)
        cs.set_values(ad, bad)
        y = cs.spmv(x)
        hit = np.zeros(s.neq, bool)
        hit[[rows[k], ja[k] - 1]] = True
        assert not np.isfinite(y[hit]).any()
        assert np.abs(y[~hit] - y0[~hit]).max() <= 1e-13 * np.abs(y0).max()
        cs.close()
    s.close()


def _dominant(ia, ja, ad, al):
    """A system of a mesh's pattern, given as a matrix alone: the mesh's values
    scaled symmetrically to entries of one size, with a constant diagonal of
    twice the largest row sum.  Its condition number is at most 3, so a residual
    of sqrt(k + 1) tol (SQMR's bound, k < 100) is an error of 30 tol."""
    import scipy.sparse as sp
    from poromec_amd.solver import CsrcSolver
    n = len(ad)
    rows = np.repeat(np.arange(n), np.diff(ia))
    L = sp.csr_matrix((al, (rows, ja - 1)), shape=(n, n))
    one = np.ones(n)
    sc = 1.0 / np.sqrt(abs(L) @ one + abs(L).T @ one + np.abs(ad))
    L.data[:] = al * sc[rows] * sc[ja - 1]
    big = 2.0 * (abs(L) @ one + abs(L).T @ one).max()
    b = np.random.default_rng(2).standard_normal(n)
    ref = np.zeros(n)
    for _ in range(60):  # Jacobi: halves the error at least
        ref = (b - L @ ref - L.T @ ref) / big
    cs = CsrcSolver(ia, ja)
    cs.set_values(np.full(n, big), L.data)
    return cs, b, ref


def check_fp32_shapes(s):
    """Every shape of the FP32 product, on the pattern of the mesh in s, by
    solvers that take their products in the set shape (SQMR and PCG have one of
    their own at these sizes): BiCGSTAB with one and two dots, GMRES with the
    rows scaled.  FP32+IR by the FP32 matrix gains five digits an outer step: an
    operator that is not that matrix, or not the same one every time, takes more
    of them, and one that fails its inner solve has FP64 products beside the
    residuals'."""
    from poromec_amd import _lib as L
    from poromec_amd.solver import SPMV_SHAPES, SolverConfig
    cs, b, ref = _dominant(*s.export_csrc())
    for solver in ("bicgstab", "gmres"):
        bits = set()
        for shape in range(SPMV_SHAPES):
            L.check(cs.lib.pm_set_spmv_shape(cs.ctx, 1, shape), "pm_set_spmv_shape")
            x, info = cs.solve(b, SolverConfig(solver=solver, tol=1e-10, precision="fp32ir"))
            assert info["outer"] <= 3 and info["spmv64"] == info["outer"], (solver, shape, info)
            assert np.linalg.norm(x - ref) <= 3e-10 * np.linalg.norm(ref), (solver, shape)
            bits.add(x.tobytes())
        assert len(bits) > 1, solver  # the set shape is the one that runs
    cs.close()


# the fused iterations' stored product by runs of columns, on blocks of <= 32
# runs (Q1/Q1) and of up to 77
@pytest.mark.parametrize("solver", ["sqmr", "pcg"])
@pytest.mark.parametrize("prec", ["fp64", "fp32ir"])
@pytest.mark.parametrize("nen,n", [(8, 18), (20, 10)])
def test_fused_iterations_by_runs(nen, n, prec, solver):
    from poromec_amd.solver import SolverConfig
    s, (ia, ja, ad, al, _), _ = _system(nen, n)
    assert s.matrix_info()["nnz"] >= 2_000_000
    cs, b, ref = _dominant(ia, ja, ad, al)
    tol = 1e-12 if prec == "fp64" else 1e-10
    x, info = cs.solve(b, SolverConfig(solver=solver, tol=tol, precision=prec))
    assert info["iters"] < 100
    assert np.linalg.norm(x - ref) <= 30 * tol * np.linalg.norm(ref)
    cs.close()
    s.close()


# the three-kernel loops, which a matrix of short runs takes above 12 million
# values (FP32: 24): 31 separate columns a side of the diagonal, 25 million
# values.  Entries of one sign and size against a diagonal of four times the
# largest row sum: condition number at most 5/3, Jacobi gains a factor four a
# sweep, and SQMR's residual of sqrt(k + 1) tol (k < 100) means an error of
# 5/3 10 tol < 30 tol.
@pytest.mark.parametrize("prec", ["fp64", "fp32ir"])
def test_three_kernel_loops(prec):
    import scipy.sparse as sp
    from poromec_amd import _lib as L
    from poromec_amd.solver import CsrcSolver, SolverConfig
    n = 400_000
    offs = np.cumsum(np.arange(2, 33))  # no two columns of a row adjacent
    rng = np.random.default_rng(7)
    Lm = sp.diags([rng.uniform(-1.0, -0.5, n - k) for k in offs], [-k for k in offs], shape=(n, n),
                  format="csr")
    Lm.sort_indices()
    one = np.ones(n)
    diag = np.full(n, 4.0 * (abs(Lm) @ one + abs(Lm).T @ one).max())
    cs = CsrcSolver(Lm.indptr.astype(np.int64) + 1, Lm.indices + 1)
    cs.set_values(diag, Lm.data)
    assert 2 * Lm.nnz + n > 24_000_000
    b = rng.standard_normal(n)
    ref = np.zeros(n)
    for _ in range(25):
        ref = (b - Lm @ ref - Lm.T @ ref) / diag
    tol = 1e-12 if prec == "fp64" else 1e-10
    for solver in ("sqmr", "pcg"):
        xs = []
        for shape in (2, 5):  # 64 lanes a row, 32
            L.check(cs.lib.pm_set_spmv_shape(cs.ctx, int(prec == "fp32ir"), shape), "shape")
            x, info = cs.solve(b, SolverConfig(solver=solver, tol=tol, precision=prec))
            assert info["iters"] < 100
            assert np.linalg.norm(x - ref) <= 30 * tol * np.linalg.norm(ref), (solver, shape)
            xs.append(x)
        assert not np.array_equal(*xs)  # the fused iterations would not see the shape
    cs.close()
