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


# the fused iterations' stored product by runs of columns, on blocks of <= 32
# runs (Q1/Q1) and of up to 77, given as a matrix alone.  The system: the
# mesh's, scaled symmetrically to entries of one size, with a constant diagonal
# of twice the largest row sum, so its condition number is at most 3 and a
# residual of sqrt(k + 1) tol (SQMR's bound, k < 100) an error of 30 tol.
@pytest.mark.parametrize("solver", ["sqmr", "pcg"])
@pytest.mark.parametrize("prec", ["fp64", "fp32ir"])
@pytest.mark.parametrize("nen,n", [(8, 18), (20, 10)])
def test_fused_iterations_by_runs(nen, n, prec, solver):
    from poromec_amd.solver import CsrcSolver, SolverConfig
    s, (ia, ja, ad, al, rows), L = _system(nen, n)
    assert s.matrix_info()["nnz"] >= 2_000_000
    one = np.ones(s.neq)
    sc = 1.0 / np.sqrt(abs(L) @ one + abs(L).T @ one + np.abs(ad))
    al = al * sc[rows] * sc[ja - 1]
    L.data[:] = al
    big = 2.0 * (abs(L) @ one + abs(L).T @ one).max()
    b = np.random.default_rng(2).standard_normal(s.neq)
    ref = np.zeros(s.neq)
    for _ in range(60):  # Jacobi: halves the error at least
        ref = (b - L @ ref - L.T @ ref) / big
    cs = CsrcSolver(ia, ja)
    cs.set_values(np.full(s.neq, big), al)
    tol = 1e-12 if prec == "fp64" else 1e-10
    x, info = cs.solve(b, SolverConfig(solver=solver, tol=tol, precision=prec))
    assert info["iters"] < 100
    assert np.linalg.norm(x - ref) <= 30 * tol * np.linalg.norm(ref)
    cs.close()
    s.close()
