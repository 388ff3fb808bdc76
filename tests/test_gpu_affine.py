"""Parallelepiped meshes, whose element loops and Krylov products run in the
element's Legendre modes (pm_affine.hip), against the oracle's Gauss loops; the
loops of distorted meshes, which keep the Gauss points, on the same decks.

Bars: the element loops' own (matrix within 1e-13 of the row's largest entry,
right-hand sides within 1e-13 of max|b|); solutions within 1e-9 of those from
the stored matrix, the bar of the marches."""
import dataclasses

import numpy as np
import pytest

from oracle import oracle as O
from poromec_amd import problem as P
from test_gpu_elmt07 import _rowwise

pytestmark = pytest.mark.gpu

SHEAR = np.array([[1.0, 0.2, -0.1], [0.15, 0.8, 0.25], [-0.2, 0.1, 1.2]])


def _deck(shape, nen, shear=True, seed=3):
    """Box under gravity, traction and flux, its vertices mapped by SHEAR."""
    d = P.heterogeneous_box_deck(max(shape), seed=seed, shape=shape, sigma_lnk=0.8, corr_len=2.0,
                                 dt=0.05, nen=nen, patch_fraction=0.7)
    if shear:
        d = dataclasses.replace(d, x=d.x @ SHEAR.T)
    d.gravity = np.array([0.5, -0.3, -10.0])
    d.e[:, 5] = 2000.0
    d.load[1] = (43, 2, 2)
    d.fload[1, 0, :2] = (0.0, 1e30)
    d.fload[1, 1, :2] = (1e-3, 1e-3)
    d.eloadp[np.arange(d.numel) % shape[0] == 0, 5] = 2
    if nen == 8:
        d.e[:, 8] = 0.25
    return d


# one element; 63, 64 and 65 of them (a workgroup takes 64); several workgroups
@pytest.mark.parametrize("nen", [20, 8])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 7, 3), (4, 4, 4), (5, 13, 1), (9, 5, 6)])
def test_element_loops(shape, nen):
    _check_loops(_deck(shape, nen))


# the Gauss loops in colours, which meshes of other elements keep: every
# interior vertex moved, and one vertex of a box alone
@pytest.mark.parametrize("nen", [20, 8])
@pytest.mark.parametrize("shape,one", [((3, 4, 3), False), ((6, 5, 4), False), ((4, 4, 4), True)])
def test_element_loops_distorted(shape, one, nen):
    d = _deck(shape, nen, shear=False)
    x = d.x.copy()
    inner = np.nonzero(np.all((x > 0) & (x < np.array(shape)), axis=1))[0]
    inner = inner[:1] if one else inner
    x[inner] += 0.08 * np.random.default_rng(2).standard_normal((len(inner), 3))
    _check_loops(dataclasses.replace(d, x=x))


def _check_loops(d):
    from poromec_amd.solver import MefSolver
    st = O.build_structure(d)
    m = O.OracleModel(d, st)
    s = MefSolver(d)
    rng = np.random.default_rng(11)
    u = rng.standard_normal((st["nnode"], 4)) * 1e-3
    dp = rng.standard_normal(st["nnode"]) * 1e-4
    u[d.nnodev:, 3] = 0.0
    dp[d.nnodev:] = 0.0
    m.u[:], m.dp[:] = u, dp
    s.set_state(u=u, u0=np.zeros_like(u), dp=dp, t=0.0)
    f = rng.standard_normal(st["neq"]) * 1e-3
    for isw, lhs in ((2, True), (2, False), (4, False)):
        m.b[:] = f
        m.env.t = 0.5
        m.assemble(isw=isw, lhs=lhs, rhs=True)
        s.set_vectors(b=f)
        s.pform(isw, lhs, True, d.dt, 0.5, target="b")
        b = s.vectors()[1]
        assert np.abs(b - m.b).max() <= 1e-13 * np.abs(m.b).max(), (isw, lhs)
    _, _, ad, al = s.export_csrc()
    assert _rowwise(st["ia"], ad, al, m.ad, m.al[: st["nad"]]) < 1e-13
    s.close()


# one lane an element (from 50,000 on), the last patch one element short of
# full: against the Gauss loops of the same mesh with a vertex moved by 1e-9
# (no parallelepipeds any more; the entries move by ~1e-9 of the largest)
@pytest.mark.parametrize("nen,shape", [(20, (37, 39, 35)), (8, (39, 37, 35))])
def test_element_loops_one_lane(nen, shape):
    from poromec_amd.solver import MefSolver
    d = _deck(shape, nen)
    assert d.numel > 50000
    moved = dataclasses.replace(d, x=d.x.copy())
    moved.x[d.nnodev // 2, 2] += 1e-9
    out = []
    rng = np.random.default_rng(12)
    for deck in (d, moved):
        s = MefSolver(deck)
        if not out:
            u = rng.standard_normal((s.nnode, 4)) * 1e-3
            u[d.nnodev:, 3] = 0.0
            dp = rng.standard_normal(s.nnode) * 1e-4
            f = rng.standard_normal(s.neq)
        s.set_state(u=u, u0=np.zeros_like(u), dp=dp, t=0.0)
        s.set_vectors(b0=np.zeros(s.neq), b=np.zeros(s.neq))
        s.pform(4, False, True, d.dt, 0.5, target="b0")
        s.pform(2, True, True, d.dt, 0.5, target="b")
        b0, b, _ = s.vectors()
        out.append((b0, b, s.spmv(f)))
        s.close()
    for a, b in zip(*out):
        scale = np.abs(b).max()
        assert np.abs(a - b).max() <= 1e-7 * scale
        assert np.median(np.abs(a - b)) <= 1e-14 * scale  # rows away from the vertex


def _stored(s):
    """The same matrix in a context that has no elements."""
    from poromec_amd.solver import CsrcSolver
    ia, ja, ad, al = s.export_csrc()
    cs = CsrcSolver(ia, ja)
    cs.set_values(ad, al)
    return cs


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


# meshes just past the size from which products run through the elements, and
# the same with one vertex moved (no longer parallelepipeds: stored matrix)
@pytest.mark.parametrize("nen,shape", [(20, (13, 13, 13)), (8, (23, 24, 22))])
@pytest.mark.parametrize("moved", [False, True])
def test_products_sqmr(nen, shape, moved):
    from poromec_amd.solver import MefSolver, SolverConfig
    d = _deck(shape, nen, shear=False)
    d.e[:, 8] = 0.0
    if moved:
        d.x[np.argmin(np.abs(d.x - 0.5 * np.array(shape)).sum(1)), 2] += 0.05
    s = MefSolver(d)
    s.pform(2, True, False, d.dt, d.dt)
    assert s.matrix_info()["nnz"] > 4_500_000
    for use32 in (False, True):
        assert s.products_through_elements(use32) == (not moved)
    b = np.random.default_rng(5).standard_normal(s.neq)
    cs = _stored(s)
    x0, _ = cs.solve(b, SolverConfig(tol=1e-11))
    x, info = s.solve(b, SolverConfig(tol=1e-11))
    # the residual is recomputed from the stored matrix
    assert info["true_rel"] < 1e-9 and _rel(x, x0) < 1e-9, info
    x, info = s.solve(b, SolverConfig(tol=1e-10, precision="fp32ir"))
    assert info["true_rel"] < 1e-10 and _rel(x, x0) < 1e-8, info
    s.close()
    cs.close()


def test_products_other_solvers():
    from poromec_amd.solver import MefSolver, SolverConfig
    d = _deck((14, 15, 15), 20)
    d.idv[:, 3] = 1  # K = K_uu, positive definite
    s = MefSolver(d)
    s.pform(2, True, False, d.dt, d.dt)
    assert s.products_through_elements(False)
    b = np.random.default_rng(6).standard_normal(s.neq)
    cs = _stored(s)
    x0, _ = cs.solve(b, SolverConfig(solver="pcg", tol=1e-12))
    for solver, precond in (("pcg", 2), ("bicgstab", 2), ("minres", 5)):
        x, _ = s.solve(b, SolverConfig(solver=solver, precond=precond, tol=1e-12))
        assert _rel(x, x0) < 1e-9, solver
    # GMRES stops on the scaled residual; its rows' scales differ by < 100
    x, info = s.solve(b, SolverConfig(solver="gmres", tol=1e-7, maxit=20))
    assert info["true_rel"] < 1e-5
    s.close()
    cs.close()


# the fused iterations (two passes) against the oracle's loops: one row block
# per workgroup wavefront and more, breakdown, the iteration limit
@pytest.mark.parametrize("nen,shape", [(20, (1, 1, 1)), (20, (4, 5, 3)), (8, (1, 1, 2)),
                                       (8, (9, 8, 7))])
@pytest.mark.parametrize("solver", ["sqmr", "pcg"])
def test_fused_iterations(nen, shape, solver):
    from poromec_amd._lib import PmError
    from poromec_amd.solver import MefSolver, SolverConfig
    d = _deck(shape, nen, shear=False)
    d.e[:, 8] = 0.0
    st = O.build_structure(d)
    m = O.OracleModel(d, st)
    m.assemble(isw=2, lhs=True, rhs=False)
    s = MefSolver(d)
    s.pform(2, True, False, d.dt, d.dt)
    b = np.random.default_rng(8).standard_normal(s.neq)
    it, x_o, _ = O.solv(st, m.ad, m.al[: st["nad"]], b, solver={"sqmr": 11, "pcg": 1}[solver],
                        tol=1e-12, maxit=50000)
    x, info = s.solve(b, SolverConfig(solver=solver, tol=1e-12))
    assert _rel(x, x_o) < 1e-9, info
    if solver == "sqmr" and nen == 20:  # the counts of equal-order systems scatter more
        assert abs(info["iters"] - it) <= 2 + 0.1 * it, (info, it)
    _, info = s.solve(b, SolverConfig(solver=solver, tol=1e-10, precision="fp32ir"))
    assert info["true_rel"] < 1e-10, info
    # stopped one iteration short: PCG reports it, SQMR hands over to GMRES
    n = info64 = s.solve(b, SolverConfig(solver=solver, tol=1e-11))[1]["iters"]
    if solver == "pcg" and n > 1:
        with pytest.raises(PmError):
            s.solve(b, SolverConfig(solver=solver, tol=1e-11, maxit=n - 1))
    assert s.solve(b, SolverConfig(solver=solver, tol=1e-11, maxit=n))[1]["iters"] == info64
    if solver == "sqmr":  # A 0 . 0 = 0: the reference's breakdown stop
        with pytest.raises(PmError):
            s.solve(np.zeros(s.neq), SolverConfig(tol=1e-11))
    s.close()


# the batched solve through the elements: boxes of different sizes, the middle
# one with a zero right-hand side, against each box alone (RCM numbers every
# box as it does alone, one range after the other)
@pytest.mark.parametrize("nen,ns", [(20, (9, 3, 12)), (8, (18, 5, 20))])
@pytest.mark.parametrize("solver,prec", [("sqmr", "fp64"), ("sqmr", "fp32ir"), ("pcg", "fp64")])
def test_batch_through_elements(nen, ns, solver, prec):
    from poromec_amd.solver import MefSolver, SolverConfig
    decks = [P.heterogeneous_box_deck(n, seed=n, corr_len=n / 2, dt=0.1, nen=nen) for n in ns]
    big, off = P.concat_decks(decks)
    s = MefSolver(big)
    s.batch_define(off)
    s.pform(2, True, False, big.dt, big.dt)
    assert s.products_through_elements(prec == "fp32ir")
    rng = np.random.default_rng(9)
    singles = [MefSolver(d) for d in decks]
    bs = [rng.standard_normal(o.neq) if k != 1 else np.zeros(o.neq) for k, o in enumerate(singles)]
    # fp32ir cannot meet much less than 1e-10 of a random load
    tol = 1e-12 if prec == "fp64" else 1e-10
    cfg = SolverConfig(solver=solver, tol=tol, precision=prec)
    for _ in range(2):  # the second solve reuses the first one's buffers
        x, info = s.solve(np.concatenate(bs), cfg)
    at = 0
    for k, o in enumerate(singles):
        part = x[at: at + o.neq]
        at += o.neq
        if k == 1:
            assert not part.any()
        else:
            o.pform(2, True, False, big.dt, big.dt)
            ref, _ = o.solve(bs[k], SolverConfig(tol=1e-12))
            assert _rel(part, ref) < (1e-9 if prec == "fp64" else 1e-7), k
        o.close()
    if prec == "fp64":
        assert s.batch_iters()[1] == 0
    else:
        assert info["true_rel"] < 1e-10
    s.close()


# one lane an element (from 50,000 on): the solvers' products against the
# residual recomputed from the stored matrix; K = K_uu, positive definite.
# MINRES and GMRES stop on a scaled residual; the rows' scales differ by < 100
@pytest.mark.parametrize("nen", [20, 8])
def test_products_one_lane(nen):
    from poromec_amd.solver import MefSolver, SolverConfig
    d = _deck((37, 38, 36), nen)
    assert d.numel >= 50000
    d.idv[:, 3] = 1
    s = MefSolver(d)
    s.pform(2, True, False, d.dt, d.dt)
    assert s.products_through_elements(False) and s.products_through_elements(True)
    b = np.random.default_rng(6).standard_normal(s.neq)
    for solver, precond, prec, tol, bar in (("pcg", 2, "fp64", 1e-11, 1e-9),
                                            ("pcg", 2, "fp32ir", 1e-10, 1e-10),
                                            ("bicgstab", 2, "fp64", 1e-11, 1e-9),
                                            ("minres", 5, "fp64", 1e-10, 1e-8),
                                            ("gmres", 2, "fp64", 1e-6, 1e-4)):
        x, info = s.solve(b, SolverConfig(solver=solver, precond=precond, tol=tol, precision=prec))
        assert info["true_rel"] < bar, (solver, prec, info)
    s.close()


# the batched passes with one lane an element, the two boxes' element counts
# (27,000 and 24,389) each below that line: against each box alone
@pytest.mark.parametrize("nen", [20, 8])
@pytest.mark.parametrize("solver", ["sqmr", "pcg"])
def test_batch_one_lane(nen, solver):
    from poromec_amd.solver import MefSolver, SolverConfig
    decks = [P.heterogeneous_box_deck(n, seed=n, corr_len=8.0, dt=0.1, nen=nen) for n in (30, 29)]
    big, off = P.concat_decks(decks)
    assert big.numel >= 50000
    s = MefSolver(big)
    s.batch_define(off)
    s.pform(2, True, False, big.dt, big.dt)
    assert s.products_through_elements(False)
    rng = np.random.default_rng(9)
    singles = [MefSolver(d) for d in decks]
    bs = [rng.standard_normal(o.neq) for o in singles]
    x, _ = s.solve(np.concatenate(bs), SolverConfig(solver=solver, tol=1e-12))
    s.close()
    at = 0
    for k, o in enumerate(singles):
        o.pform(2, True, False, big.dt, big.dt)
        ref, _ = o.solve(bs[k], SolverConfig(tol=1e-12))
        assert _rel(x[at: at + o.neq], ref) < 1e-9, k
        at += o.neq
        o.close()


# two boxes that meet in a plane of restrained nodes: no equation couples them,
# but their elements are neighbours, and a patch must not take from both (nine
# elements a layer, sixteen a patch: the one at the plane would).  Supports
# every twelve layers keep the system's condition that of a short column.
def test_batch_boxes_sharing_restrained_nodes():
    from poromec_amd.solver import MefSolver, SolverConfig
    shape, cut = (3, 3, 1700), 501
    d = P.heterogeneous_box_deck(3, seed=6, shape=shape, corr_len=4.0, dt=0.1, nen=8)
    d.idv[d.x[:, 2] % 12 == 0, :3] = 1
    d.idv[d.x[:, 2] == cut] = 1
    s = MefSolver(d, reorder=False)  # as read: one box's equations after the other's
    s.pform(2, True, False, d.dt, d.dt)
    assert s.products_through_elements(False) and s.products_through_elements(True)
    b = np.random.default_rng(10).standard_normal(s.neq)
    cs = _stored(s)
    x0, _ = cs.solve(b, SolverConfig(tol=1e-12))
    s.batch_define([0, 9 * cut, d.numel])
    x, info = s.solve(b, SolverConfig(tol=1e-12))
    assert _rel(x, x0) < 1e-9, info
    x, info = s.solve(b, SolverConfig(tol=1e-10, precision="fp32ir"))
    assert info["true_rel"] < 1e-10, info
    s.close()
    cs.close()


# FP32+IR through the elements reads no FP32 values: none are made, and the
# solve without allocations takes the same matrix
def test_fp32ir_through_elements_makes_no_fp32_values():
    import ctypes as C
    from poromec_amd import _lib as L
    from poromec_amd.solver import MefSolver, SolverConfig
    d = _deck((14, 14, 14), 20, shear=False)
    s = MefSolver(d)
    s.pform(2, True, False, d.dt, d.dt)
    assert s.products_through_elements(True)
    b = np.random.default_rng(5).standard_normal(s.neq)
    s.solve(b, SolverConfig(tol=1e-6))  # the work vectors
    cfg = SolverConfig(tol=1e-8, precision="fp32ir")

    def free():
        f, total = C.c_size_t(), C.c_size_t()
        assert s.lib.hipMemGetInfo(C.byref(f), C.byref(total)) == 0
        return f.value

    def noalloc():
        x = np.zeros(s.neq)
        rc = s.lib.pm_solve_noalloc(s.ctx, C.byref(cfg.c()), L.ptr(b), L.ptr(x), None)
        return rc, x

    assert noalloc()[0] == -8  # no FP32+IR solve of this matrix yet
    before = free()
    x, info = s.solve(b, cfg)
    assert info["true_rel"] < 1e-8
    assert before - free() < 2 * s.matrix_info()["nnz"]
    rc, y = noalloc()
    assert rc == 0 and np.array_equal(x, y)
    s.set_ordered(True)  # takes the stored values: made now, for the call that cannot
    assert before - free() > 3 * s.matrix_info()["nnz"]
    s.set_ordered(False)
    s.pform(2, True, False, d.dt, d.dt)
    assert noalloc()[0] == -8
    s.close()
