"""The workloads this framework's speed is measured on, each through the
public entry points of ``poromec_amd.solver``.

A case is a dict of plain values.  Its ``kind`` names the call:

``step``      one backward-Euler step of the ``solv`` macro from a given state
              (``set_state``, ``step``, ``state``), the unit of every march
``batch``     the same step for many independent boxes in one context
``vprop``     the same step with properties at the integration points
``assemble``  the element loops and the product: ``pform`` isw 4 and isw 2 into
              given load vectors, then ``spmv``
``stress``    stresses and Darcy flux of a state (``tform``)
``adjoint``   a short march with its gradients (``adjoint``)
``dropin``    ``solv_pm`` for a caller that assembles its own CSRC matrix
              (``CsrcSolver``: values in, solution out)

``nen`` is 20 for the hexa20/8 element and 8 for the equal-order Q1/Q1 element;
``nx, ny, nz`` are cells.  Meshes, materials, loads and tolerances are those of
the benchmark configurations (``poromec_amd.problem``); the 87^3 and 128^3 boxes
of the headline take a minute a step, so the largest box here is 64^3.
"""
import math

import numpy as np
import torch

from poromec_amd import problem as P
from poromec_amd.solver import CsrcSolver, MefSolver, SolverConfig

TOL = 1.0e-10  # the benchmark configurations' Krylov tolerance


def listed():
    def case(name, kind, nen, shape, **kw):
        return dict(name=name, kind=kind, nen=nen, nx=shape[0], ny=shape[1], nz=shape[2],
                    **kw)

    return [
        # the consolidation column of the first configuration: the smallest
        # march, every launch and synchronisation counts
        case("column_hexa20_fp64", "step", 20, (4, 4, 40), deck="column", precision="fp64"),
        # a deck of the size of the reference's shipped examples, odd in every
        # direction, heterogeneous
        case("box_hexa20_16_fp64", "step", 20, (17, 15, 16), deck="box", precision="fp64"),
        # the upper end of the batch's boxes, mixed precision
        case("box_hexa20_24_fp32ir", "step", 20, (24, 24, 24), deck="box", precision="fp32ir"),
        # the Q1/Q1 element at an ordinary size
        case("box_q1_32_fp64", "step", 8, (32, 31, 33), deck="box", precision="fp64"),
        # the second configuration's box at its nominal 1.1 million dofs
        case("box_q1_64_fp32ir", "step", 8, (64, 64, 64), deck="box", precision="fp32ir"),
        # independent boxes of different sizes in one batched step
        case("batch_hexa20_8_boxes", "batch", 20, (0, 0, 0), nbox=8, nmin=8, nmax=12,
             precision="fp64"),
        # Kozeny-Carman, density and Hashin-Shtrikman at the integration points
        case("vprop_hexa20_10", "vprop", 20, (10, 9, 8), deck="box", precision="fp64"),
        # the element loops alone: re-assembly after new materials or a new dt
        case("assemble_hexa20_40", "assemble", 20, (40, 40, 40), deck="box"),
        case("assemble_q1_64", "assemble", 8, (63, 64, 65), deck="box"),
        # the printed fields of one output step
        case("stress_hexa20_40", "stress", 20, (40, 39, 41), deck="box"),
        # inversion: misfit and gradient of a short march
        case("adjoint_q1_8", "adjoint", 8, (8, 8, 8), deck="box", nsteps=5, nsens=64),
        # a Fortran host that keeps its own assembly and hands over the matrix
        case("dropin_csrc_pcg", "dropin", 8, (12, 13, 11), deck="box", solver="pcg"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "vprop", "assemble", "assemble",
                       "stress", "adjoint", "dropin"])
    if kind == "batch":
        nmin = rng.randint(4, 10)
        return dict(kind=kind, nen=rng.choice([8, 20]), nx=0, ny=0, nz=0,
                    nbox=rng.randint(2, 12), nmin=nmin, nmax=nmin + rng.randint(0, 4),
                    precision=rng.choice(["fp64", "fp32ir"]))
    if kind == "step":
        nen = rng.choice([8, 20])
        lo, hi = (5, 56) if nen == 8 else (4, 22)
    elif kind == "vprop":
        nen, lo, hi = 20, 4, 12
    elif kind == "assemble":
        nen = rng.choice([8, 20])
        lo, hi = (8, 66) if nen == 8 else (5, 42)
    elif kind == "stress":
        nen = rng.choice([8, 20])
        lo, hi = (8, 64) if nen == 8 else (5, 42)
    elif kind == "adjoint":
        nen, lo, hi = 8, 4, 9
    else:
        nen, lo, hi = 8, 5, 13
    n = _log_int(rng, lo, hi)
    shape = [max(lo, min(hi, n + rng.randint(-2, 2))) for _ in range(3)]
    c = dict(kind=kind, nen=nen, nx=shape[0], ny=shape[1], nz=shape[2], deck="box")
    if kind == "step":
        c["precision"] = rng.choice(["fp64", "fp32ir"])
    elif kind == "vprop":
        c["precision"] = "fp64"
    elif kind == "adjoint":
        c.update(nsteps=rng.randint(2, 5), nsens=rng.randint(4, 64))
    elif kind == "dropin":
        c["solver"] = rng.choice(["sqmr", "pcg"])
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _deck(case, seed):
    shape = (case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng([seed, 17])
    if case["deck"] == "column":
        d = P.column_deck(*shape, E=10.0 * rng.uniform(0.8, 1.25), nu=0.3,
                          load_mpa=1.0e-3 * rng.uniform(0.5, 2.0), dt=0.01, nen=case["nen"])
    else:
        d = P.heterogeneous_box_deck(max(shape), seed=seed, shape=shape, dt=0.1, nen=case["nen"],
                                     corr_len=min(8.0, max(shape) / 2))
    d.e[:, 7] = 0.2  # porosity
    return d


def _batch_decks(case, seed):
    """``problem.batch_decks`` with the box sizes fixed by the case: every seed
    gives the same boxes other materials."""
    ns = np.random.default_rng([case["nbox"], case["nmin"], case["nmax"]]).integers(
        case["nmin"], case["nmax"] + 1, size=case["nbox"])
    rng = np.random.default_rng([seed, 41])
    return [P.heterogeneous_box_deck(int(n), seed=int(rng.integers(2**31)),
                                     sigma_lnk=rng.uniform(0.5, 1.5), dt=0.1,
                                     corr_len=min(8.0, n / 2), nen=case["nen"]) for n in ns]


def _field(d, nnode, rng):
    """A smooth nodal state (u, v, w [m], p [MPa]) and dp of the size a loaded
    box has, zero at the restrained vertices; mid-edge nodes follow later."""
    u = np.zeros((nnode, 4))
    x = d.x / max(d.nx, d.ny, d.nz)
    for j in range(4):
        for _ in range(3):
            k = rng.integers(1, 4, size=3)
            ph = rng.uniform(0, 2 * np.pi, size=3)
            u[: d.nnodev, j] += rng.uniform(0.2, 1.0) * np.prod(np.sin(x * k * np.pi + ph), axis=1)
    u[:, :3] *= 1.0e-4
    u[:, 3] *= 1.0e-3
    u[: d.nnodev][d.idv == 1] = 0.0
    return u


def _state_field(d, nen, seed):
    """Full nodal state of a promoted mesh: mid-edge displacements are their
    edge's average plus a small bubble."""
    rng = np.random.default_rng([seed, 29])
    ix, nnode = _promote(d.ix[:, :8].astype(np.int64) - 1, d.nnodev) if nen == 20 \
        else (d.ix[:, :8].astype(np.int64) - 1, d.nnodev)
    u = _field(d, nnode, rng)
    if nen == 20:
        fixed = np.zeros((nnode, 3), bool)
        for a, b, m in _EDGES:
            mid = ix[:, m]
            u[mid, :3] = 0.5 * (u[ix[:, a], :3] + u[ix[:, b], :3]) * 1.001
            fixed[mid] = (d.idv[ix[:, a], :3] == 1) & (d.idv[ix[:, b], :3] == 1)
        u[:, :3][fixed] = 0.0
    return u, 0.5 * u[:, 3]


def _zero_state(s):
    return dict(u=np.zeros((s.nnode, 4)), u0=np.zeros((s.nnode, 4)), dp=np.zeros(s.nnode),
                porosity=np.full(s.nnode, 0.2))


def _cfg(case, **kw):
    kw.setdefault("tol", TOL)
    return SolverConfig(precision=case.get("precision", "fp64"), **kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        big, off = P.concat_decks(_batch_decks(case, seed))
        big.e[:, 7] = 0.2
        s = MefSolver(big)
        s.batch_define(off)
        return dict(kind=kind, s=s, cfg=_cfg(case), z=_zero_state(s))
    d = _deck(case, seed)
    if kind == "dropin":
        ia, ja, ad, al, b = _csrc(d, seed)
        return dict(kind=kind, s=CsrcSolver(ia, ja), ad=ad, al=al, b=b,
                    cfg=_cfg(case, solver=case["solver"], tol=1e-12))
    if kind == "vprop":
        d.e[:, 5] = 2000.0
        d.e[:, 7] = np.random.default_rng([seed, 7]).uniform(0.25, 0.35, d.e.shape[0])
    s = MefSolver(d)
    if kind == "step":
        return dict(kind=kind, s=s, cfg=_cfg(case), z=_zero_state(s))
    if kind == "vprop":
        s.set_vprop([18] * d.e.shape[0], (1, 1, 1, 1))
        return dict(kind=kind, s=s, deck=d, cfg=_cfg(case), z=_zero_state(s))
    if kind == "adjoint":
        rng = np.random.default_rng([seed, 3])
        free = np.nonzero(d.idv[:, 3] == 0)[0]
        node = rng.choice(free, size=min(case["nsens"], len(free)), replace=False)
        target = 1.0e-3 * rng.uniform(0.0, 0.5, size=(case["nsteps"], len(node)))
        return dict(kind=kind, s=s, cfg=_cfg(case, tol=1e-13, maxit=200000), z=_zero_state(s),
                    nsteps=case["nsteps"], sensors=[(int(v), 3) for v in node], target=target)
    u, dp = _state_field(d, case["nen"], seed)
    s.set_state(u=u, u0=0.5 * u, dp=dp, porosity=np.full(s.nnode, 0.2), t=0.1)
    if kind == "stress":
        return dict(kind=kind, s=s)
    rng = np.random.default_rng([seed, 5])
    return dict(kind=kind, s=s, dt=d.dt, f=1.0e-3 * rng.standard_normal(s.neq),
                x=rng.standard_normal(s.neq))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind, s = state["kind"], state["s"]
    if kind in ("step", "batch", "vprop"):
        if kind == "vprop":  # the points' properties back to the start's
            s.set_materials(state["deck"])
            s.set_vprop([18] * state["deck"].e.shape[0], (1, 1, 1, 1))
        s.set_state(**state["z"], t=0.0)
        s.step(state["cfg"])
        st = s.state()
        return dict(u=st["u"], dp=st["dp"], porosity=st["porosity"])
    if kind == "assemble":
        s.set_vectors(b0=state["f"], b=state["f"])
        s.pform(4, False, True, state["dt"], 0.1 + state["dt"], target="b0")
        s.pform(2, True, True, state["dt"], 0.1 + state["dt"], target="b")
        b0, b, _ = s.vectors()
        return dict(b0=b0, b=b, y=s.spmv(state["x"]))
    if kind == "stress":
        tx, txe, txb, flux = s.tform()
        return dict(tx=tx, txe=txe, txb=txb, flux=flux)
    if kind == "adjoint":
        s.set_state(**state["z"], t=0.0)
        J, gE, gk = s.adjoint(state["nsteps"], state["sensors"], state["target"], state["cfg"])
        return dict(J=J, grad_logE=gE, grad_logk=gk)
    s.set_values(state["ad"], state["al"])
    x, _ = s.solve(state["b"], state["cfg"])
    return x


# ---------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------
def _sizes(case, shape=None):
    """cells, equations (before restraints) and stored matrix values of a box"""
    nx, ny, nz = shape or (case["nx"], case["ny"], case["nz"])
    c = P.box_counts(nx, ny, nz, nen=case["nen"])
    per = 108 if case["nen"] == 8 else 200  # stored values of an equation's row
    return c["numel"], c["dofs"], c["dofs"] * per, c["nnode"], c["nnodev"]


def _step_work(case, shape, steps=1, solves=1):
    """A step: the matrix is written once, the mesh and the state are read and
    written once, and every Krylov iteration reads and writes its five vectors
    once; the iterations are those the solver is known to need on these decks
    (proportional to the longest side)."""
    nel, n, nnz, nn, _ = _sizes(case, shape)
    long = max(shape)
    its = long * (114 if case["nen"] == 8 else 290) if case.get("deck") != "column" else 92
    w = 4 if case.get("precision") == "fp32ir" else 8
    loc = 32 if case["nen"] == 8 else 68
    gp = 8 if case["nen"] == 8 else 64
    by = steps * (8 * nnz + 80 * nn + 4 * nel * case["nen"]) + solves * its * 80 * n
    fl = steps * nel * gp * loc * loc * 6 + solves * its * (2 * nnz + 12 * n)
    return by, fl, w


def work(case):
    kind = case["kind"]
    shape = (case["nx"], case["ny"], case["nz"])
    if kind == "batch":
        m = (case["nmin"] + case["nmax"]) / 2
        by, fl, _ = _step_work(case, (int(m),) * 3)
        return dict(bytes=by * case["nbox"], flops=fl * case["nbox"])
    if kind in ("step", "vprop"):
        by, fl, _ = _step_work(case, shape)
        return dict(bytes=by, flops=fl)
    if kind == "adjoint":
        by, fl, _ = _step_work(case, shape, case["nsteps"], 2 * case["nsteps"])
        return dict(bytes=by, flops=fl)
    nel, n, nnz, nn, nv = _sizes(case)
    if kind == "stress":  # 8 corners an element; state, mesh and materials in, 21 values out
        return dict(bytes=40 * nn + 24 * nv + nel * (4 * case["nen"] + 120) + 168 * nn,
                    flops=nel * 8 * (1600 if case["nen"] == 20 else 600))
    if kind == "assemble":  # matrix written once and read once by the product
        loc = 32 if case["nen"] == 8 else 68
        gp = 8 if case["nen"] == 8 else 64
        return dict(bytes=16 * nnz + 40 * n + 72 * nn + nel * (4 * case["nen"] + 120),
                    flops=nel * gp * (loc * loc * 6 + loc * 20) + 2 * nnz)
    its = max(shape) * 114
    return dict(bytes=8 * nnz + its * 64 * n, flops=its * (2 * nnz + 10 * n))


# ---------------------------------------------------------------------------
# the same in plain numpy, 64 bits
# ---------------------------------------------------------------------------
_EDGES = [(0, 1, 8), (1, 2, 9), (2, 3, 10), (3, 0, 11), (4, 5, 12), (5, 6, 13), (6, 7, 14),
          (7, 4, 15), (0, 4, 16), (1, 5, 17), (2, 6, 18), (3, 7, 19)]
_RST8 = np.array([[1, 1, 1], [-1, 1, 1], [-1, -1, 1], [1, -1, 1],
                  [1, 1, -1], [-1, 1, -1], [-1, -1, -1], [1, -1, -1]], float)
_RST20 = np.vstack([_RST8] + [0.5 * (_RST8[a] + _RST8[b]) for a, b, _ in _EDGES])


def _promote(v, nnodev):
    """hexa20 connectivity of a hexa8 one: mid-edge nodes numbered after the
    vertices in the order the elements first meet them."""
    key = np.stack([np.minimum(v[:, a], v[:, b]) * np.int64(nnodev) + np.maximum(v[:, a], v[:, b])
                    for a, b, _ in _EDGES], axis=1)
    _, first, inv = np.unique(key.ravel(), return_index=True, return_inverse=True)
    rank = np.empty(len(first), np.int64)
    rank[np.argsort(first)] = np.arange(len(first))
    return np.hstack([v, nnodev + rank[inv].reshape(key.shape)]), nnodev + len(first)


def _shape8(p):
    f = 1.0 + _RST8[None] * p[:, None]  # (point, node, axis)
    N = f.prod(2) / 8
    dN = np.stack([_RST8[None, :, i] * f[:, :, (i + 1) % 3] * f[:, :, (i + 2) % 3]
                   for i in range(3)], 2) / 8
    return N, dN


def _shape20(p):
    r = _RST20
    f = 1.0 + r[None] * p[:, None]
    N = np.empty((len(p), 20))
    dN = np.empty((len(p), 20, 3))
    for k in range(20):
        g, R = f[:, k], r[k]
        if k < 8:
            q = (R * p).sum(1) - 2
            N[:, k] = g.prod(1) * q / 8
            for i in range(3):
                o = g[:, (i + 1) % 3] * g[:, (i + 2) % 3]
                dN[:, k, i] = R[i] * o * (q + g[:, i]) / 8
        else:
            z = int(np.nonzero(R == 0)[0][0])
            i, j = (z + 1) % 3, (z + 2) % 3
            m = 1 - p[:, z] ** 2
            N[:, k] = m * g[:, i] * g[:, j] / 4
            dN[:, k, z] = -2 * p[:, z] * g[:, i] * g[:, j] / 4
            dN[:, k, i] = m * R[i] * g[:, j] / 4
            dN[:, k, j] = m * g[:, i] * R[j] / 4
    return N, dN


class _Box:
    """Element matrices and the assembled dense system of a small deck."""

    def __init__(self, d, nen):
        self.d, self.nen = d, nen
        v = d.ix[:, :8].astype(np.int64) - 1
        self.ix, self.nnode = _promote(v, d.nnodev) if nen == 20 else (v, d.nnodev)
        self.v = v
        self.mat = d.e[d.ix[:, 20] - 1]
        E, nu = self.mat[:, 0], self.mat[:, 1]
        self.lam = E * nu / ((1 + nu) * (1 - 2 * nu))
        self.mu = E / (2 * (1 + nu))
        self.alpha, self.im = self.mat[:, 4], 1 / self.mat[:, 3]
        self.perm = self.mat[:, 2] / (self.mat[:, 6] * 1e-6 * d.gravity_mod)
        nd = np.zeros((self.nnode, 4), bool)  # free dofs
        nd[: d.nnodev] = d.idv == 0
        if nen == 20:
            fixed = np.zeros((self.nnode, 3), bool)
            for a, b, m in _EDGES:
                fixed[self.ix[:, m]] = (d.idv[v[:, a], :3] == 1) & (d.idv[v[:, b], :3] == 1)
            nd[d.nnodev:, :3] = ~fixed[d.nnodev:]
        self.eq = np.full((self.nnode, 4), -1)
        self.eq[nd] = np.arange(nd.sum())
        self.neq = int(nd.sum())
        self.ld = np.hstack([self.eq[self.ix][:, :, :3].reshape(len(v), -1), self.eq[v][:, :, 3]])

    def grads(self, pts):
        """shape values and global derivatives of u and p nodes, det J"""
        N8, d8 = _shape8(pts)
        Nu, du = _shape20(pts) if self.nen == 20 else (N8, d8)
        xv = self.d.x[self.v]
        J = np.einsum("gki,ekj->egij", d8, xv)
        Ji = np.linalg.inv(J)
        gu = np.einsum("egai,gki->egka", Ji, du)
        gp = np.einsum("egai,gki->egka", Ji, d8)
        return Nu, gu, N8, gp, np.linalg.det(J)

    def parts(self):
        """K_uu, K_pu (= K_up^T), storage S and permeability L (all positive forms)"""
        g, w = np.polynomial.legendre.leggauss(4 if self.nen == 20 else 2)
        pts = np.array([[r, s, t] for t in g for s in g for r in g])
        wt = np.array([a * b * c for c in w for b in w for a in w])
        Nu, gu, N8, gp, det = self.grads(pts)
        W = wt[None] * det
        m = gu.shape[2]
        ne = len(self.v)
        K = np.zeros((ne, m, 3, m, 3))
        G = np.einsum("eg,egia,egjb->eiajb", W, gu, gu, optimize=True)
        K += self.lam[:, None, None, None, None] * G
        K += self.mu[:, None, None, None, None] * G.transpose(0, 1, 4, 3, 2)
        tr = np.einsum("eiaja->eij", G)
        for a in range(3):
            K[:, :, a, :, a] += self.mu[:, None, None] * tr
        Q = -self.alpha[:, None, None, None] * np.einsum("eg,gi,egjb->eijb", W, N8, gu,
                                                         optimize=True)
        S = self.im[:, None, None] * np.einsum("eg,gi,gj->eij", W, N8, N8, optimize=True)
        Lk = self.perm[:, None, None] * np.einsum("eg,egia,egja->eij", W, gp, gp, optimize=True)
        return K.reshape(ne, 3 * m, 3 * m), Q.reshape(ne, 8, 3 * m), S, Lk

    def matrices(self, dt):
        Kuu, Q, S, Lk = self.parts()
        ne, m = Kuu.shape[0], Kuu.shape[1]
        K = np.zeros((ne, m + 8, m + 8))
        K[:, :m, :m] = Kuu
        K[:, m:, :m] = Q
        K[:, :m, m:] = Q.transpose(0, 2, 1)
        K[:, m:, m:] = -(S + dt * Lk)
        C = np.zeros_like(K)
        C[:, m:, :m] = Q
        C[:, m:, m:] = -S
        return K, C, Kuu, Lk

    def dense(self, Ke):
        A = np.zeros((self.neq + 1, self.neq + 1))
        ld = self.ld  # -1: the last row and column, dropped
        np.add.at(A, (ld[:, :, None], ld[:, None, :]), Ke)
        return A[:-1, :-1]

    def load(self):
        """The uniform traction on the top faces (a type-40 face load on face 1)."""
        F = np.zeros(self.neq + 1)
        t = self.d.fload[0, 1:4, 0]
        face = [0, 1, 2, 3] + ([8, 9, 10, 11] if self.nen == 20 else [])
        g, w = np.polynomial.legendre.leggauss(3)
        pts = np.array([[r, s, 1.0] for s in g for r in g])
        wt = np.array([a * b for b in w for a in w])
        Nf = (_shape20(pts)[0] if self.nen == 20 else _shape8(pts)[0])[:, face]
        c = wt @ Nf / 4  # the face's share of each node, per unit area
        top = np.nonzero(self.d.eload[:, 0] > 0)[0]
        x = self.d.x[self.v[top]]
        area = np.abs((x[:, 0, 0] - x[:, 2, 0]) * (x[:, 0, 1] - x[:, 2, 1]))
        for k, no in enumerate(face):
            for a in range(3):
                np.add.at(F, self.eq[self.ix[top, no], a], t[a] * c[k] * area)
        return F[:-1]

    def nodal(self, s):
        u = np.zeros((self.nnode, 4))
        f = self.eq >= 0
        u[f] = s[self.eq[f]]
        return u


def _solve(A, b):
    return torch.linalg.solve(torch.from_numpy(A), torch.from_numpy(b)).numpy()


def _csrc(d, seed):
    """A caller's own symmetric system: diagonal, strict lower rows and a load."""
    B = _Box(d, 8)
    K, _, _, _ = B.matrices(d.dt)
    i = np.repeat(B.ld[:, :, None], 32, 2).ravel()
    j = np.repeat(B.ld[:, None, :], 32, 1).ravel()
    keep = (i >= 0) & (j >= 0) & (j <= i)
    key = i[keep].astype(np.int64) * B.neq + j[keep]
    u, inv = np.unique(key, return_inverse=True)
    val = np.bincount(inv, weights=K.ravel()[keep])
    row, col = u // B.neq, u % B.neq
    low = col < row
    ad = val[~low]
    ia = np.zeros(B.neq + 1, np.int64)
    np.add.at(ia, row[low] + 1, 1)
    b = B.load() + 1e-6 * np.random.default_rng([seed, 11]).standard_normal(B.neq)
    return np.cumsum(ia) + 1, (col[low] + 1).astype(np.int32), ad, val[low], b


def _exact_step(case, seed):
    d = _deck(case, seed)
    B = _Box(d, case["nen"])
    K, _, _, _ = B.matrices(d.dt)
    u = B.nodal(_solve(B.dense(K), B.load()))
    # porosity: the elements' alpha tr(eps) + dp / M at each vertex, averaged
    _, gu, _, _, _ = B.grads(_RST8)
    tr = np.einsum("egka,eka->eg", gu, u[B.ix][:, :, :3])
    dphi = B.alpha[:, None] * tr + B.im[:, None] * u[B.v, 3]
    por = np.full(B.nnode, 0.2)
    cnt = np.bincount(B.v.ravel(), minlength=d.nnodev)
    por[: d.nnodev] += np.bincount(B.v.ravel(), weights=dphi.ravel(), minlength=d.nnodev) / cnt
    return dict(u=u, dp=u[:, 3].copy(), porosity=por)


def _exact_stress(case, seed):
    d = _deck(case, seed)
    B = _Box(d, case["nen"])
    u, dp = _state_field(d, case["nen"], seed)
    tx = np.zeros((B.nnode, 6))
    txb, flux = np.zeros((B.nnode, 6)), np.zeros((B.nnode, 3))
    cnt = np.bincount(B.v.ravel(), minlength=B.nnode)[:, None]
    for g in range(8):
        _, gu, _, gp, _ = B.grads(_RST8[g:g + 1])
        G = np.einsum("eka,ekb->eba", gu[:, 0], u[B.ix][:, :, :3])  # du_b / dx_a
        e = np.stack([G[:, 0, 0], G[:, 1, 1], G[:, 2, 2], G[:, 0, 1] + G[:, 1, 0],
                      G[:, 1, 2] + G[:, 2, 1], G[:, 2, 0] + G[:, 0, 2]], 1)
        no = B.v[:, g]
        st = B.mu[:, None] * e
        st[:, :3] = 2 * st[:, :3] + (B.lam * e[:, :3].sum(1) - B.alpha * dp[no])[:, None]
        sb = st.copy()
        sb[:, :3] += (B.alpha * u[no, 3])[:, None]
        fl = -B.perm[:, None] * np.einsum("eka,ek->ea", gp[:, 0], u[B.v, 3])
        for out, val in ((tx, st), (txb, sb), (flux, fl)):
            for c in range(val.shape[1]):
                out[:, c] += np.bincount(no, weights=val[:, c], minlength=B.nnode)
    for out in (tx, txb, flux):
        out /= np.maximum(cnt, 1)
    txe = tx.copy()
    txe[:, :3] += u[:, 3:4]
    return dict(tx=tx, txe=txe, txb=txb, flux=flux)


def _exact_adjoint(case, seed):
    st = np.random.default_rng([seed, 3])
    d = _deck(case, seed)
    B = _Box(d, case["nen"])
    K, C, Kuu, Lk = B.matrices(d.dt)
    A, Cd, F = B.dense(K), B.dense(C), B.load()
    free = np.nonzero(d.idv[:, 3] == 0)[0]
    node = st.choice(free, size=min(case["nsens"], len(free)), replace=False)
    target = 1.0e-3 * st.uniform(0.0, 0.5, size=(case["nsteps"], len(node)))
    q = B.eq[node, 3]
    lu = torch.linalg.lu_factor(torch.from_numpy(A))
    solve = lambda b: torch.linalg.lu_solve(*lu, torch.from_numpy(b)[:, None])[:, 0].numpy()  # noqa: E731
    s, J, hist = np.zeros(B.neq), 0.0, []
    for n in range(case["nsteps"]):
        s = solve(F + Cd @ s)
        hist.append(s)
        J += float(((s[q] - target[n]) ** 2).sum())
    lam = np.zeros(B.neq)
    gE, gk = np.zeros(d.numel), np.zeros(d.numel)
    m = Kuu.shape[1]
    for n in reversed(range(case["nsteps"])):
        r = Cd.T @ lam
        np.add.at(r, q, 2 * (hist[n][q] - target[n]))
        lam = solve(r)
        le = np.append(lam, 0.0)[B.ld]
        se = np.append(hist[n], 0.0)[B.ld]
        gE -= np.einsum("ei,eij,ej->e", le[:, :m], Kuu, se[:, :m], optimize=True)
        gk += d.dt * np.einsum("ei,eij,ej->e", le[:, m:], Lk, se[:, m:], optimize=True)
    return dict(J=J, grad_logE=gE, grad_logk=gk)


def exact(case, seed):
    """Direct solutions and closed forms for the cases small enough for a dense
    matrix (about 10,000 equations), and for the stresses.  The larger solves and
    the assembly in the library's own ordering have none that is quick enough; the
    per-point property updates have none outside the element itself."""
    kind = case["kind"]
    if kind == "stress":
        return _exact_stress(case, seed)
    if kind in ("batch", "vprop", "assemble"):
        return None
    if _sizes(case)[1] > 12500:
        return None
    if kind == "adjoint":
        return _exact_adjoint(case, seed)
    if kind == "step":
        return _exact_step(case, seed)
    d = _deck(case, seed)
    B = _Box(d, 8)
    _, _, _, _, b = _csrc(d, seed)
    return _solve(B.dense(B.matrices(d.dt)[0]), b)
