"""One multigrid V-cycle against its restatement with sparse matrices.

A solve of one Picard iteration whose Krylov method (GCR) may take one step
returns x0 + a z with z = M^-1 (b - A x0) and a = (A z, r) / (A z, A z): the
V-cycle M^-1 is all that is between the system, which the oracle assembles from
the downloaded coefficients, and the velocities.  Aggregates, Galerkin products,
sweeps and the coarsest solve are restated here from their definition (the head
of csrc/mg.hip), level by level, without the kernels' splits and orders."""
import numpy as np
import pytest
import scipy.sparse as sp

import _oracle as O
import branch_cases
from imau_vel import config, geometry

pytestmark = pytest.mark.gpu

CMAX, SWEEPS = 32, 10     # the coarsest level's largest extent, its symmetric sweeps


@pytest.fixture(scope="module")
def ctx():
    from imau_vel import solver
    c = solver.Context()
    yield c
    c.close()


# 9-point pattern: offsets (dJ, dI) from a row's cell to the unknowns it may couple to
STAR = {(0, 0), (0, -1), (0, 1), (-1, 0), (1, 0)}
PATTERN = {(0, 0): STAR, (1, 1): STAR, (0, 1): {(-1, 0), (-1, 1), (0, 0), (0, 1)},
           (1, 0): {(0, -1), (0, 0), (1, -1), (1, 0)}}


class Level:
    """Unknowns (component, J, I) in any order, their matrix and colours."""

    def __init__(self, comp, J, I, A):
        self.comp, self.J, self.I, self.A = comp, J, I, A.tocsr()
        self.D = self.A.diagonal()
        self.skip = np.zeros(len(comp), bool)       # rows outside the four colours
        self.colour = 2 * comp + ((J + I) & 1)

    def update(self, x, b, idx):
        if len(idx):
            off = self.A[idx] @ x - self.D[idx] * x[idx]
            d = self.D[idx]
            x[idx] = np.where(d != 0.0, (b[idx] - off) / np.where(d != 0.0, d, 1.0), 0.0)

    def sweep(self, x, b, order):
        for c in order:
            self.update(x, b, np.flatnonzero((self.colour == c) & ~self.skip))


def coarsen(lev, agg, rows):
    """R A P of `lev`: agg[n] is the aggregate (J, I) of unknown n or None, rows
    those that are restricted; couplings outside the pattern are dropped."""
    key = {}
    for c in (0, 1):
        n = lev.extent[c]
        for J in range((n[0] + 1) // 2):
            for I in range((n[1] + 1) // 2):
                key[(c, J, I)] = len(key)
    A = lev.A.tocoo()
    r, c, v = [], [], []
    for n, m, a in zip(A.row, A.col, A.data):
        if not rows[n] or agg[n] is None or agg[m] is None:
            continue
        (Jn, In), (Jm, Im) = agg[n], agg[m]
        if (Jm - Jn, Im - In) in PATTERN[lev.comp[n], lev.comp[m]]:
            r.append(key[lev.comp[n], Jn, In])
            c.append(key[lev.comp[m], Jm, Im])
            v.append(a)
    ks = np.array(list(key))
    out = Level(ks[:, 0], ks[:, 1], ks[:, 2], sp.coo_matrix((v, (r, c)), shape=(len(key),) * 2))
    out.extent = {q: ((lev.extent[q][0] + 1) // 2, (lev.extent[q][1] + 1) // 2) for q in (0, 1)}
    out.size = ((lev.size[0] + 1) // 2, (lev.size[1] + 1) // 2)
    n = len(lev.comp)
    up = [key[lev.comp[q], agg[q][0], agg[q][1]] if agg[q] is not None else -1 for q in range(n)]
    lev.P = sp.coo_matrix((np.ones(sum(u >= 0 for u in up)), ([q for q in range(n) if up[q] >= 0],
                                                             [u for u in up if u >= 0])), shape=(n, len(key))).tocsr()
    lev.R = sp.diags(np.array(rows, float)) @ lev.P
    lev.R = lev.R.T.tocsr()
    return out


def hierarchy(g, A):
    nx, ny = g.nx, g.ny
    unk = [(c, j, i) for i in range(nx) for j in range(ny) for c in (0, 1)
           if (i < nx - 1 if c == 0 else j < ny - 1)]
    comp, J, I = (np.array(a) for a in zip(*unk))
    fine = Level(comp, J, I, A)
    fine.extent, fine.size = {0: (ny, nx - 1), 1: (ny - 1, nx)}, (ny, nx)
    edge = np.where(comp == 0, (I == 0) | (I == nx - 2) | (J == 0) | (J == ny - 1),
                    (I == 0) | (I == nx - 1) | (J == 0) | (J == ny - 2))
    nnz = np.diff(fine.A.indptr)
    rows = ~edge & (nnz > 1)                       # free and calving-front rows; zero rows are a single 1
    agg = [(J[n] >> 1, I[n] >> 1) if rows[n] else None for n in range(len(unk))]
    for n in np.flatnonzero(edge & (nnz == 2)):    # 'infinite': the aggregate of the source
        cols = fine.A.indices[fine.A.indptr[n]:fine.A.indptr[n + 1]]
        src = int(cols[cols != n][0])
        assert not edge[src]
        if rows[src]:
            agg[n] = (J[src] >> 1, I[src] >> 1)
    fine.skip = edge
    levels = [fine, coarsen(fine, agg, rows)]
    while max(levels[-1].size) > CMAX:
        l = levels[-1]
        levels.append(coarsen(l, [(a >> 1, b >> 1) for a, b in zip(l.J, l.I)], np.ones(len(l.J), bool)))
    return levels


def vcycle(levels, y):
    rhs, x = [y], []
    for q, l in enumerate(levels):
        z = np.zeros(len(l.D))
        if q + 1 == len(levels):
            for _ in range(SWEEPS):
                l.sweep(z, rhs[q], (0, 1, 2, 3, 3, 2, 1, 0))
        else:
            l.sweep(z, rhs[q], (0, 1, 2, 3))
            l.update(z, rhs[q], np.flatnonzero(l.skip))
            rhs.append(l.R @ (rhs[q] - l.A @ z))
        x.append(z)
    for q in range(len(levels) - 2, -1, -1):
        l = levels[q]
        x[q] += l.P @ x[q + 1]
        l.sweep(x[q], rhs[q], (3, 2, 1, 0))
        l.update(x[q], rhs[q], np.flatnonzero(l.skip))
    return x[0]


def case(kind):
    if kind == "BC":
        _, g, cfg, st = branch_cases.bc_margin_case()
    elif kind in ("channel", "sans"):
        kw = dict(include_SSADIVA_crossterms=0) if kind == "sans" else None
        g, cfg, st = geometry.channel(nx=61, ny=21, dx=8e3, seed=3, **(dict(cfg=geometry.synthetic_config(**kw)) if kw else {}))
    else:
        g, cfg, st = geometry.random_geometry(*kind, seed=sum(kind), beta_sq=1e4)
    c2 = type(cfg).from_buffer_copy(cfg)
    config.set_config(c2, DIVA_visc_it_nit=6, DIVA_visc_it_norm_dUV_tol=0.0)
    O.solve("diva", g, c2, st, O.LIN_BANDED_LU)    # a state with velocities
    return g, cfg, st


# one, two and three coarse levels, odd and even extents, fronts, 'zero' sides, the form without cross terms
@pytest.mark.parametrize("kind", [(29, 31), (64, 65), (71, 66), (131, 40), "channel", "sans", "BC"],
                         ids=lambda k: str(k).replace(" ", ""))
@pytest.mark.parametrize("precision,tol", [("fp64", 5e-13), ("mixed", 2.7e-5)])
def test_vcycle(ctx, kind, precision, tol):
    """tol: each of the few hundred row updates of a cycle divides by a dominant
    diagonal, so it passes rounding on without growth: 500 x 9 terms x 1.1e-16 in
    FP64, and a tenth of 500 x 9 x 6e-8 in FP32 (signs average out; the sum alone
    would hide a lost coupling), relative to the largest change.  Measured 6e-15
    and 3e-7."""
    g, cfg, st = case(kind)
    config.set_config(cfg, stop_rule=0, DIVA_visc_it_nit=1, DIVA_visc_it_norm_dUV_tol=0.0, DIVA_visc_it_relax=1.0,
                      DIVA_vel_max=1e12, DIVA_choice_matrix_solver="PETSc", ksp_type=1, mg_levels=0, anderson_m=0,
                      precision=precision)
    st.DIVA_PETSc_rtol, st.DIVA_PETSc_abstol, st.DIVA_SOR_nit = 1e-14, 0.0, 1
    u0, v0 = st["u_vav_cx"].copy(), st["v_vav_cy"].copy()
    ctx.solve_diva(g, cfg, st)
    ptr, idx, val, b, x0 = O.assemble_csr(g, cfg, st, u0, v0)
    A = sp.csr_matrix((val, idx, ptr), shape=(len(b),) * 2)
    r = b - A @ x0
    z = vcycle(hierarchy(g, A), r)
    q = A @ z
    step = (q @ r) / (q @ q) * z
    unk = [(c, j, i) for i in range(g.nx) for j in range(g.ny) for c in (0, 1)
           if (i < g.nx - 1 if c == 0 else j < g.ny - 1)]
    got = np.array([st["u_vav_cx"][j, i] if c == 0 else st["v_vav_cy"][j, i] for c, j, i in unk])
    err = np.abs(got - x0 - step).max() / np.abs(step).max()
    print(kind, precision, "levels", len(hierarchy(g, A)), "err %.2e" % err)
    assert err <= tol, err
