"""Solves that prefer a form with more device memory still run, with the same
results, where the context's budget holds only the form with less."""
import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M
from mprgp_amd import problems
from tests.common import scene_qp

pytestmark = pytest.mark.gpu


def beam():
    sc = problems.beam_scene("b", 12, 4, 4, seed=3, tol=1e-8)
    A, b, node, normal, c, x0 = scene_qp(sc)
    Jc, cc = problems.self_contact_rows(sc, np.random.default_rng(2), 6)
    return A, b, sp.vstack([problems.rows_to_J(node, normal, sc.n_nodes), Jc]).tocsr(), np.concatenate([c, cc]), x0


def on_budget(A, b, x0, call, extra=None):
    """call(qp) on a context of its own; extra: bytes allowed beyond the matrix and the QP."""
    ctx = M.Context(0)
    try:
        q = ctx.matrix_csr(A).qp()
        used = ctx.memory()[0]
    finally:
        ctx.close()
    ctx = M.Context(0, hbm_budget=0 if extra is None else used + extra)
    try:
        q = ctx.matrix_csr(A).qp()
        q.set_rhs(b)
        q.set_x(x0)
        out = call(q)
        return out, q.get_x()
    finally:
        ctx.close()


def lower_levels(A):
    """Blocks below the diagonal and dependency levels of the forward sweep."""
    P = sp.csr_matrix(A).tobsr((3, 3))
    level = np.zeros(A.shape[0] // 3, int)
    n_lo = 0
    for i in range(level.size):
        lo = P.indices[P.indptr[i]:P.indptr[i + 1]]
        lo = lo[lo < i]
        n_lo += lo.size
        level[i] = level[lo].max() + 1 if lo.size else 0
    return n_lo, level.max() + 1


def test_ica_without_room_for_the_ring(ctx):
    A, b, J, c, x0 = beam()
    n, nn, m, nnz = A.shape[0], A.shape[0] // 3, J.shape[0], J.nnz
    n_lo, levels = lower_levels(A)
    parts = (n + 255) // 256 + 1
    least = 8 * (9 * nn + 9 * n_lo + 2 * nnz + 2 * m + parts + 8) + \
        4 * (levels + 1 + 2 * nn + 1 + 2 * n_lo + m + 1 + 2 * nnz + n + 1) + 1024

    def call(q):
        rc, st, lam, sweeps = M.ica_solve(q, J, c, tol=1e-6, max_it=30, gs_max_it=20, gs_tol=1e-8)
        return rc, st["iterations"], st["residual"], sweeps, lam.tobytes()
    free, xf = on_budget(A, b, x0, call)
    tight, xt = on_budget(A, b, x0, call, least)
    assert tight == free
    np.testing.assert_array_equal(xt, xf)
    with pytest.raises(M.MprgpError) as e:
        on_budget(A, b, x0, call, least - 2048)
    assert e.value.code == -7


def test_coupled_solve_without_room_for_the_one_workgroup_loop(ctx):
    A, b, J, c, x0 = beam()
    n, m, nnz = A.shape[0], J.shape[0], J.nnz
    parts = (n + 255) // 256 + 1
    least = 4 * (m + 1 + nnz + n + 1 + nnz) + 8 * (2 * nnz + 5 * (m + 1) + 8 * parts + 16) + 1024

    def call(q):
        rc, st = M.general_solve(q, J, c, tol=1e-9, max_it=60, alpha_bar=1e-3, project_first=1)
        return [rc] + [st[f] for f in ("iterations", "num_cg", "num_exp", "num_prop", "active", "residual")], \
            st["launches"]
    (free, loop), xf = on_budget(A, b, x0, call)
    (tight, host), xt = on_budget(A, b, x0, call, least)
    assert loop > 0 and host == 0
    assert tight == free
    np.testing.assert_array_equal(xt, xf)
    with pytest.raises(M.MprgpError) as e:
        on_budget(A, b, x0, call, least - 1)
    assert e.value.code == -7


@pytest.mark.parametrize("material", [M.LINEAR, M.COROTATIONAL])
def test_fem_body_without_room_for_its_tet_lists(ctx, material):
    sc = problems.beam_scene("b", 12, 4, 4, seed=3, tol=1e-8, material=material)
    # nodes in no order, so that the lists are long
    order = np.random.default_rng(5).permutation(sc.n_nodes)
    X0, tets = sc.X0[order], np.argsort(order)[sc.tets].astype(np.int32)
    x, v = 1.01 * X0.ravel(), sc.v_n[order].ravel()

    filler = sp.eye(60000, format="csr")  # held while the body is made, given back before it is used

    def system(room=None):
        c = M.Context(0)
        try:
            c.matrix_csr(filler)
            held = c.memory()[0]
        finally:
            c.close()
        c = M.Context(0, hbm_budget=0 if room is None else held + room)
        try:
            fill = c.matrix_csr(filler)
            before = c.memory()[0]
            fem = M.Fem(c, X0, tets, sc.young, sc.poisson, sc.density)
            made = c.memory()[0]
            fill.close()
            q = fem.matrix.qp()
            fem.set_damping(0.1, 0.02)
            fem.assemble(q, x, v, sc.gravity, sc.h, material)
            rowptr, colidx, blocks = fem.matrix.get_bsr3()
            return made - before, (rowptr, colidx, blocks, q.get_rhs())
        finally:
            c.close()
    made, want = system()
    c = M.Context(0)
    try:
        empty = c.memory()[0]
        P = sp.bsr_matrix((np.ones((len(want[1]), 3, 3)), want[1], want[0]))
        A = c.matrix_csr((P + sp.eye(P.shape[0])).tocsr())
        matrix = c.memory()[0] - empty
        A.close()
    finally:
        c.close()
    N, T, nb = sc.n_nodes, len(tets), len(want[1])
    body = 256 * 17 + 16 * T + 8 * 21 * T + 16 * N + 4 * (nb + 1 + 16 * T + 2 * nb + N + 1 + 4 * T)
    assert made > matrix + body  # the lists
    least, got = system(matrix + body)
    assert least == matrix + body
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
    with pytest.raises(M.MprgpError) as e:
        system(matrix + body - 1)
    assert e.value.code == -7
