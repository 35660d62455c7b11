"""Both main loops of the coupled solve against the oracle: the one-workgroup
loop on small systems, and the host-driven loop on the same rows with a
component of seven rows, at rest, on nodes of their own (stats launches says
which ran).  Then what the one-workgroup loop does where J J^T is singular on
the rows a step needs: the error of the oracle and of the host-driven loop.

Bars, as in the coupled solve's other tests: the enumerated minimiser to 1e-8,
the oracle's solution to 1e-8 relative."""
import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M
import oracle
from mprgp_amd import problems
from tests.test_gpu_general import beam_with_contacts, qp_of
from tests.test_oracle_general import brute_qp, tiny_coupled_qp

pytestmark = pytest.mark.gpu
REST = 3


def with_rest(A, b, J, c, x0):
    """The problem beside REST nodes at rest (A = I, b = 0) with seven rows off their bounds."""
    n = A.shape[0]
    A2 = sp.block_diag([sp.csr_matrix(A), sp.eye(3 * REST)]).tocsr()
    A2.sort_indices()
    J7 = np.random.default_rng(7).standard_normal((7, 3 * REST))
    J2 = sp.block_diag([sp.csr_matrix(J), J7]).tocsr()
    return A2, np.concatenate([b, np.zeros(3 * REST)]), J2, np.concatenate([c, np.full(7, -1.0)]), \
        np.concatenate([x0, np.zeros(3 * REST)]), n


@pytest.mark.parametrize("seed", [0, 1, 3, 6, 7])
def test_both_loops_reach_the_enumerated_minimiser(ctx, seed):
    A, b, J, c, x0 = tiny_coupled_qp(seed)
    best = brute_qp(A, b, J, c)
    q = qp_of(ctx, A, b, x0)
    rc, st = M.general_solve(q, J, c, tol=1e-11, max_it=3000, project_first=1)
    assert rc == 0 and st["launches"] > 0
    np.testing.assert_allclose(q.get_x(), best, atol=1e-8)
    A2, b2, J2, c2, x2, n = with_rest(A, b, J, c, x0)
    q = qp_of(ctx, A2, b2, x2)
    rc, st = M.general_solve(q, J2, c2, tol=1e-11, max_it=3000, project_first=1)
    assert rc == 0 and st["launches"] == 0
    np.testing.assert_allclose(q.get_x()[:n], best, atol=1e-8)


def test_both_loops_match_the_oracle_on_a_beam(ctx):
    sc, A, b, J, c, x0, m_ground = beam_with_contacts()
    ab = 2.0 / oracle.spec_rad(A, 1e-10)[0]
    kw = dict(tol=1e-9, max_it=3000, alpha_bar=ab)
    code, xr, sr = oracle.general_solve(A, b, J, c, x0, **kw)
    assert code == 0
    q = qp_of(ctx, A, b, x0)
    rc, st = M.general_solve(q, J, c, project_first=1, **kw)
    assert rc == 0 and st["launches"] > 0
    assert np.linalg.norm(q.get_x() - xr) <= 1e-8 * np.linalg.norm(xr)
    A2, b2, J2, c2, x2, n = with_rest(A, b, J, c, x0)
    q = qp_of(ctx, A2, b2, x2)
    rc, st = M.general_solve(q, J2, c2, project_first=1, **kw)
    assert rc == 0 and st["launches"] == 0
    assert np.linalg.norm(q.get_x()[:n] - xr) <= 1e-8 * np.linalg.norm(xr)


def doubled(J, c, rows):
    J = J.toarray()[rows]
    return sp.csr_matrix(np.vstack([J, J])), np.concatenate([c[rows], c[rows]])


def and_zero_row(J, c, bound):
    """Row 0 and a row of stored zeros: J J^T is 0 on it."""
    r = sp.csr_matrix(J.toarray()[:1])
    n = J.shape[1]
    return sp.csr_matrix((np.concatenate([r.data, np.zeros(3)]), np.concatenate([r.indices, np.arange(3)]),
                          [0, r.nnz, r.nnz + 3]), shape=(2, n)), np.array([c[0], bound])


# a component of several rows: an active factor or a projection's block that
# is singular; a row by itself: a projection that needs it, a face that holds it
@pytest.mark.parametrize("seed,rows", [(0, [0, 1, 2]), (1, [0, 1, 2]), (3, [0]), (3, [0, 1]), (0, "zero row, 0.5"),
                                       (0, "zero row, 0.0"), (0, "zero row, -0.5")])
def test_singular_rows_fail_in_the_one_workgroup_loop(ctx, seed, rows):
    A, b, J, c, x0 = tiny_coupled_qp(seed)
    if isinstance(rows, str):
        Js, cs = and_zero_row(J, c, float(rows.split(",")[1]))
    else:
        Js, cs = doubled(J, c, rows)
    kw = dict(tol=1e-8, max_it=100, alpha_bar=0.01)
    code, xr, sr = oracle.general_solve(A, b, Js, cs, x0, project_first=1, **kw)
    q = qp_of(ctx, A, b, x0)
    ends = []
    for project_first in (1, 0):  # without it the loop itself meets the rows first
        q.reset_x()
        try:
            rc, st = M.general_solve(q, Js, cs, project_first=project_first, **kw)
            assert st["launches"] > 0
            ends.append(st["code"])
        except M.MprgpError as e:
            assert "J J^T" in M.last_error()
            ends.append(e.code)
    print(f"seed {seed}, {rows}: oracle {code}, {ends}", flush=True)
    assert ends[0] == code
    A2, b2, J2, c2, x2, n = with_rest(A, b, Js, cs, x0)
    q = qp_of(ctx, A2, b2, x2)
    for project_first, end in zip((1, 0), ends):
        q.reset_x()
        try:
            rc, st = M.general_solve(q, J2, c2, project_first=project_first, **kw)
            got = st["code"]
        except M.MprgpError as e:
            got = e.code
        assert got == end
    # the QP is usable afterwards
    q = qp_of(ctx, A, b, x0)
    rc, st = M.general_solve(q, J, c, tol=1e-11, max_it=3000, project_first=1)
    assert rc == 0
    np.testing.assert_allclose(q.get_x(), brute_qp(A, b, J, c), atol=1e-8)
