"""The coupled solve's one-workgroup main loop against its host-driven loop,
which the oracle's tests pin: the same iterates, so bit for bit the same x and
the same counters.  A component of seven rows on nodes of their own, at rest
off their bounds, sends the same problem to the host-driven loop.  Sizes:
components of one row to the largest taken, systems around a slice of 64
nodes, more rows than threads, the largest system, and iteration limits at
the end of a launch's share of 256."""
import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M

pytestmark = pytest.mark.gpu

REST = 3  # nodes without load, coupled to nothing


def chain(rng, n):
    """A chain of n nodes (3x3 blocks, condition about 1e4) and REST nodes apart."""
    lap = sp.diags([-np.ones(n - 1), 2.0 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1]) + 1e-3 * sp.eye(n)
    q = np.eye(3) + 0.3 * np.ones((3, 3))
    A = sp.block_diag([sp.kron(lap, q), sp.eye(3 * REST)]).tocsr()
    A.sort_indices()
    b = np.concatenate([0.05 * rng.standard_normal(3 * n) - 0.02, np.zeros(3 * REST)])
    return A, b


def rows_on(rng, n, k, count):
    """count components of k rows: row i of a component on nodes base and base + i."""
    J = sp.lil_matrix((k * count, 3 * (n + REST)))
    for q in range(count):
        base = q * (n // count)
        for i in range(k):
            for node in {base, min(base + i, n - 1)}:
                J[q * k + i, 3 * node:3 * node + 3] = rng.standard_normal(3)
    return J.tocsr(), rng.uniform(-0.5, 0.1, k * count)


@pytest.mark.parametrize("precond", [1, 0])
@pytest.mark.parametrize("n,k,count,max_it", [
    (1, 1, 1, 500), (1, 2, 1, 500), (21, 2, 3, 500), (61, 3, 8, 500), (62, 4, 7, 500), (125, 5, 20, 500),
    (700, 6, 40, 400), (2597, 2, 600, 300), (2597, 1, 1100, 257), (300, 5, 12, 256), (300, 5, 12, 257),
    (300, 5, 12, 1), (300, 5, 12, 0)])
def test_both_loops_give_the_same_bits(ctx, n, k, count, max_it, precond):
    rng = np.random.default_rng(n + k)
    A, b = chain(rng, n)
    J, c = rows_on(rng, n, k, count)
    J7 = sp.csr_matrix(np.hstack([np.zeros((7, 3 * n)), rng.standard_normal((7, 3 * REST))]))
    q = ctx.matrix_csr(A).qp()
    q.set_rhs(b)
    got = []
    for rows, bounds in ((J, c), (sp.vstack([J, J7]).tocsr(), np.concatenate([c, np.full(7, -1e-8)]))):
        q.set_x(np.zeros(A.shape[0]))
        rc, st = M.general_solve(q, rows, bounds, tol=1e-12, max_it=max_it, alpha_bar=0.25, project_first=1,
                                 preconditioned=precond)
        got.append((rc, [st[f] for f in ("iterations", "num_cg", "num_exp", "num_prop", "active", "residual")],
                    q.get_x()))
    print(f"n {n}, {count} components of {k}: {got[0][:2]}", flush=True)
    assert got[0][0] == got[1][0] and got[0][1] == got[1][1]
    assert np.array_equal(got[0][2], got[1][2])
