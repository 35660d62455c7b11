"""Which of the coupled solve's two main loops runs (stats launches: the
one-workgroup loop's, 0 where the host drives it): the one-workgroup loop for
small systems with few components of several rows, the host-driven one where
the matrix or the components would take one CU longer than the launches they
save.  On either side of the line both give the same bits."""
import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M
from tests.test_gpu_general_loop import REST, chain, rows_on

pytestmark = pytest.mark.gpu


def solve(ctx, A, b, J, c, max_it=40):
    q = ctx.matrix_csr(A).qp()
    q.set_rhs(b)
    q.set_x(np.zeros(A.shape[0]))
    rc, st = M.general_solve(q, J, c, tol=1e-12, max_it=max_it, alpha_bar=0.25, project_first=1)
    return st, q.get_x()


# nodes, rows of a component, components, one workgroup
@pytest.mark.parametrize("n,k,count,one", [(1, 1, 1, True), (300, 5, 12, True), (300, 6, 128, False),
                                           (1200, 6, 32, True), (1200, 3, 256, False), (2597, 2, 60, True),
                                           (2597, 2, 600, False), (2597, 6, 16, True), (2597, 6, 128, False),
                                           (2598, 1, 5, False)])
def test_components_decide(ctx, n, k, count, one):
    rng = np.random.default_rng(n + k + count)
    A, b = chain(rng, n)
    J, c = rows_on(rng, n, k, count)
    st, x = solve(ctx, A, b, J, c)
    print(f"{n} nodes, {count} components of {k}: {st['iterations']} iterations, {st['launches']} launches", flush=True)
    assert (st["launches"] > 0) == one
    J7 = sp.csr_matrix(np.hstack([np.zeros((7, 3 * n)), rng.standard_normal((7, 3 * REST))]))
    s7, x7 = solve(ctx, A, b, sp.vstack([J, J7]).tocsr(), np.concatenate([c, np.full(7, -1e-8)]))
    assert s7["launches"] == 0
    assert [s7[f] for f in ("iterations", "num_cg", "num_exp", "num_prop", "residual")] == \
        [st[f] for f in ("iterations", "num_cg", "num_exp", "num_prop", "residual")]
    np.testing.assert_array_equal(x, x7)


@pytest.mark.parametrize("n,band,one", [(100, 49, True), (600, 20, True), (600, 80, False), (1200, 7, True),
                                        (1200, 60, False), (2600, 1, True), (2600, 30, False)])
def test_matrix_decides(ctx, n, band, one):
    off = np.arange(-band, band + 1)
    lap = sp.diags([np.full(n - abs(o), -1.0 / band if o else 2.2) for o in off], off)
    A = sp.kron(lap, np.eye(3) + 0.3 * np.ones((3, 3))).tocsr()
    A.sort_indices()
    rng = np.random.default_rng(n + band)
    J = sp.lil_matrix((2, 3 * n))
    J[0, 0:6], J[1, 3:6] = rng.standard_normal(6), rng.standard_normal(3)
    st, _ = solve(ctx, A, 0.05 * rng.standard_normal(3 * n), J.tocsr(), np.array([-0.1, 0.1]), max_it=10)
    assert (st["launches"] > 0) == one


def test_without_iterations_no_loop_is_launched(ctx):
    rng = np.random.default_rng(1)
    A, b = chain(rng, 300)
    J, c = rows_on(rng, 300, 5, 12)
    st, _ = solve(ctx, A, b, J, c, max_it=0)
    assert st["launches"] == 0 and st["iterations"] == 0
