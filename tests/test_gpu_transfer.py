"""Host vectors of one call through the context's pinned memory: round trips
and projections are exact for small calls and at the sizes where that memory
is given up for plain copies (4 MB a call: one vector of 174,762 nodes; a
projection's two vectors and its sum, 87,380 nodes), each after larger and
smaller calls on the same context."""
import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M

pytestmark = pytest.mark.gpu


def body(ctx, n):
    q = ctx.matrix_csr(sp.identity(3 * n, format="csr")).qp()
    q.set_rows(np.arange(n), np.tile([0.0, 1.0, 0.0], (n, 1)), np.zeros(n))
    return q


@pytest.mark.parametrize("sizes", [(1, 2730, 2731, 5462, 1), (87380, 87381, 21), (174762, 174763, 2)])
def test_vectors_arrive_whole(sizes):
    ctx = M.Context(0)
    qps = [body(ctx, n) for n in sizes]
    rng = np.random.default_rng(0)
    for _ in range(2):
        for q, n in zip(qps, sizes):
            x, b = rng.standard_normal(3 * n), rng.standard_normal(3 * n)
            q.set_x(x)
            q.set_rhs(b)
            assert np.array_equal(q.get_x(), x) and np.array_equal(q.get_rhs(), b)
            y = x.reshape(-1, 3).copy()
            y[:, 1] = np.maximum(y[:, 1], 0.0)
            assert np.array_equal(q.project(x), y.ravel())
            assert not q.is_feasible(x - 1.0) and q.is_feasible(y.ravel())
            q.set_x(b)
            q.reset_x()
            assert np.array_equal(q.get_x(), b)
