"""The two forms of the ICA sweep at the sizes where they can go wrong: x in
the LDS ring (levels wider than a workgroup's 128 nodes, rows with more lower
blocks than are loaded ahead, more nodes than the ring holds) and the form
that reads x from memory (columns further back than the ring).  A few
iterations against the oracle, which sums every row in the same order: the
bound of the other ICA tests, 1e-10 relative."""
import numpy as np
import pytest
import scipy.sparse as sp

from mprgp_amd import problems
from tests.test_gpu_ica import both

pytestmark = pytest.mark.gpu


def banded_system(rng, n, reach, per_row, far=0):
    """Block-diagonally dominant matrix: each node coupled to per_row nodes up
    to `reach` before it, and the first `far` of the last nodes to node 0."""
    i = np.repeat(np.arange(n), per_row)
    j = i - rng.integers(1, reach + 1, size=i.size)
    i, j = i[j >= 0], j[j >= 0]
    i = np.concatenate([i, n - 1 - np.arange(far)]).astype(int)
    j = np.concatenate([j, np.zeros(far)]).astype(int)
    pairs = np.unique(np.array([i, j]), axis=1)
    rows, cols, vals = [], [], []
    for d in range(3):
        for e in range(3):
            rows.append(3 * pairs[0] + d)
            cols.append(3 * pairs[1] + e)
            vals.append(rng.normal(size=pairs.shape[1]) * 0.2)
    L = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))), shape=(3 * n, 3 * n))
    S = (L + L.T).tocsr()
    A = (S + sp.diags(np.abs(S).sum(axis=1).A1 * 1.1 + 1.0)).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("n,reach,per_row,far", [(1, 1, 1, 0), (700, 690, 1, 0), (900, 60, 14, 0), (7001, 120, 4, 0),
                                                 (7001, 120, 4, 3)])
def test_sweep_forms_match_the_oracle(ctx, n, reach, per_row, far):
    rng = np.random.default_rng(n + far)
    A = banded_system(rng, n, reach, per_row, far)
    node = np.sort(rng.choice(n, size=max(1, n // 10), replace=False)).astype(np.int32)
    normal = rng.normal(size=(node.size, 3))
    J = problems.rows_to_J(node, normal, n)
    x0 = rng.normal(size=3 * n)
    c = J @ x0 - 0.3 * rng.random(node.size)
    both(ctx, A, rng.normal(size=3 * n), J, c, x0, tol=1e-13, max_it=4, gs_max_it=50, gs_tol=1e-14)
    both(ctx, A, rng.normal(size=3 * n), sp.csr_matrix((0, 3 * n)), np.zeros(0), x0, tol=1e-13, max_it=2)
