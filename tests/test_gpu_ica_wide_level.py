"""The ICA sweep where a level has more nodes than the LDS ring has slots
(6,400): nodes that couple to none before them, then a few that read the last
of them, in the ring.  Against the oracle, with the bound of the other ICA
tests."""
import numpy as np
import pytest
import scipy.sparse as sp

from mprgp_amd import problems
from tests.test_gpu_ica import both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [6399, 6400, 6401, 6528, 13000])
def test_level_wider_than_the_ring(ctx, wide):
    rng = np.random.default_rng(wide)
    last, n = 40, wide + 40
    i = np.repeat(np.arange(wide, n), 3)
    j = wide - 1 - np.array([rng.choice(200, 3, replace=False) for _ in range(last)]).ravel()
    S = sp.lil_matrix((3 * n, 3 * n))
    for a, b in zip(i, j):
        S[3 * a:3 * a + 3, 3 * b:3 * b + 3] = 0.2 * rng.normal(size=(3, 3))
    S = (S + S.T).tocsr()
    A = (S + sp.diags(np.asarray(abs(S).sum(axis=1)).ravel() * 1.1 + 1.0)).tocsr()
    A.sort_indices()
    node = np.sort(rng.choice(n, size=n // 20, replace=False)).astype(np.int32)
    J = problems.rows_to_J(node, rng.normal(size=(node.size, 3)), n)
    x0 = rng.normal(size=3 * n)
    both(ctx, A, rng.normal(size=3 * n), J, J @ x0 - 0.3 * rng.random(node.size), x0, tol=1e-13, max_it=3,
         gs_max_it=30, gs_tol=1e-14)
