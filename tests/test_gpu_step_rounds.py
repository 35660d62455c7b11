"""The step kernel where its loops end raggedly: block rows of every length
around the SpMV's rounds (full rounds, a last round of the blocks left, none),
slices with idle lanes, and numbers of tiles around the reductions' columns of
64.  Random block matrices with rows on none, some or all of the nodes; the
first steps of the solve (CG entry, CG steps, expansions) against the oracle's.

Bound: on well-conditioned systems the iterates of the two sides differ by the
rounding of a few products, about 1e-15 relative per step (measured on the
525-node beam: 9.4e-16 after 55 steps); 1e-12 leaves three digits."""
import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M
import oracle
from mprgp_amd import problems

pytestmark = pytest.mark.gpu


def ragged_system(rng, n, frac):
    """SPD block matrix whose rows have 1 .. about 24 blocks, b, rows, x0."""
    i, j = [], []
    for a in range(n):
        for b in rng.integers(max(0, a - 40), a + 1, size=int(rng.integers(0, 11))):
            if b < a:
                i.append(a)
                j.append(int(b))
    pairs = np.unique(np.array([i, j]).reshape(2, -1), axis=1)
    blk = rng.normal(size=(pairs.shape[1], 3, 3)) * 0.3
    r, c = [], []
    for d in range(3):
        for e in range(3):
            r.append(3 * pairs[0] + d)
            c.append(3 * pairs[1] + e)
    L = sp.csr_matrix((blk.transpose(1, 2, 0).reshape(-1), (np.concatenate(r), np.concatenate(c))),
                      shape=(3 * n, 3 * n)) if pairs.shape[1] else sp.csr_matrix((3 * n, 3 * n))
    S = L + L.T
    A = (S + sp.diags(np.abs(S).sum(axis=1).A1 * 1.05 + rng.uniform(1.0, 3.0, 3 * n))).tocsr()
    A.sort_indices()
    node = np.sort(rng.choice(n, size=int(round(frac * n)), replace=False)).astype(np.int32)
    normal = rng.normal(size=(node.size, 3))
    x0 = rng.normal(size=3 * n)
    c = np.einsum("ij,ij->i", normal, x0.reshape(-1, 3)[node]) - np.abs(rng.normal(size=node.size)) * 0.5
    return A, rng.normal(size=3 * n) * 4.0, node, normal, c, x0


@pytest.mark.parametrize("tail", [1, 1 << 30])
@pytest.mark.parametrize("n,tiles,frac", [(1, 1, 1.0), (63, 1, 0.5), (65, 2, 1.0), (130, 4, 0.0), (321, 8, 0.3),
                                          (64 * 64, 1, 0.1), (64 * 65 + 1, 1, 0.2), (64 * 129 + 5, 1, 0.05),
                                          (64 * 450 + 3, 1, 0.05)])
def test_first_steps_match_the_oracle(ctx, n, tiles, frac, tail):
    rng = np.random.default_rng(n)
    A, b, node, normal, c, x0 = ragged_system(rng, n, frac)
    J = problems.rows_to_J(node, normal, n) if node.size else sp.csr_matrix((0, 3 * n))
    q = ctx.matrix_csr(A).qp()
    q.set_rows(node, normal, c)
    q.set_rhs(b)
    q.set_x(x0)
    ab = 1.9 / float(np.abs(A).sum(axis=1).max())
    seen = np.zeros(3, int)
    for k in (1, 2, 3, 5, 9):
        _, xr, so, _ = oracle.decoupled_solve(A, b, J, c, x0, tol=1e-13, max_it=k, alpha_bar=ab)
        rc, st = q.solve(M.params(tol=1e-13, max_it=k, alpha_bar=ab, project_first=1, from_x0=1, tiles=tiles,
                                  tail_tiles=tail))
        x = q.get_x()
        counts = [st["num_cg"], st["num_exp"], st["num_prop"]]
        assert counts == [so["num_cg"], so["num_exp"], so["num_prop"]], (n, k)
        assert np.linalg.norm(x - xr) <= 1e-12 * np.linalg.norm(xr), (n, k)
        seen = np.maximum(seen, counts)
    assert seen[0] >= 1
