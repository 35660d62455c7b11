"""Where a launch's tiles are placed changes no result: the tile counts at
which the runs of tiles per XCD and the launch size change (8, 16 and 32 tiles,
a tile per CU, four per CU), rotated or in chunks, and by the solve that
builds its tile table on the device."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import mprgp_amd as M
from mprgp_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [1, 8, 9, 16, 17, 32, 33, 256, 257, 1024, 1025])
def test_placements_give_the_same_bits(ctx, tiles):
    n = 64 * (tiles - 1) + 1  # the last slice holds one node
    rng = np.random.default_rng(tiles)
    lap = sp.diags([-np.ones(n - 1), 2.2 * np.ones(n), -np.ones(n - 1)], [-1, 0, 1])
    q = ctx.matrix_csr(sp.kron(lap, np.eye(3) + 0.2 * np.ones((3, 3))).tocsr()).qp()
    q.set_rhs(rng.standard_normal(3 * n) - 0.5)
    q.set_rows(np.arange(0, n, 2), np.tile([0.0, 1.0, 0.0], ((n + 1) // 2, 1)), rng.uniform(-1.0, 0.0, (n + 1) // 2))
    out = []
    for how in ("rotated", "chunks", "device table"):
        q.set_x(np.zeros(3 * n))
        p = M.params(tol=1e-8, max_it=60, project_first=1, tiles=1, alpha_bar=0.2, xcd_layout=int(how == "chunks"))
        if how == "device table":
            st = M.Stats()
            _lib.load().mprgp_qp_solve_noalloc(q.h, C.byref(p), C.byref(st))
            st = st.as_dict()
        else:
            _, st = q.solve(p)
        out.append((q.get_x(), st["iterations"], st["residual"]))
    for o in out[1:]:
        assert np.array_equal(o[0], out[0][0]) and o[1:] == out[0][1:]
