"""The XCD a context's launches start on changes no result: solves on nine
contexts alive at once (one more than the XCDs), one after the other and all
at the same time, from the context's tables and from those built on the
device, and through an engine beside them."""
import ctypes as C
import threading

import numpy as np
import pytest

import mprgp_amd as M
from mprgp_amd import _lib, problems, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(20, 4, 4), (40, 9, 9)])
def test_contexts_alive_at_once_give_the_same_bits(dims):
    ctxs = [M.Context(0) for _ in range(9)]
    try:
        qps = [workloads.DeviceQP(c, problems.beam_scene("b", *dims, seed=1, tol=1e-6)) for c in ctxs]
        kw = dict(tol=1e-6, max_it=300, project_first=1)
        out = []

        def solve(i, device_table):
            q = qps[i].qp
            q.reset_x()
            if device_table:
                p, st = M.params(**kw), M.Stats()
                _lib.load().mprgp_qp_solve_noalloc(q.h, C.byref(p), C.byref(st))
                return q.get_x(), st.as_dict()["iterations"]
            _, st = q.solve(**kw)
            return q.get_x(), st["iterations"]
        for i in range(9):
            out += [solve(i, False), solve(i, True)]
        res = [None] * 9
        threads = [threading.Thread(target=lambda i=i: res.__setitem__(i, solve(i, False))) for i in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        out += res[:8]
        for x, it in out[1:]:
            assert it == out[0][1]
            np.testing.assert_array_equal(x, out[0][0])
        eng = M.Engine(ctxs[0], max_active=4, tiles=1)
        try:
            qps[0].qp.reset_x()
            eng.wait(eng.submit(qps[0].qp, **kw))
            np.testing.assert_array_equal(qps[0].qp.get_x(), out[0][0])
        finally:
            eng.close()
    finally:
        for c in ctxs:
            c.close()
