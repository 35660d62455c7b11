"""The FP64 CG step with P(y) stored by a launch of its own (small launches of
large tiles) against the same step with P(y) formed at the product's gathers:
tail_tiles decides between them launch by launch, and the results are the same
bits.  Sizes: one slice, a tile's end, several tiles, and a batch whose
launches pass from one form to the other as QPs finish; alone and beside
mixed-form QPs."""
import numpy as np
import pytest

import mprgp_amd as M
from mprgp_amd import problems, workloads

pytestmark = pytest.mark.gpu
CG_PY = workloads.OPS.index("CG_PY")


def results(ctx, qps, tail, tiles, spw, precisions, max_it=400):
    for q in qps:
        q.qp.reset_x()
    ps = [M.params(tol=1e-7, max_it=max_it, alpha_bar=q.ab, project_first=1, precision=pr, tiles=tiles,
                   slices_per_wave=spw, tail_tiles=tail, graph_steps=4) for q, pr in zip(qps, precisions)]
    _, st = M.solve_batch(ctx, [q.qp for q in qps], per_qp=ps)
    return ([q.qp.get_x() for q in qps], [[s[k] for k in ("iterations", "num_cg", "num_exp", "residual")] for s in st],
            [int(q.qp.op_counts()[CG_PY]) for q in qps])


def device_qps(ctx, dims):
    qps = []
    for k, d in enumerate(dims):
        q = workloads.DeviceQP(ctx, problems.beam_scene("b", *d, seed=k, tol=1e-7))
        q.ab = q.qp.solve(M.params(tol=1e-7, max_it=0))[1]["alpha_bar"]
        qps.append(q)
    return qps


@pytest.mark.parametrize("tiles,spw,split", [(8, 1, True), (1, 2, True), (8, 2, True), (4, 1, False), (1, 1, False)])
@pytest.mark.parametrize("dims", [[(3, 2, 2)], [(20, 4, 4)], [(30, 7, 7)], [(12, 3, 3), (30, 7, 7), (40, 8, 8)]])
def test_both_forms_give_the_same_bits(ctx, dims, tiles, spw, split):
    qps = device_qps(ctx, dims)
    fp64 = [M.FP64] * len(qps)
    own = results(ctx, qps, 1 << 30, tiles, spw, fp64)
    gathered = results(ctx, qps, 1, tiles, spw, fp64)
    both = results(ctx, qps, 3, tiles, spw, fp64)  # changes over as the batch empties
    assert all(n > 0 for n in own[2]) == split
    for other in (gathered, both):
        assert other[1] == own[1]
        for a, b in zip(own[0], other[0]):
            np.testing.assert_array_equal(a, b)
    if len(qps) > 1:
        mixed = [M.MIXED if k == 1 else M.FP64 for k in range(len(qps))]
        m = [results(ctx, qps, tail, tiles, spw, mixed) for tail in (1 << 30, 1)]
        assert m[0][1] == m[1][1] and m[0][2][1] == 0
        for a, b in zip(m[0][0], m[1][0]):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(m[0][0][0], own[0][0])
