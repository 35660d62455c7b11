"""Device assembly where the lists of tets that a workgroup keeps in LDS end:
tets around one edge (its block sums all of them, 96 held at a time), so that
lists are shorter than one run, one run exactly, one more, and several runs,
with blocks below and above a workgroup's 256; LINEAR and COROTATIONAL, with
and without stiffness damping.

Bars, against the oracle's assembly: 1e-12 of |A||x| and of max |b|.  A tet of
the narrowest fan has an angle of 2 pi / 200, so D_m^-1 is off by about
60 eps = 7e-15 relative; the strains are about 0.05, so the forces are off by
1.5e-13 of their own size."""
import types

import numpy as np
import pytest

import mprgp_amd as M
import oracle
from mprgp_amd import problems
from tests.test_gpu_fem import check_system

pytestmark = pytest.mark.gpu


def fan(n, closed):
    """n tets around the edge of nodes 0 and 1, closed to a ring or not."""
    k = n if closed else n + 1
    a = 2.0 * np.pi * np.arange(k) / 200.0 if not closed else 2.0 * np.pi * np.arange(k) / k
    ring = np.stack([np.cos(a), np.sin(a), np.full(k, 0.5)], 1)
    X0 = np.concatenate([[[0.0, 0.0, 0.0], [0.0, 0.0, 1.0]], ring])
    i = np.arange(n)
    tets = np.stack([np.zeros(n, int), np.ones(n, int), 2 + i, 2 + (i + 1) % k], 1)
    rng = np.random.default_rng(n)
    sc = types.SimpleNamespace(X0=X0, tets=tets.astype(np.int32), n_nodes=k + 2, young=rng.uniform(1e5, 2e5, n),
                               poisson=rng.uniform(0.2, 0.4, n), density=1000.0, gravity=np.array([0.0, -9.8, 0.0]),
                               h=0.01, v_n=0.1 * rng.standard_normal(X0.shape))
    Q = problems.random_rotation(rng)
    return sc, (X0 @ (np.eye(3) + 0.05 * rng.standard_normal((3, 3)))) @ Q.T


@pytest.mark.parametrize("mtype", [M.LINEAR, M.COROTATIONAL])
@pytest.mark.parametrize("n,closed", [(1, False), (20, True), (95, False), (96, False), (97, False), (192, False),
                                      (200, True)])
def test_fans_match_the_oracle(ctx, n, closed, mtype):
    sc, x = fan(n, closed)
    check_system(ctx, sc, x, mtype)


@pytest.mark.parametrize("n", [1, 127, 128, 129])
def test_damped_fans_match_the_oracle(ctx, n):
    """At the Newton iterate x1: the damping forces K c of every tet."""
    sc, x = fan(n, False)
    rng = np.random.default_rng(n + 1)
    x1 = x + 1e-3 * rng.standard_normal(x.shape)
    tets, d, vol, mass = oracle.fem_setup(sc.n_nodes, sc.tets, sc.X0)
    A, b = oracle.fem_build_system(sc.n_nodes, tets, d, vol, mass, sc.young, sc.poisson, sc.density, x.ravel(),
                                   sc.v_n.ravel(), sc.gravity, sc.h, M.LINEAR, x1=x1.ravel(), alpha_k=0.1, alpha_m=0.02)
    fem = M.Fem(ctx, sc.X0, sc.tets, sc.young, sc.poisson, sc.density)
    fem.set_damping(0.1, 0.02)
    q = fem.matrix.qp()
    fem.assemble_at(q, x.ravel(), sc.v_n.ravel(), x1.ravel(), sc.gravity, sc.h, M.LINEAR)
    assert np.abs(q.get_rhs() - b).max() <= 1e-12 * np.abs(b).max()
