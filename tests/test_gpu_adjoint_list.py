"""The force adjoint from interaction lists against the numpy frozen-tree VJP
(tests/test_gpu_adjoint.py's checker and tolerance) at body counts around a
wave's 8 bodies and a group of 64, at softenings inside and outside the range
of the unscaled divisions, and with every list overflowing (theta = 0, where
the tree's adjoint is the direct sum's)."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import adjoint_ref as ar
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 9, 63, 65, 200])
@pytest.mark.parametrize("quad", [True, False])
@pytest.mark.parametrize("eps2", [1e-3, 2.0 ** 201])
def test_vjp_at_group_edges(n, quad, eps2):
    pos, vel, m = plummer_bodies(n, seed=n)
    m = m * np.random.default_rng(7).uniform(0.5, 1.5, n)
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, theta=0.6, useQuad=quad,
                             allowIncest=True)
    st = nb.NBodyState(ctx, None, pos, vel, m)
    G = np.random.default_rng(8).normal(size=(n, 3))
    gx, gm = st.gravity_vjp(G)
    o = orc.Oracle(orc.make_ctx(eps2=eps2, theta=0.6, use_quad=quad, allow_incest=True), pos,
                   vel, m)
    o.gravity()
    t = o.tree()
    rx, rm = ar.frozen_vjp(pos, m, t, ar.tree_children(t), ar.walk_lists(t), eps2, G, quad)
    assert np.abs(gx - rx).max() <= 1e-11 * np.abs(rx).max()
    assert np.abs(gm - rm).max() <= 1e-11 * np.abs(rm).max()
    st.close()


def test_vjp_with_overflowing_lists():
    n, eps2 = 9000, 1e-3
    pos, vel, m = plummer_bodies(n, seed=3)
    G = np.random.default_rng(9).normal(size=(n, 3))
    out = []
    for crit, theta in (("bh86", 0.0), ("exact", -1.0)):
        ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, theta=theta,
                                 criterion=crit)
        st = nb.NBodyState(ctx, None, pos, vel, m)
        out.append(st.gravity_vjp(G))
        st.close()
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max()
