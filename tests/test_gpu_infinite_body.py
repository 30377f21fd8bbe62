"""A body at an infinite x: the state reports an error, and the accelerations
of that evaluation are what IEEE arithmetic makes of the reference's
expressions.  The term of anything at infinity is m / inf / inf = 0 times its
displacement: no number in x, 0 in y and z.  In the direct sum the other
bodies' sums in y and z stay (the oracle's bits); in the tree it is the root,
which every body accepts."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_direct_sum_with_an_infinite_body(sign):
    n, eps2 = 500, 1e-4
    pos, vel, m = plummer_bodies(n, seed=n)
    pos = pos.copy()
    pos[7, 0] = sign * np.inf
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=eps2, criterion="exact")
    st = nb.NBodyState(ctx, None, pos, vel, m, prestep=False)
    assert nb.status_is_fatal(st.lib.nbhip_gravity(st._h))
    a = st.bodies()[2]
    st.close()
    keep = np.arange(n) != 7
    o = orc.Oracle(orc.make_ctx(eps2=eps2, theta=ctx.theta, timestep=ctx.timestep,
                                criterion="exact"), pos[keep], vel[keep], m[keep])
    assert o.gravity() == 0
    assert np.isnan(a[:, 0]).all()
    assert np.array_equal(a[keep, 1:], o.acc[:, 1:])


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("n", [2, 100, 5000])
def test_tree_with_an_infinite_body(n, sign):
    pos, vel, m = plummer_bodies(n, seed=n)
    pos = pos.copy()
    pos[n // 3, 0] = sign * np.inf
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=1e-4, theta=0.5, useQuad=False)
    st = nb.NBodyState(ctx, None, pos, vel, m, prestep=False)
    assert nb.status_is_fatal(st.lib.nbhip_gravity(st._h))
    a = st.bodies()[2]
    st.close()
    keep = np.arange(n) != n // 3
    assert np.isnan(a[:, 0]).all()
    assert (a[keep, 1:] == 0.0).all()
