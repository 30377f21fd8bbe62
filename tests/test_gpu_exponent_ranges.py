"""FP64 interactions at the ends of the range that takes unscaled divisions
(nbh_plain_range): softenings, masses and root sizes just inside and just
outside it, against the oracle's IEEE arithmetic.  Inside and outside must
both give the oracle's bits: the tolerance is zero."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# (log2 of the position scale, log2 of the masses, eps2, log2 of one odd mass or None)
CASES = [(0, -4, 1e-4, None), (0, -4, 2.0 ** -200, None), (0, -4, 2.0 ** -201, None),
         (0, -4, 0.0, None), (0, -4, 2.0 ** 200, None), (0, -4, 2.0 ** 201, None),
         (86, -4, 2.0 ** 150, None), (92, -4, 2.0 ** 150, None), (0, 300, 1e-4, None),
         (0, 301, 1e-4, None), (0, -300, 1e-4, None), (0, -301, 1e-4, None),
         (0, -4, 1e-4, -301), (0, -4, 1e-4, 301)]


@pytest.mark.parametrize("criterion", ["bh86", "exact"])
@pytest.mark.parametrize("scale,mass,eps2,odd", CASES)
def test_range_ends_match_oracle(criterion, scale, mass, eps2, odd):
    if criterion == "exact" and eps2 == 0.0:
        pytest.skip("the direct sum's self term needs a softening")
    n = 300
    pos, vel, _ = plummer_bodies(n, seed=5)
    pos = pos * 2.0 ** scale
    m = np.full(n, 2.0 ** mass) * (1.0 + np.arange(n) / 1024.0 if mass != 300 else 1.0)
    if odd is not None:
        m[17] = 2.0 ** odd
    rsize = 4.0 * 2.0 ** scale
    theta = 0.5 if criterion == "bh86" else -1.0
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=eps2, theta=theta,
                             criterion=criterion, treeRSize=rsize)
    st = nb.NBodyState(ctx, None, pos, vel, m)
    o = orc.Oracle(orc.make_ctx(eps2=eps2, theta=ctx.theta, timestep=ctx.timestep,
                                criterion=criterion, use_quad=ctx.useQuad, tree_rsize=rsize),
                   pos, vel, m)
    assert o.gravity() == 0
    assert np.isfinite(o.acc).all()
    assert np.array_equal(st.accelerations(), o.acc)
    st.close()
