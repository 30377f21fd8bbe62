"""The FP64 list walk where factors of its quadrupole terms leave the range of
the numbers, against the oracle, bit for bit (tolerance zero): softenings
whose reciprocal fifth power overflows, and cells whose quadrupole overflows
though no body interacts with them."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _check(bodies, eps2, quad, rsize=4.0, theta=0.5):
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=eps2, theta=theta, useQuad=quad,
                             treeRSize=rsize)
    st = nb.NBodyState(ctx, None, *bodies)
    o = orc.Oracle(orc.make_ctx(eps2=eps2, theta=theta, timestep=ctx.timestep, use_quad=quad,
                                tree_rsize=rsize), *bodies)
    assert o.gravity() == 0
    assert np.isfinite(o.acc).all()
    assert np.array_equal(st.accelerations(), o.acc)
    st.close()


@pytest.mark.parametrize("eps2", [1e-120, 1e-130, 1e-150, 1e-180, 1e-204])
@pytest.mark.parametrize("quad", [True, False])
@pytest.mark.parametrize("n", [2, 300, 9001])
def test_tiny_softenings(n, quad, eps2):
    _check(plummer_bodies(n, seed=n), eps2, quad)


def test_quadrupoles_that_overflow_unused():
    """Close pairs of heavy bodies far apart: the root's quadrupole is
    infinite, the pairs' are not, and every body opens the root."""
    rng = np.random.default_rng(4)
    centre = rng.permutation(8)[:, None] >> np.arange(3) & 1
    pos = (centre * 2.0 - 1.0) * rng.uniform(1500.0, 2000.0, (8, 3))
    pos = np.repeat(pos, 2, 0) + rng.uniform(0.0, 2.0 ** -12, (16, 3))
    m = 2.0 ** 1005 * rng.uniform(0.5, 1.0, 16)
    _check((pos, np.zeros_like(pos), m), 1.0, True, rsize=8192.0)
