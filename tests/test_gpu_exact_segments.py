"""Exact forces against the oracle's one sum around the counts where the
number of segments changes: the same bits below 4096 bodies, beyond that the
rounding of sums of n terms in another order (n eps times the sum of the
terms' sizes, which a Plummer sphere keeps within a hundred times the sum)."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 4095, 4096, 4351, 8191, 8192, 8449])
def test_segments(n):
    bodies = plummer_bodies(n, seed=n)
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=1e-4, criterion="exact",
                             allowIncest=True)
    o = orc.Oracle(orc.make_ctx(eps2=1e-4, theta=0.0, timestep=1e-3, criterion="exact",
                                allow_incest=True), *bodies)
    o.gravity()
    st = nb.NBodyState(ctx, None, *bodies)
    a = st.accelerations()
    st.close()
    if n < 4096:
        assert np.array_equal(a, o.acc)
    else:
        size = np.linalg.norm(o.acc, axis=1)
        tol = 100 * n * np.finfo(float).eps * np.maximum(size, np.median(size))
        assert (np.linalg.norm(a - o.acc, axis=1) <= tol).all()
