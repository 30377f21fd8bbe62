"""The force adjoint from interaction lists at separations whose reciprocal
ninth power overflows: a body has no quadrupole, so nothing that grows like
that may enter its terms.  One body per octant of the root (its only cell),
opened by every body (theta = 0), against the direct sum's adjoint.
Tolerance: both sides add at most eight terms of a few roundings each, 1e-12
of the largest entry."""
import numpy as np
import pytest

from milkywayathome_client_amd import nbody as nb
from oracle import adjoint_ref as ar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 5, 8])
@pytest.mark.parametrize("scale,eps2", [(-130, 1e-90), (-125, 1e-77), (-3, 1e-90)])
@pytest.mark.parametrize("quad", [True, False])
def test_close_bodies_without_quadrupoles(n, scale, eps2, quad):
    rng = np.random.default_rng(8)
    octant = np.array([[(k >> d & 1) * 2.0 - 1.0 for d in range(3)] for k in range(8)])[:n]
    pos = octant * rng.uniform(0.1, 0.9, (n, 3)) * 2.0 ** scale
    m = rng.uniform(0.5, 1.5, n)
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, theta=0.0, useQuad=quad,
                             treeRSize=4.0 * 2.0 ** scale)
    st = nb.NBodyState(ctx, None, pos, np.zeros_like(pos), m)
    assert st.last_status == 0
    G = rng.normal(size=(n, 3))
    gx, gm = st.gravity_vjp(G)
    rx, rm = ar.direct_adj(pos, m, eps2, G)
    assert np.isfinite(rx).all() and np.isfinite(rm).all()
    assert np.abs(gx - rx).max() <= 1e-12 * np.abs(rx).max()
    assert np.abs(gm - rm).max() <= 1e-12 * np.abs(rm).max()
    st.close()
