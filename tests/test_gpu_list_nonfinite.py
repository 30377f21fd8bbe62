"""A body with a coordinate that is no number, in a state that walks lists:
the state reports an error, and the accelerations of that evaluation are what
IEEE arithmetic makes of the reference's expressions, as in the streaming
walk."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu

NBHIP_ERROR = 2


@pytest.mark.parametrize("n", [2, 100, 5000])
@pytest.mark.parametrize("quad", [True, False])
def test_a_body_that_is_no_number_reaches_every_body(n, quad):
    """No cell that holds it is ever accepted (its distance compares with
    nothing), so each walk interacts with the body itself, whose distance is
    no number either."""
    pos, vel, m = plummer_bodies(n, seed=n)
    pos = pos.copy()
    pos[n // 3, 0] = np.nan
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=1e-4, theta=0.5, useQuad=quad)
    st = nb.NBodyState(ctx, None, pos, vel, m, prestep=False)
    rc = st.lib.nbhip_gravity(st._h)
    assert nb.status_is_fatal(rc)
    if n == 2:
        assert rc == NBHIP_ERROR           # both bodies meet themselves: no incest
    assert np.isnan(st.bodies()[2]).all()
    st.close()
