"""The tree of an evaluation that reported an error (a body with a coordinate
that is no number, at the sizes where the summaries notice): a table whose
records were not all written is refused, or every body it names exists."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [13, 5000, 100000])
@pytest.mark.parametrize("fresh", [True, False])
def test_tree_after_error(n, fresh):
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=1e-4, theta=0.5)
    pos, vel, m = plummer_bodies(n, seed=n)
    bad = pos.copy()
    bad[n // 3] = np.nan
    if not fresh:                      # memory that another state has used
        nb.NBodyState(ctx, None, pos, vel, m).close()
    st = nb.NBodyState(ctx, None, bad, vel, m, prestep=False)
    assert nb.status_is_fatal(st.lib.nbhip_gravity(st._h))
    try:
        t = st.tree()
    except nb.NBodyError:
        t = None
    if t is not None:
        assert ((t["ref"] >= -1) & (t["ref"] < n)).all()
    st.close()
