"""The FP64 walk and its workgroup size: the bits of the streaming walk do not
depend on it (states of more bodies than lists are kept for, and states whose
lists do not fit, against the oracle), and where lists are walked, whose launch
it does not shape, the autotuner keeps the setting it finds."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,theta", [(131073, 0.9), (140001, 0.9), (12001, 0.2), (40001, 0.25)])
def test_blocks_of_the_streaming_walk(n, theta):
    bodies = plummer_bodies(n, seed=11)
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1e-2, eps2=1e-4, theta=theta,
                             allowIncest=True)
    st = nb.NBodyState(ctx, None, *bodies)
    o = orc.Oracle(orc.make_ctx(eps2=1e-4, theta=ctx.theta, timestep=ctx.timestep,
                                use_quad=ctx.useQuad, allow_incest=True), *bodies)
    o.gravity()
    for block in (64, 128, 256):
        st.set_tune(block, 1024)
        assert np.array_equal(st.walk_accel(), o.acc), block
    best, trials = st.autotune()
    assert best in trials and best[2] == min(t[2] for t in trials)
    st.close()


def test_autotune_keeps_the_setting_of_list_walks():
    ctx = nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1e-2, eps2=1e-4, theta=0.5)
    st = nb.NBodyState(ctx, None, *plummer_bodies(3000, seed=11))
    for _ in range(3):
        for block in (64, 128, 256):
            st.set_tune(block, 1024)
            best, trials = st.autotune()
            assert best[:2] == (block, 1024)
            assert best in trials and len(trials) == 3
    st.close()
