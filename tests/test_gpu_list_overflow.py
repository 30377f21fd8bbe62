"""The FP64 walk of states whose interaction lists do not fit (8192 nodes a
group), which stream with 8, 16, 32 or 64 bodies a wave, against the oracle,
bit for bit (tolerance zero): around the sizes where the number changes, in a
batch where one simulation's lists do not fit, and in a state that goes from
bodies whose lists fit to others and back."""
import ctypes as C

import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _ctx(theta, quad=True):
    return nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=1e-4, theta=theta, useQuad=quad)


def _oracle(bodies, theta, quad=True):
    o = orc.Oracle(orc.make_ctx(eps2=1e-4, theta=theta, timestep=1e-3, use_quad=quad), *bodies)
    assert o.gravity() == 0
    return o


@pytest.mark.parametrize("n,theta", [(1000, 0.0), (8191, 0.1), (8192, 0.1), (8193, 0.1),
                                     (16383, 0.2), (16384, 0.2), (16385, 0.2), (32768, 0.25),
                                     (32769, 0.25), (65537, 0.35)])
@pytest.mark.parametrize("quad", [True, False])
def test_body_counts(n, theta, quad):
    bodies = plummer_bodies(n, seed=n)
    st = nb.NBodyState(_ctx(theta, quad), None, *bodies)
    o = _oracle(bodies, theta, quad)
    assert np.array_equal(st.accelerations(), o.acc)
    assert np.array_equal(st.walk_accel(), o.acc)
    st.close()


def test_one_simulation_of_a_batch():
    members = [plummer_bodies(n, seed=n) for n in (500, 12000, 77)]
    bt = nb.NBodyBatch(_ctx(0.2), None, members)
    for k, mem in enumerate(members):
        assert np.array_equal(bt.sim_bodies(k)[2], _oracle(mem, 0.2).acc), k
    bt.close()


def test_there_and_back():
    """Eager forces and replayed steps over bodies whose lists fit (clumps far
    from each other), then do not (one sphere), then do again."""
    n, theta = 16000, 0.25
    sphere = plummer_bodies(n, seed=1)
    at = np.random.default_rng(2).integers(-6, 7, (160, 3)) * 1.5
    clumps = (sphere[0] * 0.05 + np.repeat(at, 100, 0), sphere[1], sphere[2])
    st = nb.NBodyState(_ctx(theta), None, *clumps)
    for bodies in (clumps, sphere, clumps, sphere):
        p = [np.ascontiguousarray(a, dtype=np.float64).ctypes.data_as(C.POINTER(C.c_double))
             for a in bodies]
        assert st.lib.nbhip_upload(st._h, *p) == 0
        st.set_graph(False)
        assert st.gravity() == 0
        o = _oracle(bodies, theta)
        assert np.array_equal(st.accelerations(), o.acc)
        st.set_graph(True)
        for _ in range(2):
            assert st.steps(1) == 0 and o.step() == 0
            x, v, a = st.bodies()
            assert np.array_equal(x, o.pos) and np.array_equal(v, o.vel)
            assert np.array_equal(a, o.acc)
    st.close()
