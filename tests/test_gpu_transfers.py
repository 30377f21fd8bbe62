"""Bodies to the device and back, bit for bit, around the largest state that
leaves through page-locked memory, whole and per simulation of a batch."""
import numpy as np
import pytest

from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu


def _bodies(n, seed):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(n, 3)), rng.normal(size=(n, 3)), rng.uniform(0.5, 1.5, n) / max(n, 1)


def _ctx():
    return nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=1e-4, theta=0.5,
                              allowIncest=True)


@pytest.mark.parametrize("n", [1, 85, 86, 4095, 4096, 4097, 100001])
def test_round_trip(n):
    bodies = _bodies(n, n)
    st = nb.NBodyState(_ctx(), None, *bodies)
    before = st.walk_accel()
    pos, vel, acc = st.bodies()
    assert np.array_equal(pos, bodies[0]) and np.array_equal(vel, bodies[1])
    assert np.array_equal(acc, before)
    assert np.array_equal(st.walk_accel(), before)        # the tree is still there
    st.close()


@pytest.mark.parametrize("sizes", [(1, 7, 2000), (3000, 1, 2500)])
def test_round_trip_of_a_batch(sizes):
    members = [_bodies(n, n) for n in sizes]
    bt = nb.NBodyBatch(_ctx(), None, members, eps2=[1e-4] * len(sizes))
    for k, (pos, vel, _) in enumerate(members):
        p, v, _ = bt.sim_bodies(k)
        assert np.array_equal(p, pos) and np.array_equal(v, vel)
    bt.close()
