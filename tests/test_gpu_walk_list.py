"""The FP64 list walk against the oracle, bit for bit (tolerance zero): body
counts around a group of 64, a wave's 4 or 8 bodies, the change of batch
width and the largest state with lists; every criterion; lists that overflow
beside lists that do not; groups shared by several simulations and massless
bodies."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _ctx(theta=0.5, criterion="bh86", quad=True, eps2=1e-4, incest=False):
    c = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, theta=theta,
                           criterion=criterion, useQuad=quad, allowIncest=incest)
    o = orc.make_ctx(eps2=eps2, theta=c.theta, timestep=c.timestep, criterion=criterion,
                     use_quad=c.useQuad, allow_incest=incest)
    return c, o


def _check(bodies, **kw):
    ctx, octx = _ctx(**kw)
    st = nb.NBodyState(ctx, None, *bodies)
    o = orc.Oracle(octx, *bodies)
    rc = o.gravity()
    assert np.array_equal(st.accelerations(), o.acc)
    assert bool(st.last_status) == bool(rc)
    assert np.array_equal(st.walk_accel(), o.acc)
    st.close()


@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 9, 63, 64, 65, 67, 127, 128, 129, 1000, 8191, 8192,
                               8193, 8197])
def test_body_counts(n):
    _check(plummer_bodies(n, seed=n))


@pytest.mark.parametrize("n", [24575, 24576, 24577, 24583])
@pytest.mark.parametrize("quad", [True, False])
def test_end_of_the_fetch_ahead(n, quad):
    _check(plummer_bodies(n, seed=n), theta=0.8, quad=quad, incest=True)


@pytest.mark.parametrize("n", [131071, 131072, 131073])
def test_largest_states_with_lists(n):
    _check(plummer_bodies(n, seed=4), theta=0.8, incest=True)   # above 1/sqrt 3 bodies meet no self


@pytest.mark.parametrize("criterion,theta", [("bh86", 0.5), ("bh86", 1.0), ("sw93", 0.7),
                                             ("treecode", 0.8)])
@pytest.mark.parametrize("quad", [True, False])
@pytest.mark.parametrize("eps2", [1e-4, 0.0])
def test_criteria(criterion, theta, quad, eps2):
    _check(plummer_bodies(9001, seed=8), criterion=criterion, theta=theta, quad=quad, eps2=eps2,
           incest=True)


@pytest.mark.parametrize("n,theta", [(3000, 0.0), (12000, 0.3), (20000, 0.2), (20000, 0.12)])
def test_lists_that_overflow(n, theta):
    """Up to 8192 nodes a group: none, some and all of the groups beyond."""
    _check(plummer_bodies(n, seed=6), theta=theta)


def test_two_far_clumps():
    """A group whose box spans both clumps decides by the bodies' tests."""
    a, b = plummer_bodies(1000, seed=1), plummer_bodies(1031, seed=2)
    pos = np.concatenate([a[0] + 30.0, b[0] - 30.0])
    _check((pos, np.concatenate([a[1], b[1]]), np.concatenate([a[2], b[2]])))


@pytest.mark.parametrize("sizes", [(1, 1, 1, 2, 3), (60, 10, 70, 1, 200), (3000, 40, 4000, 2500)])
def test_groups_shared_by_simulations(sizes):
    ctx, _ = _ctx()
    members, eps2 = [], []
    for k, n in enumerate(sizes):
        pos, vel, m = plummer_bodies(n, seed=50 + k, position=(0.3 * k, 0.0, -0.2 * k))
        m = m.copy()
        if n > 50:
            m[::9] = 0.0                     # massless: sorted after every massive body
        members.append((pos, vel, m))
        eps2.append(1e-4 * (k + 1))
    bt = nb.NBodyBatch(ctx, None, members, eps2=eps2, prestep=False)
    bt.lib.nbhip_gravity(bt._h)              # massless bodies report incest, as in the reference
    for k, mem in enumerate(members):
        octx = orc.make_ctx(eps2=eps2[k], theta=ctx.theta, timestep=ctx.timestep)
        o = orc.Oracle(octx, *mem)
        o.gravity()
        assert np.array_equal(bt.sim_bodies(k)[2], o.acc), k
    bt.close()


def test_replayed_steps():
    """Graph replays against the oracle's steps, with eager work between."""
    bodies = plummer_bodies(5003, seed=12)
    ctx, octx = _ctx()
    st = nb.NBodyState(ctx, None, *bodies)
    o = orc.Oracle(octx, *bodies)
    assert o.gravity() == 0
    st.set_graph(True)
    for _ in range(3):
        assert st.steps(2) == 0
        for _ in range(2):
            assert o.step() == 0
        x, v, a = st.bodies()
        assert np.array_equal(x, o.pos) and np.array_equal(v, o.vel) and np.array_equal(a, o.acc)
        st.walk_accel()
    st.close()
