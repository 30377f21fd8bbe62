"""The force adjoint where interaction lists fit for some groups of 64 bodies
and not for others, or for none, and where a group holds bodies of several
simulations, against evaluations without either: the same bodies as the first simulation
of a batch too large for lists, and each simulation in a state of its own.
Tolerance: the same terms in another order, 1e-11 of the largest entry (the
tolerance of the other adjoint tests)."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu

LIST_BODIES = 131072


def _ctx(theta, eps2=1e-3):
    return nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, theta=theta,
                              allowIncest=True)


def _close(a, b):
    assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()


@pytest.mark.parametrize("n,theta", [(9001, 0.35), (9001, 0.2), (12000, 0.25),
                                     (20000, 0.3), (20000, 0.2), (50000, 0.35)])
def test_lists_that_do_not_fit(n, theta):
    bodies = plummer_bodies(n, seed=6)
    G = np.random.default_rng(9).normal(size=(n, 3))
    st = nb.NBodyState(_ctx(theta), None, *bodies)
    gx, gm = st.gravity_vjp(G)
    st.close()
    rest = LIST_BODIES + 1 - n
    filler = (np.random.default_rng(2).uniform(-1.0, 1.0, (rest, 3)), np.zeros((rest, 3)),
              np.full(rest, 1e-9))
    bt = nb.NBodyBatch(_ctx(theta), None, [bodies, filler])
    rx, rm = bt.gravity_vjp(np.concatenate([G, np.zeros((rest, 3))]))
    bt.close()
    _close(gx, rx[:n])
    _close(gm, rm[:n])


@pytest.mark.parametrize("sizes", [(1, 1, 1, 2, 3), (60, 10, 70, 1, 200), (3000, 40, 4000, 2500)])
def test_groups_shared_by_simulations(sizes):
    members = [plummer_bodies(n, seed=50 + k, position=(0.3 * k, 0.0, -0.2 * k))
               for k, n in enumerate(sizes)]
    eps2 = [1e-3 * (k + 1) for k in range(len(sizes))]
    G = np.random.default_rng(9).normal(size=(sum(sizes), 3))
    bt = nb.NBodyBatch(_ctx(0.6), None, members, eps2=eps2)
    gx, gm = bt.gravity_vjp(G)
    bt.close()
    at = 0
    for k, n in enumerate(sizes):
        st = nb.NBodyState(_ctx(0.6, eps2[k]), None, *members[k])
        rx, rm = st.gravity_vjp(G[at:at + n])
        st.close()
        _close(gx[at:at + n], rx)
        _close(gm[at:at + n], rm)
        at += n
