"""A simulation that has gone wrong (coordinates that are no numbers, infinite
or huge, masses near the end of the range) shares groups of 64 bodies and
waves with others: those keep their own results, bit for bit the oracle's in
FP64 and a single run's in the mixed forms, their statuses, and their force
adjoint (the same terms in another order, 1e-11 of the largest entry)."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SIZES = (60, 10, 70, 1, 200, 33)


def _members(wrong, first):
    members = [plummer_bodies(n, seed=70 + k, position=(0.3 * k, 0.0, -0.2 * k))
               for k, n in enumerate(SIZES)]
    bad = 0 if first else 2
    pos, vel, m = (a.copy() for a in members[bad])
    if wrong == "nan":
        pos[5, 0] = np.nan
    elif wrong == "inf":
        pos[5, 1] = -np.inf
    elif wrong == "wide":
        pos *= 1e40
    elif wrong == "heavy":
        m[:] = 1e300
        pos *= 1e10
    members[bad] = (pos, vel, m)
    return members, bad


def _ctx(criterion, quad):
    return nb.NBodyCtx.create(timestep=1e-4, timeEvolve=1.0, eps2=1e-4, theta=0.6,
                              criterion=criterion, useQuad=quad)


@pytest.mark.parametrize("wrong", ["nan", "inf", "wide", "heavy"])
@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("criterion,quad", [("bh86", True), ("bh86", False), ("sw93", True)])
def test_fp64_neighbours(wrong, first, criterion, quad):
    members, bad = _members(wrong, first)
    ctx = _ctx(criterion, quad)
    bt = nb.NBodyBatch(ctx, None, members, prestep=False)
    bt.lib.nbhip_gravity(bt._h)
    G = np.random.default_rng(9).normal(size=(sum(SIZES), 3))
    gx, gm = bt.gravity_vjp(G)
    off = np.concatenate([[0], np.cumsum(SIZES)])
    for k, mem in enumerate(members):
        if k == bad:
            continue
        o = orc.Oracle(orc.make_ctx(eps2=1e-4, theta=0.6, timestep=ctx.timestep,
                                    criterion=criterion, use_quad=quad), *mem)
        assert o.gravity() == 0
        assert np.array_equal(bt.sim_bodies(k)[2], o.acc), k
        assert bt.statuses()[k] == 0, k
        st = nb.NBodyState(ctx, None, *mem)
        rx, rm = st.gravity_vjp(G[off[k]:off[k + 1]])
        st.close()
        for a, b in ((gx[off[k]:off[k + 1]], rx), (gm[off[k]:off[k + 1]], rm)):
            assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max(), k
    bt.close()


@pytest.mark.parametrize("wrong", ["nan", "inf", "wide"])
@pytest.mark.parametrize("precision", ["mixed", "mixed_coherent"])
def test_mixed_neighbours(wrong, precision):
    """Waves that hold several simulations interact as waves of one do only in
    the per-lane form; the coherent one's bodies have to stay finite."""
    members, bad = _members(wrong, False)
    ctx = _ctx("bh86", True)
    bt = nb.NBodyBatch(ctx, None, members, precision=precision, prestep=False)
    bt.lib.nbhip_gravity(bt._h)
    for k, mem in enumerate(members):
        if k == bad:
            continue
        st = nb.NBodyState(ctx, None, *mem, precision=precision)
        a, b = bt.sim_bodies(k)[2], st.accelerations()
        st.close()
        assert np.isfinite(a).all(), k
        if precision == "mixed":
            assert np.array_equal(a, b), k
    bt.close()
