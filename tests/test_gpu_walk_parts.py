"""The mixed walks cut into parts: the same bits as one wave gives (the
simulation inside a batch too large to be cut), from fewer node blocks than
parts to the largest state that is cut; and the oracle's accelerations."""
import numpy as np
import pytest

from helpers import plummer_bodies
from milkywayathome_client_amd import nbody as nb
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

FILL = 262145                            # bodies that make a batch too large to be cut


@pytest.mark.parametrize("precision", ["mixed", "mixed_coherent"])
@pytest.mark.parametrize("n,criterion,quad,batch", [
    (1, "bh86", True, None), (64, "bh86", True, 64), (1000, "bh86", True, None),
    (1000, "sw93", False, 16), (10007, "bh86", True, 128), (30000, "treecode", True, 1 << 20),
    (262144, "bh86", True, None)])
def test_parts_equal_one_wave(precision, n, criterion, quad, batch):
    if precision == "mixed_coherent":
        n = (n + 63) // 64 * 64          # whole waves, so that the batch groups them alike
    theta = {"bh86": 0.5, "sw93": 0.7, "treecode": 0.8}[criterion]
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=1e-4, theta=theta,
                             criterion=criterion, useQuad=quad, allowIncest=True)
    bodies = plummer_bodies(n, seed=n)
    fill = plummer_bodies(FILL, seed=7)
    st = nb.NBodyState(ctx, None, *bodies, precision=precision)
    bt = nb.NBodyBatch(ctx, None, [bodies, fill], eps2=[1e-4, 1e-4], precision=precision)
    if batch:
        for x in (st, bt):
            x.set_tune(block=128, batch=batch)
    a, b = st.walk_accel(), bt.walk_accel()[:n]
    st.close()
    bt.close()
    assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [64, 5000, 40000])
def test_parts_match_the_oracle(n):
    """FP32 interactions (2^-24 each, a few of them per term) summed in
    blocks: 2e-6 of the acceleration at the median, 1e-5 at 99 %."""
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=1e-4, theta=0.5)
    bodies = plummer_bodies(n, seed=n)
    o = orc.Oracle(orc.make_ctx(eps2=1e-4, theta=0.5, timestep=1e-3), *bodies)
    o.gravity()
    st = nb.NBodyState(ctx, None, *bodies, precision="mixed")
    e = np.linalg.norm(st.accelerations() - o.acc, axis=1) / np.linalg.norm(o.acc, axis=1)
    st.close()
    assert np.median(e) <= 2e-6 and np.percentile(e, 99) <= 1e-5
