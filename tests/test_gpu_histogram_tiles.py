"""The histograms' tiles at their edges: dispersions for body counts around a
tile of 1024 and a chunk of 32 tiles, with one bin, few and more bins than
bodies; raw counts where a thread takes eight bodies.  Against the numpy
restatements (the sums differ in association only: 34000 terms of one sign
lose at most ~1e-13 relative, averages near zero ~1e-13 absolute)."""
import numpy as np
import pytest

from milkywayathome_client_amd import histogram as H
from milkywayathome_client_amd import nbody as nb
from oracle import histogram_ref as R

pytestmark = pytest.mark.gpu


def _ring(n, seed):
    rng = np.random.default_rng(seed)
    t = rng.uniform(0, 2 * np.pi, n)
    pos = np.stack([30 * np.cos(t), 30 * np.sin(t), rng.normal(0, 3, n)], 1)
    vel = rng.normal(0, 10, (n, 3))
    vel[rng.random(n) < 0.01] *= 20.0
    return pos, vel, np.full(n, 1e-3)


def _state(bodies):
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=1e-3, theta=0.5)
    return nb.NBodyState(ctx, None, *bodies, prestep=False)


@pytest.mark.parametrize("bins", [(1, 1), (50, 1), (3000, 2)])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 32 * 1024, 33 * 1024 + 5])
def test_dispersions_at_tile_edges(n, bins):
    hp = H.HistogramParams(lambdaBins=bins[0], betaBins=bins[1])
    if bins == (1, 1):
        hp = H.HistogramParams(lambdaBins=1, betaBins=1, lambdaStart=-180.5, lambdaEnd=180.5,
                               betaStart=-90.5, betaEnd=90.5)
    bodies = _ring(n, 100 + n)
    ignore = np.zeros(n, dtype=bool)
    ignore[3::7] = True
    st = _state(bodies)
    st.set_ignore(ignore)
    got = st.histogram_dispersion(hp)
    ref = R.dispersions(bodies[0], bodies[1], hp, ignore=ignore)
    for k in range(1, 8):
        for g, r in zip(got[k], ref[k]):
            np.testing.assert_allclose(g, r, rtol=1e-11, atol=1e-11)
    st.close()


def test_dispersions_with_no_binned_body():
    n = 1500
    st = _state(_ring(n, 3))
    st.set_ignore(np.ones(n, dtype=bool))
    got = st.histogram_dispersion(H.HistogramParams())
    for k in range(1, 8):
        assert np.all(got[k][0] == 0.0)
        assert np.all(got[k][1] == (-1.0 if k >= 3 else 0.0))
    st.close()


@pytest.mark.parametrize("n", [256 * 2048 - 1, 256 * 2048, 256 * 2048 + 1])
def test_counts_at_eight_bodies_a_thread(n):
    hp = H.HistogramParams(lambdaBins=100, betaBins=3)
    bodies = _ring(n, 9)
    ignore = np.arange(n) % 3 == 0
    st = _state(bodies)
    st.set_ignore(ignore)
    counts, totals = st.histogram(hp)
    ref, tot = H.create_histogram(bodies[0], hp, ignore)
    assert totals[0] == tot and counts[0].sum() == tot
    # a body within 1e-9 degrees of a bin's edge may fall either side: none expected, two allowed
    assert np.abs(counts[0] - np.round(ref * tot)).sum() <= 4
    st.close()
