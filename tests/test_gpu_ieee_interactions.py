"""One FP64 interaction a body, against numpy's IEEE square roots and
divisions, bit for bit: the interactions take their root and quotients from
one reciprocal square root, and must round as those operators do.  Two massive
bodies, and massless ones that accept a cell holding both (monopole and
quadrupole) or, in the direct sum, meet one massive body; at sizes, masses and
softenings from one end of the range without scaling to the other.  3.2
million square roots, 7.4 million quotients and a million reciprocals of the
fifth power.  (A divisor whose significand is all ones may round differently:
one in 2^52, none here.)"""
import numpy as np
import pytest

from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu

# log2 of the size, log2 of the masses, softening^2
RANGE = [(0, 0, 1e-4), (3, -4, 1e-8), (0, -300, 1e-4), (0, 299, 1e-4), (80, 0, 2.0 ** 100),
         (-45, 0, 2.0 ** -200), (-10, 250, 2.0 ** -199), (60, -280, 2.0 ** 199), (84, 290, 1.0),
         (-44, -295, 2.0 ** -150)]
# cells this small are a structure error, direct sums are not
SMALL = [(-80, 0, 2.0 ** -200), (-90, -295, 1e-50)]
COUNT = 100000


def _far(rng, scale):
    u = rng.normal(size=(COUNT, 3))
    r = rng.uniform(1.0, 8.0, (COUNT, 1)) * 2.0 ** scale
    return u / np.linalg.norm(u, axis=1)[:, None] * r


def _run(pos, m, eps2, scale, **kw):
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, treeRSize=2.0 ** (scale + 3),
                             allowIncest=True, **kw)
    st = nb.NBodyState(ctx, None, pos, np.zeros_like(pos), m)
    a = st.accelerations()
    t = st.tree() if kw.get("theta") else None
    st.close()
    return a, t


@pytest.mark.parametrize("scale,mass,eps2", RANGE + SMALL)
def test_one_body(scale, mass, eps2):
    rng = np.random.default_rng(scale + 1000)
    far = _far(rng, scale)
    pos = np.concatenate([[[0.25 * 2.0 ** scale] * 3], far])
    m = np.concatenate([[1.37 * 2.0 ** mass], np.zeros(COUNT)])
    a, _ = _run(pos, m, eps2, scale, criterion="exact")
    d = pos[0] - far
    r2 = d[:, 2] * d[:, 2] + (d[:, 1] * d[:, 1] + d[:, 0] * d[:, 0]) + eps2
    assert np.array_equal(a[1:], ((m[0] / np.sqrt(r2)) / r2)[:, None] * d)


@pytest.mark.parametrize("quad", [True, False])
@pytest.mark.parametrize("scale,mass,eps2", RANGE)
def test_one_cell(scale, mass, eps2, quad):
    rng = np.random.default_rng(scale + 2000)
    far = _far(rng, scale)
    pair = np.array([[0.30, 0.20, -0.10], [0.32, 0.25, -0.17]]) * 2.0 ** scale
    pos = np.concatenate([pair, far])
    m = np.concatenate([np.array([1.3, 0.7]) * 2.0 ** mass, np.zeros(COUNT)])
    a, t = _run(pos, m, eps2, scale, theta=1.0, useQuad=quad)
    want = np.full((COUNT, 3), np.nan)
    left = np.ones(COUNT, bool)
    for q in np.flatnonzero(t["kind"] == 0):          # the chain of cells, root first
        d = t["pos"][q] - far
        sq = d[:, 2] * d[:, 2] + (d[:, 1] * d[:, 1] + d[:, 0] * d[:, 0])
        take = left & (sq >= t["rcrit2"][q])
        left &= ~take
        d, r2 = d[take], sq[take] + eps2
        r = np.sqrt(r2)
        w = ((t["mass"][q] / r) / r2)[:, None] * d
        if quad:
            xx, xy, xz, yy, yz, zz = t["quad"][q]
            x, y, z = d.T
            v = np.stack([xx * x + xy * y + xz * z, xy * x + yy * y + yz * z,
                          xz * x + yz * y + zz * z], 1)
            dqd = v[:, 0] * x + v[:, 1] * y + v[:, 2] * z
            d5 = 1.0 / ((r2 * r2) * r)
            w = w + ((2.5 * (d5 * dqd)) / r2)[:, None] * d
            w = w - d5[:, None] * v
        want[take] = w
    assert left.sum() < COUNT // 4                    # the others open every cell
    left = ~left
    assert np.array_equal(a[2:][left], want[left])
