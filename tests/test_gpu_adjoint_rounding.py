"""Rounding of the list adjoint's interaction: two massive bodies and massless
ones far away, each of which accepts one cell that holds the two, so that
its gradient is one interaction's.  The powers of the distance are rounded as
IEEE square roots and quotients round them, in the streaming adjoint's order:
the same bits as that expression in numpy (tolerance zero)."""
import numpy as np
import pytest

from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu


def _interaction(d, M, Q, g, eps2, quad):
    """The streaming adjoint's expressions for d = node - body."""
    dx, dy, dz = d.T
    g0, g1, g2 = g.T
    s2 = (dz * dz + (dy * dy + dx * dx)) + eps2
    s3 = (1.0 / np.sqrt(s2)) / s2
    s5 = s3 / s2
    dg = dx * g0 + dy * g1 + dz * g2
    cg = M * s3
    cd = -3.0 * M * s5 * dg
    if not quad:
        return np.stack([cg * g0 + cd * dx, cg * g1 + cd * dy, cg * g2 + cd * dz], 1)
    qxx, qxy, qxz, qyy, qyz, qzz = Q
    ux = qxx * dx + qxy * dy + qxz * dz
    uy = qxy * dx + qyy * dy + qyz * dz
    uz = qxz * dx + qyz * dy + qzz * dz
    wx = qxx * g0 + qxy * g1 + qxz * g2
    wy = qxy * g0 + qyy * g1 + qyz * g2
    wz = qxz * g0 + qyz * g1 + qzz * g2
    dQd = ux * dx + uy * dy + uz * dz
    ug = ux * g0 + uy * g1 + uz * g2
    s7 = s5 / s2
    s9 = s7 / s2
    cg = cg + 2.5 * dQd * s7
    cd = cd + (-17.5 * dQd * s9 * dg + 5.0 * s7 * ug)
    cu = 5.0 * s7 * dg
    return np.stack([cg * g0 + cd * dx + cu * ux - s5 * wx,
                     cg * g1 + cd * dy + cu * uy - s5 * wy,
                     cg * g2 + cd * dz + cu * uz - s5 * wz], 1)


@pytest.mark.parametrize("quad", [True, False])
@pytest.mark.parametrize("eps2", [1e-4, 0.3])
@pytest.mark.parametrize("count", [200, 20000])
def test_one_interaction_each(count, eps2, quad):
    rng = np.random.default_rng(3)
    pair = np.array([[0.3, 0.2, -0.1], [0.31, 0.22, -0.13]])
    u = rng.normal(size=(count, 3))
    far = u / np.linalg.norm(u, axis=1)[:, None] * rng.uniform(20.0, 60.0, (count, 1))
    pos = np.concatenate([pair, far])
    m = np.concatenate([[1.3, 0.7], np.zeros(count)])
    ctx = nb.NBodyCtx.create(timestep=1e-3, timeEvolve=1.0, eps2=eps2, theta=1.0, useQuad=quad,
                             treeRSize=4.0, allowIncest=True)
    st = nb.NBodyState(ctx, None, pos, np.zeros_like(pos), m)
    g = np.concatenate([np.zeros((2, 3)), rng.normal(size=(count, 3))])
    gx, _ = st.gravity_vjp(g)
    t = st.tree()
    st.close()
    want = np.full((count, 3), np.nan)
    left = np.ones(count, bool)
    for q in np.flatnonzero(t["kind"] == 0):          # the chain of cells, root first
        d = t["pos"][q] - far
        sq = d[:, 2] * d[:, 2] + (d[:, 1] * d[:, 1] + d[:, 0] * d[:, 0])
        take = left & (sq >= t["rcrit2"][q])
        want[take] = -_interaction(d[take], t["mass"][q], t["quad"][q], g[2:][take], eps2, quad)
        left &= ~take
    assert not left.any()
    assert np.array_equal(gx[2:], want)
