"""The sampler's radii against a scalar restatement of the rejection: body i's
radius is its first accepted trial, trial t drawing Philox block t of the
body's stream, however the trials are dealt out over a wave.  Sizes around a
wave's end; both acceptance rates (a Plummer sphere cut at 50 radii accepts
one trial in 140, an NFW halo one in three)."""
import numpy as np
import pytest

from milkywayathome_client_amd import nbody as nb

pytestmark = pytest.mark.gpu

SEED = 0x1234567890


def _first_radius(body, bound, dens, peak):
    key = (SEED & 0xFFFFFFFF, SEED >> 32)
    for t in range(1 << 16):
        o = nb.philox4x32_10((body, t, 0, 0x64776172), key)
        u = [((((o[2 * k] << 32) | o[2 * k + 1]) >> 11) + 0.5) * 2.0 ** -53 for k in (0, 1)]
        r = u[0] * bound
        if r > 0.0 and r * r * dens(r) / peak > u[1]:
            return r
    raise AssertionError("no radius")


@pytest.mark.parametrize("comp", ["light", "dark"])
@pytest.mark.parametrize("n", [4, 63, 64, 65, 257])
def test_radii_are_the_first_accepted_trials(comp, n):
    if comp == "light":
        a, bound = 0.2, 50.0 * (0.2 + 0.8)
        dens = lambda r: (1.0 + (r / a) ** 2) ** -2.5                     # noqa: E731
        peak = (2.0 / 3.0) * a * a * dens(np.sqrt(2.0 / 3.0) * a)
    else:
        a, bound = 0.8, 5.0 * np.cbrt(60.0 / 0.568910904587397184785763397846734505)
        dens = lambda r: 1.0 / ((r / a) * (1.0 + r / a) ** 2)             # noqa: E731
        peak = a * a * dens(a)
    pos, _, _, _, _ = nb.mixed_dwarf(n, n if comp == "light" else 0, seed=SEED)
    r = np.array([_first_radius(i, bound, dens, peak) for i in range(n)])
    # the bodies are shifted by their centre of mass c: |pos + c| = r; the differences of the
    # squares are linear in c, and the radii themselves then check it (the first one is spare)
    sq = (pos ** 2).sum(1)
    c = np.linalg.lstsq(2.0 * (pos[1:] - pos[0]), (r[1:] ** 2 - r[0] ** 2) - (sq[1:] - sq[0]),
                        rcond=None)[0]
    np.testing.assert_allclose(np.linalg.norm(pos + c, axis=1), r, rtol=0, atol=1e-9)
