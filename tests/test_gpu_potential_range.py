"""The tree potential with one particle far beyond all others."""
import numpy as np
import pytest

from test_gpu_direct import reference

pytestmark = pytest.mark.gpu


def potential(ag2, ps, theta, e0):
    E = ag2.engine
    with E.Engine(E.make_params(theta=theta, e0=e0, massInH=1.0, split_threshold=100), ps.n) as eng:
        eng.upload(ps)
        eng.build_tree()
        return eng.energy(with_potential=True)["potential"]


def test_potential_with_a_particle_far_away(ag2):
    """Every node opened: 0.5 sum m phi of the direct sum, the far particle's
    share in it included, to the rounding of n terms."""
    n, e0 = 1500, 0.05 * ag2.units.KPC
    ps = ag2.ics.config1_plummer(n, seed=4)
    ps.y[700] = 2.0 ** 400
    want, _ = reference(ps, np.arange(n), e0, ag2.units.G)
    want = 0.5 * np.sum(ps.m.astype(np.longdouble) * want[3])
    assert abs(potential(ag2, ps, 0.0, e0) - want) <= 2 * n * 2.0 ** -53 * abs(want)


def test_potential_past_the_squares_range(ag2):
    """A particle so far away that r^2 overflows leaves nothing in the root cube
    (the mean of |x|^2 is not finite): every target meets the root alone, at
    2^600 / n metres, and the potential is finite and nearly nothing."""
    n, e0 = 1500, 0.05 * ag2.units.KPC
    ps = ag2.ics.config1_plummer(n, seed=4)
    ps.y[700] = 2.0 ** 600
    got = potential(ag2, ps, 0.5, e0)
    assert abs(got) <= ag2.units.G * ps.m.sum() ** 2 / 2.0 ** 580
