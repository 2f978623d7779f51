"""The direct sum far from the scales of a galaxy.

One particle far away (2^200, 2^400, 2^600 metres; r^2 itself overflows from
2^512 on), whole sets at radii near 2^366 and 2^-264 metres, and a pair 1e-150
metres apart: against the same sums in extended precision, within (n + 16) 2^-53
of the sum of the terms' magnitudes (each term carries a few roundings, the sum
of n terms at most n)."""
import numpy as np
import pytest

from test_gpu_direct import reference

pytestmark = pytest.mark.gpu


def sums(ag2, ps, tg, e0):
    E = ag2.engine
    with E.Engine(E.make_params(theta=0.5, e0=e0, massInH=1.0), ps.n) as eng:
        eng.upload(ps)
        return eng.direct_sum(tg, with_potential=True), eng.direct_sum(tg)


def check(ag2, ps, tg, e0):
    with_pot, without = sums(ag2, ps, tg, e0)
    want, mag = reference(ps, tg, e0, ag2.units.G)
    tol = (ps.n + 16) * 2.0 ** -53
    for got in (with_pot, without):
        for c in range(3):
            assert (np.abs(got[c] - want[c]) <= tol * mag[0]).all(), c
    assert (np.abs(with_pot[3] - want[3]) <= tol * mag[1]).all()


@pytest.mark.parametrize("power", [150, 200, 400, 600])
def test_one_particle_far_away(ag2, power):
    ps = ag2.ics.config1_plummer(1500, seed=4)
    ps.y[700] = 2.0 ** power
    # (r^2 of the far particle's own pairs overflows past 2^512)
    check(ag2, ps, np.arange(0 if power < 512 else 1, 1500, 7), 0.05 * ag2.units.KPC)


@pytest.mark.parametrize("power", [300, -330])
def test_sets_at_any_scale(ag2, power):
    ps = ag2.ics.config1_plummer(1500, seed=4)
    s = 2.0 ** power
    for a in (ps.x, ps.y, ps.z):
        a *= s
    ps.x[1], ps.y[1], ps.z[1] = ps.x[0], ps.y[0], ps.z[0]
    check(ag2, ps, np.arange(0, 1500, 7), 0.05 * ag2.units.KPC * s)


@pytest.mark.parametrize("e0", [1e-3, 1.0, 1e18])
def test_a_pair_hardly_apart(ag2, e0):
    """Coordinates within a few e0 of the origin, two of them 1e-150 apart."""
    ps = ag2.ics.config1_plummer(300, seed=6)
    unit = np.abs(ps.x).max()
    for a in (ps.x, ps.y, ps.z):
        a *= 3.0 * e0 / unit
    for k, d in ((10, 0.0), (11, 1e-150)):
        ps.x[k], ps.y[k], ps.z[k] = d, -d, d
    check(ag2, ps, np.arange(300), e0)
