"""The gravity walk where its queues, groups and chunks have edges: particle
counts around a group of targets and a chunk of 64 entries, opening angles
from nearly everything opened (long partial chunks) to wide (short lists), with
and without gas, in both precision forms, against the oracle's force step.

Counts are exact.  FP64: within 1e-10 of each acceleration, as in the parity
tests.  Split form: the walk leaves pairs closer than 2^-8 of the FP32 offset
sum to the FP64 steps, so a pair's offset, rounded to 2^-24 of target and entry,
is off by at most 2^-15 of the distance per component, sqrt(3) 2^-15 in length,
and its force by up to four times that (r^-3 and the direction): 2^-12 of the
sum of the contributions' magnitudes."""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu


def check(ag2, orc, ps, theta, precision, thr=800):
    E, U = ag2.engine, ag2.units
    e0, mih = 0.1 * U.KPC, ag2.ics.mass_in_h(ps)
    with E.Engine(E.make_params(theta=theta, e0=e0, massInH=mih, split_threshold=thr, precision=precision), ps.n) as eng:
        eng.upload(ps)
        eng.init_forces()
        got = eng.download(ps.copy())
        d = eng.diagnostics()
    want = ps.copy()
    scale = np.zeros(ps.n)
    st = orc.force_step(want, orc.params(theta, e0, mih, thr), scale=scale)
    assert d["interactions"] == st["interactions"]
    assert d["sph_pairs"] == st["sph_interactions"]
    if precision == E.AG2_FP64:
        err = vec_rel_err(got.ax, got.ay, got.az, want.ax, want.ay, want.az)
        assert err.max() < 1e-10, err.max()
    else:
        off = np.sqrt((got.ax - want.ax) ** 2 + (got.ay - want.ay) ** 2 + (got.az - want.az) ** 2)
        assert (off <= 2.0 ** -12 * scale).all(), (off / np.where(scale > 0, scale, 1)).max()
    assert np.array_equal(got.h, want.h)
    s = np.abs(want.dUdt).max()
    if s > 0:
        assert np.abs(got.dUdt - want.dUdt).max() / s < 1e-10
    return got, d


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("theta", [0.05, 0.5, 1.2])
@pytest.mark.parametrize("n", [5, 8, 9, 16, 17, 64, 65, 127, 129, 700, 4099])
def test_counts_around_groups_and_chunks(ag2, orc, n, theta, precision):
    nh, nd = n // 2, n // 4
    check(ag2, orc, ag2.ics.disk_galaxy(nh, nd, n - nh - nd, seed=n), theta, precision)


@pytest.mark.parametrize("precision", [0, 1])
def test_gas_free_sphere(ag2, orc, precision):
    check(ag2, orc, ag2.ics.config1_plummer(3001, seed=5), 0.4, precision)


@pytest.mark.parametrize("n,precision", [(32768, 0), (32769, 1), (200000, 1), (200001, 1), (400000, 0), (400001, 0)])
def test_group_size_limits(ag2, orc, n, precision):
    """Either side of the particle counts where the walk's groups change size
    (8, 16, 64 targets)."""
    nh, nd = n // 2, (3 * n) // 10
    check(ag2, orc, ag2.ics.disk_galaxy(nh, nd, n - nh - nd, seed=2), 0.5, precision)


@pytest.mark.parametrize("n", [3000, 33000, 400001])
def test_potential_in_every_group_size(ag2, n):
    """The tree potential with every node opened is the direct sum's: 0.5 sum
    m phi, all terms of one sign, so both are within n 2^-53 of it (each target
    adds its n terms), in groups of 8, 16 and 64 targets."""
    ps = ag2.ics.config1_plummer(n, seed=3)
    E = ag2.engine
    with E.Engine(E.make_params(theta=0.0, e0=0.05 * ag2.units.KPC, massInH=1.0, split_threshold=800), n) as eng:
        eng.upload(ps)
        eng.build_tree()
        tree = eng.energy(with_potential=True)["potential"]
        phi = eng.direct_sum(np.arange(n), with_potential=True)[3]
    want = 0.5 * np.sum(ps.m.astype(np.longdouble) * phi)
    assert abs(tree - want) <= 2 * n * 2.0 ** -53 * abs(want)


@pytest.mark.parametrize("n,precision", [(9000, 0), (60000, 1), (200000, 1)])
def test_long_sph_lists(ag2, orc, n, precision):
    """A small opening angle accepts more SPH candidates than a target's list
    holds (256): they go on in spill chunks, in every group size.  Two
    evaluations are bit-identical, whichever chunk a target got."""
    ps = ag2.ics.disk_galaxy(n // 4, n // 4, n - 2 * (n // 4), seed=8)
    a, da = check(ag2, orc, ps, 0.2, precision)
    b, _ = check(ag2, orc, ps, 0.2, precision)
    assert da["sph_overflow"] > 0
    for f in ("ax", "ay", "az", "dUdt"):
        assert np.array_equal(getattr(a, f), getattr(b, f)), f


@pytest.mark.parametrize("n,power", [(500, 0), (500, 300), (500, -330), (40000, -330)])
def test_fp64_forces_at_any_scale(ag2, orc, n, power):
    """Radii near 2^66, 2^366 (r^2 (r^2 + e^2)^2 of the one-root form
    overflows) and 2^-264 metres (the softening branch is live), with a
    coincident pair."""
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n)
    s = 2.0 ** power
    for a in (ps.x, ps.y, ps.z):
        a *= s
    ps.x[1], ps.y[1], ps.z[1] = ps.x[0], ps.y[0], ps.z[0]   # one coincident pair
    e0 = 0.1 * U.KPC * s
    with E.Engine(E.make_params(theta=0.5, e0=e0, split_threshold=100), n) as eng:
        eng.upload(ps)
        eng.init_forces()
        got = eng.download(ps.copy())
        d = eng.diagnostics()
    want = ps.copy()
    st = orc.force_step(want, orc.params(0.5, e0, 1.0, 100))
    assert d["interactions"] == st["interactions"]
    unit = max(np.abs(getattr(want, f)).max() for f in ("ax", "ay", "az"))
    assert 0 < unit < np.inf
    err = vec_rel_err(*[getattr(p, f) / unit for p in (got, want) for f in ("ax", "ay", "az")])
    assert err.max() < 1e-10
