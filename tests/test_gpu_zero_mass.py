"""Particles of mass zero are skipped as targets (Node.cpp:249-257): their
acceleration is exactly zero, whatever group of targets they share, in both
precision forms, every group size of the walk (8, 16 and 64 targets), with and
without gas, inside their group's box and far outside it, and in a batched walk.

The other targets match the oracle: counts exactly, FP64 within 1e-10, the split
form within 2^-12 of the sum of the contributions' magnitudes (pairs closer than
2^-8 of the FP32 offset sum are left to the FP64 steps, so a pair's offset is off
by at most sqrt(3) 2^-15 of the distance and its force by four times that)."""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu


def particles(ag2, n, gas):
    if gas:
        ps = ag2.ics.disk_galaxy(n // 2, n // 4, n - n // 2 - n // 4, seed=n)
    else:
        ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n)
    # (gas keeps its mass: the density of massless gas is a matter of its own)
    ps.m[::11] = np.where(ps.type[::11] == ag2.units.TYPE_GAS, ps.m[::11], 0.0)
    # some of them where a massive particle is, some far from all others
    ps.x[22:220:22], ps.y[22:220:22], ps.z[22:220:22] = ps.x[23:221:22], ps.y[23:221:22], ps.z[23:221:22]
    ps.x[231:331:11] *= 3.0
    assert (ps.m == 0).sum() > n // 20
    return ps


def params(ag2, ps, precision, **more):
    U = ag2.units
    return ag2.engine.make_params(theta=0.5, e0=0.1 * U.KPC, massInH=ag2.ics.mass_in_h(ps), split_threshold=800,
                                  precision=precision, **more)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,gas", [(1500, False), (1500, True), (33000, True), (410001, False), (410001, True)])
def test_massless_targets(ag2, orc, n, gas, precision):
    E, U = ag2.engine, ag2.units
    ps = particles(ag2, n, gas)
    with E.Engine(params(ag2, ps, precision), n) as eng:
        eng.upload(ps)
        eng.init_forces()
        got = eng.download(ps.copy())
        d = eng.diagnostics()
    none = ps.m == 0
    for f in ("ax", "ay", "az"):
        assert not getattr(got, f)[none].any(), f
    want, scale = ps.copy(), np.zeros(n)
    st = orc.force_step(want, orc.params(0.5, 0.1 * U.KPC, ag2.ics.mass_in_h(ps), 800), scale=scale)
    assert d["interactions"] == st["interactions"]
    assert d["sph_pairs"] == st["sph_interactions"]
    if precision == E.AG2_FP64:
        assert vec_rel_err(got.ax, got.ay, got.az, want.ax, want.ay, want.az).max() < 1e-10
    else:
        off = np.sqrt((got.ax - want.ax) ** 2 + (got.ay - want.ay) ** 2 + (got.az - want.az) ** 2)
        assert (off <= 2.0 ** -12 * scale).all(), (off / np.where(scale > 0, scale, 1)).max()


def test_massless_targets_in_a_batched_walk(ag2):
    """Massless particles feel no force: in a pool they drift with their first
    velocity, as on an engine of their own."""
    E, U = ag2.engine, ag2.units
    dt, steps = 0.01 * U.MYR, 3
    with E.Pool(max_jobs=4) as pool:
        jobs = []
        for n, gas in ((1500, True), (20000, False), (40000, True)):
            ps = particles(ag2, n, gas)
            jobs.append((pool.submit(params(ag2, ps, E.AG2_FP32_SPLIT, min_dt=dt, max_dt=dt), ps, steps), ps))
        while any(pool.status(j)[0] != E.JOB_DONE for j, _ in jobs):
            pool.step()
        for j, ps in jobs:
            got = pool.result(j, ag2.ics.ParticleSet(ps.n))
            none = ps.m == 0
            for a, v in (("ax", "vx"), ("ay", "vy"), ("az", "vz")):
                assert not getattr(got, a)[none].any()
                assert np.array_equal(getattr(got, v)[none], getattr(ps, v)[none])
