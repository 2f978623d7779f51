"""Upload and download of the particle state where a transfer changes its
shape: single copies, blocks just past one pinned piece (4 MiB), several
pieces, more pieces than the ring holds and host helpers; whole and partial
field lists.  Values come back bit for bit in caller order, before and after a
tree build has put the device's state in key order, and fields left out of an
upload take their defaults."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INPUTS = ("x", "y", "z", "vx", "vy", "vz", "m", "U", "mu", "type")


def random_state(ag2, n):
    g = np.random.default_rng(n)
    ps = ag2.ics.ParticleSet(n)
    for f in ag2.engine.Engine.ALL:
        if f == "type":
            ps.type[:] = g.integers(1, 4, n)
        else:
            getattr(ps, f)[:] = g.normal(size=n)
    ps.m[:] = np.abs(ps.m) + 1.0
    return ps


@pytest.mark.parametrize("n", [1, 3, 1000, 30615, 30616, 52428, 61231, 262145, 650001])
def test_round_trip(ag2, n):
    E = ag2.engine
    ps = random_state(ag2, n)
    with E.Engine(E.make_params(theta=0.5, e0=1.0e20), n) as eng:
        eng.upload(ps)
        for built in (False, True):
            got = eng.download(ag2.ics.ParticleSet(n))
            for f in E.Engine.ALL:
                assert np.array_equal(getattr(got, f), getattr(ps, f)), (f, built)
            part = ag2.ics.ParticleSet(n)
            eng.download(part, ("y", "type"))
            assert np.array_equal(part.y, ps.y) and np.array_equal(part.type, ps.type)
            only = ag2.ics.ParticleSet(n)
            only.type[:] = 9
            eng.download(only, ("type",))
            assert np.array_equal(only.type, ps.type)
            eng.build_tree()
        eng.upload(ps, ("x", "y", "z", "m"))
        got = eng.download(ag2.ics.ParticleSet(n))
        for f in E.Engine.ALL:
            want = getattr(ps, f) if f in ("x", "y", "z", "m") else \
                np.full(n, 0.58) if f == "mu" else np.ones(n, np.uint8) if f == "type" else np.zeros(n)
            assert np.array_equal(getattr(got, f), want), f
