"""What rounding the gravity walk adds: small sets with every node opened
against the FP64 direct sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_near_pairs_and_a_wide_group(ag2):
    """Eight targets on a line of length R, two of them too close for FP32
    offsets from the group's centre, and eight sources a sixtieth of R beyond
    the line's end.  A group that has met such a pair carries the offsets'
    remainders from then on: what is left is the FP32 arithmetic of a pair,
    eight roundings of 2^-24 (offsets alone would be 2^-25 of R, up to thirty
    times as much at the line's end)."""
    E, U = ag2.engine, ag2.units
    R = 1e21
    worst = 0.0
    for seed in range(40):
        g = np.random.default_rng(seed)
        ps = ag2.ics.ParticleSet(16)
        x = np.concatenate([[-1.0, -0.8, -0.62, -0.45, -0.45 + 1e-5, -0.3, -0.13, -0.002], g.uniform(0.0165, 0.03, 8)])
        ps.x[:] = R * x * (1 + 1e-3 * g.uniform(size=16))
        ps.x[0] = -R
        ps.y[:8], ps.z[:8] = -1e-5 * R * g.uniform(size=8), -1e-5 * R * g.uniform(size=8)
        ps.y[8:], ps.z[8:] = 4e-3 * R * g.uniform(size=8), 4e-3 * R * g.uniform(size=8)
        ps.m[:8], ps.m[8:] = 1e36, 1e38
        with E.Engine(E.make_params(theta=0.0, e0=1e-5 * R, split_threshold=800, precision=E.AG2_FP32_SPLIT), 16) as eng:
            eng.upload(ps)
            eng.init_forces()
            got = eng.download(ag2.ics.ParticleSet(16), ("ax", "ay", "az"))
            order = eng.order()[0]
            want = eng.direct_sum(np.arange(16))
        assert sorted(order[:8]) == list(range(8))   # the line is one group
        last = 7   # the target at the line's end
        off = [getattr(got, f)[last] - want[c][last] for c, f in enumerate(("ax", "ay", "az"))]
        worst = max(worst, np.sqrt(np.sum(np.square(off)) / np.sum(np.square([w[last] for w in want[:3]]))))
    assert worst <= 8 * 2.0 ** -24, worst
