"""The direct sum where its launch changes shape: one source, source counts
around its block of 256, target counts around a wave, a context too small for
all parts at once (many targets, few particles), repeated targets; and pairs
on every branch of the potential's angle: at r == 0, far inside, around and far
outside the softening length.

Against the same sums in extended precision.  Each term carries a few roundings
and a sum of n terms at most n: within (n + 16) 2^-53 of the sum of the terms'
magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(ps, tg, e0, G):
    L = np.longdouble
    x, y, z, m = (getattr(ps, f).astype(L) for f in ("x", "y", "z", "m"))
    e = L(e0)
    out, mag = np.zeros((4, len(tg)), L), np.zeros((2, len(tg)), L)
    for k, i in enumerate(tg):
        dx, dy, dz = x - x[i], y - y[i], z - z[i]
        r2 = dx * dx + dy * dy + dz * dz
        on = r2 != 0
        r = np.sqrt(r2[on])
        f = L(G) * m[on] / ((r2[on] + e * e) * r)
        ph = -(L(G) * m[on] / e) * np.arctan2(e, r)
        out[:, k] = (f * dx[on]).sum(), (f * dy[on]).sum(), (f * dz[on]).sum(), ph.sum()
        mag[:, k] = (f * r).sum(), -ph.sum()
    return out, mag


@pytest.mark.parametrize("e_scale", [1e-3, 1.0, 30.0])
@pytest.mark.parametrize("n,nt", [(1, 1), (1, 40), (2, 7), (255, 63), (256, 64), (257, 65), (1500, 300), (70, 3000)])
def test_direct_sum_shapes(ag2, n, nt, e_scale):
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.config1_plummer(n, seed=n)
    if n > 100:   # two particles at one position, one a hair away
        ps.x[11], ps.y[11], ps.z[11] = ps.x[7], ps.y[7], ps.z[7]
        ps.x[13], ps.y[13], ps.z[13] = ps.x[7] * (1 + 1e-12), ps.y[7], ps.z[7]
    tg = np.random.default_rng(nt).integers(0, n, nt).astype(np.int64)
    e0 = e_scale * U.KPC
    with E.Engine(E.make_params(theta=0.5, e0=e0, massInH=1.0), n) as eng:
        eng.upload(ps)
        with_pot = eng.direct_sum(tg, with_potential=True)
        without = eng.direct_sum(tg)
    want, mag = reference(ps, tg, e0, U.G)
    tol = (n + 16) * 2.0 ** -53
    for got in (with_pot, without):
        for c in range(3):
            assert (np.abs(got[c] - want[c]) <= tol * mag[0]).all(), c
    assert (np.abs(with_pot[3] - want[3]) <= tol * mag[1]).all()
