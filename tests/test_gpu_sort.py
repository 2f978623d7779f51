"""The key sort either side of the particle counts where it changes (one launch
pair over tiles of 2048 and 4096 keys, radix passes), on the first build after
an upload (caller order) and on builds after steps (nearly sorted): particles
stand in the order of their octant paths, coincident ones by caller index."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def octants(x, y, z, R, first, last):
    """Octant digits of levels first .. last by the reference's descent."""
    c, r, out = [0.0, 0.0, 0.0], R, []
    for level in range(1, last + 1):
        up = [x > c[0], y > c[1], z > c[2]]
        if level >= first:
            out.append(up[0] + 2 * up[1] + 4 * up[2])
        c = [c[k] + r * (0.5 if up[k] else -0.5) for k in range(3)]
        r /= 2
    return tuple(out)


def check_order(ag2, eng, n):
    perm, hi, lo = eng.order()
    assert len(perm) <= n and len(np.unique(perm)) == len(perm)
    now = eng.download(ag2.ics.ParticleSet(n))
    R = eng.diagnostics()["R"]
    same = (hi[1:] == hi[:-1]) & (lo[1:] == lo[:-1])
    assert (same | (hi[1:] > hi[:-1]) | ((hi[1:] == hi[:-1]) & (lo[1:] > lo[:-1]))).all()
    # particles that share all 42 levels: the deeper levels, then the caller index
    for k in np.flatnonzero(same):
        a, b = int(perm[k]), int(perm[k + 1])
        ka = octants(now.x[a], now.y[a], now.z[a], R, 43, 126) + (a,)
        kb = octants(now.x[b], now.y[b], now.z[b], R, 43, 126) + (b,)
        assert ka < kb


@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 4097, 16385, 39999, 40000, 40001, 45057, 80000, 80001, 131073])
def test_order(ag2, n):
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.shuffled(ag2.ics.hernquist(n, seed=n), n)
    if n > 4000:   # runs sharing the sorted bytes, and one position twice
        ps.x[3:20], ps.y[3:20], ps.z[3:20] = ps.x[2] * (1 + 1e-13 * np.arange(17)), ps.y[2], ps.z[2]
        ps.x[2100], ps.y[2100], ps.z[2100] = ps.x[5], ps.y[5], ps.z[5]
    dt = 2.0 * U.MYR
    with E.Engine(E.make_params(theta=0.7, e0=0.05 * U.KPC, split_threshold=800, min_dt=dt, max_dt=dt), n) as eng:
        eng.upload(ps)
        eng.build_tree()
        check_order(ag2, eng, n)
        eng.init_forces()
        for _ in range(3):
            eng.step()
            check_order(ag2, eng, n)
