"""The key sort either side of the particle counts where it changes (merge sort
over tiles of 1024, 2048 and 4096 keys, sample sort, radix passes), on the first
build after an upload (caller order) and on builds after steps (nearly sorted): particles
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


@pytest.mark.parametrize("n", [1024, 1025, 16384, 16385, 59999, 60000, 60001, 262144, 262145, 524288, 524289, 1048576, 1048577, 2097152, 2097153])
def test_order_at_limits(ag2, n):
    """Either side of the merge sort's tiles, the sample sort's range and its
    steps."""
    E = ag2.engine
    ps = ag2.ics.shuffled(ag2.ics.hernquist(n, seed=n), n)
    with E.Engine(E.make_params(theta=0.7, e0=0.05 * ag2.units.KPC, split_threshold=800), n) as eng:
        for order in (slice(None), slice(None, None, -1)):
            for a in (ps.x, ps.y, ps.z):
                a[:] = a[order].copy()
            eng.upload(ps)
            eng.build_tree()
            check_order(ag2, eng, n)


def test_order_overfull_bucket(ag2):
    """128 tiles of 2048 particles on a line, each with 15 particles between
    two of its samples in one and the same stretch: more than a bucket holds."""
    E, tiles, tile, step = ag2.engine, 128, 2048, 16
    n = tiles * tile
    ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=3)
    g = np.random.default_rng(7)
    for t in range(tiles):
        first = int(f"{t % step:04b}"[::-1], 2) + 1024   # this tile's sample below the stretch
        x = np.concatenate([g.uniform(0.1, 0.5, first + 1), g.uniform(0.5, 0.5001, step - 1),
                            g.uniform(0.5001, 0.9, tile - first - step)])
        ps.x[t * tile:(t + 1) * tile] = g.permutation(x) * ag2.units.KPC
    ps.y[:] = ps.z[:] = 0.3 * ag2.units.KPC
    with E.Engine(E.make_params(theta=0.7, e0=0.05 * ag2.units.KPC, split_threshold=800), n) as eng:
        eng.upload(ps)
        eng.build_tree()
        check_order(ag2, eng, n)
        perm = eng.order()[0]
        assert (np.diff(ps.x[perm]) >= 0).all() and len(perm) == n


def test_batch_with_large_job(ag2):
    """A serving round whose largest job is past the merge sort's range."""
    from test_gpu_serving import close, run_pool, solo
    dt = 0.1 * ag2.units.MYR
    prm = ag2.engine.make_params(theta=0.7, e0=0.05 * ag2.units.KPC, split_threshold=800, min_dt=dt, max_dt=dt)
    jobs = [(ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n), prm, 2) for n in (2, 63, 2049, 60001, 130000)]
    res, _ = run_pool(ag2, jobs, max_jobs=8)
    assert len(res) == len(jobs)
    for i, (ps, prm, steps) in enumerate(jobs):
        assert close(res[i], solo(ag2, ps, prm, steps)) is None, i
