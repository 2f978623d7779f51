"""The pool's memory budget and the SPH spill chunks of small opening angles:
they are taken where the budget has room, refuse no job, balance when they go,
and a job's result does not depend on the size of the context it got."""
import numpy as np
import pytest

from test_gpu_serving import close, solo

pytestmark = pytest.mark.gpu


def job(ag2, n, theta, k=64, seed=1):
    U = ag2.units
    ps = ag2.ics.disk_galaxy(n // 4, n // 4, n - 2 * (n // 4), seed=seed)
    dt = 2e-4 * U.MYR
    prm = ag2.engine.make_params(theta=theta, e0=0.1 * U.KPC, massInH=ag2.ics.mass_in_h(ps, k), split_threshold=800,
                                 precision=ag2.engine.AG2_FP32_SPLIT, min_dt=dt, max_dt=dt)
    return ps, prm


def run(ag2, pool, jobs, steps=2):
    ids = [pool.submit(prm, ps, steps) for ps, prm in jobs]
    used = []
    while any(pool.status(i)[0] != ag2.engine.JOB_DONE for i in ids):
        pool.step()
        used.append(pool.stats()["hbm_used"])
    return [pool.result(i, ag2.ics.ParticleSet(ps.n)) for i, (ps, _) in zip(ids, jobs)], used


def context_bytes(ag2, ps):
    return ag2.engine.load_library().ag2_context_bytes(ps.n, int((ps.type == 2).sum()))


def test_a_job_of_the_budgets_size_is_taken_at_any_angle(ag2):
    """Without room for chunks its long lists are left to the overflow walk."""
    ps, prm = job(ag2, 20000, 0.15)
    budget = context_bytes(ag2, ps)
    with ag2.engine.Pool(max_jobs=2, hbm_budget=budget) as pool:
        (got,), used = run(ag2, pool, [(ps, prm)])
    assert max(used) <= budget
    assert close(got, solo(ag2, ps, prm, 2)) is None


def test_what_is_used_balances(ag2):
    """One context serves jobs of any angle one after another: what is used does
    not grow after the smallest angle, and stays within the budget."""
    with ag2.engine.Pool(max_jobs=1, hbm_budget=1 << 30) as pool:
        last = []
        for theta in (0.5, 0.15, 0.5, 0.2, 0.15, 0.7, 0.15):
            _, used = run(ag2, pool, [job(ag2, 16000, theta)], 1)
            last.append(used[-1])
    assert last[0] < last[1] and set(last[1:]) == {last[1]}
    assert last[1] <= 1 << 30


def test_chunks_run_out_for_the_set_alone(ag2):
    """A set with more long lists than the chunks provided for its gas, but
    fewer than those of the larger context a pool gives it: the lists go to the
    overflow walk in both, so the results are the same bit for bit."""
    E = ag2.engine
    n, theta = 10000, 0.3
    ng = n - 2 * (n // 4)
    per = 1.5 * 75.0 * (0.5 / theta) ** 1.75 / 256 - 0.75   # provided per gas particle
    own, classed = per * ng + 64, per * 8192 + 64
    for k in range(64, 400, 8):   # gas masses in a group: longer supports, longer lists
        ps, prm = job(ag2, n, theta, k)
        with E.Engine(prm, n) as eng:
            eng.upload(ps)
            eng.init_forces()
            over = eng.diagnostics()["sph_overflow"]
        if own * 1.05 < over < classed * 0.95:
            break
    else:
        pytest.fail("no support gives lists between %d and %d" % (own, classed))
    with E.Pool(max_jobs=1) as pool:
        (got,), _ = run(ag2, pool, [(ps, prm)])
    want = solo(ag2, ps, prm, 2)
    for f in ("x", "vx", "ax", "ay", "az", "U", "dUdt"):
        assert np.array_equal(getattr(got, f), getattr(want, f)), f
