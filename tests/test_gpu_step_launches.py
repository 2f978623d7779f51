"""What a step does in its neighbours' launches (the tree width's sums in the
drift, the walk's counters in the second kick, the group count of a gas-free
set in the node kernel) against the same phases run by themselves, and the state's
move into key order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SAME = ("R", "n_in_tree", "n_nodes", "max_level", "interactions", "walk_entries", "walk_tests", "sph_pairs")


@pytest.mark.parametrize("gas", [0, 1])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 131072, 131073])
def test_step_equals_phases(ag2, n, gas):
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n)
    if gas:
        ps.type[::3] = U.TYPE_GAS
        ps.U[::3] = U.u_from_temperature(1e4)
        ps.init_temperature()
    dt = 0.1 * U.MYR
    prm = E.make_params(theta=0.7, e0=0.05 * U.KPC, massInH=48 * ps.m[0], split_threshold=800, min_dt=dt, max_dt=dt)
    with E.Engine(prm, n) as eng:
        eng.upload(ps)
        eng.init_forces()
        for _ in range(2):
            eng.step()
        a = eng.diagnostics()
        eng.build_tree()   # the second kick left the positions as they were
        eng.gas_density()
        eng.forces()
        b = eng.diagnostics()
    assert {k: a[k] for k in SAME} == {k: b[k] for k in SAME}
    assert (a["interactions"] > 0) == (n > 1)


@pytest.mark.parametrize("n", [1, 257, 131072, 131073])
def test_build_moves_whole_state(ag2, n):
    """The state goes into key order and comes back unchanged."""
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.shuffled(ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n), n)
    g = np.random.default_rng(n)
    ps.type[:] = g.integers(1, 4, n)
    for f in E.Engine.ALL:
        a = getattr(ps, f)
        if f not in ("x", "y", "z", "m", "type") and a.dtype == np.float64:
            a[:] = g.normal(size=n)
    with E.Engine(E.make_params(theta=0.7, e0=0.05 * U.KPC, split_threshold=800), n) as eng:
        eng.upload(ps)
        before = eng.download(ps.copy())
        eng.build_tree()
        after = eng.download(ps.copy())
    for f in E.Engine.ALL:
        assert np.array_equal(getattr(before, f), getattr(after, f)), f
