"""What a target's direct sum depends on: the sources alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 5000, 33333])
def test_a_target_alone_and_among_others(ag2, n):
    """A target's sum is the same bit for bit in any list: alone, among few,
    among many, in another order, and through the path without allocation."""
    E = ag2.engine
    ps = ag2.ics.config1_plummer(n, seed=n)
    e0 = 0.3 * ag2.units.KPC
    every = np.arange(n)
    with E.Engine(E.make_params(theta=0.5, e0=e0, massInH=1.0), n) as eng:
        eng.upload(ps)
        for pot in (False, True):
            cols = slice(0, 4 if pot else 3)
            whole = np.array(eng.direct_sum(every, with_potential=pot)[cols])
            g = np.random.default_rng(n)
            for tg in (every[::-1], g.permutation(n)[:100], np.array([n // 2]), every[:64], g.integers(0, n, 3 * n)):
                for call in (eng.direct_sum, eng.direct_sum_noalloc):
                    if len(tg) <= E.DIRECT_NOALLOC_MAX or call == eng.direct_sum:
                        got = np.array(call(tg, with_potential=pot)[cols])
                        assert np.array_equal(got, whole[:, tg]), (len(tg), pot)
