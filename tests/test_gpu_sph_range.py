"""The SPH pair kernel on both of its paths: supports inside and outside the
range where the short root and quotients are used, lists that end anywhere
among the lanes that share a record, against the oracle."""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("power", [0, 45, -180])   # supports near 2^65, 2^110, 2^-115 metres
@pytest.mark.parametrize("n", [9, 77, 1500])
def test_sph_pairs(ag2, orc, n, power):
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.gas_sphere(n, seed=n)
    ps.vx[:] = np.random.default_rng(n).normal(0, 2e4, n)
    s = 2.0 ** power
    for a in (ps.x, ps.y, ps.z):
        a *= s
    e0, mih = 0.02 * U.KPC * s, min(48, n // 3) * ps.m[0]
    prm = orc.params(0.5, e0, mih, 100)
    a = ps.copy()
    st = orc.force_step(a, prm)
    assert st["sph_interactions"] > 0
    with E.Engine(E.make_params(theta=0.5, e0=e0, massInH=mih, split_threshold=100), n) as eng:
        eng.upload(ps)
        eng.init_forces()
        b = eng.download(ps.copy())
        d = eng.diagnostics()
    assert d["sph_pairs"] == st["sph_interactions"]
    unit = np.abs([a.ax, a.ay, a.az]).max()   # (squares of the tightest set's accelerations overflow)
    assert np.isfinite(unit)
    assert vec_rel_err(*[v / unit for v in (b.ax, b.ay, b.az, a.ax, a.ay, a.az)]).max() < 1e-10
    assert np.abs(b.dUdt - a.dUdt).max() <= 1e-10 * np.abs(a.dUdt).max()
