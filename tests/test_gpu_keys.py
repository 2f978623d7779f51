"""Octant keys of particles on, beside and clear of cell faces, against the
reference's descent (child centres accumulated level by level)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def word0(x, y, z, R):
    c = [np.zeros_like(x) for _ in range(3)]
    r, key = R, np.zeros(len(x), np.uint64)
    for _ in range(21):
        up = [p > q for p, q in zip((x, y, z), c)]
        key = key << np.uint64(3) | sum(u.astype(np.uint64) << np.uint64(j) for j, u in enumerate(up))
        c = [q + r * np.where(u, 0.5, -0.5) for q, u in zip(c, up)]
        r /= 2
    return key


@pytest.mark.parametrize("power", [-140, 0, 66, 200])   # scales of the root cube
def test_keys_at_faces(ag2, power):
    E, n = ag2.engine, 6000
    g = np.random.default_rng(5)
    R = 1.3 * 2.0 ** power
    ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=4)
    for a in (ps.x, ps.y, ps.z):
        level = g.integers(1, 23, n)
        face = np.rint(g.uniform(-0.5, 0.5, n) * 2.0 ** level) / 2.0 ** level * R
        near = face * (1.0 + g.choice([0.0, 2.0 ** -52, -2.0 ** -52, 1e-14, -1e-13, 1e-9], n))
        a[:] = np.where(g.random(n) < 0.3, g.uniform(-0.5, 0.5, n) * R, near)
    ps.x[0], ps.y[0], ps.z[0] = R, 0.0, 0.0
    with E.Engine(E.make_params(theta=0.7, e0=R * 1e-3, split_threshold=800), n) as eng:
        eng.upload(ps)
        eng.build_tree()
        assert eng.diagnostics()["R"] == R
        perm, hi, _ = eng.order()
    assert len(perm) == n
    assert (hi == word0(ps.x[perm], ps.y[perm], ps.z[perm], R)).all()
