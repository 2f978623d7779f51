"""Nodes of the tree at the sizes where their kernels change hands: ranges
found among 64, 1024 and 65536 neighbours, sums by one lane (2..8, 9..32
particles) and by a wave over particles, 64-blocks and 4096-blocks, with and
without particles outside the root cube."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def cells(hi, lo, proot):
    """(level, first, count) of every node in pre-order from the sorted keys."""
    n = len(hi)
    shared = np.empty(n, int)
    for i in range(n - 1):
        a, b = int(hi[i] ^ hi[i + 1]), int(lo[i] ^ lo[i + 1])
        shared[i] = (63 - a.bit_length()) // 3 if a else 21 + (63 - b.bit_length()) // 3
    shared[n - 1] = 0 if n == 1 and proot else -1
    assert shared.max() < 42, "the inputs hold no particles at one position"
    level, first, count, stack = [], [], [], []
    prev = -1
    for i in range(n):
        while stack and level[stack[-1]] > prev:   # the cells that ended before i
            k = stack.pop()
            count[k] = i - first[k]
        for lv in range(prev + 1, shared[i] + 1):
            stack.append(len(level))
            level.append(lv), first.append(i), count.append(0)
        level.append(max(prev, shared[i]) + 1), first.append(i), count.append(1)
        prev = shared[i]
    for k in stack:
        count[k] = n - first[k]
    return np.array(level), np.array(first), np.array(count)


@pytest.mark.parametrize("spread", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 32, 33, 63, 64, 65, 257, 1023, 1025, 4096, 4097, 8257, 20000, 70001])
def test_nodes(ag2, n, spread):
    E, U = ag2.engine, ag2.units
    ps = ag2.ics.shuffled(ag2.ics.hernquist(n, seed=n), n)
    rng = np.random.default_rng(n)
    ps.m *= rng.uniform(0.5, 2.0, n)
    ps.type[:] = np.where(rng.random(n) < 0.4, 2, 1)
    if spread and n > 2:   # a few far away: the root cube leaves them out, or long chains of cells
        k = max(1, n // 100)
        for a in (ps.x, ps.y, ps.z):
            a[:k] *= 300.0
    dt = 2.0 * U.MYR
    with E.Engine(E.make_params(theta=0.7, e0=0.05 * U.KPC, split_threshold=2, min_dt=dt, max_dt=dt), n) as eng:
        eng.upload(ps)
        eng.build_tree()
        perm, hi, lo = eng.order()
        t = eng.tree()
    proot, nin = n >= 2, len(perm)
    level, first, count = cells(hi, lo, proot)
    assert (t["level"] == level).all() and (t["first"] == first).all() and (t["count"] == count).all()
    order = np.concatenate([perm, np.setdiff1d(np.arange(n), perm)])
    m, gas = ps.m[order], ps.m[order] * (ps.type[order] == 2)
    rows = [m, m * ps.x[order], m * ps.y[order], m * ps.z[order],
            gas, gas * ps.vx[order], gas * ps.vy[order], gas * ps.vz[order]]
    u = 2.0 ** -53
    sample = range(len(level)) if n < 10000 else [*range(40), *range(40, len(level), 17)]
    for k in sample:
        a, b = (0, n) if k == 0 and proot else (first[k], first[k] + count[k])
        c = b - a
        s = [math.fsum(r[a:b]) for r in rows]
        # c - 1 additions in any order (and a product) against the exact sum
        assert abs(t["mass"][k] - s[0]) <= (c + 1) * u * s[0]
        assert abs(t["gas"][k] - s[4]) <= (c + 1) * u * s[4]
        for j in range(3):
            scale = math.fsum(np.abs(rows[1 + j][a:b])) / s[0]
            assert abs(t["com"][k][j] - s[1 + j] / s[0]) <= (2 * c + 4) * u * scale
            if s[4] > 0 and count[k] > 1:
                scale = math.fsum(np.abs(rows[5 + j][a:b])) / s[4]
                assert abs(t["mvel"][k][j] - s[5 + j] / s[4]) <= (2 * c + 4) * u * scale
