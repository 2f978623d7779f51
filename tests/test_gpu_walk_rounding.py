"""What rounding the gravity walk adds to its own tree: the engine's tree walked
in extended precision for a sample of targets, and small sets with every node
opened against the FP64 direct sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = np.longdouble


def exact_walk(tree, order, R, ps, e0, G, theta, tg):
    """Accelerations of targets tg from the engine's nodes (pre-order)."""
    level, leaf = tree["level"], tree["count"] == 1
    nn = len(level)
    skip = np.empty(nn, np.int64)   # the next node that is not below
    stack = []
    for i in range(nn - 1, -1, -1):
        while stack and level[stack[-1]] > level[i]:
            stack.pop()
        skip[i] = stack[-1] if stack else nn
        stack.append(i)
    own = np.where(leaf, order[np.minimum(tree["first"], len(order) - 1)], -1)
    radius = R * np.ldexp(1.0, -level.astype(int))
    pos = [getattr(ps, f)[tg] for f in ("x", "y", "z")]
    acc = np.zeros((3, len(tg)), L)
    at, live = np.zeros(len(tg), np.int64), np.arange(len(tg))
    while len(live):
        k = at[live]
        d = [tree["com"][k, c] - pos[c][live] for c in range(3)]
        r = np.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
        self = own[k] == tg[live]
        with np.errstate(divide="ignore"):
            take = ~self & (r != 0) & (leaf[k] | (radius[k] / r < theta))
        t, q = live[take], k[take]
        d = [tree["com"][q, c].astype(L) - pos[c][t] for c in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        f = L(G) * tree["mass"][q].astype(L) / ((r2 + L(e0) * L(e0)) * np.sqrt(r2))
        for c in range(3):
            acc[c, t] += f * d[c]
        at[live] = np.where(take | self, skip[k], k + 1)
        live = live[at[live] < nn]
    return acc


def errors(ag2, ps, e0, precision, sample):
    """Per sampled target: the relative error's length, and its part along the force."""
    E, U = ag2.engine, ag2.units
    tg = np.random.default_rng(5).choice(ps.n, sample, replace=False)
    with E.Engine(E.make_params(theta=0.5, e0=e0, split_threshold=800, precision=precision), ps.n) as eng:
        eng.upload(ps)
        eng.init_forces()
        out = eng.download(ag2.ics.ParticleSet(ps.n), ("ax", "ay", "az"))
        want = exact_walk(eng.tree(), eng.order()[0], eng.diagnostics()["R"], ps, e0, U.G, 0.5, tg)
    off = np.stack([out.ax[tg], out.ay[tg], out.az[tg]]) - want
    size = np.sqrt((want * want).sum(0))
    return ((np.sqrt((off * off).sum(0)) / size).astype(float),
            ((off * want).sum(0) / (size * size)).astype(float))


@pytest.mark.parametrize("n", [33333, 150001, 410001])
def test_fp64_pairs_have_no_bias(ag2, n):
    """Every step of a pair rounds to nearest: over a thousand targets the
    errors along the force cancel (half of 2^-53 allowed), and the sums, formed
    in chunks of at most 64 entries, keep the median error below 2^-52."""
    ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n)
    err, along = errors(ag2, ps, 0.05 * ag2.units.KPC, ag2.engine.AG2_FP64, 1000)
    assert abs(np.median(along)) < 2.0 ** -54, np.median(along)
    assert np.median(err) < 2.0 ** -52, np.median(err)


# median relative errors of the same targets with every chunk's entries summed
# under their masks, about 26 of 64 at a time
MASKED = {410001: 5.842e-8, 700001: 6.031e-8}


@pytest.mark.parametrize("n", [410001, 700001])
def test_split_form_sums_few_terms_plainly(ag2, n):
    """Full chunks, where every lane takes every entry, round no more than
    chunks swept under masks did."""
    ps = ag2.ics.plummer(n, 1e10, 1.0, 20.0, seed=n)
    err, _ = errors(ag2, ps, 0.05 * ag2.units.KPC, ag2.engine.AG2_FP32_SPLIT, 2000)
    assert np.median(err) < MASKED[n], np.median(err)


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
