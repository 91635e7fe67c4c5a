"""Steps of the mixed form whose hard stars (PN1_HARD_K: sums in FP64) change
from one evaluation to the next.  k_fin reads this evaluation's hard stars while
it writes the next one's, and a star's FP64 sums are found by counting the hard
stars before it in its row: the two must not share memory.  Massless stars cross
the threshold inwards and outwards near the centre of a point-symmetric cluster,
six to a row in all of its groups of 16, over k_fin's three forms, with the sums
in the pair kernel's chunks (the automatic plan) and in k_fin (variant 0)."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

C = np.array([1.0, 0.5, -0.25])
EPS, DT, STEPS = 0.1, 2.0**-6, 5


def state(stars, seed=1):
    """Equal masses around C, symmetric under cyclic permutations and sign
    changes of the axes (the field at C then vanishes to second order), and six
    massless stars near C in each of three rows."""
    rng = np.random.default_rng(stars + seed)
    count = (stars - 18) // 24
    last = (18 + 24 * count - 64) // 64
    near = 1 + np.array(sorted({row * 64 + k for row in (0, 1, last) for k in (3, 9, 20, 40, 44, 60)}))
    g = rng.normal(size=(count, 3)) * 0.5
    g[0] = (0.18, 0.12, 0.07)                   # the core's share, also with few stars
    r = np.concatenate([np.roll(g, k, axis=1) * (s1, s2, s3) for k in range(3)
                        for s1 in (1, -1) for s2 in (1, -1) for s3 in (1, -1)])
    n = 1 + len(near) + len(r)
    x, v, m = np.zeros((n, 3)), np.zeros((n, 3)), np.full(n, 2.0 / len(r))
    m[0] = 1e-6
    m[near] = 0.0
    x[np.setdiff1d(np.arange(1, n), near)] = C + rng.permutation(r)
    for q, i in enumerate(near):
        d = rng.normal(size=3)
        d /= np.linalg.norm(d)
        # along a line through C, 0.03 per step (v dt / 2): they come in, pass
        # the centre and leave at different steps
        x[i] = C + d * (0.09 - 0.013 * (7 * q % 18))
        v[i] = d * 0.03 * 2 / DT
    return x, v, m, near


def hard(x, a, m, near):
    """Whether each star of `near` cancels beyond PN1_HARD_K = 30."""
    w2 = 1.0 / (((x[1:, None] - x[None, near]) ** 2).sum(-1) + EPS * EPS)
    return (m[1:, None] * w2).sum(0) > 30.0 * np.linalg.norm(a[near], axis=1)


def crossings(states, near):
    """Changes of the hard stars between steps, of the FP64 run."""
    flags = np.array([hard(x, a, m, near) for x, a, m in states])
    d = np.diff(flags.astype(int), axis=0)
    return (d > 0).sum(), (d < 0).sum(), flags.any(axis=0).sum()


# Each evaluation's acceleration is within 1e-6 of FP64 (the mixed form's bound;
# hard stars far closer), a step adds dt / 2 times such accelerations to the
# velocity (its weights), and the error fed back through the positions is dt^2
# smaller: STEPS * DT / 2 * 1e-6 * max |a|, with room of 2.  One wrong sum of a
# hard star (|a| ~ 0.2) moves its velocity by dt / 6 |a| ~ 1e-3.
def bound(a):
    return STEPS * DT * 1e-6 * np.linalg.norm(a[1:], axis=1).max()


@pytest.mark.parametrize("stars,tuning", [(300, (0, 0, -1)), (1024, (0, 0, -1)), (3000, (0, 0, -1)),
                                          (70000, (0, 0, -1)), (1024, (16, 0, 0)), (3000, (16, 0, 0)),
                                          (70000, (32, 0, 0))])
def test_hard_stars_change_between_steps(stars, tuning):
    x, v, m, near = state(stars)
    n = len(m)
    with pn.Context(n) as ctx:
        ctx.set_params(EPS, 50.0, DT, pn.FP64)
        ctx.upload(x, v, m)
        seen = []
        for _ in range(STEPS):
            seen.append((ctx.download()[0], ctx.force(), m))
            ctx.step(1)
        xe, ve = ctx.download()
        ins, outs, count = crossings(seen, near)
        print(f"case: {n} particles, {ins} become hard, {outs} stop, {count} ever", flush=True)
        assert ins >= 2 and outs >= 2
        tol = bound(seen[0][1])
        ctx.set_params(EPS, 50.0, DT, pn.MIXED)
        ctx.set_tuning(*tuning)
        runs = []
        for calls in ([STEPS], [STEPS], [1] * STEPS):
            ctx.upload(x, v, m)
            for k in calls:
                ctx.step(k)
            runs.append(ctx.download())
    for xs, vs in runs:
        assert np.abs(vs - ve).max() <= tol, (np.abs(vs - ve).max(), tol)
        assert np.abs(xs - xe).max() <= tol
        assert np.array_equal(xs, runs[0][0]) and np.array_equal(vs, runs[0][1])


@pytest.mark.parametrize("clusters,variant", [(6, -1), (220, -1), (6, 0), (220, 0)])
def test_hard_stars_of_an_ensemble_change_between_steps(clusters, variant):
    """A workgroup per row, and a wave per row (more than 1024 rows)."""
    cl = [state(300 + 32 * (k % 3), k) for k in range(clusters)]
    with pn.Ensemble(sum(len(c[2]) for c in cl), clusters) as ens:
        ens.set_params(EPS, 50.0, DT, pn.FP64)
        ens.upload([c[:3] for c in cl])
        seen = []
        for _ in range(STEPS):
            seen.append((ens.download()[0], ens.force()))
            ens.step(1)
        xe, ve = ens.download()
        cross = [crossings([(xs[k], a[k], cl[k][2]) for xs, a in seen], cl[k][3])
                 for k in range(min(clusters, 6))]
        print(f"case: {clusters} clusters, crossings {cross}", flush=True)
        assert all(i >= 1 and o >= 1 for i, o, _ in cross)
        ens.set_params(EPS, 50.0, DT, pn.MIXED)
        ens.set_tuning(0, 0, variant)
        runs = []
        for _ in range(2):
            ens.upload([c[:3] for c in cl])
            ens.step(STEPS)
            runs.append(ens.download())
    for xs, vs in runs:
        for k in range(clusters):
            tol = bound(seen[0][1][k])
            assert np.abs(vs[k] - ve[k]).max() <= tol, (k, np.abs(vs[k] - ve[k]).max(), tol)
            assert np.abs(xs[k] - xe[k]).max() <= tol
            assert np.array_equal(xs[k], runs[0][0][k]) and np.array_equal(vs[k], runs[0][1][k])
