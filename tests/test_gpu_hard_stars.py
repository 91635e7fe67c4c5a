"""Stars whose pair terms cancel (PN1_HARD_K) take their sums in FP64: the first
two of a row of 64 in the pair kernel's chunks, any more in k_fin.  Massless
stars at and around the centre of a point-symmetric cluster, one to four to a
row, over k_fin's three forms, and shards, which must equal the full rows."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

C = np.array([1.0, 0.5, -0.25])


def state(stars):
    """Pairs of stars at C +- r; the hard ones replace the middle of the list's
    rows, so that the others stay symmetric."""
    rng = np.random.default_rng(stars)
    half = stars // 2
    r = rng.normal(size=(half, 3)) * 0.5
    x = np.concatenate([np.zeros((1, 3)), C + r, C - r])
    v = np.concatenate([np.zeros((1, 3)), rng.normal(size=(2 * half, 3)) * 0.1])
    m = np.full(2 * half + 1, 1.0 / half)
    m[0] = 1e-6
    hard = []
    for row, cnt in ((0, 4), (1, 1), (half // 64, 3), ((half - 1) // 64, 2)):
        for k in range(cnt):
            i = row * 64 + 7 + 13 * k
            if i < half:
                hard.append(i)
    for n, i in enumerate(sorted(set(hard))):
        for j in (1 + i, 1 + half + i):                 # the pair: both massless
            x[j] = C + 1e-3 * rng.normal(size=3) * (n % 3)
            m[j] = 0.0
    x[1 + half:][hard] += 5.0                           # the second one elsewhere
    return x, v, m, 1 + np.array(sorted(set(hard)))


def rel(a, b):
    return np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)


@pytest.mark.parametrize("stars", [300, 700, 1024, 3000, 10240, 70000])
def test_hard_stars(stars):
    """Mixed against FP64: every star <= 1e-6, the mixed form's bound, the hard
    ones <= 1e-9 (their sums are FP64: rounding of cancelling terms alone)."""
    x, v, m, hard = state(stars)
    n = len(m)
    print(f"case: {n} particles, hard {hard}", flush=True)
    with pn.Context(n) as ctx:
        ctx.set_params(1e-3, 50.0, 2.0**-10, pn.FP64)
        ctx.upload(x, v, m)
        exact = ctx.force()
        w2 = 1.0 / (((x[1:, None] - x[None, hard]) ** 2).sum(-1) + 1e-6)
        terms = (m[1:, None] * w2).sum(0)
        assert np.all(terms > 30.0 * np.linalg.norm(exact[hard], axis=1)), "not hard"
        ctx.set_params(1e-3, 50.0, 2.0**-10, pn.MIXED)
        ctx.upload(x, v, m)
        for _ in range(2):
            err = rel(ctx.force(), exact)
            assert err[1:].max() <= 1e-6
            assert err[hard].max() <= 1e-9, err[hard]
        ctx.set_tuning(16, 0, -1)
        ctx.upload(x, v, m)
        full = ctx.force()
        assert rel(full, exact)[hard].max() <= 1e-9
        for a, b in ((1, 257), (257, min(n, 1025)), (1, n)):
            assert np.array_equal(ctx.force_range(a, b), full[a:b])
        ctx.set_tuning(0, 0, -1)                        # the shard's own split
        for a, b in ((1, 257), (257, min(n, 1025))):
            err = rel(ctx.force_range(a, b), exact[a:b])
            inside = hard[(hard >= a) & (hard < b)] - a
            assert err.max() <= 1e-6 and (err[inside] <= 1e-9).all()


def test_hard_stars_of_an_ensemble():
    """The automatic plan of clusters of one and of several chunks, against each
    cluster's FP64 forces, as above."""
    cl = [state(k) for k in (300, 10240, 700, 3000)]
    exact = []
    with pn.Ensemble(sum(len(c[2]) for c in cl), len(cl)) as ens:
        ens.set_params(1e-3, 50.0, 2.0**-10, pn.FP64)
        ens.upload([c[:3] for c in cl])
        exact = ens.force()
        ens.set_params(1e-3, 50.0, 2.0**-10, pn.MIXED)
        ens.upload([c[:3] for c in cl])
        for _ in range(2):
            for a, e, c in zip(ens.force(), exact, cl):
                err = rel(a, e)
                assert err[1:].max() <= 1e-6
                assert err[c[3]].max() <= 1e-9, err[c[3]]
