"""The automatic launch plan around its change from 16 equal to 24 tapered
chunks per row: the forces of an explicit split's kernels, masses over six
decades."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu


def cluster(stars, seed):
    x, v, m = pn.ic_plummer(stars, seed, a=1.0, m_bh=0.05)
    m[1:] *= 10.0 ** np.random.default_rng(seed).uniform(-3, 3, stars)
    return x, v, m


@pytest.mark.parametrize("stars", [8191, 8192, 8193])
@pytest.mark.parametrize("mode,bound", [(pn.FP64, 1e-12), (pn.MIXED, 2e-6)])
def test_automatic_plan_against_explicit_split(stars, mode, bound):
    """Around the change of the automatic plan: the same forces as the
    256-star kernels of an explicit split give.  FP64: the sums' order alone,
    the parity bound; mixed: each within 1e-6 of FP64."""
    x, v, m = cluster(stars, 77)
    print(f"case: {stars} stars, mode {mode}", flush=True)
    with pn.Context(stars + 1) as ctx:
        ctx.set_params(1e-3, 50.0, 2.0**-10, mode)
        ctx.upload(x, v, m)
        a = ctx.force()
        ctx.set_tuning(16, 0, -1)
        b = ctx.force()
    assert (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)).max() <= bound


@pytest.mark.parametrize("mode,bound", [(pn.FP64, 1e-12), (pn.MIXED, 2e-6)])
def test_ensemble_plan_against_items(mode, bound):
    """The ensemble's automatic plan (rows of 64 stars) against its 256-star
    items: an explicit chunk, and a variant set and taken back after the upload,
    which changes the tables under a captured step.  Sizes at the edges of rows,
    chunks and parts, and a cluster without stars."""
    sizes = [1, 63, 64, 65, 255, 256, 257, 511, 513, 1025, 4097]
    cl = []
    for k in sizes:
        x, v, m = cluster(k, 500 + k)
        x[1:] += (0.5, 0.25, -0.125)          # one star alone is at the BH's place
        cl.append((x, v, m))
    cl.insert(3, (np.zeros((1, 3)), np.ones((1, 3)), np.array([2.0])))
    n = sum(len(m) for _, _, m in cl)

    def worst(a, b):
        return max((np.linalg.norm(p - q, axis=1) / np.maximum(np.linalg.norm(q, axis=1), 1e-300)).max()
                   for p, q in zip(a, b))

    with pn.Ensemble(n, len(cl)) as ens:
        ens.set_params(1e-2, 50.0, 2.0**-10, mode)
        ens.upload(cl)
        a = ens.force()
        ens.step(2)
        x0, v0 = ens.download()
        ens.set_tuning(0, 0, 0)               # 256-star items from here on
        ens.upload(cl)
        b = ens.force()
        ens.set_tuning(0, 0, -1)
        a2 = ens.force()
        ens.set_tuning(0, 0, 1)
        b2 = ens.force()
        ens.set_tuning(0, 0, -1)
        ens.upload(cl)
        assert all(np.array_equal(p, q) for p, q in zip(ens.force(), a))
        ens.step(1)
        ens.set_tuning(0, 0, 0)
        ens.force()
        ens.set_tuning(0, 0, -1)
        ens.step(1)
        x1, v1 = ens.download()
        ens.set_tuning(128, 0, -1)
        ens.upload(cl)
        d = ens.force()
    for other in (b, a2, b2, d):
        assert worst(other, a) <= bound
    # FP64: the same step from the same state; mixed: its first evaluation's
    # pair thresholds come from another evaluation of the same accuracy
    for p, q in zip(x0 + v0, x1 + v1):
        assert np.abs(p - q).max() <= (1e-12 if mode == pn.FP64 else 1e-6) * max(1.0, np.abs(q).max())


@pytest.mark.parametrize("mode,bound", [(pn.FP64, 1e-12), (pn.MIXED, 2e-6)])
@pytest.mark.parametrize("stars", [2, 64, 65, 700, 2049])
def test_explicit_splits(stars, mode, bound):
    """Splits at the edges of the row kernels' range (2 to 32, at most one chunk
    per star) against the 256-star kernels of the same split."""
    x, v, m = cluster(stars, 600 + stars)
    with pn.Context(stars + 1) as ctx:
        ctx.set_params(1e-2, 50.0, 2.0**-10, mode)
        for split in (1, 2, 15, 16, 17, 24, 32, 33):
            print(f"case: {stars} stars, split {split}, mode {mode}", flush=True)
            ctx.set_tuning(split, 0, -1)
            ctx.upload(x, v, m)
            a = ctx.force()
            ctx.set_tuning(split, 0, 0)
            b = ctx.force()
            err = np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
            assert err.max() <= bound, (split, err.max())
