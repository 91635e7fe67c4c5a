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
