"""The automatic launch plan (rows of 64 stars) against the 256-star kernels,
which an explicit variant selects: edges of rows and blocks, and both sides of
the plan's change from 16 equal to 24 tapered chunks, masses over six decades."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stars", [2, 65, 257, 1025, 8191, 8192, 8193])
@pytest.mark.parametrize("mode,bound", [(pn.FP64, 1e-12), (pn.MIXED, 2e-6)])
def test_automatic_plan_against_the_256_star_kernels(stars, mode, bound):
    """FP64: the sums' order alone, the parity bound; mixed: each within 1e-6 of
    FP64."""
    x, v, m = pn.ic_plummer(stars, 77, a=1.0, m_bh=0.05)
    m[1:] *= 10.0 ** np.random.default_rng(77).uniform(-3, 3, stars)
    with pn.Context(stars + 1) as ctx:
        ctx.set_params(1e-3, 50.0, 2.0**-10, mode)
        ctx.upload(x, v, m)
        a = ctx.force()
        for shape in ((8, 0, 0), (16, 0, 0), (64, 0, 0), (24, 0, 1)):
            print(f"case: {stars} stars, mode {mode}, {shape}", flush=True)
            ctx.set_tuning(*shape)
            ctx.upload(x, v, m)
            b = ctx.force()
            err = np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)
            assert err.max() <= bound, (shape, err.max())
