"""k_fin by groups of 16 stars (up to 16 rows of 64 with 8 partials or more):
star counts at the edges of groups, rows and of the rule, with stars close to
the BH and tight pairs (their masks are shared by a row's four groups), against
the whole-row form, which a split of 4 chunks takes."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu


def state(stars):
    x, v, m = pn.ic_plummer(stars, 700 + stars, a=1.0, m_bh=0.05)
    for k, r in ((3, 2e-4), (17, 5e-4), (stars - 1, 3e-4)):     # close to the BH
        x[1 + k % stars] = x[0] + r * np.array([0.6, -0.48, 0.64])
    for k in (5, 33, 50, stars // 2):                            # tight pairs
        x[1 + (k + 1) % stars] = x[1 + k] + np.array([1e-4, -2e-4, 1e-4])
    return x, v, m


@pytest.mark.parametrize("stars", [255, 256, 257, 271, 272, 273, 512, 1007, 1023, 1024, 1025])
def test_groups_against_rows(stars):
    """FP64: the sums' order alone, <= 1e-12 relative (the parity bound); mixed:
    each evaluation within 1e-6 of FP64, so <= 2e-6, the second one with the
    thresholds and lists of the first.  Two calls of a step equal one of two."""
    x, v, m = state(stars)
    print(f"case: {stars} stars", flush=True)

    def rel(a, b):
        return (np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)).max()

    with pn.Context(stars + 1) as ctx:
        exact = None
        for mode in (pn.FP64, pn.MIXED):
            ctx.set_params(1e-3, 50.0, 2.0**-16, mode)
            got = []
            for split in (4, 0):
                ctx.set_tuning(split, 0, -1)
                ctx.upload(x, v, m)
                got.append([ctx.force(), ctx.force()])
            if mode == pn.FP64:
                exact = got[0][0]
                assert rel(got[1][0], exact) <= 1e-12
            else:
                for a in got[0] + got[1]:
                    assert rel(a, exact) <= 1e-6
            ctx.step(2)
            one = ctx.download()
            ctx.upload(x, v, m)
            ctx.force()
            ctx.force()
            ctx.step(1)
            ctx.step(1)
            two = ctx.download()
            assert np.array_equal(one[0], two[0]) and np.array_equal(one[1], two[1])
