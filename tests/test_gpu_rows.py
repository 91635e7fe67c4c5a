"""The O(n) kernels take stars in rows of 64, eight to a workgroup, and their
last workgroup adds the sums over all stars and finishes the BH.  Star counts
at the edges of rows and workgroups: forces and steps against the oracle, and
step calls that continue one another."""
import numpy as np
import pytest

import oracle_bind as ob
from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

EPS, C, DT = 1e-3, 50.0, 2.0**-10


def rel_err(a, b):
    return np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)


@pytest.mark.parametrize("stars", [3, 63, 64, 65, 511, 512, 513, 1025])
def test_row_edges(stars):
    """FP64 forces <= 1e-12 of the oracle's (the parity bound), mixed <= 1e-6;
    two steps <= 1e-12; two calls of one step equal one call of two, bit for
    bit (the second call prepares its first evaluation anew)."""
    x, v, m = pn.ic_plummer(stars, 900 + stars, a=1.0, m_bh=0.05)
    print(f"case: {stars} stars", flush=True)
    ref = ob.orc_force(x, v, m, EPS, C)
    with pn.Context(len(m) + 7) as ctx:
        for mode, bound in ((pn.FP64, 1e-12), (pn.MIXED, 1e-6)):
            ctx.set_params(EPS, C, DT, mode)
            ctx.upload(x, v, m)
            assert rel_err(ctx.force(), ref).max() <= bound, mode
            ctx.upload(x, v, m)
            ctx.step(2)
            x2, v2 = ctx.download()
            ctx.upload(x, v, m)
            ctx.step(1)
            ctx.step(1)
            x11, v11 = ctx.download()
            assert np.array_equal(x2, x11) and np.array_equal(v2, v11), mode
            if mode == pn.FP64:
                xo, vo = ob.orc_q1_steps(x, v, m, EPS, C, DT, 2)
                assert max(np.abs(x2 - xo).max(), np.abs(v2 - vo).max()) <= 1e-12


@pytest.mark.parametrize("mode", [pn.FP64, pn.MIXED])
def test_ensemble_with_clusters_of_no_star(mode):
    """A cluster that is its BH alone keeps its row of zeros: the BH drifts by
    v dt / 2 per step (the driver's weights), and its neighbours step as
    they do alone with the same chunk."""
    cl = [pn.ic_plummer(ns, 950 + ns, a=1.0, m_bh=0.05) for ns in (65, 600)]
    lone = (np.array([[1.0, 2.0, 3.0]]), np.array([[0.5, -0.25, 0.125]]), np.array([0.1]))
    with pn.Ensemble(800, 4) as ens:
        ens.set_params(EPS, C, DT, mode)
        ens.set_tuning(4096, 0, -1)
        ens.upload([lone, cl[0], lone, cl[1]])
        ens.step(2)
        xs, vs = ens.download()
        for k in (0, 2):
            # per step three roundings of sums up to 18, divided by 6
            assert np.allclose(xs[k], lone[0] + lone[1] * DT, rtol=0, atol=4e-15)
            assert np.allclose(vs[k], lone[1], rtol=0, atol=4e-15)
        ens.upload(cl)
        ens.step(2)
        xa, va = ens.download()
    for k, q in ((0, 1), (1, 3)):
        assert np.array_equal(xa[k], xs[q]) and np.array_equal(va[k], vs[q])
