"""The VJP's pair kernel where a tile of 64 records does not line up with a
wave's 64 stars: ensemble chunk lengths that are no multiple of 64 (the self
pairs then meet in the middle of a tile), and star counts at the edges of
tiles, rows and 256-star blocks, against the complex-step oracle."""
import numpy as np
import pytest

import oracle_bind as ob
from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

EPS, C = 1e-3, 50.0


@pytest.mark.parametrize("chunk", [33, 100, 129, 4096])
def test_chunks_off_the_tiles(chunk):
    """<= 1e-12 of the largest component (the bound the chunkings of a single
    context are held to) between ensemble chunks and a single context."""
    cl = [pn.ic_plummer(ns, 700 + ns, a=1.0, m_bh=0.02) for ns in (63, 65, 257, 600)]
    rng = np.random.default_rng(71)
    us = [rng.normal(size=(len(m), 3)) for _, _, m in cl]
    with pn.Ensemble(sum(len(m) for _, _, m in cl), len(cl)) as ens:
        ens.set_params(EPS, C, 2.0**-10, pn.FP64)
        ens.set_tuning(chunk, 0, -1)
        ens.upload(cl)
        gxs, gvs, gm0 = ens.force_vjp(us)
    for k, (x, v, m) in enumerate(cl):
        with pn.Context(len(m)) as ctx:
            ctx.set_params(EPS, C, 2.0**-10, pn.FP64)
            ctx.upload(x, v, m)
            gx, gv, g0 = ctx.force_vjp(us[k])
        scale = max(np.abs(gx).max(), np.abs(gv).max(), abs(g0))
        err = max(np.abs(gxs[k] - gx).max(), np.abs(gvs[k] - gv).max(), abs(gm0[k] - g0)) / scale
        print(f"chunk {chunk} stars {len(m) - 1}: {err:.2e}", flush=True)
        assert err <= 1e-12


@pytest.mark.parametrize("stars", [3, 64, 65, 256, 258])
def test_edges_vs_complex_step(stars):
    """<= 1e-12 of the largest sampled component."""
    x, v, m = pn.ic_plummer(stars, 800 + stars, a=1.0, m_bh=0.02)
    n = len(m)
    u = np.random.default_rng(72).normal(size=x.shape)
    with pn.Context(n) as ctx:
        ctx.set_params(EPS, C, 2.0**-10, pn.FP64)
        ctx.upload(x, v, m)
        gx, gv, g0 = ctx.force_vjp(u)
    coords = [("m0",), ("x", 0, 0), ("x", 1, 1), ("v", 1, 2), ("x", n - 1, 0), ("v", n - 1, 1),
              ("v", n // 2, 0)]
    ref = ob.cs_force_vjp(x, v, m, u, EPS, C, coords)
    got = np.array([g0 if c[0] == "m0" else (gx if c[0] == "x" else gv)[c[1], c[2]]
                    for c in coords])
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"{stars} stars: {err:.2e}", flush=True)
    assert err <= 1e-12
