"""The energy kernel evaluates each pair of stars once: rows of 64 stars meet
the following half of the rows cyclically and their own stars above each
lane's, split into chunks and waves.  Star counts at the edges of rows (even
and odd numbers of them), of the waves' parts and of the chunk counts, with
masses over six decades, against the oracle's direct double sums, alone and
as clusters of an ensemble."""
import numpy as np
import pytest

import oracle_bind as ob
from conftest import energy_atol
from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

EPS, C = 1e-2, 20.0
# Each term is ~20 roundings and is summed in chains of at most a few hundred
# here and of n in the oracle (n 2^-53 <= 5e-13 of the sum of magnitudes); the
# star terms keep one sign except pot_pn2's, whose largest parts cancel to no
# less than a tenth for these states.  energy_atol: the oracle's self pairs.
RTOL = 1e-11


def cluster(stars, seed):
    x, v, m = pn.ic_plummer(stars, seed, a=1.0, m_bh=0.05)
    x[1:] += (0.5, 0.25, -0.125)          # one star alone is at the BH's place
    m[1:] *= 10.0 ** np.random.default_rng(seed).uniform(-3, 3, stars)
    return x, v, m


STARS = [1, 2, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 511, 512, 513, 1024, 1025, 4097]


def test_energy_row_edges():
    cl = [cluster(k, 300 + k) for k in STARS]
    refs = [ob.orc_energy_terms(x, v, m, EPS, C) for x, v, m in cl]
    alone = []
    with pn.Context(4200) as ctx:
        for (x, v, m), ref in zip(cl, refs):
            print(f"case: {len(m) - 1} stars", flush=True)
            ctx.set_params(EPS, C, 2.0**-10, pn.FP64)
            ctx.upload(x, v, m)
            e = ctx.energy()
            alone.append(e)
            tol = RTOL * np.abs(ref).max() + energy_atol(dict(m=m, eps=EPS), ref)
            assert np.all(np.abs(e - ref) <= tol), (len(m), e, ref)
    with pn.Ensemble(sum(STARS) + len(STARS) + 1, len(STARS) + 1) as ens:
        ens.set_params(EPS, C, 2.0**-10, pn.FP64)
        lone = (np.zeros((1, 3)), np.array([[3.0, 0.0, 4.0]]), np.array([2.0]))
        ens.upload(cl + [lone])
        for _ in range(2):                     # the counters return to zero
            e = ens.energy()
            assert np.array_equal(e[:-1], np.array(alone))
            assert np.array_equal(e[-1], [25.0, 0.0, 0.0, 0.0, 25.0])
