"""What pn1_get_tuning, pn1_ens_get_tuning and the tuners report, set on another
object with the same state, runs the same kernels: the same bits (the automatic
plan, the row form and the 256-star kernels add in different orders)."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

EPS, C, DT = 1e-3, 50.0, 2.0**-10


def context(n, mode, shape, st, tune=False):
    with pn.Context(n) as ctx:
        ctx.set_params(EPS, C, DT, mode)
        ctx.set_tuning(*shape)
        ctx.upload(*st)
        got = ctx.autotune(1) if tune else None
        if tune:
            ctx.upload(*st)                     # the thresholds as after an upload
        return ctx.get_tuning(), ctx.force(), got


@pytest.mark.parametrize("mode", [pn.FP64, pn.MIXED])
@pytest.mark.parametrize("stars", [2, 300, 4097, 10240])
def test_context(stars, mode):
    st = pn.ic_plummer(stars, 40 + stars, a=1.0, m_bh=0.05)
    for shape in ((0, 0, -1), (0, 16, -1), (0, 0, 0), (0, 0, 1), (1, 0, -1), (2, 0, -1), (24, 0, -1),
                  (33, 0, -1), (192, 0, -1), (64, 32, 5), (16, 0, 0)):
        print(f"case: {stars} stars, mode {mode}, tuning {shape}", flush=True)
        said, a, _ = context(stars + 1, mode, shape, st)
        again, b, _ = context(stars + 1, mode, said, st)
        assert again == said and np.array_equal(a, b), (shape, said, again)
        if shape[0] == 0 and shape[2] < 0:
            assert said[0] == 0 and said[2] == -1
    said, a, (S, var, _) = context(stars + 1, mode, (0, 0, -1), st, tune=True)
    assert (S, var) == (said[0], said[2])
    again, b, _ = context(stars + 1, mode, (S, 0, var), st)
    assert again == said and np.array_equal(a, b)


@pytest.mark.parametrize("mode", [pn.FP64, pn.MIXED])
@pytest.mark.parametrize("sizes", [(300, 40, 700), (3000, 9000, 2000)])
def test_ensemble(sizes, mode):
    cl = [pn.ic_plummer(ns, 60 + ns, a=1.0, m_bh=0.05) for ns in sizes]

    def ensemble(shape, tune=False):
        with pn.Ensemble(sum(sizes) + len(sizes), len(sizes)) as e:
            e.set_params(EPS, C, DT, mode)
            e.set_tuning(*shape)
            e.upload(cl)
            got = e.autotune(1) if tune else None
            if tune:
                e.upload(cl)
            return e.get_tuning(), np.concatenate(e.force()), got

    for shape in ((0, 0, -1), (0, 16, -1), (0, 0, 0), (0, 0, 1), (128, 0, -1), (4096, 0, 1)):
        print(f"case: {sizes}, mode {mode}, tuning {shape}", flush=True)
        said, a, _ = ensemble(shape)
        again, b, _ = ensemble(said)
        assert again == said and np.array_equal(a, b), (shape, said, again)
        assert (said[2] == -1) == (shape[0] == 0 and shape[2] < 0)
    said, a, (L, var, _) = ensemble((0, 0, -1), tune=True)
    assert (L, var) == (said[0], said[2])
    again, b, _ = ensemble((L, 0, var))
    assert again == said and np.array_equal(a, b)
