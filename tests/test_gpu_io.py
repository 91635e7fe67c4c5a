"""States pass between AoS host arrays and the SoA device buffers two doubles
at a time through one kernel each way: every particle count parity and the
edges of its workgroups, bit for bit; refused uploads leave the state that
was there; uploads that overtake running work do not disturb it."""
import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu


def state(n, seed):
    rng = np.random.default_rng(seed)
    x, v = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
    return x, v, rng.uniform(0.5, 1.0, n)


@pytest.mark.parametrize("n", [1, 2, 3, 85, 86, 170, 171, 512, 1365, 1366, 50001])
def test_round_trip(n):
    x, v, m = state(n, n)
    with pn.Context(n + n % 3) as ctx:
        ctx.set_params(1e-2, 10.0, 2.0**-10, pn.FP64)
        ctx.upload(x, v, m)
        a, b = ctx.download()
        assert np.array_equal(a, x) and np.array_equal(b, v)
        if n > 1:
            u = np.random.default_rng(0).normal(size=(n, 3))
            z = ctx.force_vjp(np.zeros((n, 3)))            # the cotangent's v part alone
            assert not np.any(z[0]) and not np.any(z[1]) and z[2] == 0.0
            g = ctx.force_vjp(u)
            assert all(np.array_equal(p, q) for p, q in zip(g, ctx.force_vjp(u)))


def test_refused_upload_keeps_the_state():
    x, v, m = state(300, 1)
    with pn.Context(300) as ctx, pn.Ensemble(600, 3) as ens:
        ctx.set_params(1e-2, 10.0, 2.0**-10, pn.FP64)
        ens.set_params(1e-2, 10.0, 2.0**-10, pn.FP64)
        ctx.upload(x, v, m)
        ens.upload([(x, v, m), (x, v, m)])
        a, e = ctx.force(), ens.force()
        for k, what in ((np.nan, "non-finite position"), (np.inf, "non-finite position"),
                        (-np.inf, "non-finite position"), (x[0, 1], "exactly on the black hole")):
            y = x + 1.0
            y[0] = x[0]
            if np.isfinite(k):
                y[299] = x[0]
            else:
                y[299, 1] = k
            with pytest.raises(pn.Pn1Error, match=what):
                ctx.upload(y, v, m)
            with pytest.raises(pn.Pn1Error, match="cluster 1: .*" + what):
                ens.upload([(x, v, m), (y, v, m)])
        w = m.copy()
        w[7] = np.nan
        with pytest.raises(pn.Pn1Error, match="non-finite mass at particle 7"):
            ctx.upload(x, v, w)
        w[7], w[0] = 1.0, 0.0
        with pytest.raises(pn.Pn1Error, match="black hole mass"):
            ctx.upload(x, v, w)
        # distinct positions whose squared distance underflows are no error
        y = x.copy()
        y[0] = 0.0
        y[5] = (1e-200, 0.0, 0.0)
        assert np.array_equal(ctx.force(), a)
        assert all(np.array_equal(p, q) for p, q in zip(ens.force(), e))
        ctx.upload(y, v, m)
        assert np.array_equal(ctx.download()[0], y)


@pytest.mark.parametrize("mode", [pn.FP64, pn.MIXED])
def test_uploads_behind_running_steps(mode):
    """Upload, step and upload again without waiting: each result is that of
    the same calls one at a time."""
    states = [state(k, 10 + k) for k in (700, 300, 701)]
    with pn.Context(701) as ctx:
        ctx.set_params(1e-1, 10.0, 2.0**-12, mode)
        alone = []
        for s in states:
            ctx.upload(*s)
            ctx.sync()
            ctx.step(3)
            ctx.sync()
            alone.append(ctx.download())
        for s, want in zip(states, alone):
            ctx.upload(*states[0])
            ctx.step(5)
            ctx.upload(*s)
            ctx.step(3)
            got = ctx.download()
            assert all(np.array_equal(p, q) for p, q in zip(got, want))
