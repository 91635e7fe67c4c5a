"""More clusters than a launch holds workgroups of 512 threads (2^23): every
entry point of the ensemble against a few of the clusters alone."""
import ctypes

import numpy as np
import pytest

from pn_amd import lib as pn

pytestmark = pytest.mark.gpu

NC = (1 << 23) + 3


@pytest.mark.timeout(240)
def test_two_body_clusters():
    """A star and its BH each, the 256-star items' own form (no chunk of the
    automatic plan fits).  Every cluster's arithmetic is its own: the same bits
    as the sample's, over 1024 clusters, which take the same items and the same
    form of k_fin (the one for few rows rounds some accelerations otherwise)."""
    rng = np.random.default_rng(5)
    n = 2 * NC
    x, v, u = (rng.normal(size=(n, 3)) for _ in range(3))
    m = rng.uniform(0.1, 1.0, n)
    off = np.arange(0, n + 1, 2, dtype=np.int32)
    pick = np.unique(np.concatenate([[0, 1, NC // 2, (1 << 22) - 1, 1 << 22, (1 << 22) + 1,
                                      (1 << 23) - 1, 1 << 23, NC - 1], rng.integers(0, NC, 1100)]))
    rows = np.stack([2 * pick, 2 * pick + 1], 1).ravel()

    def run(x, v, m, u, off, tuning):
        nc = len(off) - 1
        with pn.Ensemble(len(m), nc) as e:
            L, h, p = e._L, e._h, pn.ptr
            e.set_params(1e-2, 10.0, 2.0**-8, pn.FP64)
            if tuning:
                e.set_tuning(*tuning)
            e._chk(L.pn1_ens_upload(h, nc, off.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                    p(x), p(v), p(m)), "upload")
            print(f"case: {nc} clusters uploaded", flush=True)
            out = [np.empty((len(m), 3)) for _ in range(5)]
            en, gm = np.empty((nc, 5)), np.empty(nc)
            e._chk(L.pn1_ens_force(h, p(out[0])), "force")
            print("force", flush=True)
            e._chk(L.pn1_ens_energy(h, p(en)), "energy")
            print("energy", flush=True)
            e._chk(L.pn1_ens_force_vjp(h, p(u), p(out[1]), p(out[2]), p(gm)), "vjp")
            print("vjp", flush=True)
            e._chk(L.pn1_ens_step(h, 1), "step")
            e._chk(L.pn1_ens_download(h, p(out[3]), p(out[4])), "download")
            print("step", flush=True)
        return out, en, gm

    few, en1, gm1 = run(*(np.ascontiguousarray(a[rows]) for a in (x, v, m, u)),
                        np.arange(0, len(rows) + 1, 2, dtype=np.int32), (0, 0, 0))
    many, en, gm = run(x, v, m, u, off, None)
    for a, b in zip(many, few):
        assert np.isfinite(a).all()
        assert (a[rows] == b).all()
    assert np.array_equal(en[pick], en1) and np.array_equal(gm[pick], gm1)
