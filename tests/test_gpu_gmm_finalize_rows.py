"""GmmFinalize's sums over the accumulate's partial rows, at row counts around the 32 rows that a
thread loads at once: a row group (256 / (2 D + 1) of them) with one row, 31 to 33 and 65.

Tolerance: a sum of P binary64 terms in any order is within P 2^-53 of the sum of their absolute
values; the variance is a difference of two quotients of such sums, (P + 4) 2^-53 each.
"""
import numpy as np
import pytest

from ptask_amd import gmm, paths

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,K", [(1, 3), (16, 5), (32, 2)])
@pytest.mark.parametrize("rows", [(0, 1), (1, 0), (32, -1), (32, 0), (32, 1), (65, 0)])
def test_rows_are_summed(hip, D, K, rows):
    G = 256 // (2 * D + 1)
    P = rows[0] * G + rows[1]
    print(f"case gmm finalize D={D} K={K} rows={P}", flush=True)
    rng = np.random.default_rng(100 * D + P)
    o = gmm.model_offsets(D, K, 1)
    N = 1000 * P
    model = np.zeros(gmm.model_elems(D, K, 1))
    model[1:4] = (N, D, K)
    model[o["mu"]:o["var"]] = rng.uniform(-2, 2, K * D)
    model[o["var"]:o["frac"]] = 1
    model[o["frac"]:o["ll"]] = 1.0 / K
    gmm.fill_table(model, D, K, 1)
    cen = model[o["table"]:].view(np.float32)[:2 * K * gmm.dpad(D)].reshape(K, 2, -1)[:, 0, :D].astype(np.float64)
    w = rng.uniform(0.5, 2, (P, K))
    s1 = rng.uniform(-0.5, 0.5, (P, K, D))
    s2 = rng.uniform(1, 2, (P, K, D))
    ll = rng.uniform(-5, -1, P)
    part = np.concatenate([w, s1.reshape(P, -1), s2.reshape(P, -1), ll[:, None]], 1)
    assert part.shape[1] == gmm.partial_stride(D, K)
    dM, dP = hip.DeviceBuffer(model.nbytes), hip.DeviceBuffer(part.nbytes)
    dM.upload(model)
    dP.upload(np.ascontiguousarray(part))
    hip.launch(hip.Module(paths.kernel_path("gmm.hsaco")).function("GmmFinalize"), (K + 1, 1, 1), (256, 1, 1),
               hip.ArgPack().ptr(dM.ptr).ptr(dP.ptr).raw(bytes(gmm.Dims(N, D, K, P, 1))))
    hip.synchronize()
    got = np.empty_like(model)
    dM.download(got)
    W = w.sum(0)[:, None]
    dm, q = s1.sum(0) / W, s2.sum(0) / W
    eps = (P + 8) * 2.0 ** -53
    tm = np.abs(s1).sum(0) / W + np.abs(cen + dm)
    assert np.all(np.abs(got[o["mu"]:o["var"]].reshape(K, D) - (cen + dm)) <= 2 * eps * tm)
    assert np.all(np.abs(got[o["var"]:o["frac"]].reshape(K, D) - (q - dm * dm)) <= 4 * eps * (q + tm * tm + dm * dm))
    assert np.all(np.abs(got[o["frac"]:o["ll"]] - W[:, 0] / N) <= 2 * eps * W[:, 0] / N)
    assert abs(got[o["ll"]] - ll.sum()) <= eps * np.abs(ll).sum()
    assert got[0] == 1
