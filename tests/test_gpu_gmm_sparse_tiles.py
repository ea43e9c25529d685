"""The accumulate kernels on tiles at both sides of the rule that passes over points without a
responsibility: at most five responsibilities that are not 0 for four points of a tile.

Every point lies within 0.02 of one mean, and reciprocal variances are 1e10, so a responsibility is 0
except in the components of that mean: one for most means, two for the twins (equal means, 1/2 each).
Four rows of one tile each: single points only, one twin below the limit and one above (a full tile's
160 counts), and a ragged tile.  A sum is off by 132 binary32 roundings of the sum of absolute values
(128 additions, the difference, the product and the conversion) and, for twins, by the 3 of the
responsibility's own (the log of 2, its sum with the log density and the exponential: the log density's
rounding cancels, as both twins have the same).  The log density itself is up to 1e10 * D * 4e-4 / 2, so its
sum with log 2 rounds by up to 2^-24 of that, which enters the exponent: twins lie exactly on their mean,
where the log density is -ln(var) D / 2.
"""
import numpy as np
import pytest

from ptask_amd import gmm, paths

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", ["GmmAccumulate", "GmmAccumulateMfma"])
@pytest.mark.parametrize("D,K", [(32, 64), (12, 44), (9, 50), (32, 17), (8, 64), (3, 6)])
def test_sparse_and_dense_tiles(hip, kernel, D, K):
    print(f"case gmm sparse tiles {kernel} D={D} K={K}", flush=True)
    rng = np.random.default_rng(100 * D + K)
    mu = rng.uniform(-1, 1, (K, D)).astype(np.float32).astype(np.float64)
    mu[1] = mu[0]  # the twins
    mu[K - 1] = mu[K - 2]
    twins = np.array([0, 1, K - 2, K - 1])
    single = np.setdiff1d(np.arange(K), twins)
    comp, X = [], []
    for n, t in ((128, 0), (128, 32), (128, 33), (101, 26)):  # 101 points: the limit is 126, the count 127
        c = np.concatenate([rng.choice(twins, t), rng.choice(single, n - t)])
        x = mu[c].copy()
        x[t:] += rng.uniform(-0.02, 0.02, (n - t, D))
        order = rng.permutation(n)
        comp.append(c[order])
        X.append(x[order].astype(np.float32))
    N = sum(len(c) for c in comp)
    o = gmm.model_offsets(D, K, 1)
    model = np.zeros(gmm.model_elems(D, K, 1))
    model[1:4] = (N, D, K)
    model[o["mu"]:o["var"]] = mu.ravel()
    model[o["var"]:o["frac"]] = 1e-10
    model[o["frac"]:o["ll"]] = 1.0 / K
    gmm.fill_table(model, D, K, 1)
    part = np.full(4 * gmm.partial_stride(D, K), np.nan)
    bufs = []
    for a in (np.concatenate(X), model, part):
        b = hip.DeviceBuffer(a.nbytes)
        b.upload(a)
        bufs.append(b)
    hip.launch(hip.Module(paths.kernel_path("gmm.hsaco")).function(kernel), (4, 1, 1), (256, 1, 1),
               hip.ArgPack().ptr(bufs[0].ptr).raw(bytes(gmm.Dims(N, D, K, 4, 1))).ptr(bufs[1].ptr).ptr(bufs[2].ptr))
    hip.synchronize()
    bufs[2].download(part)
    lp0 = 0.5 * D * np.log(1e10) + np.log(K)  # the largest term of a twin's log density, at its mean
    eps = 2.0 ** -24
    for row, c, x in zip(part.reshape(4, -1), comp, X):
        x = x.astype(np.float64)
        r = (c[:, None] == np.arange(K)).astype(np.float64)
        for a, b in ((0, 1), (K - 2, K - 1)):
            r[:, a] = r[:, b] = 0.5 * (r[:, a] + r[:, b])
        d = x[:, None, :] - mu[None]
        want = np.concatenate([r.sum(0), (r[:, :, None] * d).sum(0).ravel(), (r[:, :, None] * d * d).sum(0).ravel()])
        size = np.concatenate([r.sum(0), (r[:, :, None] * np.abs(d)).sum(0).ravel(),
                               (r[:, :, None] * d * d).sum(0).ravel()])
        tol = (132 + 2 * lp0 + 4) * eps  # 2 lp0: the two roundings at lp0's size in a twin's exponent
        # GmmAccumulateMfma sums about one component's mean, up to 2 away from another, in binary64: 128
        # additions and 4 operations of the conversion, at up to 4 per responsibility
        mid = 132 * 2.0 ** -53 * 4 * len(c)
        assert np.all(np.abs(row[:-1] - want) <= tol * size + mid), (D, K)
