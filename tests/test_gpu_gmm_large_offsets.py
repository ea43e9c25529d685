"""GmmAccumulateMfma on points far from the origin: squares of the coordinates themselves overflow binary32,
squares of the distances (a hundred roundings of a coordinate) do not.  A dimension past D and a point past
the last must not reach a sum, whatever is in memory there.  Tolerance as in test_gpu_gmm_tiles."""
import numpy as np
import pytest

from ptask_amd import gmm, paths
from test_gpu_gmm_tiles import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0.0, 1e20, -2e22])
@pytest.mark.parametrize("N,blocks", [(1, 1), (17, 1), (1311, 3)])
@pytest.mark.parametrize("D,K", [(1, 3), (5, 17), (8, 16), (13, 40), (20, 64), (31, 33)])
def test_offsets(hip, D, K, N, blocks, offset):
    print(f"case gmm offsets D={D} K={K} N={N} offset={offset}", flush=True)
    sd = max(1.0, abs(offset) * 1e-5)
    rng = np.random.default_rng(N + D)
    X = (offset + sd * rng.uniform(-2, 2, (N, D))).astype(np.float32)
    o = gmm.model_offsets(D, K, 1)
    model = np.zeros(gmm.model_elems(D, K, 1))
    model[1:4] = (N, D, K)
    model[o["mu"]:o["var"]] = offset + sd * rng.uniform(-2, 2, K * D)
    model[o["var"]:o["frac"]] = sd * sd * rng.uniform(0.5, 2, K * D)
    model[o["frac"]:o["ll"]] = 1.0 / K
    gmm.fill_table(model, D, K, 1)
    tab = model[o["table"]:].view(np.float32)
    Dp = gmm.dpad(D)
    rows = tab[:2 * K * Dp].reshape(K, 2, Dp)
    mu, iv, C = rows[:, 0, :D], rows[:, 1, :D].astype(np.float64), tab[2 * K * Dp:2 * K * Dp + K].astype(np.float64)
    part = np.full(blocks * gmm.partial_stride(D, K), np.nan)
    bufs = []
    for a in (X, model, part):
        b = hip.DeviceBuffer(max(a.nbytes, 16))
        b.upload(a)
        bufs.append(b)
    hip.launch(hip.Module(paths.kernel_path("gmm.hsaco")).function("GmmAccumulateMfma"), (blocks, 1, 1), (256, 1, 1),
               hip.ArgPack().ptr(bufs[0].ptr).raw(bytes(gmm.Dims(N, D, K, blocks, 1))).ptr(bufs[1].ptr).ptr(bufs[2].ptr))
    hip.synchronize()
    bufs[2].download(part)
    got = part.reshape(blocks, -1).sum(0)
    # the kernel's centre: the mean of the means, rounded to binary32
    g = mu.astype(np.float64).mean(0).astype(np.float32).astype(np.float64)
    want, ll, S, scale, big = reference(X, mu, iv, C, g)
    W, eps = 8 * -(-D // 8), 2.0 ** -24
    assert np.all(np.abs(got[:-1] - want) <= (2 * (2 * W + 4) * S + 160) * eps * scale + 1e-30)
    assert abs(got[-1] - ll) <= ((2 * W + 8) * S + 4 * big) * eps * N
