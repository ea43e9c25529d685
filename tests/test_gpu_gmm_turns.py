"""GmmAccumulateMfma with many tiles per row, where its waves take turns at the block's sums: more than four
16 x 16 tiles of moments (fewer stay in registers), 9 to 20 point tiles per row and a ragged last one, so
that every wave has several turns.  Eight launches give the same bits, and the sums are binary64's within the
tolerance of test_gpu_gmm_tiles."""
import numpy as np
import pytest

from ptask_amd import gmm, paths
from test_gpu_gmm_tiles import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles,blocks", [(9, 1), (37, 3), (55, 5), (20, 1), (513 * 9, 768)])
@pytest.mark.parametrize("D,K", [(32, 64), (24, 33), (17, 48), (9, 64)])
def test_turns(hip, D, K, tiles, blocks):
    print(f"case gmm turns D={D} K={K} tiles={tiles} blocks={blocks}", flush=True)
    N = 128 * tiles - 37
    rng = np.random.default_rng(tiles + D)
    X = rng.uniform(-2, 2, (N, D)).astype(np.float32)
    o = gmm.model_offsets(D, K, 1)
    model = np.zeros(gmm.model_elems(D, K, 1))
    model[1:4] = (N, D, K)
    model[o["mu"]:o["var"]] = rng.uniform(-2, 2, K * D)
    model[o["var"]:o["frac"]] = rng.uniform(0.5, 2, K * D)
    model[o["frac"]:o["ll"]] = 1.0 / K
    gmm.fill_table(model, D, K, 1)
    nan = np.full(blocks * gmm.partial_stride(D, K), np.nan)
    dX, dM, dP = (hip.DeviceBuffer(a.nbytes) for a in (X, model, nan))
    dX.upload(X)
    dM.upload(model)
    fn = hip.Module(paths.kernel_path("gmm.hsaco")).function("GmmAccumulateMfma")
    runs = []
    for _ in range(8):
        dP.upload(nan)
        hip.launch(fn, (blocks, 1, 1), (256, 1, 1),
                   hip.ArgPack().ptr(dX.ptr).raw(bytes(gmm.Dims(N, D, K, blocks, 1))).ptr(dM.ptr).ptr(dP.ptr))
        hip.synchronize()
        part = np.empty_like(nan)
        dP.download(part)
        runs.append(part)
    assert all(np.array_equal(runs[0].view(np.uint64), r.view(np.uint64)) for r in runs[1:])
    if N > 10_000:  # the reference holds N x K x D values
        assert np.isfinite(runs[0]).all()
        w = runs[0].reshape(blocks, -1)[:, :K].sum()
        assert abs(w - N) <= 160 * 2.0 ** -24 * N  # each point's responsibilities add up to 1
        return
    tab = model[o["table"]:].view(np.float32)
    Dp = gmm.dpad(D)
    rows = tab[:2 * K * Dp].reshape(K, 2, Dp)
    mu, iv, C = rows[:, 0, :D], rows[:, 1, :D].astype(np.float64), tab[2 * K * Dp:2 * K * Dp + K].astype(np.float64)
    want, ll, S, scale, big = reference(X, mu, iv, C, mu.astype(np.float64).mean(0))
    got = runs[0].reshape(blocks, -1).sum(0)
    W, eps = 8 * -(-D // 8), 2.0 ** -24
    assert np.all(np.abs(got[:-1] - want) <= (2 * (2 * W + 4) * S + 160) * eps * scale + 1e-30)
    assert abs(got[-1] - ll) <= ((2 * W + 8) * S + 4 * big) * eps * N
