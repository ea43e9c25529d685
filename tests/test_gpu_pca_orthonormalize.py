"""PcaOrthonormalize alone against binary64, at the edges of its groups: 4 and 16 components held in
registers, one more, 64; columns around a thread's two and four, one thread to all of them; numbers of
partial rows around its group of eight.

Tolerance: everything is binary64 but the stored result, so a component is off by its rounding to
binary32 (2^-24 of itself) plus the binary64 sums' (4096 terms of 1.1e-16, against the unit norm).
"""
import ctypes as C

import numpy as np
import pytest

from ptask_amd import paths

pytestmark = pytest.mark.gpu


class Dims(C.Structure):
    _fields_ = [(f, C.c_int) for f in ("M", "N", "K", "J", "ld", "Mp", "G", "GR", "k", "center", "pad0", "pad1")]


@pytest.mark.parametrize("N,K,k,GR", [(1, 1, 0, 1), (8, 7, 6, 3), (64, 64, 60, 8), (66, 20, 15, 9), (700, 20, 16, 8),
                                      (700, 20, 17, 8), (2047, 40, 33, 7), (2048, 5, 4, 8), (2049, 20, 19, 16),
                                      (4096, 64, 63, 8), (4093, 3, 1, 1)])
def test_component(hip, N, K, k, GR):
    print(f"case orthonormalize N={N} K={K} k={k} GR={GR}", flush=True)
    rng = np.random.default_rng(N + 100 * k)
    ld = (N + 3) & ~3
    d = Dims(64, N, K, 1, ld, 64, GR, GR, k, 1, 0, 0)
    off_red = 8 * ((K + 1) & ~1) + 8 * ((GR + 1) & ~1)
    off_p = off_red + 8 * GR * ld
    S = np.zeros(off_p + 4 * K * ld + 4 * GR * ld, np.uint8)
    red = np.zeros((GR, ld))
    red[:, :N] = rng.standard_normal((GR, N))
    P = np.zeros((K, ld), np.float32)
    if k:
        q, _ = np.linalg.qr(rng.standard_normal((N, k)))
        P[:k, :N] = q.T
    S[off_red:off_p] = red.reshape(-1).view(np.uint8)
    S[off_p:off_p + 4 * K * ld] = P.reshape(-1).view(np.uint8)
    b = hip.DeviceBuffer(S.nbytes)
    b.upload(S)
    fn = hip.Module(paths.kernel_path("pca.hsaco")).function("PcaOrthonormalize")
    hip.launch(fn, (1, 1, 1), (1024, 1, 1), hip.ArgPack().ptr(b.ptr).raw(bytes(d)))
    hip.synchronize()
    out = np.empty_like(S)
    b.download(out)
    got = out[off_p:off_p + 4 * K * ld].view(np.float32).reshape(K, ld)
    p = red.sum(0)
    q = P[:k].astype(np.float64)
    p = p - q.T @ (q @ p)
    want = p / np.linalg.norm(p)
    # the norm left after projection scales the binary64 errors of the sums
    scale = np.abs(red.sum(0)).max() * np.sqrt(N) / np.linalg.norm(p)
    assert np.all(np.abs(got[k] - want) <= 2.0 ** -24 * np.abs(want) * 1.01 + 4096 * 1.2e-16 * scale + 2.0 ** -149)
    assert np.array_equal(got[:k], P[:k]) and not got[k, N:].any()
    rest = out.copy()
    rest[off_p + 4 * k * ld:off_p + 4 * (k + 1) * ld] = S[off_p + 4 * k * ld:off_p + 4 * (k + 1) * ld]
    assert np.array_equal(rest, S)
