"""The direct groupby calls of few rows (one block) and around the row and key counts where the launch
changes, exact against the oracle: rows a thread, partly filled waves, all rows dropped, one key, runs of
every length, keys whose offsets the block forms itself and more, two and three radix passes, in place."""
import numpy as np
import pytest

from ptask_amd import groupby as GB
from test_groupby_api import check_against_oracle, run_direct

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 63, 64, 65, 1023, 1025, 4095, 4096, 4097, 8191, 8192, 8193]
KEYS = [0, 1, 255, 256, 4094, 4095, 4096, 65_535, 65_536, GB.MAX_KEYS - 1]


def rows_of(kind, n, nk, seed):
    rng = np.random.default_rng(seed)
    K = nk + 1
    if kind == "one":
        keys = np.full(n, nk)
    elif kind == "dropped":
        keys = np.where(rng.random(n) < 0.5, -1, K)
    elif kind == "mixed":
        keys = rng.integers(0, K, n)
        bad = rng.random(n) < 0.1
        keys[bad] = rng.choice([-1, K, 2**31 - 1, -2**31], bad.sum())
    else:
        keys = np.minimum((rng.random(n) ** 4 * K).astype(np.int64), nk)
    return keys.astype(np.int32), rng.integers(-2**31, 2**31, n, dtype=np.int64).astype(np.int32)


@pytest.mark.parametrize("nk", KEYS)
@pytest.mark.parametrize("n", ROWS)
def test_few_rows(hip, n, nk):
    for i, kind in enumerate(("skewed", "mixed", "one", "dropped")):
        print(f"case few rows n={n} nk={nk} {kind}", flush=True)
        keys, vals = rows_of(kind, n, nk, seed=n + nk + i)
        check_against_oracle(keys, vals, nk, run_direct(hip, keys, vals, nk, fn="run" if i % 2 else "noalloc"))


def test_outputs_over_inputs(hip):
    import oracle
    L = GB.lib()
    for n, nk in ((3000, 500), (8000, 70_000), (16_000, 4095), (20_000, 500)):
        print(f"case in place n={n} nk={nk}", flush=True)
        keys, vals = rows_of("mixed", n, nk, seed=n)
        g, head, eoff, eok, eov = oracle.groupby(keys, vals, nk)
        k, v = hip.DeviceBuffer(keys.nbytes), hip.DeviceBuffer(vals.nbytes)
        k.upload(keys)
        v.upload(vals)
        off, grp = hip.DeviceBuffer(8 * (nk + 1)), hip.DeviceBuffer(8 * (3 + 3 * (nk + 1)))
        nb = L.ptk_groupby_workspace_bytes(n, nk)
        ws = hip.DeviceBuffer(nb)
        assert L.ptk_groupby_run(k.ptr, v.ptr, n, nk, ws.ptr, nb, off.ptr, grp.ptr, k.ptr, v.ptr, None) == 0
        hip.synchronize()
        ok, ov = np.zeros(n, np.int32), np.zeros(n, np.int32)
        k.download(ok)
        v.download(ov)
        rows = int(head[1])
        assert np.array_equal(ok[:rows], eok[:rows]) and np.array_equal(ov[:rows], eov[:rows])
