"""GroupbyPartition on more blocks than chunks (a quarter chunk each), in the full pipeline against the
oracle: row counts around quarters and chunks, grids from one block more than the chunks to more than the
quarters, both bucket-number widths, invalid keys in every quarter."""
import numpy as np
import pytest

import oracle
from ptask_amd import groupby as GB
from ptask_amd import paths
from test_gpu_groupby_kernels import make_keys, run_kernels

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gmod(hip):
    return hip.Module(paths.kernel_path("groupby.hsaco"))


@pytest.mark.parametrize("nk", [0, 1000, 65_535, 200_000])
@pytest.mark.parametrize("n", [1, 4096, 4097, 12_288, 16_384, 16_385, 50_001])
def test_quarters(hip, gmod, monkeypatch, n, nk):
    chunks = GB.chunks(n)
    keys, vals = make_keys("invalid", n, nk, seed=n + nk)
    g, head, offsets, eok, eov = oracle.groupby(keys, vals, nk)
    rows = int(head[1])
    for grid in (chunks + 1, 4 * chunks, 4 * chunks + 3):
        print(f"case quarters n={n} nk={nk} grid={grid}", flush=True)
        # the histogram's and the partition's grids (and the scratch, which may be larger) follow chunks()
        monkeypatch.setattr(GB, "chunks", lambda rows, grid=grid: grid)
        got = run_kernels(hip, gmod, keys, vals, nk, [None] * 7)
        assert np.array_equal(got["groups"][:3], head)
        assert np.array_equal(got["groups"][3:3 + g.size], g.reshape(-1))
        assert np.array_equal(got["offsets"], offsets)
        assert np.array_equal(got["ok"][:rows], eok[:rows])
        assert np.array_equal(got["ov"][:rows], eov[:rows])
