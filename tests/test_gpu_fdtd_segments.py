"""How the three-step FDTD launches cut tiles into segments, bit for bit against the oracle: whole
tiles per block with a remainder, slabs of one tile per block, equal runs that cross tiles, slabs of a
single plane, in the persistent kernel and in the batched executor (any number of virtual blocks)."""
import ctypes as C

import numpy as np
import pytest

import oracle
from ptask_amd import batch as BT
from ptask_amd import fdtd as FD
from ptask_amd import paths
from test_gpu_fdtd_kernels import assert_parity, run_fused

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fmod(hip):
    return hip.Module(paths.kernel_path("fdtd_fused.hsaco"))


# (shape, grid): tiles of 58 x 10 columns
CASES = [((130, 29, 40), 4),    # 9 tiles, two whole ones per block and one cut into four slabs
         ((130, 29, 40), 9),    # one whole tile per block, none left
         ((130, 29, 40), 10),   # fewer tiles than blocks: nine slabs of the whole depth
         ((58, 9, 90), 3),      # two tiles on three blocks: runs that cross from tile to tile
         ((57, 9, 90), 7),      # one tile in seven slabs
         ((57, 9, 12), 256),    # more blocks than planes: slabs of one plane and empty ones
         ((64, 64, 64), 256), ((61, 33, 47), 64), ((2, 2, 2), 5)]


@pytest.mark.parametrize("shape,grid", CASES)
def test_persistent_segments(hip, fmod, shape, grid):
    nx, ny, nz = shape
    print(f"case segments shape={shape} grid={grid}", flush=True)
    F = oracle.init_fields(nx, ny, nz, seed=17 + nz)
    got = run_fused(hip, fmod, "FdtdThreeStepPersistent", F, FD.make_params(nx, ny, nz), 2,
                    ((grid, 1, 1), (64, 16, 1)))
    assert_parity(got, oracle.fdtd_run(F, oracle.make_params(nx, ny, nz, 0.5), 6))


@pytest.mark.parametrize("blocks", [1, 5, 37, 256, 700])
def test_batched_segments(hip, blocks):
    print(f"case batched segments blocks={blocks}", flush=True)
    shapes = [(16, 16, 16), (40, 23, 31), (90, 12, 7), (5, 33, 60), (1, 1, 1)]
    with BT.Executor(64 << 20) as ex:
        t = (C.c_int * 5)(0, 8, 256, 3, blocks)
        assert BT.lib().ptk_batch_set_tuning(ex.h, t) == 0, BT.lib().ptk_batch_last_error()
        ids = [ex.submit_fdtd(*s, 6, 1000 + i, keep=True) for i, s in enumerate(shapes)]
        ex.drain()
        for i, s in zip(ids, shapes):
            F = oracle.init_fields(*s, seed=1000 + ids.index(i))
            ref = oracle.fdtd_run(F, oracle.make_params(*s, 0.5), 6)
            for f in range(6):
                a = ex.read(i, f, np.float32)
                assert np.array_equal(a.view(np.uint32), np.asarray(ref[f], np.float32).reshape(-1).view(np.uint32)), (s, f)
