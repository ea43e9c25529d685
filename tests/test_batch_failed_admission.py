"""A launch that fails while the executor admits instances: none of that call's instances is admitted, all
stay queued with their slots and arena ranges given back, and the next call admits each of them once.

Runs the executor on the CPU over a stand-in for libptk_hip.so that keeps memory on the host, computes
nothing and fails a named kernel's n-th launch when told to; a process of its own, so that the real library
is not the one already loaded."""
import json
import shutil
import subprocess
import sys

import pytest

from ptask_amd import paths

STUB = r"""
#include <stdlib.h>
#include <string.h>
#include "ptk_hip.h"
#define OK PTK_HIP_OK
static char fail_name[64];
static int fail_after = -1, count[256];
static const char *names[256];
static int nnames;
void stub_fail(const char *name, int after) { strncpy(fail_name, name, 63); fail_after = after; }
int stub_launches(const char *name) {
    for (int i = 0; i < nnames; ++i) if (!strcmp(names[i], name)) return count[i];
    return 0;
}
int ptk_hip_get_device(int *d) { *d = 0; return OK; }
int ptk_hip_get_device_props(int d, ptk_hip_device_props_t *p) { memset(p, 0, sizeof *p); p->compute_units = 256; return OK; }
int ptk_hip_malloc(void **p, size_t n) { *p = calloc(1, n ? n : 1); return OK; }
int ptk_hip_free(void *p) { free(p); return OK; }
int ptk_hip_host_malloc(void **p, size_t n) { *p = calloc(1, n ? n : 1); return OK; }
int ptk_hip_host_free(void *p) { free(p); return OK; }
int ptk_hip_memcpy_htod_async(void *d, const void *s, size_t n, ptk_hip_stream st) { memcpy(d, s, n); return OK; }
int ptk_hip_memcpy_dtoh_async(void *d, const void *s, size_t n, ptk_hip_stream st) { memcpy(d, s, n); return OK; }
int ptk_hip_memcpy_htod(void *d, const void *s, size_t n) { memcpy(d, s, n); return OK; }
int ptk_hip_memcpy_dtoh(void *d, const void *s, size_t n) { memcpy(d, s, n); return OK; }
int ptk_hip_stream_create(ptk_hip_stream *s) { *s = (ptk_hip_stream)1; return OK; }
int ptk_hip_stream_destroy(ptk_hip_stream s) { return OK; }
int ptk_hip_stream_synchronize(ptk_hip_stream s) { return OK; }
int ptk_hip_event_create(ptk_hip_event *e, int t) { *e = (ptk_hip_event)1; return OK; }
int ptk_hip_event_destroy(ptk_hip_event e) { return OK; }
int ptk_hip_event_record(ptk_hip_event e, ptk_hip_stream s) { return OK; }
int ptk_hip_event_synchronize(ptk_hip_event e) { return OK; }
int ptk_hip_event_elapsed_ms(float *ms, ptk_hip_event a, ptk_hip_event b) { *ms = 0; return OK; }
int ptk_hip_module_load(ptk_hip_module *m, const char *path) { *m = (ptk_hip_module)1; return OK; }
int ptk_hip_module_unload(ptk_hip_module m) { return OK; }
int ptk_hip_module_get_function(ptk_hip_function *f, ptk_hip_module m, const char *name) {
    int i = 0;
    while (i < nnames && strcmp(names[i], name)) ++i;
    if (i == nnames) names[nnames++] = strdup(name);
    *f = (ptk_hip_function)(size_t)(i + 1);
    return OK;
}
int ptk_hip_launch(ptk_hip_function f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz,
                   unsigned lds, ptk_hip_stream s, void *args, size_t n) {
    const int i = (int)(size_t)f - 1;
    if (!strcmp(names[i], fail_name) && fail_after >= 0 && fail_after-- == 0) return PTK_HIP_ERR_RUNTIME;
    ++count[i];
    return OK;
}
int ptk_hip_stream_begin_capture(ptk_hip_stream s) { return OK; }
int ptk_hip_stream_end_capture(ptk_hip_stream s, ptk_hip_graph *g) { *g = (ptk_hip_graph)1; return OK; }
int ptk_hip_graph_launch(ptk_hip_graph g, ptk_hip_stream s) { return OK; }
int ptk_hip_graph_destroy(ptk_hip_graph g) { return OK; }
const char *ptk_hip_last_error_string(void) { return "told to fail"; }
"""

SCRIPT = r"""
import ctypes, json, sys
sys.path.insert(0, sys.argv[2])
from ptask_amd import batch, paths
paths.LIB_DIR = sys.argv[1]
stub = ctypes.CDLL(sys.argv[1] + "/libptk_hip.so", mode=ctypes.RTLD_GLOBAL)
mode, kernel, after = int(sys.argv[3]), sys.argv[4].encode(), int(sys.argv[5])
ex = batch.Executor(64 << 20, mode)
ids = [ex.submit_fdtd(8 + i % 3, 9, 7, 4, i, keep=True) for i in range(40)]
ids += [ex.submit_groupby(1000, 99, 0.0, 5, keep=True), ex.submit_gmm(500, 3, 4, 2, 6, keep=True)]
ids += [ex.submit_fdtd(6, 6, 6, 3, i, keep=True) for i in range(3)]
used = sum(batch.footprint(batch.FDTD, 8 + i % 3, 9, 7, 4) for i in range(40)) + batch.footprint(batch.GROUPBY, 1000, 99)
used += batch.footprint(batch.GMM, 500, 3, 4, 2) + 3 * batch.footprint(batch.FDTD, 6, 6, 6, 3)
out = {}
stub.stub_fail(kernel, after)
try:
    ex.run(1)
    out["raised"] = ""
except batch.BatchError as e:
    out["raised"] = str(e)
out["states"] = [ex.status(i)[0] for i in ids]
out["used"] = ex.stats()["arena_used"]
iters, active, completed = ex.run(1)
out["active_and_completed"] = active + completed
out["used_later"], out["want"] = ex.stats()["arena_used"], used
ex.drain()
out["done"] = [ex.status(i)[0] for i in ids]
for i in ids:
    ex.release(i)
out["used_end"] = ex.stats()["arena_used"]
# every slot is back: as many instances as before fit again
more = [ex.submit_fdtd(8, 9, 7, 3, i) for i in range(60)]
ex.drain()
out["more"] = [ex.status(i)[0] for i in more]
ex.close()
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def libdir(tmp_path_factory):
    d = tmp_path_factory.mktemp("stub")
    (d / "stub.c").write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-I", paths.include_dir(), "-o", str(d / "libptk_hip.so"),
                    str(d / "stub.c")], check=True)
    shutil.copy(paths.lib_path("libptk_batch.so"), d)
    return str(d)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("kernel,after", [("BatchInitFdtd", 0), ("BatchInitFdtd", 1), ("BatchInitGroupby", 0),
                                          ("BatchInitGmm", 0), ("BatchInitGmmModel", 0)])
def test_failed_admission_is_taken_back(libdir, mode, kernel, after):
    p = subprocess.run([sys.executable, "-c", SCRIPT, libdir, paths.REPO_DIR, str(mode), kernel, str(after)],
                       capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-2000:]
    r = json.loads(p.stdout.splitlines()[-1])
    assert "told to fail" in r["raised"]
    assert set(r["states"]) == {0}  # queued
    assert r["used"] == 0
    assert r["active_and_completed"] == len(r["states"])
    assert r["used_later"] == r["want"]
    assert set(r["done"]) == {2}
    assert r["used_end"] == 0
    assert set(r["more"]) == {3}
