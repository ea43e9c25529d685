"""The framework's main paths as measurable cases: what a program that drives the task kernels, the
direct groupby library and the batched executor has them do, from the smallest calls to the largest.

Kinds of case:

  groupby  one ptk_groupby_run call (libptk_groupby.so) on rows in device memory.
  fdtd     a run of Yee time steps from device-resident fields: either the fastest graph form
           (FdtdThreeStepPersistent, the remainder steps in one more launch) or the reference's six
           update tasks per step, with the launch geometry the graph application gives its tasks.
  gmm      an EM run: GmmAccumulateMfma and GmmFinalize per step on the application's grid.
  pca      the Gram-Schmidt PCA graph's tasks in the order the application dispatches them.
  scan     the two-task exclusive prefix sum.
  batch    many uneven graph instances through the batched executor: submit, drain, read back.

The chains of task launches are recorded once into a HIP graph, as Graph::EnableLaunchCapture does
for a graph that runs more than once, and a pass replays that graph on the current stream.
"""
import ctypes as C
import math

import numpy as np
import torch

from ptask_amd import batch as BT
from ptask_amd import fdtd as FD
from ptask_amd import gmm as GM
from ptask_amd import groupby as GB
from ptask_amd import hip as H
from ptask_amd import paths

F64 = torch.float64
F32 = torch.float32


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # a served request of a few thousand rows: launches and latency are all that counts
        {"name": "groupby_4k", "kind": "groupby", "n": 4000, "keys": 1023, "dist": "uniform"},
        # an ordinary table with a skewed key column, rows not a multiple of anything
        {"name": "groupby_500k", "kind": "groupby", "n": 500_003, "keys": 65535, "dist": "zipf"},
        # the repository's groupby workload: 8M Zipf rows over 65536 keys
        {"name": "groupby_8m", "kind": "groupby", "n": 8_000_000, "keys": 65535, "dist": "zipf"},
        # the small FDTD configuration (64^3) as one short run
        {"name": "fdtd_64", "kind": "fdtd", "form": "steps3", "nx": 64, "ny": 64, "nz": 64, "steps": 50},
        # a user's own ragged cavity on the reference's task interface, six launches per step
        {"name": "fdtd_six_ragged", "kind": "fdtd", "form": "six", "nx": 201, "ny": 117, "nz": 93, "steps": 10},
        # the headline grid: 384^3, steps that are not a multiple of three
        {"name": "fdtd_384", "kind": "fdtd", "form": "steps3", "nx": 384, "ny": 384, "nz": 384, "steps": 20},
        # a mixture of the size a served request carries
        {"name": "gmm_50k", "kind": "gmm", "n": 50_001, "d": 16, "k": 24, "steps": 20},
        # the repository's GMM workload
        {"name": "gmm_2m", "kind": "gmm", "n": 2_000_000, "d": 32, "k": 64, "steps": 25},
        # a small ragged matrix: a chain of short dependent tasks
        {"name": "pca_3000x700", "kind": "pca", "m": 3000, "n": 700, "k": 4, "j": 8},
        # the repository's PCA workload
        {"name": "pca_65536x2048", "kind": "pca", "m": 65536, "n": 2048, "k": 16, "j": 10},
        # offsets over a column of counts
        {"name": "scan_8m", "kind": "scan", "n": 8_000_000},
        # uneven small graphs executed together (FDTD of edge 16..40, 50 steps, and groupbys)
        {"name": "batch_mix", "kind": "batch", "fdtd": 24, "edge_min": 16, "edge_max": 40, "steps": 50,
         "groupby": 4, "rows": 60_000, "keys": 4095},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["groupby", "groupby", "fdtd", "fdtd", "gmm", "gmm", "pca", "scan", "batch"])
    if kind == "groupby":
        return {"kind": kind, "n": _log(rng, 500, 8_000_000), "keys": _log(rng, 15, 262143),
                "dist": rng.choice(["uniform", "zipf"])}
    if kind == "fdtd":
        form = rng.choice(["steps3", "steps3", "six"])
        return {"kind": kind, "form": form, "nx": rng.randint(24, 320), "ny": rng.randint(24, 320),
                "nz": rng.randint(24, 320), "steps": rng.randint(3, 18) if form == "steps3" else rng.randint(2, 10)}
    if kind == "gmm":
        return {"kind": kind, "n": _log(rng, 10_000, 1_500_000), "d": rng.randint(4, 32), "k": rng.randint(4, 64),
                "steps": rng.randint(5, 20)}
    if kind == "pca":
        return {"kind": kind, "m": _log(rng, 500, 40_000), "n": _log(rng, 64, 2500), "k": rng.randint(2, 12),
                "j": rng.randint(3, 10)}
    if kind == "scan":
        return {"kind": kind, "n": _log(rng, 10_000, 16_000_000)}
    lo = rng.randint(10, 24)
    return {"kind": kind, "fdtd": rng.randint(8, 28), "edge_min": lo, "edge_max": lo + rng.randint(4, 22),
            "steps": rng.randint(12, 60), "groupby": rng.randint(1, 5), "rows": _log(rng, 2000, 120_000),
            "keys": _log(rng, 100, 20_000)}


# ---- shared helpers ----------------------------------------------------------------------------

_modules = {}


def _fn(code_object, name):
    if code_object not in _modules:
        _modules[code_object] = H.Module(paths.kernel_path(code_object))
    return _modules[code_object].function(name)


def _stream():
    """The current stream as the C ABI takes it (None: the null stream)."""
    return torch.cuda.current_stream().cuda_stream or None


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


class _Recorded:
    """A chain of kernel launches recorded once as a HIP graph."""

    def __init__(self, launches):
        L = H.lib()
        torch.cuda.synchronize()
        s = H.Stream()
        H.check(L.ptk_hip_stream_begin_capture(s.handle), "begin_capture")
        for fn, grid, block, args in launches:
            H.launch(fn, grid, block, args, s)
        self.graph = C.c_void_p()
        H.check(L.ptk_hip_stream_end_capture(s.handle, C.byref(self.graph)), "end_capture")
        s.destroy()

    def __call__(self):
        H.check(H.lib().ptk_hip_graph_launch(self.graph, _stream()), "graph_launch")

    def __del__(self):
        try:
            H.lib().ptk_hip_graph_destroy(self.graph)
        except Exception:
            pass


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


# ---- groupby -----------------------------------------------------------------------------------

def _groupby_keys(case, g):
    n, K = case["n"], case["keys"] + 1
    if case["dist"] == "uniform":
        return torch.randint(0, K, (n,), generator=g, device="cuda", dtype=torch.int32)
    p = torch.arange(1, K + 1, device="cuda", dtype=F64) ** -1.1
    cdf = torch.cumsum(p / p.sum(), 0)
    r = torch.searchsorted(cdf, torch.rand(n, generator=g, device="cuda", dtype=F64)).clamp_(max=K - 1)
    return ((r * 40503) % K).to(torch.int32)


def _groupby_prepare(case, seed):
    n, nk = case["n"], case["keys"]
    g = _gen(seed)
    keys = _groupby_keys(case, g)
    vals = torch.randint(-2**31, 2**31 - 1, (n,), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    ws = int(GB.lib().ptk_groupby_workspace_bytes(n, nk))
    i64 = dict(dtype=torch.int64, device="cuda")
    return {"keys": keys, "vals": vals, "ws": torch.empty(ws, dtype=torch.uint8, device="cuda"),
            "offsets": torch.zeros(nk + 1, **i64), "groups": torch.zeros(3 + 3 * (nk + 1), **i64),
            "outKeys": torch.zeros_like(keys), "outVals": torch.zeros_like(vals)}


def _groupby_run(case, s):
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    rc = GB.lib().ptk_groupby_run(p(s["keys"]), p(s["vals"]), case["n"], case["keys"], p(s["ws"]), s["ws"].numel(),
                                  p(s["offsets"]), p(s["groups"]), p(s["outKeys"]), p(s["outVals"]), _stream())
    if rc:
        raise RuntimeError(GB.lib().ptk_groupby_last_error().decode())
    return {k: s[k] for k in ("offsets", "groups", "outKeys", "outVals")}


# ---- FDTD --------------------------------------------------------------------------------------

def _shape(f, c):
    d1, d2, d3 = FD.extent(f, c["nx"], c["ny"], c["nz"])
    return (d3, d2, d1)  # i fastest


def _fdtd_fields(case, seed):
    g = _gen(seed)
    return [torch.rand(_shape(f, case), generator=g, device="cuda", dtype=F32) * 2 - 1 for f in range(6)]


def _fdtd_prepare(case, seed):
    nx, ny, nz, steps = case["nx"], case["ny"], case["nz"], case["steps"]
    p = FD.make_params(nx, ny, nz)
    src = _fdtd_fields(case, seed)
    sets = [[torch.zeros_like(a) for a in src] for _ in range(2)]
    cur, launches, turn = list(src), [], 0
    if case["form"] == "six":
        for s in range(steps):
            for name, own, a, b in FD.TASKS:
                out = sets[s % 2][own]
                grid, block = FD.default_geometry(*FD.extent(own, nx, ny, nz))
                launches.append((_fn("fdtd.hsaco", name), grid, block,
                                 FD.pack_task_args(H, cur[own].data_ptr(), cur[a].data_ptr(), cur[b].data_ptr(), p,
                                                   out.data_ptr())))
                cur[own] = out
    else:
        def whole(name, grid, block, out):
            args = H.ArgPack()
            for t in cur:
                args.ptr(t.data_ptr())
            args.raw(bytes(p), 4)
            for t in out:
                args.ptr(t.data_ptr())
            launches.append((_fn("fdtd_fused.hsaco", name), grid, block, args))

        for _ in range(steps // 3):
            whole("FdtdThreeStepPersistent", (_cus(), 1, 1), (64, 16, 1), sets[turn])
            cur, turn = sets[turn], turn ^ 1
        if steps % 3 == 2:
            whole("FdtdTwoStepOverlap", ((nx + 60) // 60, (ny + 12) // 12, (nz + 16) // 16), (64, 16, 1), sets[turn])
            cur, turn = sets[turn], turn ^ 1
        elif steps % 3 == 1:
            whole("FdtdStepOverlap8", ((nx + 62) // 62, (ny + 6) // 6, (nz + 8) // 8), (64, 8, 1), sets[turn])
            cur, turn = sets[turn], turn ^ 1
    return {"src": src, "sets": sets, "out": list(cur), "graph": _Recorded(launches)}


def _fdtd_run(case, s):
    s["graph"]()
    return s["out"]


def _yee(E, Hf, p, N, steps):
    """`steps` Yee steps in 64 bits; arrays indexed [k, j, i]."""
    nx, ny, nz = N
    cH, cE, Cx, Cy, Cz = p.Dt / p.mu0, p.Dt / p.eps0, p.Cx, p.Cy, p.Cz
    Ex, Ey, Ez = E
    Hx, Hy, Hz = Hf
    for _ in range(steps):
        Hx += cH * ((Ey[1:] - Ey[:-1]) * Cz - (Ez[:, 1:] - Ez[:, :-1]) * Cy)
        Hy += cH * ((Ez[:, :, 1:] - Ez[:, :, :-1]) * Cx - (Ex[1:] - Ex[:-1]) * Cz)
        Hz += cH * ((Ex[:, 1:] - Ex[:, :-1]) * Cy - (Ey[:, :, 1:] - Ey[:, :, :-1]) * Cx)
        if ny > 1 and nz > 1:
            Ex[1:-1, 1:-1] += cE * ((Hz[1:-1, 1:] - Hz[1:-1, :-1]) * Cy - (Hy[1:, 1:-1] - Hy[:-1, 1:-1]) * Cz)
        if nx > 1 and nz > 1:
            Ey[1:-1, :, 1:-1] += cE * ((Hx[1:, :, 1:-1] - Hx[:-1, :, 1:-1]) * Cz
                                       - (Hz[1:-1, :, 1:] - Hz[1:-1, :, :-1]) * Cx)
        if nx > 1 and ny > 1:
            Ez[:, 1:-1, 1:-1] += cE * ((Hy[:, 1:-1, 1:] - Hy[:, 1:-1, :-1]) * Cx
                                       - (Hx[:, 1:, 1:-1] - Hx[:, :-1, 1:-1]) * Cy)
    return [Hx, Hy, Hz, Ex, Ey, Ez]


def _fdtd_exact(case, seed):
    f = [a.to(F64) for a in _fdtd_fields(case, seed)]
    N = (case["nx"], case["ny"], case["nz"])
    return _yee(f[3:], f[:3], FD.make_params(*N), N, case["steps"])


def _cells(case):
    return sum(FD.elems(f, case["nx"], case["ny"], case["nz"]) for f in range(6))


# ---- GMM ---------------------------------------------------------------------------------------

def _gmm_data(case, seed):
    """Points of a seeded mixture (means U[-10,10), sd U[0.5,2)) and one initial mean per
    generating component, as the executor draws its GMM requests."""
    n, d, k = case["n"], case["d"], case["k"]
    g = _gen(seed)
    u = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=F32)  # noqa: E731
    means, sd = u(k, d) * 20 - 10, u(k, d) * 1.5 + 0.5
    c = torch.randint(0, k, (n,), generator=g, device="cuda")
    c[:k] = torch.arange(k, device="cuda")
    x = means[c] + sd[c] * torch.randn(n, d, generator=g, device="cuda", dtype=F32)
    return x.contiguous(), x[:k].to(F64)


def _gmm_prepare(case, seed):
    n, d, k, steps = case["n"], case["d"], case["k"], case["steps"]
    x, mu0 = _gmm_data(case, seed)
    o = GM.model_offsets(d, k, steps)
    m = np.zeros(GM.model_elems(d, k, steps))
    m[1:4] = (n, d, k)
    m[o["mu"]:o["var"]] = mu0.cpu().numpy().ravel()
    m[o["var"]:o["frac"]] = 1e-10
    m[o["frac"]:o["ll"]] = 1.0 / k
    GM.fill_table(m, d, k, steps)
    start = torch.from_numpy(m).cuda()
    model = start.clone()
    tiles = -(-n // 128)
    blocks = max(1, min(tiles, 768))
    part = torch.empty(blocks * GM.partial_stride(d, k), dtype=F64, device="cuda")
    dims = bytes(GM.Dims(n, d, k, blocks, steps))
    acc, fin = _fn("gmm.hsaco", "GmmAccumulateMfma"), _fn("gmm.hsaco", "GmmFinalize")
    launches = []
    for _ in range(steps):
        launches.append((acc, (blocks, 1, 1), (256, 1, 1),
                         H.ArgPack().ptr(x.data_ptr()).raw(dims).ptr(model.data_ptr()).ptr(part.data_ptr())))
        launches.append((fin, (k + 1, 1, 1), (256, 1, 1),
                         H.ArgPack().ptr(model.data_ptr()).ptr(part.data_ptr()).raw(dims)))
    return {"x": x, "start": start, "model": model, "part": part, "graph": _Recorded(launches)}


def _gmm_run(case, s):
    s["model"].copy_(s["start"])  # the initial model of this run
    s["graph"]()
    o, m = GM.model_offsets(case["d"], case["k"], case["steps"]), s["model"]
    return {"mu": m[o["mu"]:o["var"]], "var": m[o["var"]:o["frac"]], "frac": m[o["frac"]:o["ll"]],
            "loglike": m[o["ll"]:o["ll"] + case["steps"]]}


def _gmm_exact(case, seed):
    n, d, k, steps = case["n"], case["d"], case["k"], case["steps"]
    x32, mu = _gmm_data(case, seed)
    x = x32.t().to(F64).contiguous()  # D x N: every reduction below runs along contiguous rows
    var = torch.full((k, d), 1e-10, dtype=F64, device="cuda")
    frac = torch.full((k,), 1.0 / k, dtype=F64, device="cuda")
    ll = []
    for _ in range(steps):
        r = torch.empty(k, n, dtype=F64, device="cuda")
        for c in range(k):
            q = ((x - mu[c][:, None]).square_() * (1.0 / var[c])[:, None]).sum(0)
            r[c] = -0.5 * q - 0.5 * var[c].log().sum() + frac[c].log()
        t = torch.logsumexp(r, 0)
        ll.append(t.sum())
        r = r.sub_(t).exp_()
        w = r.sum(1)
        mu = torch.stack([(x * r[c]).sum(1) / w[c] for c in range(k)])
        var = torch.stack([((x - mu[c][:, None]).square_() * r[c]).sum(1) / w[c] for c in range(k)])
        frac = w / n
    return {"mu": mu.reshape(-1), "var": var.reshape(-1), "frac": frac, "loglike": torch.stack(ll)}


# ---- PCA ---------------------------------------------------------------------------------------

class _PcaDims(C.Structure):
    """PCA_DIMS (include/ptk_pca.h)."""
    _fields_ = [(f, C.c_int) for f in ("M", "N", "K", "J", "ld", "Mp", "G", "GR", "k", "center", "pad0", "pad1")]


def _pca_data(case, seed):
    """A matrix of decaying factors plus noise, column-major (M fastest)."""
    m, n = case["m"], case["n"]
    g = _gen(seed)
    q = min(24, n)
    w = 0.8 ** torch.arange(q, device="cuda", dtype=F32)
    a = torch.randn(n, q, generator=g, device="cuda", dtype=F32) * w
    b = torch.randn(q, m, generator=g, device="cuda", dtype=F32)
    return (a @ b + 0.3 * torch.randn(n, m, generator=g, device="cuda", dtype=F32)).contiguous()


def _pca_prepare(case, seed):
    M, N, K, J = case["m"], case["n"], case["k"], case["j"]
    x = _pca_data(case, seed)
    d = _PcaDims()
    d.M, d.N, d.K, d.J, d.center = M, N, K, J, 1
    d.ld, d.Mp = (N + 3) & ~3, (M + 63) // 64 * 64
    slabs = d.Mp // (8 if (d.ld // 4 + 255) // 256 <= 2 else 4)
    d.G = min(slabs, 3 * _cus() // 2)
    d.GR = min(d.G, 8)
    off_red = 8 * ((K + 1) & ~1) + 8 * ((d.G + 1) & ~1)
    off_p = off_red + 8 * d.GR * d.ld
    total = off_p + 4 * K * d.ld + 4 * d.G * d.ld
    R = torch.empty(d.Mp, d.ld, dtype=F32, device="cuda")
    T = torch.empty(K, d.Mp, dtype=F32, device="cuda")
    S = torch.zeros(total, dtype=torch.uint8, device="cuda")

    launches = []

    def add(name, bufs, k, grid, block):
        d.k = k
        a = H.ArgPack()
        if name == "PcaLoad":
            a.ptr(x.data_ptr()).raw(bytes(d)).ptr(R.data_ptr()).ptr(T.data_ptr()).ptr(S.data_ptr())
        else:
            for b in bufs:
                a.ptr(b.data_ptr())
            a.raw(bytes(d))
        launches.append((_fn("pca.hsaco", name), grid, block, a))

    rows, b256 = (d.G, 1, 1), (256, 1, 1)
    add("PcaLoad", (), 0, (d.Mp // 64, 1, 1), b256)
    for k in range(K):
        add("PcaStart", (R, T, S), k, rows, b256)
        if k > 0:
            add("PcaFinish", (S,), k - 1, (1, 1, 1), b256)
        for j in range(1, J + 1):
            add("PcaReduce", (S,), k, ((d.ld + 63) // 64, d.GR, 1), b256)
            add("PcaOrthonormalize", (S,), k, (1, 1, 1), (1024, 1, 1))
            if j < J:
                add("PcaGram", (R, S), k, rows, b256)
    add("PcaDeflate", (R, T, S), K - 1, rows, b256)
    add("PcaFinish", (S,), K - 1, (1, 1, 1), b256)
    L = S[:8 * K].view(F64)
    P = S[off_p:off_p + 4 * K * d.ld].view(F32).reshape(K, d.ld)
    return {"x": x, "R": R, "T": T, "S": S, "P": P, "L": L, "graph": _Recorded(launches)}


def _pca_run(case, s):
    s["graph"]()
    return {"R": s["R"], "T": s["T"], "P": s["P"], "L": s["L"]}


def _pca_exact(case, seed):
    M, N, K, J = case["m"], case["n"], case["k"], case["j"]
    r = _pca_data(case, seed).to(F64)  # N x M
    r -= r.mean(0)
    ld, Mp = (N + 3) & ~3, (M + 63) // 64 * 64
    T = torch.zeros(K, Mp, dtype=F64, device="cuda")
    P = torch.zeros(K, ld, dtype=F64, device="cuda")
    L = torch.zeros(K, dtype=F64, device="cuda")
    for k in range(K):
        t = r[k].clone()
        for _ in range(J):
            p = r.mv(t)
            if k:
                q = P[:k, :N]
                p = p - q.t().mv(q.mv(p))
            p = p / p.norm()
            t = p @ r
            L[k] = t.norm()
            t = t / L[k]
        r.addr_(p, t, alpha=-float(L[k]))
        T[k, :M], P[k, :N] = L[k] * t, p
    R = torch.zeros(Mp, ld, dtype=F64, device="cuda")
    R[:M, :N] = r.t()
    return {"R": R, "T": T, "P": P, "L": L}


# ---- scan --------------------------------------------------------------------------------------

def _scan_prepare(case, seed):
    n = case["n"]
    x = torch.randint(0, 200, (n,), generator=_gen(seed), device="cuda", dtype=torch.int32)
    out = torch.zeros_like(x)
    tiles = -(-n // 4096)
    sums = torch.empty(tiles, dtype=torch.int32, device="cuda")
    grid = (min(tiles, 2048), 1, 1)
    a = H.ArgPack().ptr(x.data_ptr()).i32(n).ptr(sums.data_ptr())
    b = H.ArgPack().ptr(x.data_ptr()).i32(n).ptr(sums.data_ptr()).ptr(out.data_ptr())
    return {"x": x, "out": out, "sums": sums,
            "graph": _Recorded([(_fn("scan.hsaco", "PfxScanReduce"), grid, (1024, 1, 1), a),
                                (_fn("scan.hsaco", "PfxScanApply"), grid, (1024, 1, 1), b)])}


def _scan_run(case, s):
    s["graph"]()
    return s["out"]


# ---- batch -------------------------------------------------------------------------------------

def _edges(case):
    n, lo, hi = case["fdtd"], case["edge_min"], case["edge_max"]
    return [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)]


def _instance_seed(seed, i):
    return (seed ^ ((i + 1) * 0x9E3779B97F4A7C15)) & (2**64 - 1)


def _batch_prepare(case, seed):
    need = sum(BT.footprint(BT.FDTD, e, e, e, case["steps"]) for e in _edges(case))
    need += case["groupby"] * BT.footprint(BT.GROUPBY, case["rows"], case["keys"])
    return {"ex": BT.Executor(need + (need >> 4) + (64 << 20)), "seed": seed}


def _batch_run(case, s):
    ex, seed = s["ex"], s["seed"]
    ids = [ex.submit_fdtd(e, e, e, case["steps"], _instance_seed(seed, i), keep=True)
           for i, e in enumerate(_edges(case))]
    gids = [ex.submit_groupby(case["rows"], case["keys"], 1.1, _instance_seed(seed, 1000 + i), keep=True)
            for i in range(case["groupby"])]
    ex.drain()
    fields = [np.concatenate([ex.read(i, f, np.float32) for f in range(6)]) for i in ids]
    tables = [[ex.read(i, w, t) for w, t in ((3, np.int64), (4, np.int32), (5, np.int32))] for i in gids]
    for i in ids + gids:
        ex.release(i)
    return {"fdtd": fields, "groupby": tables}


def _splitmix(x):
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def _batch_exact(case, seed):
    out = []
    with np.errstate(over="ignore"):
        for i, e in enumerate(_edges(case)):
            c = {"nx": e, "ny": e, "nz": e}
            f = []
            for q in range(6):  # uniform on [-1, 1): the top 24 bits of the counter-based generator
                key = np.uint64((_instance_seed(seed, i) ^ (q * 0xD1B54A32D192ED03)) & (2**64 - 1))
                r = _splitmix(_splitmix(np.array([key])) + np.arange(FD.elems(q, e, e, e), dtype=np.uint64))
                a = (r >> np.uint64(40)).astype(np.float64) / 8388608.0 - 1.0
                f.append(torch.from_numpy(a.reshape(_shape(q, c))))
            f = _yee(f[3:], f[:3], FD.make_params(e, e, e), (e, e, e), case["steps"])
            out.append(np.concatenate([t.numpy().reshape(-1) for t in f]))
    return {"fdtd": out, "groupby": [[None] * 3 for _ in range(case["groupby"])]}


# ---- the interface -----------------------------------------------------------------------------

_PREPARE = {"groupby": _groupby_prepare, "fdtd": _fdtd_prepare, "gmm": _gmm_prepare, "pca": _pca_prepare,
            "scan": _scan_prepare, "batch": _batch_prepare}
_RUN = {"groupby": _groupby_run, "fdtd": _fdtd_run, "gmm": _gmm_run, "pca": _pca_run, "scan": _scan_run,
        "batch": _batch_run}
_EXACT = {"fdtd": _fdtd_exact, "gmm": _gmm_exact, "pca": _pca_exact, "batch": _batch_exact}


def prepare(case, seed):
    return {"case": case, **_PREPARE[case["kind"]](case, seed)}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](case, state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, seed) if f else None


def work(case):
    kind = case["kind"]
    if kind == "groupby":
        K = case["keys"] + 1
        return {"bytes": 16 * case["n"] + 8 * K + 24 * min(K, case["n"]), "flops": 0}
    if kind == "fdtd":
        return {"bytes": 8 * _cells(case), "flops": 7 * _cells(case) * case["steps"]}
    if kind == "gmm":
        return {"bytes": 4 * case["n"] * case["d"], "flops": 8 * case["n"] * case["d"] * case["k"] * case["steps"]}
    if kind == "pca":
        mn = case["m"] * case["n"]
        return {"bytes": 8 * mn + 4 * case["k"] * (case["m"] + case["n"]),
                "flops": mn * case["k"] * (4 * case["j"] + 2)}
    if kind == "scan":
        return {"bytes": 8 * case["n"], "flops": case["n"]}
    cells = sum(_cells({"nx": e, "ny": e, "nz": e}) for e in _edges(case))
    return {"bytes": 4 * cells + case["groupby"] * (16 * case["rows"] + 8 * (case["keys"] + 1)),
            "flops": 7 * cells * case["steps"]}


def tolerance(case):
    """About four times the largest error against 64 bits seen over the ranges that draw() covers
    (rel: 2-norm; max: the largest difference over the result's root mean square)."""
    kind = case["kind"]
    if kind in ("groupby", "scan"):
        return "exact"
    if kind in ("fdtd", "batch"):  # 1.5e-6 after 50 steps
        return {"rel": 6e-6, "max": 1e-4}
    if kind == "gmm":  # 8.3e-7 and 3.7e-6 (mixing fractions of 64 overlapping components in 4-D)
        return {"rel": 4e-6, "max": 2e-5}
    return {"rel": 2e-6, "max": 3e-5}  # PCA: 3.8e-7 and 6.8e-6 (the residual)
