"""Performance cases of the library: what its users run, through the public
Python objects (the device builder through its C entry point), on matrices
of the library's generators with torch tensors as vectors.

A case is a dict: `op` (spmv, adjoint, fwd_adj, spmm, batch, build), the
matrix (`matrix`, `n` and the generator's parameters) and the plan's format
and options.  Plans, like a user's, are made once in `prepare`; `run` is one
call on them.
"""
import ctypes

import numpy as np
import torch

import gpu_spmv_amd as ax
from gpu_spmv_amd import _lib

_FORMATS = {
    "csr": (ax.FMT_CSR, dict(kernel=ax.KER_STREAM)),
    "k1": (ax.FMT_K1, {}),
    "axc": (ax.FMT_AXC, {}),
    "axt": (ax.FMT_AXT, {}),
    "axt_h4": (ax.FMT_AXT, dict(thw=64, th=4)),
    "axt_com": (ax.FMT_AXT, dict(thw=64, th=1, mode=ax.AXT_COM)),
    "rct": (ax.FMT_RCT, {}),
}


def listed():
    return [
        # One SpMV of a small Poisson problem (the 256^2 Laplacian): a Krylov
        # solver's inner call, bound by the launch.
        dict(name="laplace_256_csr", op="spmv", matrix="laplace", n=256, format="csr", f32=False),
        # The 2^20-row power-law matrix of the benchmark (a graph): FP64 SpMV
        # with the format meant for it ...
        dict(name="powerlaw_1m_rct", op="spmv", matrix="powerlaw", n=1 << 20, format="rct", f32=False),
        # ... and with the reference's own AXT layout, the default of a plan.
        dict(name="powerlaw_1m_axt", op="spmv", matrix="powerlaw", n=1 << 20, format="axt", f32=False),
        # A 3D mesh in scattered numbering (permuted 27-point stencil),
        # renumbered inside the plan.
        dict(name="stencil_100_rct_reorder", op="spmv", matrix="stencil", n=100, normal=False, permute=True, format="rct", f32=False,
             reorder=True),
        # The adjoint (a backward pass alone) of an unstructured matrix with
        # FP32 values in the K1 format, an odd number of rows.
        dict(name="random_300k_k1_f32_adjoint", op="adjoint", matrix="random", n=300007, lo=4, hi=40, format="k1", f32=True),
        # Forward + adjoint + value gradient of a least-squares loss: a
        # training step's work, on a graph ...
        dict(name="powerlaw_700k_rct_fwd_adj", op="fwd_adj", matrix="powerlaw", n=700001, format="rct", f32=False),
        # ... and on a mesh with learned weights, value gradient in CSR order.
        dict(name="stencil_80_axt_fwd_adj", op="fwd_adj", matrix="stencil", n=80, normal=True, permute=True, format="axt", f32=False,
             reorder=True),
        # Many right-hand sides on a graph: a few columns ...
        dict(name="powerlaw_600k_rct_spmm8", op="spmm", matrix="powerlaw", n=600000, format="rct", f32=False, k=8, tile_rows=1024, ktile=8),
        # ... and a feature matrix (tile options as the autotuner picks them).
        dict(name="powerlaw_400k_rct_spmm32", op="spmm", matrix="powerlaw", n=400003, format="rct", f32=False, k=32, tile_rows=256, ktile=16),
        # A block of vectors on a mesh in natural order, the default plan.
        dict(name="stencil_64_axt_spmm16", op="spmm", matrix="stencil", n=64, normal=False, permute=False, format="axt", f32=False, k=16),
        # Many uneven banded systems in one call.
        dict(name="banded_48_batch_rct", op="batch", matrix="banded", n=100000, count=48, hbw=64, format="rct", f32=False),
        # The AXT arrays (with x) rebuilt on the device from a device CSR, as
        # when a matrix changes every step; caller's arrays, no allocation.
        dict(name="powerlaw_256k_axt_build", op="build", matrix="powerlaw", n=1 << 18, thw=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_matrix(rng, most):
    """A matrix of about 16 x 1024 to `most` nonzeros."""
    kind = rng.choice(["laplace", "stencil", "powerlaw", "powerlaw", "banded", "random"])
    nnz = _log_int(rng, 16384, most)
    if kind == "laplace":
        return dict(matrix=kind, n=max(32, int((nnz / 5) ** 0.5)))
    if kind == "stencil":
        return dict(matrix=kind, n=max(9, int((nnz ** (1 / 3) + 2) / 3)), normal=rng.random() < 0.5, permute=rng.random() < 0.5)
    if kind == "powerlaw":
        return dict(matrix=kind, n=max(4097, nnz // 20))
    if kind == "banded":
        hbw = rng.randint(1, 64)
        return dict(matrix=kind, n=max(1000, int(nnz / (0.3 * (2 * hbw + 1)))) if nnz > 60 * hbw else 1000, hbw=hbw)
    lo = rng.randint(0, 12)
    hi = lo + rng.randint(1, 40)
    return dict(matrix=kind, n=max(1001, 2 * nnz // (lo + hi)), lo=lo, hi=hi)


def draw(rng):
    most = 0.9 * max(work(c)["bytes"] for c in listed())
    while True:
        c = _draw(rng)
        if work(c)["bytes"] <= most:
            return c


def _draw(rng):
    op = rng.choice(["spmv", "spmv", "spmv", "adjoint", "fwd_adj", "spmm", "spmm", "batch", "build"])
    f32 = rng.random() < 0.3
    if op == "batch":
        return dict(op=op, matrix="banded", n=_log_int(rng, 1001, 100000), count=_log_int(rng, 4, 48), hbw=rng.randint(1, 64),
                    format=rng.choice(["axt", "rct"]), f32=f32)
    if op == "build":
        return dict(op=op, thw=rng.choice([2, 4, 8, 16]), **_draw_matrix(rng, 5_000_000))
    if op == "spmm":
        c = dict(op=op, f32=f32, **_draw_matrix(rng, 8_000_000))
        c["k"] = rng.choice([rng.randint(1, 16), rng.randint(8, 32)])
        c["format"] = rng.choice(["rct", "rct", "axt", "csr", "axc"])
        if c["format"] == "rct":
            c["ktile"] = 8 if c["k"] <= 8 else 16
            c["tile_rows"] = 1024 if c["k"] <= 8 else rng.choice([256, 512])
        return c
    c = dict(op=op, f32=f32, **_draw_matrix(rng, 14_000_000 if op == "fwd_adj" else 20_000_000))
    c["format"] = rng.choice(["rct", "axt"]) if op == "fwd_adj" else rng.choice(["rct", "rct", "axt", "csr", "k1", "axc", "axt_h4", "axt_com"])
    if c["matrix"] == "stencil" and c["permute"]:
        c["reorder"] = rng.random() < 0.7
    return c


# ---------------------------------------------------------------- inputs
def _one_matrix(case, seed):
    kind, n = case["matrix"], case["n"]
    if kind == "laplace":
        return ax.laplace2d(n)
    if kind == "stencil":
        m = ax.stencil27(n, permute=case["permute"], seed=seed)
        if case["normal"]:
            ax.fill_values_normal(m, 1.0, 0.1, seed + 1)
        return m
    if kind == "powerlaw":
        return ax.powerlaw(n, 2.0, 2048, 20.0, seed=seed)
    if kind == "banded":
        return ax.banded(n, case["hbw"], 0.3, seed=seed)
    return ax.random_sparse(n, case["lo"], case["hi"], seed=seed)


def _shapes(case):
    """(rows, half-bandwidth) of a batch's members, the same for every seed."""
    rng = np.random.default_rng(5)
    return [(int(rng.integers(max(1, case["n"] // 100), case["n"] + 1)), int(rng.integers(1, case["hbw"] + 1)))
            for _ in range(case["count"])]


def _matrices(case, seed):
    if case["op"] in ("fwd_adj", "build"):  # one pattern, new values: what training and a changing matrix have
        m = _one_matrix(case, 11)
        ax.fill_values_normal(m, 1.0 if case.get("normal") else 0.0, 0.1 if case.get("normal") else 1.0, seed)
        return [m]
    if case["op"] != "batch":
        return [_one_matrix(case, seed)]
    return [ax.banded(n, h, 0.3, seed=1000 * seed + i) for i, (n, h) in enumerate(_shapes(case))]


def _vectors(case, seed, nrows, ncols):
    """The case's input tensors, U[-1, 1)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def u(n):
        return torch.rand(n, dtype=torch.float64, device="cuda", generator=g) * 2 - 1

    op = case["op"]
    if op == "adjoint":
        return dict(ybar=u(nrows))
    if op == "fwd_adj":
        return dict(x=u(ncols), b=u(nrows))
    if op == "spmm":
        return dict(X=u(ncols * case["k"]))
    return dict(x=u(ncols))


def _empty(n, dtype=torch.float64):
    return torch.empty(n, dtype=dtype, device="cuda")


def _device_csr(m):
    return (torch.from_numpy(m.row.view(np.int32)).cuda(), torch.from_numpy(m.col.view(np.int32)).cuda(),
            torch.from_numpy(m.val).cuda())


def prepare(case, seed):
    mats = _matrices(case, seed)
    m = mats[0]
    nrows, ncols = sum(a.nrows for a in mats), sum(a.ncols for a in mats)
    v = _vectors(case, seed, nrows, ncols)
    op = case["op"]
    if op == "build":
        row, col, val = _device_csr(m)
        thw = case["thw"]
        tiles = int(((np.diff(m.row.astype(np.int64)) + thw - 1) // thw).sum())
        out = dict(ax=_empty(2 * thw * tiles), sec=_empty(tiles, torch.int32), con=_empty(nrows + 1, torch.int32),
                   plane=_empty(thw * tiles, torch.int32))
        f = _lib.Dfmt(lenAX=2 * thw * tiles, lenSEC=tiles, lenCON=nrows, lenMAPX=thw * tiles,
                      **{k: t.data_ptr() for k, t in out.items()})
        a = _lib.Dcsr(nrows, ncols, m.nnz, 0, row.data_ptr(), col.data_ptr(), val.data_ptr())
        return dict(op=op, a=a, f=f, thw=thw, out=out, keep=(row, col, val), **v)
    fmt, opts = _FORMATS[case["format"]]
    opts = dict(opts, vtype=ax.F32 if case["f32"] else ax.F64, **{k: case[k] for k in ("tile_rows", "ktile") if k in case})
    if op == "batch":
        return dict(op=op, batch=ax.Batch(mats, fmt=fmt, **opts), y=_empty(nrows), **v)
    flags = (ax.PLAN_REORDER if case.get("reorder") else 0) | (ax.PLAN_TRANSPOSE if op in ("adjoint", "fwd_adj") else 0)
    s = dict(op=op, plan=ax.Plan(m, fmt, flags=flags, **opts), **v)
    if op == "spmv":
        s.update(y=_empty(nrows))
    elif op == "adjoint":
        s.update(xbar=_empty(ncols))
    elif op == "fwd_adj":
        s.update(y=_empty(nrows), r=_empty(nrows), xbar=_empty(ncols), vbar=_empty(m.nnz))
    else:
        s.update(k=case["k"], Y=_empty(nrows * case["k"]))
    return s


def run(s):
    op = s["op"]
    stream = torch.cuda.current_stream().cuda_stream
    if op == "spmv":
        s["plan"].spmv(s["x"], s["y"], stream=stream)
        return s["y"]
    if op == "adjoint":
        s["plan"].adjoint(s["ybar"], s["xbar"], stream=stream)
        return s["xbar"]
    if op == "fwd_adj":
        s["plan"].fwd_adj(s["x"], s["b"], s["y"], s["r"], s["xbar"], s["vbar"], stream=stream)
        return {k: s[k] for k in ("y", "r", "xbar", "vbar")}
    if op == "spmm":
        s["plan"].spmm(s["k"], s["X"], s["Y"], stream=stream)
        return s["Y"]
    if op == "batch":
        s["batch"].spmv(s["x"], s["y"], stream=stream)
        return s["y"]
    _lib.call("axspmv_dev_build_axt_noalloc", ctypes.byref(s["a"]), s["x"].data_ptr(), 256, s["thw"], 1, ax.AXT_UNC, stream,
              ctypes.byref(s["f"]))
    return s["out"]


# ------------------------------------------------------------------ work
def _size(case):
    """(rows, nonzeros): exact for the meshes, the expected count elsewhere."""
    kind, n = case["matrix"], case["n"]
    if kind == "laplace":
        return n * n, 5 * n * n - 4 * n
    if kind == "stencil":
        return n ** 3, (3 * n - 2) ** 3
    if kind == "powerlaw":
        return n, 20 * n
    if kind == "banded":
        shapes = _shapes(case) if case["op"] == "batch" else [(n, case["hbw"])]
        return sum(r for r, _ in shapes), sum(0.3 * (r * (2 * h + 1) - h * (h + 1)) for r, h in shapes)
    return n, n * (case["lo"] + case["hi"]) / 2


def work(case):
    """CSR bytes of the matrix, every vector once; multiply-adds."""
    n, nnz = _size(case)
    op = case["op"]
    if op == "build":  # CSR and x in; slots of a value, an x value and a column, a header per tile, row starts out
        return dict(bytes=12 * nnz + 4 * n + 8 * n + nnz * (20 + 4 / case["thw"]) + 4 * n, flops=0)
    matrix = (8 if case["f32"] else 12) * nnz + 4 * (n + 1)
    if op == "fwd_adj":  # x, b in; y, r, x_bar out; one gradient per nonzero
        return dict(bytes=matrix + 5 * 8 * n + 8 * nnz, flops=5 * nnz)
    k = case.get("k", 1)
    return dict(bytes=matrix + 16 * n * k, flops=2 * nnz * k)


# ----------------------------------------------------------------- exact
def exact(case, seed):
    op = case["op"]
    if op == "build":
        return None  # copies of values: compared byte for byte
    y = []
    mats = _matrices(case, seed)
    v = _vectors(case, seed, sum(m.nrows for m in mats), sum(m.ncols for m in mats))
    x0 = 0
    for m in mats:
        row, col, val = _device_csr(m)
        if case["f32"]:
            val = val.to(torch.float32).to(torch.float64)
        col = col.long()
        rid = torch.repeat_interleave(torch.arange(m.nrows, device="cuda"), (row[1:] - row[:-1]).long())
        zr, zc = torch.zeros(m.nrows, dtype=torch.float64, device="cuda"), torch.zeros(m.ncols, dtype=torch.float64, device="cuda")
        if op == "adjoint":
            return zc.index_add_(0, col, val * v["ybar"][rid])
        if op == "spmm":
            k = case["k"]
            X = v["X"].view(m.ncols, k)
            cols = [torch.zeros_like(zr).index_add_(0, rid, val * X[:, j].contiguous()[col]) for j in range(k)]
            return torch.stack(cols, dim=1).reshape(-1)
        x = v["x"][x0:x0 + m.ncols]
        x0 += m.ncols
        y.append(zr.index_add_(0, rid, val * x[col]))
        if op == "fwd_adj":
            r = y[0] - v["b"]
            # the RCT plans' gradient has the plan's entry order, a reordered plan's too
            plain = case["format"] != "rct" and not case.get("reorder")
            return dict(y=y[0], r=r, xbar=zc.index_add_(0, col, val * r[rid]), vbar=r[rid] * x[col] if plain else None)
    return torch.cat(y)
