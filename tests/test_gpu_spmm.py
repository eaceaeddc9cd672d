"""GPU: SpMM kernels at the sizes where they can go wrong -- row lengths
around a batch of entries and around the long-row limit, odd and even numbers
of right-hand sides, operands off 16 bytes, X beyond 32-bit byte offsets --
against the oracle's spmm.  Tolerance: FP64 sums of at most 2600 products,
1e-12 of the largest entry as in the other parity tests."""
import numpy as np
import pytest

import gpu_spmv_amd as ax
from conftest import rel_err
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
TOL = 1e-12


def edge_rows():
    lens = [0, 1, 7, 8, 9, 15, 16, 17, 0, 31, 32, 33, 255, 256, 257, 271, 272, 273, 2600, 0, 4] + [3, 5, 8, 16, 2] * 20
    rng = np.random.default_rng(3)
    row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    n = 3001
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens]).astype(np.uint32)
    return ax.CsrMatrix(row, col, rng.standard_normal(col.size), ncols=n)


EDGE = edge_rows()
BAND = ax.banded(3001, 3, 0.5, seed=6)  # narrow band: 16-bit keys
RCT = [("packed", EDGE, dict(tile_rows=256)), ("s4", EDGE, dict(tile_rows=200, slices=4)),
       ("split_f32", EDGE, dict(tile_rows=300, flags=ax.PLAN_RCT_SPLIT, vtype=ax.F32)), ("k16", BAND, dict(tile_rows=128)),
       ("block64", EDGE, dict(tile_rows=64, block=64))]
ROWWISE = [(ax.FMT_AXT, dict(thw=4)), (ax.FMT_CSR, {}), (ax.FMT_AXC, dict(hbs=2, vtype=ax.F32))]


def spmm(plan, m, X, off=0):
    """Y of one call with X and Y `off` doubles past their buffers' start;
    the words before and after Y must stay untouched."""
    k = X.shape[1]
    n = m.nrows * k
    dX = ax.DeviceBuffer.from_array(np.concatenate([np.full(off, np.nan), X.ravel()]))
    dY = ax.DeviceBuffer.from_array(np.full(n + off + 1, np.nan))
    plan.spmm(k, dX.ptr + 8 * off, dY.ptr + 8 * off)
    ax._lib.call("axspmv_device_sync")
    Y = dY.download(np.float64, n + off + 1)
    assert np.isnan(Y[-1]) and np.all(np.isnan(Y[:off]))
    return Y[off:-1].reshape(m.nrows, k)


def f32_values(m, kw):
    if kw.get("vtype") != ax.F32:
        return m
    return ax.CsrMatrix(m.row, m.col, m.val.astype(np.float32).astype(np.float64), ncols=m.ncols)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("k,kt", [(1, 0), (2, 0), (7, 0), (8, 0), (16, 0), (17, 16), (18, 16), (32, 0), (33, 32), (64, 0), (66, 64)])
@pytest.mark.parametrize("fmt,kw", ROWWISE, ids=["axt", "csr", "axc_f32"])
def test_rowwise_edges(fmt, kw, k, kt, off):
    X = ax.uniform(70 + k, EDGE.ncols * k).reshape(EDGE.ncols, k)
    Y = spmm(ax.Plan(EDGE, fmt, ktile=kt, **kw), EDGE, X, off)
    assert rel_err(orc.spmm(f32_values(EDGE, kw), X), Y) <= TOL


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("k,kt", [(1, 0), (2, 8), (7, 8), (8, 8), (16, 16), (17, 16), (18, 16), (32, 32), (33, 32), (64, 64), (66, 64)])
@pytest.mark.parametrize("m,kw", [r[1:] for r in RCT], ids=[r[0] for r in RCT])
def test_rct_edges(m, kw, k, kt, off):
    X = ax.uniform(90 + k, m.ncols * k).reshape(m.ncols, k)
    Y = spmm(ax.Plan(m, ax.FMT_RCT, ktile=kt, **kw), m, X, off)
    assert rel_err(orc.spmm(f32_values(m, kw), X), Y) <= TOL


@pytest.mark.parametrize("fmt,kw", ROWWISE + [(ax.FMT_RCT, dict(tile_rows=4, slices=2))], ids=["axt", "csr", "axc_f32", "rct"])
def test_x_of_4_gb(fmt, kw):
    """X of 4.3 GB: row offsets beyond 32 bits."""
    ncols, k = (1 << 23) + 5, 64
    rng = np.random.default_rng(8)
    lens = np.array([0, 5, 300, 40, 17])
    row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    col = np.concatenate([np.sort(rng.choice(ncols, n, replace=False)) for n in lens]).astype(np.uint32)
    col[-1] = ncols - 1
    m = ax.CsrMatrix(row, col, rng.standard_normal(col.size), ncols=ncols)
    # only the X rows that the matrix reads are filled
    used = np.unique(col)
    X = ax.uniform(9, used.size * k).reshape(used.size, k)
    dX = ax.DeviceBuffer(8 * ncols * k)
    for c, xr in zip(used, X):
        ax._lib.call("axspmv_memcpy_h2d", dX.ptr + 8 * k * int(c), xr.ctypes.data, xr.nbytes, None)
    ax._lib.call("axspmv_device_sync")
    dY = ax.DeviceBuffer.from_array(np.full(m.nrows * k, np.nan))
    ax.Plan(m, fmt, **kw).spmm(k, dX, dY)
    xs, val = X[np.searchsorted(used, col)], f32_values(m, kw).val
    ref = np.stack([val[a:b] @ xs[a:b] for a, b in zip(row[:-1].astype(int), row[1:].astype(int))])
    assert rel_err(ref, dY.download(np.float64, m.nrows * k).reshape(m.nrows, k)) <= TOL


# ------------------------------------------- heavy rows (RCT plans for SpMM)
def heavy_matrix():
    """70,001 rows, over 65,536 columns, a fifteenth of the rows holding most
    of the entries, the first and the last row among them."""
    n = 70001
    rng = np.random.default_rng(12)
    lens = rng.integers(0, 6, n)
    big = np.concatenate([[0, n - 1], rng.choice(np.arange(1, n - 1), n // 15, replace=False)])
    lens[big] = rng.integers(32, 200, big.size)
    lens[0] = 2500
    row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    col = rng.integers(0, n, int(row[-1])).astype(np.uint32)  # unsorted, repeats: every entry is summed
    return ax.CsrMatrix(row, col, rng.standard_normal(col.size), ncols=n)


HEAVY = heavy_matrix()
HEAVY_PLANS = [dict(tile_rows=1024), dict(tile_rows=250, slices=4), dict(tile_rows=512, flags=ax.PLAN_RCT_SPLIT),
               dict(tile_rows=2048, slices=2, vtype=ax.F32, block=256)]


def has_heavy(plan, kw):
    return plan.info()["nblocks"] > -(-HEAVY.nrows // kw["tile_rows"]) * kw.get("slices", 1)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("k", [1, 6, 16, 21])
@pytest.mark.parametrize("kw", HEAVY_PLANS, ids=["r1024", "r250_s4", "split", "f32_s2"])
def test_heavy_rows_spmm(kw, k, off):
    X = ax.uniform(110 + k, HEAVY.ncols * k).reshape(HEAVY.ncols, k)
    p = ax.Plan(HEAVY, ax.FMT_RCT, **kw)
    assert has_heavy(p, kw)
    for _ in range(2):  # the second call's heavy rows start from the first one's sums: cleared
        assert rel_err(orc.spmm(f32_values(HEAVY, kw), X), spmm(p, HEAVY, X, off)) <= TOL


@pytest.mark.parametrize("kw", HEAVY_PLANS, ids=["r1024", "r250_s4", "split", "f32_s2"])
def test_heavy_rows_spmv_and_fwd_adj(kw):
    m = HEAVY
    ref_m = f32_values(m, kw)
    x, b = ax.uniform(5, m.ncols), ax.uniform(6, m.nrows)
    p = ax.Plan(m, ax.FMT_RCT, **dict(kw, flags=kw.get("flags", 0) | ax.PLAN_TRANSPOSE))
    assert has_heavy(p, kw)
    y = orc.ncsr(ref_m, x)
    for _ in range(2):
        assert rel_err(y, ax.spmv_host(p, x)) <= TOL
    dx, db = ax.DeviceBuffer.from_array(x), ax.DeviceBuffer.from_array(b)
    dy, dr, dxb = (ax.DeviceBuffer.from_array(np.full(m.nrows, np.nan)) for _ in range(3))
    dv = ax.DeviceBuffer(8 * m.nnz)
    for fused in (True, False):
        p.fwd_adj(dx, db, dy, dr, dxb, dv, fused=fused)
        assert rel_err(y, dy.download(np.float64, m.nrows)) <= TOL
        r = dr.download(np.float64, m.nrows)
        assert np.array_equal(r, dy.download(np.float64, m.nrows) - b)
        assert rel_err(orc.ncsr_t(ref_m, r, m.ncols), dxb.download(np.float64, m.ncols)) <= TOL
        assert np.array_equal(p.vbar_csr(dv.download(np.float64, m.nnz)), r[m.row_ids()] * x[m.col])


def test_heavy_rows_graph():
    """Replays of a captured SpMM clear the heavy rows each time."""
    k = 8
    X = ax.uniform(120, HEAVY.ncols * k).reshape(HEAVY.ncols, k)
    p = ax.Plan(HEAVY, ax.FMT_RCT, tile_rows=1024)
    dX, dY = ax.DeviceBuffer.from_array(X), ax.DeviceBuffer(8 * HEAVY.nrows * k)
    g = ax.Graph.of_plan(p, ax._lib.OP_SPMM, repeats=2, X=dX, Y=dY, k=k)
    ref = orc.spmm(HEAVY, X)
    for _ in range(3):
        dY.upload(np.full(HEAVY.nrows * k, np.nan))
        g.launch()
        ax._lib.call("axspmv_device_sync")
        assert rel_err(ref, dY.download(np.float64, HEAVY.nrows * k).reshape(HEAVY.nrows, k)) <= TOL


@pytest.mark.parametrize("vtype", [ax.F64, ax.F32])
@pytest.mark.parametrize("fmt", [ax.FMT_AXT, ax.FMT_CSR, ax.FMT_AXC])
def test_short_rows_of_scattered_columns(fmt, vtype):
    """More than 65,536 columns read without locality by short rows only: one
    right-hand side per lane at k-tile 8, whole and partial tiles."""
    m = ax.random_sparse(66001, 0, 9, seed=14)
    ref = m if vtype == ax.F64 else ax.CsrMatrix(m.row, m.col, m.val.astype(np.float32).astype(np.float64), ncols=m.ncols)
    for k in (1, 7, 8, 16):
        X = ax.uniform(15, m.ncols * k).reshape(m.ncols, k)
        p = ax.Plan(m, fmt, vtype=vtype, ktile=8)
        dX, dY = ax.DeviceBuffer.from_array(X), ax.DeviceBuffer.from_array(np.full(m.nrows * k, np.nan))
        p.spmm(k, dX, dY)
        assert rel_err(orc.spmm(ref, X), dY.download(np.float64, m.nrows * k).reshape(m.nrows, k)) <= 1e-12


# Heavy rows are for plans meant for SpMM.
GRAPH = ax.powerlaw(100001, 2.0, 2048, 20.0, seed=31)


@pytest.mark.parametrize("kw,heavy", [
    (dict(), False), (dict(flags=ax.PLAN_TRANSPOSE), False), (dict(slices=4), False),
    (dict(ktile=8), True), (dict(ktile=8, vtype=ax.F32), True), (dict(tile_rows=448), True),
    (dict(ktile=8, flags=ax.PLAN_DETERMINISTIC), False), (dict(tile_rows=448, slices=4, flags=ax.PLAN_DETERMINISTIC), False)])
def test_heavy_rows_by_intent(kw, heavy):
    """Neither the default plan nor a deterministic one keeps heavy rows apart:
    one launch per SpMV, with column slices partials and their merge."""
    p = ax.Plan(GRAPH, ax.FMT_RCT, **kw)
    info = p.info()
    S = kw.get("slices", 1)
    assert (info["nblocks"] > 1.05 * GRAPH.nrows / int(info["name"].split("_")[1][1:]) * S + S) == heavy, info
    assert info["launches"] == (2 if heavy or S > 1 else 1)
    assert heavy or not info["name"].endswith("_atomic")
    mv = f32_values(GRAPH, kw)
    x = ax.uniform(32, GRAPH.ncols)
    assert rel_err(orc.ncsr(mv, x), ax.spmv_host(p, x)) <= TOL
    X = ax.uniform(33, GRAPH.ncols * 5).reshape(GRAPH.ncols, 5)
    assert rel_err(orc.spmm(mv, X), spmm(p, GRAPH, X)) <= TOL


def test_heavy_rows_not_beside_automatic_slices():
    """Column slices that the plan chooses itself replace heavy rows; slices
    that the caller asks for do not."""
    m = ax.powerlaw(270001, 2.0, 2048, 20.0, seed=34)
    X = ax.uniform(35, m.ncols * 3).reshape(m.ncols, 3)
    for kw, heavy in ((dict(ktile=8), False), (dict(ktile=8, tile_rows=2112), False), (dict(ktile=8, slices=2), True)):
        p = ax.Plan(m, ax.FMT_RCT, **kw)
        info = p.info()
        assert info["name"].startswith("rct_r2112_s2"), info
        assert (info["nblocks"] > 1.05 * m.nrows / 2112 * 2 + 2) == heavy, (kw, info)
        assert rel_err(orc.spmm(m, X), spmm(p, m, X)) <= TOL


@pytest.mark.parametrize("n,signs,kw,saved_bits", [
    (300001, False, dict(tile_rows=1024), 8),                    # 72 MB: 24-bit keys
    (450001, False, dict(tile_rows=1024, vtype=ax.F32), 8),
    (100001, True, dict(tile_rows=448), 0),                      # values from a table, 32-bit keys
    (200001, True, dict(tile_rows=1024), 8),                     # both (73 MB in 32-bit keys)
    (100001, True, dict(tile_rows=448, flags=ax.PLAN_RCT_SPLIT), 0),
], ids=["k24", "k24_f32", "table", "k24_table", "split_table"])
def test_heavy_rows_with_short_keys_and_tables(n, signs, kw, saved_bits):
    """Heavy rows, whose tiles lie after the ordinary ones, with every way of
    storing a key and a value: SpMM, SpMV, forward + adjoint."""
    if n == 200001:  # 25 entries a row, 600 in one of 12
        rng = np.random.default_rng(n)
        lens = np.where(np.arange(n) % 12 == 5, 600, 25)
        row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
        m = ax.CsrMatrix(row, rng.integers(0, n, int(row[-1])).astype(np.uint32), rng.standard_normal(int(row[-1])), ncols=n)
    else:
        m = ax.powerlaw(n, 2.0, 2048, 20.0, seed=n)
    plain = ax.Plan(m, ax.FMT_RCT, **kw).info()
    if signs:
        m = ax.CsrMatrix(m.row, m.col, np.where(m.val < 0, -1.0, 1.0), ncols=m.ncols)
    flags = kw.get("flags", 0)
    p = ax.Plan(m, ax.FMT_RCT, **dict(kw, flags=flags | ax.PLAN_TRANSPOSE))
    info = p.info()
    wide = ax.Plan(m, ax.FMT_RCT, **dict(kw, flags=flags | ax.PLAN_RCT_WIDE_KEY)).info()
    assert info["nblocks"] > 1.05 * n / kw["tile_rows"] + 1
    assert abs(8 * (wide["stream_bytes"] - info["stream_bytes"]) / m.nnz - saved_bits) < 0.3
    if signs:  # 8 bytes a value before, 1 now
        assert info["stream_bytes"] < plain["stream_bytes"] - 6.5 * m.nnz
    mv = f32_values(m, kw)
    for k in (2, 5):
        X = ax.uniform(130 + k, n * k).reshape(n, k)
        assert rel_err(orc.spmm(mv, X), spmm(p, m, X)) <= TOL
    x, b = ax.uniform(136, n), ax.uniform(137, n)
    dx, db = ax.DeviceBuffer.from_array(x), ax.DeviceBuffer.from_array(b)
    dy, dr, dxb = (ax.DeviceBuffer.from_array(np.full(n, np.nan)) for _ in range(3))
    dv = ax.DeviceBuffer(8 * m.nnz)
    p.fwd_adj(dx, db, dy, dr, dxb, dv)
    y, r = dy.download(np.float64, n), dr.download(np.float64, n)
    assert rel_err(orc.ncsr(mv, x), y) <= TOL and np.array_equal(r, y - b)
    assert rel_err(orc.ncsr_t(mv, r, n), dxb.download(np.float64, n)) <= TOL
    assert np.array_equal(p.vbar_csr(dv.download(np.float64, m.nnz)), r[m.row_ids()] * x[m.col])


BIG, MID = (ax.powerlaw(n, 2.0, 2048, 20.0, seed=38) for n in (660001, 300001))
NONFINITE = [("axt", EDGE, ax.FMT_AXT, {}), ("csr", EDGE, ax.FMT_CSR, {}), ("axc", EDGE, ax.FMT_AXC, dict(hbs=2)),
             ("rct", EDGE, ax.FMT_RCT, dict(tile_rows=256)), ("rct_s4", EDGE, ax.FMT_RCT, dict(tile_rows=200, slices=4)),
             ("k16", BAND, ax.FMT_RCT, dict(tile_rows=128)), ("heavy", HEAVY, ax.FMT_RCT, dict(tile_rows=1024)),
             ("axt_seq", BIG, ax.FMT_AXT, {}), ("k24", BIG, ax.FMT_RCT, {}), ("k24_heavy", MID, ax.FMT_RCT, dict(tile_rows=1024))]


@pytest.mark.parametrize("m,fmt,kw", [c[1:] for c in NONFINITE], ids=[c[0] for c in NONFINITE])
def test_nonfinite_x_stays_in_its_rows_and_columns(m, fmt, kw):
    """X[0] = inf and X[1] = nan in one right-hand side: only the rows holding
    these columns become non-finite, and there only that right-hand side --
    not through lanes past a row's or tile's end or past the last right-hand
    side."""
    p = ax.Plan(m, fmt, **kw)
    if m is BIG or m is MID:  # the path is the one meant
        info = p.info()
        if fmt == ax.FMT_AXT:
            assert "_seq" in info["name"]
        else:
            wide = ax.Plan(m, fmt, **dict(kw, flags=ax.PLAN_RCT_WIDE_KEY)).info()
            assert info["stream_bytes"] < wide["stream_bytes"] - 0.9 * m.nnz
            assert (info["nblocks"] > 1.05 * m.nrows / 1024 + 1) == bool(kw)

    def check(ref, got):
        fin = np.isfinite(ref)
        assert fin.any() and not fin.all()
        np.testing.assert_array_equal(got[~fin], ref[~fin])
        assert rel_err(ref[fin], got[fin]) <= TOL

    x = ax.uniform(140, m.ncols)
    used = np.unique(m.col)[[0, -1]]
    x[used] = np.inf, np.nan
    check(orc.ncsr(m, x), ax.spmv_host(p, x))
    if kw.get("tile_rows", 0) == 0 and fmt == ax.FMT_RCT:
        return  # tiles too tall for SpMM
    for k, j in ((3, 0), (8, 7), (6, 3)):
        X = ax.uniform(141 + k, m.ncols * k).reshape(m.ncols, k)
        X[used, j] = np.inf, np.nan
        check(orc.spmm(m, X), spmm(p, m, X))
