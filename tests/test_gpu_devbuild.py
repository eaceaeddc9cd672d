"""GPU: format builders on the device against the host builders.

axspmv_dev_build_axt / axspmv_dev_build_axc build the reference's AXT and
AXC arrays (getFormatDataAXT cudaSpmv.cu:1391-1566, getFormatDataAXC
cudaSpmv.cu:1004-1062) with kernels.  Bar: every array equal, bit for bit,
to the host builder's (which test_builders.py pins to the reference's own
builders compiled from its sources, and to the oracle's restatement).
"""
import ctypes as C

import numpy as np
import pytest

import gpu_spmv_amd as ax
from gpu_spmv_amd import _lib as L
from conftest import FIXTURES, FixtureMatrix

pytestmark = pytest.mark.gpu


def mats():
    out = {name: FixtureMatrix(name).csr() for name in FIXTURES}
    out["powerlaw64k"] = ax.powerlaw(1 << 16, 2.0, 2048, 20.0, seed=1)
    out["stencil12p"] = ax.stencil27(12, permute=True, seed=2)
    out["banded_empty"] = ax.banded(3000, 2, 0.3, seed=6)
    out["empty"] = ax.CsrMatrix(np.zeros(6, np.uint32), np.zeros(0, np.uint32), np.zeros(0), ncols=5)
    return out


MATS = mats()
AXT = [(256, 4, 1, ax.AXT_UNC), (256, 16, 1, ax.AXT_UNC), (256, 32, 1, ax.AXT_UNC), (256, 3, 1, ax.AXT_UNC),
       (256, 32, 4, ax.AXT_UNC), (256, 64, 8, ax.AXT_UNC), (256, 32, 6, ax.AXT_UNC),
       (256, 64, 1, ax.AXT_COM), (64, 32, 1, ax.AXT_COM), (2, 4, 1, ax.AXT_COM),
       (256, 64, 4, ax.AXT_COM), (256, 32, 16, ax.AXT_COM)]


@pytest.mark.parametrize("mname", list(MATS))
@pytest.mark.parametrize("bs,thw,th,mode", AXT, ids=[f"bs{a}_thw{b}_th{c}_m{d}" for a, b, c, d in AXT])
def test_dev_build_axt_equals_host(mname, bs, thw, th, mode):
    m = MATS[mname]
    x = ax.uniform(41, max(m.ncols, 1))[:m.ncols]
    h = ax.build_axt(m, x, bs, thw, th, mode)
    d = ax.dev_build_axt(m, x, bs, thw, th, mode)
    assert d["name"] == h["name"]
    for k in ("tileN", "lenAX", "lenSEC", "lenCON", "log"):
        assert d[k] == h[k], k
    assert np.array_equal(d["ax"], h["ax"])
    assert np.array_equal(d["sec"], h["sec"])
    assert np.array_equal(d["con"], h["con"])
    assert np.array_equal(d["plane"], h["cplane"])
    assert d["ms"] > 0 or m.nrows == 0


@pytest.mark.parametrize("mname", list(MATS))
@pytest.mark.parametrize("hbs", [1, 4, 32, 64, 24])
def test_dev_build_axc_equals_host(mname, hbs):
    m = MATS[mname]
    x = ax.uniform(42, max(m.ncols, 1))[:m.ncols]
    h = ax.build_axc(m, x, hbs)
    d = ax.dev_build_axc(m, x, hbs)
    assert d["name"] == "faxc" and d["lenAX"] == h["lenAX"] and d["lenMAPX"] == h["lenMAPX"]
    assert np.array_equal(d["ax"], h["ax"])
    assert np.array_equal(d["con"], h["brp"])
    assert np.array_equal(d["plane"], h["mapx"])


def test_dev_build_without_x_leaves_x_halves_zero():
    m = MATS["plaw512"]
    x = ax.uniform(43, m.ncols)
    h = ax.build_axt(m, x, 256, 8, 1, ax.AXT_UNC)
    d = ax.dev_build_axt(m, None, 256, 8, 1, ax.AXT_UNC)
    g, gh = d["ax"].reshape(-1, 2, 8), h["ax"].reshape(-1, 2, 8)
    assert np.array_equal(g[:, 0], gh[:, 0]) and not np.any(g[:, 1])


def test_dev_build_rejects_what_the_host_rejects():
    m = MATS["toy12"]
    for args in ((256, 0, 1, ax.AXT_UNC), (256, 4, 0, ax.AXT_UNC), (3, 4, 1, ax.AXT_COM), (256, 4, 3, ax.AXT_COM),
                 (256, 4, 1, 7)):
        with pytest.raises(ax.AxspmvError):
            ax.build_axt(m, None, *args, flags=ax.BUILD_PLANES)
        with pytest.raises(ax.AxspmvError):
            ax.dev_build_axt(m, None, *args)
    with pytest.raises(ax.AxspmvError):
        ax.dev_build_axc(m, None, 0)


@pytest.mark.parametrize("case,row,col,ncols,msg", [
    ("column >= ncols", [0, 2, 3, 5], [0, 2, 1, 0, 3], 3, "column >= ncols"),
    ("offsets decrease", [0, 2, 1, 5], [0, 2, 1, 0, 2], 3, "row offsets decrease"),
    ("row[nrows] != nnz", [0, 2, 3, 4], [0, 2, 1, 0, 2], 3, "row\\[nrows\\] != nnz"),
    ("row[0] != 0", [1, 2, 3, 5], [0, 2, 1, 0, 2], 3, "row\\[0\\] != 0"),
])
def test_dev_build_checks_the_device_csr(case, row, col, ncols, msg):
    """A device CSR is checked on the device (offsets, column bounds) before
    the fill reads through its offsets: an error, nothing is built."""
    m = ax.CsrMatrix(np.array(row), np.array(col), np.ones(len(col)), ncols=ncols)
    with pytest.raises(ax.AxspmvError, match="invalid device CSR:.*" + msg):
        ax.dev_build_axt(m, None, 256, 4, 1, ax.AXT_UNC)
    with pytest.raises(ax.AxspmvError, match="invalid device CSR:.*" + msg):
        ax.dev_build_axt(m, None, 256, 64, 1, ax.AXT_COM)
    with pytest.raises(ax.AxspmvError, match="invalid device CSR:.*" + msg):
        ax.dev_build_axc(m, None, 4)


def _edge_matrix(extra):
    """A long row, a run of empty rows longer than two 64-wide search steps,
    short rows, a last row that ends the slots at 256 k + extra."""
    lens = [700, 0, 3] + [0] * 5000 + [1, 2, 5, 4, 1] * 13 + [0] * 70 + [2600]
    total = sum(lens)
    lens.append((-total) % 256 + 256 + extra)
    lens += [0] * 3
    rng = np.random.default_rng(17)
    row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    col = np.concatenate([np.sort(rng.choice(6001, n, replace=False)) for n in lens]).astype(np.uint32)
    return ax.CsrMatrix(row, col, rng.standard_normal(col.size), ncols=6001)


@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("bs,thw,th,mode", [(256, 1, 1, ax.AXT_UNC), (256, 7, 1, ax.AXT_UNC), (256, 16, 5, ax.AXT_UNC),
                                            (16, 64, 1, ax.AXT_COM), (256, 24, 8, ax.AXT_COM), (0, 32, 0, None), (0, 7, 0, None)])
def test_fill_slot_edges(extra, bs, thw, th, mode):
    """One lane per slot: slot counts around a wave's 256, rows found by
    search across long empty runs, hw that is and is not a power of two."""
    m = _edge_matrix(extra)
    x = ax.uniform(44, m.ncols)
    if mode is None:
        h, d = ax.build_axc(m, x, thw), ax.dev_build_axc(m, x, thw)
        pairs = (("ax", "ax"), ("con", "brp"), ("plane", "mapx"))
    else:
        h, d = ax.build_axt(m, x, bs, thw, th, mode), ax.dev_build_axt(m, x, bs, thw, th, mode)
        pairs = (("ax", "ax"), ("con", "con"), ("sec", "sec"), ("plane", "cplane"))
    for a, b in pairs:
        assert d[a].tobytes() == h[b].tobytes(), a


def test_dev_build_with_columns_off_16_bytes():
    """The column check's plain loads (a device CSR whose col is 4-byte aligned)."""
    m = MATS["plaw512"]
    shifted = np.concatenate([np.zeros(1, np.uint32), m.col])
    dcol = ax.DeviceBuffer.from_array(shifted)
    drow, dval = ax.DeviceBuffer.from_array(m.row), ax.DeviceBuffer.from_array(m.val)
    for bad in (False, True):
        if bad:
            shifted[-1] = m.ncols
            dcol.upload(shifted)
        a = L.Dcsr(m.nrows, m.ncols, m.nnz, 0, drow.ptr, dcol.ptr + 4, dval.ptr)
        out = C.POINTER(L.Dfmt)()
        if bad:
            with pytest.raises(ax.AxspmvError, match="column >= ncols"):
                L.call("axspmv_dev_build_axt", C.byref(a), None, 256, 4, 1, ax.AXT_UNC, None, C.byref(out))
            continue
        L.call("axspmv_dev_build_axt", C.byref(a), None, 256, 4, 1, ax.AXT_UNC, None, C.byref(out))
        plane = np.empty(out.contents.lenMAPX, np.uint32)
        L.call("axspmv_memcpy_d2h", plane.ctypes.data, out.contents.plane, plane.nbytes, None)
        L.load().axspmv_dfmt_free(out)
        assert np.array_equal(plane, ax.build_axt(m, ax.uniform(1, m.ncols), 256, 4, 1, ax.AXT_UNC)["cplane"])
