"""Sweep driver: matrix specs and the tuning database (host side only)."""
import json

import numpy as np

import gpu_spmv_amd as ax
from gpu_spmv_amd import sweep


def test_load_matrix_generators_and_files(tmp_path):
    name, m = sweep.load_matrix("laplace2d:16")
    assert name == "laplace2d_16" and m.nrows == 256 and m.nnz == 5 * 256 - 4 * 16
    p = tmp_path / "M99_toy.bin"
    m.write(str(p))
    name2, m2 = sweep.load_matrix(str(p))
    assert name2 == "M99_toy" and np.array_equal(m2.col, m.col) and np.array_equal(m2.val, m.val)


def test_best_opts_reads_database(tmp_path):
    db = dict(matrices=dict(a=dict(best=dict(label="rct_auto", format=ax.FMT_RCT, opts=dict(block=512), us=1.0)),
                            b=dict(best=None)))
    path = tmp_path / "db.json"
    path.write_text(json.dumps(db))
    assert sweep.best_opts(str(path), "a") == (ax.FMT_RCT, dict(block=512))
    assert sweep.best_opts(db, "b") is None and sweep.best_opts(db, "missing") is None


def test_candidates_cover_every_format():
    fmts = {c[1] for c in sweep.CANDIDATES}
    assert fmts == {ax.FMT_CSR, ax.FMT_K1, ax.FMT_AXC, ax.FMT_AXT, ax.FMT_RCT}
    assert sweep.BLOCKS == (32, 64, 128, 256, 512, 1024)


def _one_layout_rows():
    """(where, options) of every AXT UNC th == 1 plan that the sweep, the
    benchmark and the tuner time under a tile width of its own."""
    import bench
    rows = [("sweep " + c[0], c[2]) for c in sweep.CANDIDATES if c[1] == ax.FMT_AXT]
    rows += [("bench " + r[0], r[2]) for r in bench.OTHERS if r[1] == ax.FMT_AXT]
    rows += [(f"tuner thw{o.thw} budget{o.budget}", dict(thw=o.thw, th=o.th, mode=o.mode, slices=o.slices, flags=o.flags))
             for o in ax.autotune_defaults() if o.format == ax.FMT_AXT and o.thw != 4]
    return [(n, kw) for n, kw in rows if kw.get("th", 1) == 1 and kw.get("mode", ax.AXT_UNC) == ax.AXT_UNC and "thw" in kw
            and not kw.get("flags", 0) & (ax.PLAN_REORDER | ax.PLAN_AX_LAYOUT)]


def test_rows_named_by_tile_width_keep_it():
    """slices = 0 may run on column slices of another tile width: rows that
    differ in thw ask for one layout (or name their slices), or they would
    time one kernel under several names."""
    rows = _one_layout_rows()
    assert len(rows) > 8
    assert not [n for n, kw in rows if kw.get("slices", 0) == 0]
    # and the default is timed as well
    assert any(c[1] == ax.FMT_AXT and not c[2] for c in sweep.CANDIDATES)
    assert any(o.format == ax.FMT_AXT and o.thw == 4 and o.slices == 0 for o in ax.autotune_defaults())
