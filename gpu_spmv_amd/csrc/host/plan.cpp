// Device plans: upload a matrix in one format and run its kernel.
//
// Replaces the allocate / copy / launch / copy back / free sequence that
// every test_g*() of the reference repeats per call (cudaSpmv.cu:547-601,
// 871-929, 1100-1149, 1603-1663, 1963-2037, 2101-2170, 2213-2285): a plan
// uploads once, and axspmv_spmv() only launches.
#include <algorithm>
#include <cmath>
#include <memory>
#include <numeric>
#include <string>

#include "../hip/launch.hpp"
#include "common.hpp"
#include "plan.hpp"

using namespace axspmv;

namespace axspmv {

int hip_fail(hipError_t e, const char *what) {
    return fail(AXSPMV_E_HIP, "%s: %s", what, hipGetErrorString(e));
}

}  // namespace axspmv

void *axspmv_plan::dalloc(size_t bytes) {
    void *p = nullptr;
    if (bytes == 0) bytes = 256;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        fail(AXSPMV_E_NOMEM, "hipMalloc of %zu bytes failed", bytes);
        return nullptr;
    }
    bufs.push_back(p);
    device_bytes += bytes;
    return p;
}

int axspmv_plan::upload(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (!bytes) return AXSPMV_OK;
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e == hipSuccess ? AXSPMV_OK : hip_fail(e, "plan upload");
}

axspmv_plan::~axspmv_plan() {
    delete T;
    delete Tdet;
    delete by_slice;
    delete inner;
    for (void *p : bufs) (void)hipFree(p);
}

namespace axspmv {

// Greedy row-aligned wave blocks over units in row order: rows are packed
// into a block while the block holds at most `budget` units; a row longer
// than the budget gets a block of its own.  Long blocks go first, so the
// waves that loop longest start earliest.
std::vector<launch::Block> row_blocks(const std::vector<uint32_t> &units_per_row, uint32_t budget) {
    std::vector<launch::Block> small, big;
    uint64_t pos = 0;
    uint32_t beg = 0, cur = 0;
    bool open = false;
    for (uint32_t u : units_per_row) {
        if (u == 0) continue;
        if (u > budget) {
            if (open) small.push_back({beg, uint32_t(pos)});
            open = false;
            big.push_back({uint32_t(pos), uint32_t(pos + u)});
            pos += u;
            continue;
        }
        if (open && cur + u > budget) {
            small.push_back({beg, uint32_t(pos)});
            open = false;
        }
        if (!open) {
            beg = uint32_t(pos);
            cur = 0;
            open = true;
        }
        cur += u;
        pos += u;
    }
    if (open) small.push_back({beg, uint32_t(pos)});
    std::stable_sort(big.begin(), big.end(),
                     [](const launch::Block &a, const launch::Block &b) { return a.end - a.beg > b.end - b.beg; });
    big.insert(big.end(), small.begin(), small.end());
    return big;
}

std::vector<launch::Window> block_windows(const axspmv_csr *a, const std::vector<uint32_t> &units,
                                          const std::vector<launch::Block> &blocks) {
    const uint32_t n = a->nrows;
    std::vector<uint64_t> cum(size_t(n) + 1, 0);
    for (uint32_t r = 0; r < n; ++r) cum[r + 1] = cum[r] + units[r];
    std::vector<launch::Window> w(blocks.size(), launch::Window{0, 0});
    for (size_t i = 0; i < blocks.size(); ++i) {
        const launch::Block &b = blocks[i];
        uint32_t r = uint32_t(std::upper_bound(cum.begin(), cum.end(), uint64_t(b.beg)) - cum.begin()) - 1;
        uint32_t cmin = UINT32_MAX, cmax = 0;
        for (; r < n && cum[r] < b.end; ++r) {
            if (a->row[r + 1] == a->row[r]) continue;
            const auto mm = std::minmax_element(a->col + a->row[r], a->col + a->row[r + 1]);  // rows may be unsorted
            cmin = std::min(cmin, *mm.first);
            cmax = std::max(cmax, *mm.second);
        }
        if (cmin <= cmax) w[i] = launch::Window{cmin, cmax - cmin + 1};
    }
    return w;
}

bool worth_staging(const std::vector<launch::Window> &w) {
    size_t fit = 0;
    for (const launch::Window &x : w) fit += x.width <= launch::STAGE_COLS;
    return !w.empty() && 2 * fit >= w.size();
}

}  // namespace axspmv

namespace {

// Rows longer than this many slots are done one wave per row by SpMM.
constexpr uint32_t SPMM_LONG = 256;

// SpMM gives XCD i the i-th eighth of the rows (neighbouring rows of a mesh
// read the same X rows: one L2 instead of eight) where no eighth holds much
// more than its share of the entries; rows sorted by length, say, are dealt
// out round-robin instead.
uint32_t spmm_by_eighths(const axspmv_csr *a) {
    const uint64_t n = a->nrows;
    uint64_t most = 0;
    for (uint64_t i = 0; i < 8; ++i) most = std::max<uint64_t>(most, a->row[(i + 1) * n / 8] - a->row[i * n / 8]);
    return 8 * most <= uint64_t(a->nnz) + a->nnz / 8 ? 1 : 0;
}

bool narrow_bands(const axspmv_csr *a, uint32_t rows, uint64_t cols);

// Row-contiguous layouts: record where each row starts (device array
// `first`, uploaded here unless it is the CSR row pointer itself) for SpMM
// and the value gradient.
int setup_rowwise(Plan &p, const axspmv_csr *a, const uint32_t *d_first, const void *d_val, const uint32_t *d_col,
                  hipStream_t s) {
    if (!p.d_rowptr) {
        if (p.d_row) {
            p.d_rowptr = p.d_row;
        } else {
            p.d_rowptr = static_cast<uint32_t *>(p.dalloc(4ull * (a->nrows + 1)));
            if (!p.d_rowptr) return AXSPMV_E_NOMEM;
            AX_TRY(p.upload(p.d_rowptr, a->row, 4ull * (a->nrows + 1), s));
        }
    }
    p.d_first = const_cast<uint32_t *>(d_first);
    std::vector<uint32_t> longrows;
    for (uint32_t r = 0; r < a->nrows; ++r)
        if (a->row[r + 1] - a->row[r] > SPMM_LONG) longrows.push_back(r);
    auto *lr = static_cast<uint32_t *>(p.dalloc(4 * longrows.size()));
    if (!lr) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(lr, longrows.data(), 4 * longrows.size(), s));
    p.spmm = launch::SpmmArgs{a->nrows, p.o.vtype, SPMM_LONG, p.d_first, p.d_rowptr, d_val, d_col, lr,
                              uint32_t(longrows.size()), a->ncols, spmm_by_eighths(a),
                              longrows.empty() && a->ncols > 65536 && !narrow_bands(a, 1024, 65536)};
    p.rowwise = true;
    return AXSPMV_OK;
}

// Lanes per row for a row-per-group kernel: the power of two g in [2, 64]
// with 1.5 g >= the mean row length (CSR vector, AXC bricks).  Measured
// best or within 2 % of it on the 256^2 Laplacian, the 2^20-row power-law
// matrix and the permuted 27-point stencil for both; uniform banded rows of
// mean 19.5 prefer 8 lanes to the 16 it gives.
uint32_t lanes_for_mean(const axspmv_csr *a) {
    const double mean = a->nrows ? double(a->nnz) / a->nrows : 1.0;
    uint32_t g = 2;
    while (g < 64 && double(g) * 1.5 < mean) g *= 2;
    return g;
}

// True when the rows gather x from wide column ranges (not narrow bands).
bool wide_gathers(const axspmv_csr *a);

int plan_csr(Plan &p, const axspmv_csr *a, hipStream_t s) {
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    p.d_val = p.dalloc(vs * a->nnz);
    p.d_col = static_cast<uint32_t *>(p.dalloc(4ull * a->nnz));
    p.d_row = static_cast<uint32_t *>(p.dalloc(4ull * (a->nrows + 1)));
    if (!p.d_val || !p.d_col || !p.d_row) return AXSPMV_E_NOMEM;
    if (p.o.vtype == AXSPMV_F32) {
        std::vector<float> v(a->val, a->val + a->nnz);
        AX_TRY(p.upload(p.d_val, v.data(), 4ull * a->nnz, s));
    } else {
        AX_TRY(p.upload(p.d_val, a->val, 8ull * a->nnz, s));
    }
    AX_TRY(p.upload(p.d_col, a->col, 4ull * a->nnz, s));
    AX_TRY(p.upload(p.d_row, a->row, 4ull * (a->nrows + 1), s));
    p.slots = a->nnz;
    p.stream_bytes = (vs + 4) * a->nnz + 4ull * (a->nrows + 1);
    if (p.o.kernel == AXSPMV_KER_STREAM) {
        // lanes per row: opts.hbs, or from the mean row length
        const uint32_t g = p.o.hbs ? p.o.hbs : lanes_for_mean(a);
        if (!is_pow2(g) || g > 64) return fail(AXSPMV_E_UNSUPPORTED, "CSR vector: lanes per row %u not a power of two <= 64", g);
        p.lanes = g;
        // Non-temporal val / col loads for streams of more than twice the
        // Infinity Cache gathering wide: one box, the permuted 128^3 stencil
        // (669 MB) 797 -> 780 us; the 2^20-row power-law matrix (256 MB)
        // lost with them (259 -> 266 us), the stencil renumbered by reverse
        // Cuthill-McKee (narrow bands) stays level.
        p.seg_nt = p.stream_bytes > (512ull << 20) && wide_gathers(a) ? 1 : 0;
        p.kind = Plan::CSR_VECTOR;
        std::snprintf(p.name, sizeof p.name, "csr_vector_g%u", g);
        p.launches = 2;
        return setup_rowwise(p, a, p.d_row, p.d_val, p.d_col, s);
    }
    p.kind = Plan::CSR_NAIVE;
    std::snprintf(p.name, sizeof p.name, "csr_naive");
    return setup_rowwise(p, a, p.d_row, p.d_val, p.d_col, s);
}

int upload_planes(Plan &p, const double *vplane, const uint32_t *cplane, uint64_t nslots, hipStream_t s) {
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    p.d_vplane = p.dalloc(vs * nslots);
    p.d_cplane = static_cast<uint32_t *>(p.dalloc(4 * nslots));
    if (!p.d_vplane || !p.d_cplane) return AXSPMV_E_NOMEM;
    if (p.o.vtype == AXSPMV_F32) {
        std::vector<float> v(vplane, vplane + nslots);
        AX_TRY(p.upload(p.d_vplane, v.data(), 4 * nslots, s));
    } else {
        AX_TRY(p.upload(p.d_vplane, vplane, 8 * nslots, s));
    }
    AX_TRY(p.upload(p.d_cplane, cplane, 4 * nslots, s));
    p.slots = nslots;
    return AXSPMV_OK;
}

int upload_blocks(Plan &p, const std::vector<launch::Block> &blocks, const std::vector<uint32_t> &empty, hipStream_t s) {
    p.nblocks = uint32_t(blocks.size());
    p.d_blocks = static_cast<launch::Block *>(p.dalloc(sizeof(launch::Block) * blocks.size()));
    p.nempty = uint32_t(empty.size());
    p.d_empty = static_cast<uint32_t *>(p.dalloc(4 * empty.size()));
    if (!p.d_blocks || !p.d_empty) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(p.d_blocks, blocks.data(), sizeof(launch::Block) * blocks.size(), s));
    AX_TRY(p.upload(p.d_empty, empty.data(), 4 * empty.size(), s));
    return AXSPMV_OK;
}

// Row of CSR position q (q < nnz).
uint32_t row_of(const axspmv_csr *a, uint32_t q) {
    return uint32_t(std::upper_bound(a->row, a->row + a->nrows + 1, q) - a->row) - 1;
}

int plan_axt_com(Plan &p, const axspmv_csr *a, hipStream_t s) {
    const uint32_t thw = p.o.thw, th = p.o.th;
    axspmv_axt *m = nullptr;
    AX_TRY(axspmv_build_axt(a, nullptr, p.o.bs, thw, th, AXSPMV_AXT_COM, AXSPMV_BUILD_PLANES, &m, nullptr));
    std::unique_ptr<axspmv_axt, void (*)(axspmv_axt *)> guard(m, axspmv_axt_free);
    AX_TRY(upload_planes(p, m->vplane, m->cplane, uint64_t(m->lenAX) / 2, s));
    p.d_sec = static_cast<uint32_t *>(p.dalloc(4ull * m->lenSEC));
    if (!p.d_sec) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(p.d_sec, m->sec, 4ull * m->lenSEC, s));
    const uint32_t nnz = a->nnz;
    // Wave ranges: th == 1 in slots, a multiple of bs and of 256 (4 slots x
    // 64 lanes); th > 1 in tile columns, 4 passes of 64 columns.  A small
    // matrix gets shorter ranges (down to one pass) until about 2048 waves
    // spread over the 1024 SIMDs.
    const uint32_t units = th == 1 ? nnz : uint32_t(ceil_div(nnz, th));
    uint32_t wr = th == 1 ? std::max<uint32_t>(p.o.bs, 1024) : 256;
    const uint32_t wr_min = th == 1 ? std::max<uint32_t>(p.o.bs, 256) : 64;
    while (wr > wr_min && units / wr < 2048) wr /= 2;
    std::vector<launch::ComWave> waves;
    for (uint64_t b = 0; b < units; b += wr) {
        launch::ComWave w{uint32_t(b), uint32_t(std::min<uint64_t>(b + wr, units)), 0, 0};
        const uint64_t S = th == 1 ? w.beg : uint64_t(w.beg) * th;
        const uint64_t E = th == 1 ? w.end : std::min<uint64_t>(uint64_t(w.end) * th, nnz);
        if (S > 0 && row_of(a, uint32_t(S)) == row_of(a, uint32_t(S - 1))) w.flags |= 1;
        if (E < nnz && row_of(a, uint32_t(E - 1)) == row_of(a, uint32_t(E))) w.flags |= 2;
        waves.push_back(w);
    }
    // Rows spanning waves: (row, first wave, last wave).
    std::vector<uint32_t> span;
    bool open = false;
    uint32_t orow = 0, w0 = 0;
    for (uint32_t k = 0; k < waves.size(); ++k) {
        const uint64_t E = th == 1 ? waves[k].end : std::min<uint64_t>(uint64_t(waves[k].end) * th, nnz);
        const bool out = waves[k].flags & 2;
        const uint32_t lastrow = row_of(a, uint32_t(E - 1));
        if (open && !(out && lastrow == orow)) {
            span.insert(span.end(), {orow, w0, k});
            open = false;
        }
        if (out && !open) {
            open = true;
            orow = lastrow;
            w0 = k;
        }
    }
    std::vector<uint32_t> empty;
    for (uint32_t r = 0; r < a->nrows; ++r)
        if (a->row[r + 1] == a->row[r]) empty.push_back(r);
    auto *dw = static_cast<launch::ComWave *>(p.dalloc(sizeof(launch::ComWave) * waves.size()));
    auto *dspan = static_cast<uint32_t *>(p.dalloc(4 * span.size()));
    auto *dempty = static_cast<uint32_t *>(p.dalloc(4 * empty.size()));
    auto *head = static_cast<double *>(p.dalloc(8 * waves.size()));
    auto *tail = static_cast<double *>(p.dalloc(8 * waves.size()));
    if (!dw || !dspan || !dempty || !head || !tail) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(dw, waves.data(), sizeof(launch::ComWave) * waves.size(), s));
    AX_TRY(p.upload(dspan, span.data(), 4 * span.size(), s));
    AX_TRY(p.upload(dempty, empty.data(), 4 * empty.size(), s));
    launch::ComArgs c{};
    c.vplane = p.d_vplane;
    c.cplane = p.d_cplane;
    c.hdr = p.d_sec;
    c.waves = dw;
    c.nwaves = uint32_t(waves.size());
    c.thw = thw;
    c.th = th;
    c.bs = p.o.bs;
    c.log = m->log;
    c.nnz = nnz;
    c.vtype = p.o.vtype;
    c.head = head;
    c.tail = tail;
    c.span = dspan;
    c.nspan = uint32_t(span.size() / 3);
    c.empty = dempty;
    c.nempty = uint32_t(empty.size());
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    p.stream_bytes = (vs + 8) * p.slots + sizeof(launch::ComWave) * waves.size();
    // Non-temporal plane loads where the stream (more than 128 MB) would
    // share the Infinity Cache with the x lines the gathers reuse; th = 1 on
    // narrow bands keeps ordinary loads, as AXT UNC th = 1 does.  One box, per
    // SpMV, th = 1 / th = 4: the 2^20-row power-law matrix 271.2 -> 255.4 /
    // 251.5 -> 235.1 us, the permuted 128^3 stencil 867 -> 839.5 / 826 ->
    // 803 us, the same renumbered by reverse Cuthill-McKee 306.5 -> 311.5
    // (hence the exception) / 281.5 -> 266.3 us.
    c.nt = p.stream_bytes > (128ull << 20) && (th > 1 || wide_gathers(a)) ? 1 : 0;
    p.com = c;
    p.nblocks = c.nwaves;
    p.launches = 1 + (c.nspan > 0) + (c.nempty > 0);
    p.kind = Plan::AXT_COM;
    if (th == 1)
        std::snprintf(p.name, sizeof p.name, "axt_com_h1_thw%u_bs%u", thw, p.o.bs);
    else
        std::snprintf(p.name, sizeof p.name, "axt_com_h%u_thw%u", th, thw);
    return AXSPMV_OK;
}

// The reference's interleaved ax of AXT UNC th == 1 (values, x-halves left
// zero: every SpMV refreshes them) and the column of every value slot, with
// 0xffffffff on padding slots so the refresh writes 0 there as the builder.
int upload_ax_layout(Plan &p, const axspmv_csr *a, const axspmv_axt *m, hipStream_t s) {
    const uint32_t thw = m->tileHW;
    const uint64_t ns = uint64_t(m->lenAX) / 2;
    std::vector<double> ax(2 * ns, 0.0);
    std::vector<uint32_t> map(ns ? ns : 1, 0xffffffffu);
    for (uint64_t q = 0; q < ns; ++q) ax[(q / thw) * 2 * thw + q % thw] = m->vplane[q];
    for (uint32_t r = 0; r < a->nrows; ++r) {
        const uint64_t first = m->con[r] / 2, rl = a->row[r + 1] - a->row[r];
        for (uint64_t k = 0; k < rl; ++k) map[first + k] = m->cplane[first + k];
    }
    p.d_ax = static_cast<double *>(p.dalloc(16 * ns));
    p.d_axmap = static_cast<uint32_t *>(p.dalloc(4 * ns));
    if (!p.d_ax || !p.d_axmap) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(p.d_ax, ax.data(), 16 * ns, s));
    AX_TRY(p.upload(p.d_axmap, map.data(), 4 * ns, s));
    p.slots = ns;
    return AXSPMV_OK;
}

// AXT UNC th == 1 in S column slices: slice k holds the entries of columns
// [k C, (k + 1) C) (C = ceil(ncols / S)) and is the AXT layout of that part
// of the matrix (global column indices, so x is indexed directly).  The slices' planes and sec arrays are concatenated;
// every slice gets its own row-aligned wave blocks (unit offsets moved to the
// concatenated planes).  The dispatch list gives workgroup g (four waves,
// four blocks) slice (g % 8) % S, and workgroups run on XCD g % 8, so an XCD
// only gathers from its slice of x -- 2 MB at S = 4 on the 2^20-row matrix,
// resident in its 4 MB L2.  Rows accumulate across slices with FP64 atomic
// adds into a y cleared first.
bool narrow_bands(const axspmv_csr *a, uint32_t rows, uint64_t cols);

// AXT UNC streams its planes with non-temporal loads where the stream is
// larger than the 256 MB Infinity Cache (it comes from HBM on every SpMV
// anyway) and the rows gather x from wide column ranges (so the x lines the
// gathers share are what the cache should keep).  One box, per SpMV: the
// 2^20-row power-law matrix th = 1 218.7 -> 209.2 us (4 column slices 168.5
// -> 157.8), th = 4 / 8 226.0 -> 218.3 / 238.0 -> 227.8 us; the permuted
// 128^3 stencil th = 1 806.7 -> 784.5 us (slices 452.5 -> 412.0), th = 4 /
// 8 805.4 -> 798.4 / 822.8 -> 813.0 us; the stencil renumbered by reverse
// Cuthill-McKee, whose rows read narrow bands, lost with them (th = 1:
// 197.3 -> 204.2 us).  A 128 MB bound (K1's) would take in the power-law
// matrix with FP32 values (188 MB): th = 1 196.7 -> 192.5 us, but its
// 4-slice plan 123.0 -> 146.0 us.
bool wide_gathers(const axspmv_csr *a) {
    const uint32_t rows = uint32_t(std::min<uint64_t>(16384, ceil_div(ceil_div(uint64_t(a->nrows), 256), 64) * 64));
    return !narrow_bands(a, std::max<uint32_t>(64, rows), (2ull << 20) / 8);
}
uint32_t axt_stream_nt(const axspmv_csr *a, uint64_t stream_bytes) {
    return stream_bytes > (256ull << 20) && wide_gathers(a) ? 1 : 0;
}

// one_by_one: the slices run one after another, each on all XCDs, and add
// their row sums plainly (no atomics, the order of the additions is fixed).
int plan_axt_sliced(Plan &p, const axspmv_csr *a, bool one_by_one, hipStream_t s) {
    const uint32_t thw = p.o.thw, S = p.o.slices, n = a->nrows;
    if (S != 2 && S != 4 && S != 8) return fail(AXSPMV_E_UNSUPPORTED, "AXT column slices must be 2, 4 or 8, got %u", S);
    const uint64_t C = ceil_div(std::max<uint32_t>(a->ncols, 1), S);
    const uint32_t K = std::min<uint32_t>(4, thw);
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    // entries of each row by slice
    std::vector<uint32_t> cnt(size_t(S) * n, 0);
#pragma omp parallel for schedule(dynamic, 4096)
    for (uint32_t r = 0; r < n; ++r)
        for (uint32_t j = a->row[r]; j < a->row[r + 1]; ++j) cnt[size_t(a->col[j] / C) * n + r]++;
    // planes: first slot of every row's part of every slice, then the parts
    std::vector<std::vector<launch::Block>> sblocks(S);
    std::vector<uint32_t> at(size_t(S) * n);
    std::vector<uint32_t> units(n);
    uint64_t slots = 0;
    for (uint32_t k = 0; k < S; ++k) {
        const uint64_t s0 = slots;
        for (uint32_t r = 0; r < n; ++r) {
            const uint64_t tiles = ceil_div(cnt[size_t(k) * n + r], thw);
            at[size_t(k) * n + r] = uint32_t(slots);
            units[r] = uint32_t(tiles * (thw / K));
            slots += tiles * thw;
        }
        if (2 * (slots - s0) >= (1ull << 32) || slots >= (1ull << 32))
            return fail(AXSPMV_E_OVERFLOW, "AXT slices: %llu slots exceed 32 bits", (unsigned long long)slots);
        sblocks[k] = row_blocks(units, p.o.budget ? p.o.budget : 64);
        for (launch::Block &b : sblocks[k]) {
            b.beg += uint32_t(s0 / K);
            b.end += uint32_t(s0 / K);
        }
    }
    const std::unique_ptr<double[]> vcat(new double[slots ? slots : 1]);
    const std::unique_ptr<uint32_t[]> ccat(new uint32_t[slots ? slots : 1]), scat(new uint32_t[slots / thw + 1]);
    const uint64_t nsec = slots / thw;
#pragma omp parallel for schedule(dynamic, 4096)
    for (uint32_t r = 0; r < n; ++r) {
        uint32_t q[8];
        for (uint32_t k = 0; k < S; ++k) {
            q[k] = at[size_t(k) * n + r];
            const uint32_t c = cnt[size_t(k) * n + r], tiles = uint32_t(ceil_div(c, thw));
            for (uint32_t t = 0; t < tiles; ++t) scat[q[k] / thw + t] = r;
            for (uint32_t i = c; i < tiles * thw; ++i) {
                vcat[q[k] + i] = 0.0;
                ccat[q[k] + i] = AXSPMV_PAD_COL;
            }
        }
        for (uint32_t j = a->row[r]; j < a->row[r + 1]; ++j) {
            const uint32_t w = q[a->col[j] / C]++;
            vcat[w] = a->val[j];
            ccat[w] = a->col[j];
        }
    }
    // dispatch list: workgroup g takes blocks 4i .. 4i + 3 of slice (g % 8) % S,
    // i = (g / 8) * (8 / S) + (g % 8) / S; missing blocks are empty
    size_t most = 0;
    for (const auto &b : sblocks) most = std::max(most, b.size());
    const uint32_t per = 8 / S;
    const uint64_t groups = ceil_div(ceil_div(most, 4), per) * 8;
    std::vector<launch::Block> list(groups * 4, launch::Block{0, 0});
    for (uint64_t g = 0; g < groups; ++g) {
        const uint32_t xcd = uint32_t(g % 8), k = xcd % S;
        const uint64_t i = (g / 8) * per + xcd / S;
        for (uint32_t w = 0; w < 4; ++w)
            if (4 * i + w < sblocks[k].size()) list[4 * g + w] = sblocks[k][4 * i + w];
    }
    if (one_by_one) {  // slice after slice
        list.clear();
        p.seq.assign(1, 0);
        for (const auto &b : sblocks) {
            list.insert(list.end(), b.begin(), b.end());
            p.seq.push_back(uint32_t(list.size()));
        }
    }
    if (list.size() >= (1ull << 32) / 64) return fail(AXSPMV_E_OVERFLOW, "AXT slices: too many wave blocks");
    AX_TRY(upload_planes(p, vcat.get(), ccat.get(), slots, s));
    p.d_sec = static_cast<uint32_t *>(p.dalloc(4 * nsec));
    if (!p.d_sec) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(p.d_sec, scat.get(), 4 * nsec, s));
    // Deterministic: slice partials stored in part[k * n + r] (0 for the rows
    // without entries in slice k), summed in slice order by a merge kernel.
    const bool det = p.o.flags & AXSPMV_PLAN_DETERMINISTIC;
    std::vector<uint32_t> empty;
    if (!p.seq.empty())
        for (uint32_t r = 0; r < n; ++r)
            if (!cnt[r]) empty.push_back(r);
    if (det) {
        if (uint64_t(S) * n >= (1ull << 32)) return fail(AXSPMV_E_OVERFLOW, "AXT slices: S x nrows exceeds 32 bits");
        for (uint32_t k = 0; k < S; ++k)
            for (uint32_t r = 0; r < n; ++r)
                if (!cnt[size_t(k) * n + r]) empty.push_back(k * n + r);
        p.d_part = static_cast<double *>(p.dalloc(8ull * S * n));
        if (!p.d_part) return AXSPMV_E_NOMEM;
    }
    AX_TRY(upload_blocks(p, list, empty, s));
    p.thw = thw;
    p.th = 1;
    p.slices = S;
    p.stream_bytes = (vs + 4) * p.slots + 4 * nsec + 8ull * list.size();
    p.seg_nt = axt_stream_nt(a, p.stream_bytes);
    if (one_by_one)  // the later slices read and write the rows of y they have entries in
        for (size_t i = n; i < cnt.size(); ++i) p.stream_bytes += cnt[i] ? 16 : 0;
    p.launches = one_by_one ? S : 2;
    p.kind = Plan::AXT_UNC_H1_SLICED;
    std::snprintf(p.name, sizeof p.name, "axt_unc_h1_thw%u_%s%u%s", thw, one_by_one ? "seq" : "s", S, det ? "_det" : "");
    return AXSPMV_OK;
}

// At least half of the entries lie outside the 2 MB of x (in pieces of 64 KB)
// that their block of 16,384 rows reads most of: gathers without locality,
// wherever a local matrix has its bands or blocks.
bool scattered(const axspmv_csr *a) {
    constexpr uint32_t PIECE_LOG = 13, PIECES = 32, ROWS = 16384;
    const uint32_t np = (a->ncols >> PIECE_LOG) + 1, nb = uint32_t(ceil_div(a->nrows, ROWS));
    uint64_t far = 0;
#pragma omp parallel reduction(+ : far)
    {
        std::vector<uint32_t> cnt(np);
#pragma omp for schedule(dynamic, 1)
        for (uint32_t b = 0; b < nb; ++b) {
            std::fill(cnt.begin(), cnt.end(), 0);
            const uint32_t r1 = uint32_t(std::min<uint64_t>(a->nrows, uint64_t(b + 1) * ROWS));
            for (uint32_t j = a->row[b * ROWS]; j < a->row[r1]; ++j) cnt[a->col[j] >> PIECE_LOG]++;
            if (np <= PIECES) continue;
            std::nth_element(cnt.begin(), cnt.begin() + PIECES, cnt.end(), std::greater<uint32_t>());
            for (uint32_t k = PIECES; k < np; ++k) far += cnt[k];
        }
    }
    return 2 * far >= a->nnz;
}

// Column slices that the SpMV of an AXT UNC th == 1 plan runs one after
// another, or 1.  Where x outgrows an L2 (4 MB), row-order gathers go to the
// Infinity Cache at 54 G lines/s, whatever the kernel; a slice of at most 4
// MB is gathered from L2.  A slice costs tile padding and a pass over y: at
// least two entries per row and slice.  All slices at once, by XCD, is no
// alternative: those add with atomics (random rounding) or need partial sums
// in the plan (calls that overlap would race).  One box, FP64, without / with:
// power-law, 660,000 rows 106.5 / 105.6 us (run again and again 96.2 / 80.0),
// 750,000 129.6 / 120.7 (121.0 / 92.6), 2^20 209.5 / 163.0, 3M 920 / 550;
// permuted 100^3 stencil 270 / 194; random, 10^6 rows of 6 74.4 / 61.6.  Below
// two entries: 2M rows of 2 72.7 / 81.8; 4M of 5, 4 slices 350 / 328, 8 slices
// 350 (so 2).  Few entries read few lines of x twice, whatever the slices, and
// a launch each is all that those add (20,001 rows of 20 of 700,001 columns 7.3
// / 10.1 us, 3,001 of 300 of 5M 18.6 / 36.5, 150,001 of 9 of 3M 25.0 / 31.1):
// none under 1.4M.  Up to about 2.5M, matrices of more columns than rows still
// lose a little (300,001 of 5 of 700,001 18.4 / 18.8, 150,001 of 20 of 3M 50.9 /
// 56.3; 100,001 of 40 of 700,001 35.2 / 31.5); plans there keep the layout, and
// the order of additions, that they had.
uint32_t axt_slices(const axspmv_csr *a) {
    constexpr uint64_t SLICE = (4ull << 20) / 8;
    if (a->ncols < 5 * SLICE / 4 || a->nnz < 1400000) return 1;
    uint32_t S = 2;
    while (S < 8 && ceil_div(a->ncols, S) > SLICE) S *= 2;
    while (S > 1 && a->nnz < 2ull * S * a->nrows) S /= 2;
    return S > 1 && scattered(a) ? S : 1;
}

// The plan's SpMV in column slices (a copy of the matrix), where axt_slices
// finds it worth while and a sixteenth of the card's memory holds it.  (Of all
// its memory, not of what is free: the order of the additions then follows
// from the matrix and the options.  Where the copy cannot be allocated all the
// same the plan keeps row order, as a plan without the copy would have been
// made.)  The planes in row order stay for the value gradient and SpMM.  Streams of more than 200
// MB are loaded non-temporally (power-law, without / with, one matrix after
// another and, in brackets, one again and again: 2^20 rows 177.9 / 163.1 us,
// 900,000 151.2 / 136.8 (134.7 / 136.6), 750,000 124.8 / 112.0 (93.3 / 112.0)).
// Two slots per tile pad least: right for short rows and for the larger FP64
// streams (2^20 rows, 2 / 4 slots 163.0 / 168.6 us); else four, with half the
// load instructions (FP64, 750,000 rows 124.8 / 120.7; FP32, 2^20 rows 167.7 /
// 158.1; random rows of 6 61.7 / 65.2).
int axt_add_slices(Plan &p, const axspmv_csr *a, hipStream_t s) {
    const uint32_t S = axt_slices(a);
    if (S == 1) return AXSPMV_OK;
    size_t avail = 0, total = 0;
    const hipError_t e = hipMemGetInfo(&avail, &total);
    if (e != hipSuccess) return hip_fail(e, "plan_create: hipMemGetInfo");
    if (16ull * 16 * (a->nnz + uint64_t(S) * a->nrows) > total) return AXSPMV_OK;
    auto q = std::make_unique<Plan>();
    q->o = p.o;
    const uint64_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8, cut = uint64_t(S) * a->nrows;  // rows of all slices
    const bool nt = (vs + 4) * (a->nnz + cut / 2) > (200ull << 20);
    q->o.thw = a->nnz < 6 * cut || (nt && vs == 8) ? 2 : 4;
    q->o.slices = S;
    q->o.flags &= ~AXSPMV_PLAN_DETERMINISTIC;
    q->device = p.device;
    q->nrows = p.nrows;
    q->ncols = p.ncols;
    q->nnz = p.nnz;
    const std::string last = axspmv_last_error();
    int rc = AXSPMV_E_NOMEM;
    try {
        rc = plan_axt_sliced(*q, a, true, s);
    } catch (const std::bad_alloc &) {
    }
    if (rc == AXSPMV_E_NOMEM || rc == AXSPMV_E_OVERFLOW) {  // no room for the copy: row order, and no error
        (void)hipGetLastError();
        fail(AXSPMV_OK, "%s", last.c_str());
        return AXSPMV_OK;
    }
    if (rc) return rc;
    q->seg_nt = nt;
    // the plan's info is of the layout that SpMV runs on
    p.device_bytes += q->device_bytes;
    p.stream_bytes = q->stream_bytes;
    p.slots = q->slots;
    p.launches = S;
    std::snprintf(p.name, sizeof p.name, "%s", q->name);
    p.by_slice = q.release();
    return AXSPMV_OK;
}

int plan_axt(Plan &p, const axspmv_csr *a, hipStream_t s) {
    const uint32_t thw = p.o.thw, th = p.o.th;
    if (!is_pow2(thw) || thw > 64) return fail(AXSPMV_E_UNSUPPORTED, "AXT kernels need thw a power of two <= 64, got %u", thw);
    const bool axl = p.o.flags & AXSPMV_PLAN_AX_LAYOUT;
    if (axl && (th != 1 || p.o.mode != AXSPMV_AXT_UNC || p.o.vtype != AXSPMV_F64))
        return fail(AXSPMV_E_UNSUPPORTED, "AX layout: AXT UNC th = 1 with FP64 values only");
    if (p.o.slices > 1) {
        if (th != 1 || p.o.mode != AXSPMV_AXT_UNC || axl || (p.o.flags & AXSPMV_PLAN_STAGE_X))
            return fail(AXSPMV_E_UNSUPPORTED, "AXT column slices: UNC th = 1 only, without the AX layout or x staging");
        return plan_axt_sliced(p, a, false, s);
    }
    if (p.o.mode == AXSPMV_AXT_COM) return plan_axt_com(p, a, s);
    axspmv_axt *m = nullptr;
    AX_TRY(axspmv_build_axt(a, nullptr, p.o.bs, thw, th, p.o.mode, AXSPMV_BUILD_PLANES | AXSPMV_BUILD_PAD_COL, &m,
                           nullptr));
    std::unique_ptr<axspmv_axt, void (*)(axspmv_axt *)> guard(m, axspmv_axt_free);
    if (axl)
        AX_TRY(upload_ax_layout(p, a, m, s));
    else
        AX_TRY(upload_planes(p, m->vplane, m->cplane, uint64_t(m->lenAX) / 2, s));
    p.d_sec = static_cast<uint32_t *>(p.dalloc(4ull * m->lenSEC));
    if (!p.d_sec) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(p.d_sec, m->sec, 4ull * m->lenSEC, s));
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    std::vector<uint32_t> units(a->nrows), empty;
    const uint32_t K = std::min<uint32_t>(4, thw);
    for (uint32_t r = 0; r < a->nrows; ++r) {
        const uint32_t rl = a->row[r + 1] - a->row[r];
        if (rl == 0) empty.push_back(r);
        units[r] = th == 1 ? uint32_t(ceil_div(rl, thw) * (thw / K)) : uint32_t(ceil_div(rl, th));
    }
    // Budget in units per wave block: 64 (one pass of the wave) by default.
    // Measured against 256 (four passes): the 2^20-row power-law matrix th =
    // 1 / 4 / 8: 218 / 225 / 234 us against 227 / 240 / 271 us; the permuted
    // 27-point stencil on 128^3 th = 1 / 4: 801 / 810 against 812 / 839 us;
    // the 256^2 Laplacian (graph-timed) thw 4: 2.6 against 4.1 us.  Shorter
    // blocks balance better and, on small matrices, spread over the 1024
    // SIMDs; a banded matrix at th = 4 is the exception (5 % slower).
    const uint32_t budget = p.o.budget ? p.o.budget : 64;
    const std::vector<launch::Block> blocks = row_blocks(units, budget);
    AX_TRY(upload_blocks(p, blocks, empty, s));
    // On request, banded / stencil structure: blocks whose columns fit a
    // per-wave LDS window read x from there (not the AX layout, which reads
    // no x).
    if (!axl && (p.o.flags & AXSPMV_PLAN_STAGE_X)) {
        const std::vector<launch::Window> win = block_windows(a, units, blocks);
        if (worth_staging(win)) {
            for (const launch::Window &w : win) p.staged_blocks += w.width <= launch::STAGE_COLS;
            p.d_win = static_cast<launch::Window *>(p.dalloc(sizeof(launch::Window) * win.size()));
            if (!p.d_win) return AXSPMV_E_NOMEM;
            AX_TRY(p.upload(p.d_win, win.data(), sizeof(launch::Window) * win.size(), s));
        }
    }
    p.thw = thw;
    p.th = th;
    if (axl) {
        // refresh: map (4 B) in, x-half (8 B) out per slot; SpMV: 16 B per slot
        p.stream_bytes = 28ull * p.slots + 4ull * m->lenSEC + 8ull * p.nblocks;
        p.launches = 2;
        p.kind = Plan::AXT_UNC_H1_AX;
        std::snprintf(p.name, sizeof p.name, "axt_unc_h1_thw%u_ax", thw);
        return AXSPMV_OK;
    }
    p.stream_bytes = (vs + 4) * p.slots + 4ull * m->lenSEC + 8ull * p.nblocks;
    if (th != 1) {
        p.seg_nt = axt_stream_nt(a, p.stream_bytes);
        p.kind = Plan::AXT_UNC_H;
        std::snprintf(p.name, sizeof p.name, "axt_unc_h%u_thw%u", th, thw);
        return AXSPMV_OK;
    }
    p.kind = Plan::AXT_UNC_H1;
    p.seg_nt = axt_stream_nt(a, p.stream_bytes);
    std::snprintf(p.name, sizeof p.name, "axt_unc_h1_thw%u", thw);
    // Rows are contiguous in the planes: first slot of row r is con[r]/2.
    std::vector<uint32_t> first(a->nrows ? a->nrows : 1);
    for (uint32_t r = 0; r < a->nrows; ++r) first[r] = m->con[r] / 2;
    auto *d_first = static_cast<uint32_t *>(p.dalloc(4ull * first.size()));
    if (!d_first) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(d_first, first.data(), 4ull * first.size(), s));
    p.nunits = uint32_t(uint64_t(m->tileN) * thw / K);
    // One-pass blocks (<= 64 units) for the fused forward/adjoint kernel.
    const std::vector<launch::Block> fb = row_blocks(units, 64);
    p.nfblocks = uint32_t(fb.size());
    p.d_fblocks = static_cast<launch::Block *>(p.dalloc(sizeof(launch::Block) * fb.size()));
    if (!p.d_fblocks) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(p.d_fblocks, fb.data(), sizeof(launch::Block) * fb.size(), s));
    AX_TRY(setup_rowwise(p, a, d_first, p.d_vplane, p.d_cplane, s));
    if (!p.d_win && p.o.slices == 0) AX_TRY(axt_add_slices(p, a, s));  // (1: one layout, as asked)
    return AXSPMV_OK;
}

// Steps of one 64-lane K1 work item at most; longer chunks are split.
constexpr uint32_t K1_STEPS = 64;

int plan_k1(Plan &p, const axspmv_csr *a, hipStream_t s) {
    const uint32_t C = p.o.chunk;
    if (!is_pow2(C) || C > 64) return fail(AXSPMV_E_UNSUPPORTED, "K1 kernel needs chunk a power of two <= 64, got %u", C);
    axspmv_k1 *m = nullptr;
    AX_TRY(axspmv_build_k1(a, C, p.o.reorder ? 1 : 0, &m, nullptr));
    std::unique_ptr<axspmv_k1, void (*)(axspmv_k1 *)> guard(m, axspmv_k1_free);
    // Padding slots (steps past a row's length, and the lanes past the last
    // row) get the column AXSPMV_PAD_COL, which the kernel reads as 0.0.
#pragma omp parallel for schedule(static)
    for (uint32_t c = 0; c < m->chunkNum; ++c)
        for (uint32_t r = 0; r < C; ++r) {
            const uint64_t i = uint64_t(c) * C + r;
            const uint32_t len = i < a->nrows ? a->row[m->permi[i] + 1] - a->row[m->permi[i]] : 0;
            for (uint32_t k = len; k < m->nmc[c]; ++k) m->col[uint64_t(m->chp[c]) + uint64_t(k) * C + r] = AXSPMV_PAD_COL;
        }
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    std::vector<launch::K1Item> items;
    std::vector<uint32_t> split;
    uint32_t nslot = 0;
    for (uint32_t c = 0; c < m->chunkNum; ++c) {
        const uint32_t nm = m->nmc[c];
        if (nm <= K1_STEPS) {
            items.push_back({c, m->chp[c], 0, nm, 0xffffffffu});  // writes y directly
            continue;
        }
        const uint32_t parts = uint32_t(ceil_div(nm, K1_STEPS));
        split.insert(split.end(), {c, nslot, parts});
        for (uint32_t k = 0; k < parts; ++k)
            items.push_back({c, m->chp[c], k * K1_STEPS, std::min(nm, (k + 1) * K1_STEPS), nslot + k});
        nslot += parts;
    }
    void *val = p.dalloc(vs * m->lenVC);
    auto *col = static_cast<uint32_t *>(p.dalloc(4ull * m->lenVC));
    auto *permi = static_cast<uint32_t *>(p.dalloc(4ull * (m->chunkNum + 1) * C));
    auto *it = static_cast<launch::K1Item *>(p.dalloc(sizeof(launch::K1Item) * items.size()));
    auto *sp = static_cast<uint32_t *>(p.dalloc(4 * split.size()));
    auto *part = static_cast<double *>(p.dalloc(8ull * nslot * C));
    if (!val || !col || !permi || !it || !sp || !part) return AXSPMV_E_NOMEM;
    if (p.o.vtype == AXSPMV_F32) {
        std::vector<float> v(m->val, m->val + m->lenVC);
        AX_TRY(p.upload(val, v.data(), 4ull * m->lenVC, s));
    } else {
        AX_TRY(p.upload(val, m->val, 8ull * m->lenVC, s));
    }
    AX_TRY(p.upload(col, m->col, 4ull * m->lenVC, s));
    AX_TRY(p.upload(permi, m->permi, 4ull * (m->chunkNum + 1) * C, s));
    AX_TRY(p.upload(it, items.data(), sizeof(launch::K1Item) * items.size(), s));
    AX_TRY(p.upload(sp, split.data(), 4 * split.size(), s));
    p.k1 = launch::K1Args{it, uint32_t(items.size()), sp, uint32_t(split.size() / 3), C, a->nrows, p.o.vtype,
                          val, col, permi, part};
    p.slots = m->lenVC;
    p.stream_bytes = (vs + 4) * uint64_t(m->lenVC) + 4ull * a->nrows + sizeof(launch::K1Item) * items.size();
    // A stream of more than 128 MB shares the Infinity Cache with the x
    // lines the gathers reuse (a chunk's lanes are rows of one length, not
    // neighbours): non-temporal loads keep the cache for x.  One box, per
    // SpMV: the 2^20-row power-law matrix 226.5 -> 214.4 us, the permuted
    // 128^3 stencil 740 -> 719.6 us, the same renumbered by reverse
    // Cuthill-McKee 209.2 -> 193.2 us.
    p.k1.nt = p.stream_bytes > (128ull << 20) ? 1 : 0;
    // Short rows: fewer steps in flight (the kernel's comment has both sides).
    // x of more than 4 MB, an L2, is where scattered gathers leave it.
    const uint64_t n = a->nrows;
    if (a->nnz <= 12 * n && a->ncols > (4u << 20) / 8 && scattered(a))
        p.k1.mode = launch::K1Mode::K1_FAR;
    else if (a->nnz <= 6 * n)
        p.k1.mode = launch::K1Mode::K1_SHORT;
    p.launches = split.empty() ? 1 : 2;
    p.nblocks = uint32_t(items.size());
    p.kind = Plan::K1;
    std::snprintf(p.name, sizeof p.name, "k1_c%u%s", C, p.o.reorder ? "" : "_natural");
    return AXSPMV_OK;
}

int plan_axc(Plan &p, const axspmv_csr *a, hipStream_t s) {
    if (p.o.hbs == 0) p.o.hbs = lanes_for_mean(a);  // bricks (and lanes per row) from the mean row length
    const uint32_t G = p.o.hbs;
    if (!is_pow2(G) || G > 64) return fail(AXSPMV_E_UNSUPPORTED, "AXC kernel needs hbs a power of two <= 64, got %u", G);
    if (p.o.flags & AXSPMV_PLAN_AX_LAYOUT) {
        // AXC's ax (bricks of hbs values then hbs x values from brp[r],
        // get_axAXC cudaSpmv.cu:952-979) is the AXT UNC th = 1 layout with
        // thw = hbs, slot for slot: the same plan serves it.
        p.o.thw = G;
        p.o.th = 1;
        p.o.mode = AXSPMV_AXT_UNC;
        AX_TRY(plan_axt(p, a, s));
        std::snprintf(p.name, sizeof p.name, "axc_hbs%u_ax", G);
        return AXSPMV_OK;
    }
    axspmv_axc *m = nullptr;
    AX_TRY(axspmv_build_axc(a, nullptr, G, AXSPMV_BUILD_PLANES | AXSPMV_BUILD_PAD_COL, &m, nullptr));
    std::unique_ptr<axspmv_axc, void (*)(axspmv_axc *)> guard(m, axspmv_axc_free);
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    const uint32_t long_slots = std::max<uint32_t>(64 * G, 256);
    std::vector<uint32_t> longrows;
    for (uint32_t r = 0; r < a->nrows; ++r)
        if ((m->brp[r + 1] - m->brp[r]) / 2 > long_slots) longrows.push_back(r);
    const uint64_t nslots = m->lenAX / 2;
    void *vp = p.dalloc(vs * nslots);
    auto *mapx = static_cast<uint32_t *>(p.dalloc(4ull * m->lenMAPX));
    auto *brp = static_cast<uint32_t *>(p.dalloc(4ull * m->lenBRP));
    auto *lr = static_cast<uint32_t *>(p.dalloc(4 * longrows.size()));
    if (!vp || !mapx || !brp || !lr) return AXSPMV_E_NOMEM;
    if (p.o.vtype == AXSPMV_F32) {
        std::vector<float> v(m->vplane, m->vplane + nslots);
        AX_TRY(p.upload(vp, v.data(), 4 * nslots, s));
    } else {
        AX_TRY(p.upload(vp, m->vplane, 8 * nslots, s));
    }
    AX_TRY(p.upload(mapx, m->mapx, 4ull * m->lenMAPX, s));
    AX_TRY(p.upload(brp, m->brp, 4ull * m->lenBRP, s));
    AX_TRY(p.upload(lr, longrows.data(), 4 * longrows.size(), s));
    p.axc = launch::AxcArgs{a->nrows, G, p.o.vtype, long_slots, brp, mapx, vp, lr, uint32_t(longrows.size())};
    p.slots = nslots;
    p.stream_bytes = (vs + 4) * nslots + 4ull * m->lenBRP;
    // Non-temporal plane loads for streams of more than twice the Infinity
    // Cache gathering wide: one box, the permuted 128^3 stencil hbs 4 / 64
    // 1214.7 -> 1163.0 / 945.7 -> 914.3 us; on the 2^20-row power-law matrix
    // (streams of 300-400 MB) hbs 4 lost with them (301 -> 347 us) where hbs
    // 64 gained (400 -> 384 us); renumbered (narrow bands) level.
    p.axc.nt = p.stream_bytes > (512ull << 20) && wide_gathers(a) ? 1 : 0;
    p.launches = longrows.empty() ? 1 : 2;
    p.kind = Plan::AXC;
    std::snprintf(p.name, sizeof p.name, "axc_hbs%u", G);
    // Rows are contiguous in the value plane: first slot of row r is brp[r]/2.
    std::vector<uint32_t> first(a->nrows ? a->nrows : 1);
    for (uint32_t r = 0; r < a->nrows; ++r) first[r] = m->brp[r] / 2;
    auto *d_first = static_cast<uint32_t *>(p.dalloc(4ull * first.size()));
    if (!d_first) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(d_first, first.data(), 4ull * first.size(), s));
    return setup_rowwise(p, a, d_first, vp, mapx, s);
}

// Row-block starts for RCT: nrb blocks of about nnz / nrb nonzeros each,
// every block 1..rmax rows (nrb * rmax >= nrows).
std::vector<uint32_t> rct_row_blocks(const axspmv_csr *a, uint32_t nrb, uint32_t rmax) {
    const uint32_t n = a->nrows;
    std::vector<uint32_t> rbs(size_t(nrb) + 1, 0);
    for (uint32_t k = 1; k < nrb; ++k) {
        const uint64_t target = uint64_t(a->nnz) * k / nrb;
        uint64_t r = uint64_t(std::lower_bound(a->row, a->row + n + 1, target) - a->row);
        const uint64_t lo = std::max<uint64_t>(uint64_t(rbs[k - 1]) + 1,
                                               n > uint64_t(nrb - k) * rmax ? n - uint64_t(nrb - k) * rmax : 0);
        const uint64_t hi = std::min<uint64_t>(uint64_t(rbs[k - 1]) + rmax, n - (nrb - k));
        rbs[k] = uint32_t(std::min(std::max(r, lo), hi));
    }
    rbs[nrb] = n;
    return rbs;
}

// True when the rows, cut into blocks of `rows`, read narrow column bands:
// at most 1/8 of the nonzeros lie in blocks whose column span (max - min + 1)
// exceeds `cols`.  Such a matrix (banded, a stencil in natural order) keeps
// each block's x within one L2 already, and column slices would only leave
// most tiles empty.
bool narrow_bands(const axspmv_csr *a, uint32_t rows, uint64_t cols) {
    uint64_t wide = 0;
    for (uint64_t r0 = 0; r0 < a->nrows; r0 += rows) {
        const uint32_t r1 = uint32_t(std::min<uint64_t>(a->nrows, r0 + rows));
        const uint32_t b = a->row[r0], e = a->row[r1];
        if (b == e) continue;
        const auto mm = std::minmax_element(a->col + b, a->col + e);
        if (uint64_t(*mm.second) - *mm.first + 1 > cols) wide += e - b;
        if (wide * 8 > a->nnz) return false;
    }
    return true;
}

// The rows of an RCT plan for SpMM that get blocks of their own, in column
// slices (one per XCD), or none.  On random columns every entry reads its own
// line of X past the L2; rows of many entries are the exception, if they are
// worked on together: the tiles that an XCD holds in LDS at once (64 of them)
// then read each X row of their slice several times while it is in L2.  A
// heavy row costs an atomic add per slice, as much traffic as a few lines, so
// it needs at least 32 entries; the split is made where such rows are few (at
// most 1/8 of the rows) but hold a good part of the entries (1/4, and at
// least 4 per column), and the rows reach over more than 65,536 columns (X of
// 8 right-hand sides and more does not fit an L2).  Power-law matrices, FP64,
// one box, without / with: 600,000 rows, k = 8, 1024-row tiles 222 / 148 us;
// 400,003 rows, k = 32, 256-row tiles 323 / 236 us; SpMV on 10^6 rows and
// 1024-row tiles 195 / 133 us.  (With 4 column slices for the other rows, k =
// 8: 184 / 185 us.)
std::vector<uint32_t> heavy_rows(const axspmv_csr *a) {
    constexpr uint32_t LONG = 32;
    std::vector<uint32_t> rows;
    if (a->ncols <= 65536) return rows;
    uint64_t nnz = 0;
    for (uint32_t r = 0; r < a->nrows; ++r) {
        const uint32_t l = a->row[r + 1] - a->row[r];
        if (l < LONG) continue;
        rows.push_back(r);
        nnz += l;
    }
    if (8 * rows.size() > a->nrows || 4 * nnz < a->nnz || nnz < 4ull * a->ncols || narrow_bands(a, 1024, 65536)) rows.clear();
    return rows;
}

// The matrix's values as indices into a table of at most 256 (bit for bit; of
// the FP32 values with f32), or false.  Meshes with constant coefficients and
// graphs without weights have a handful; an entry then takes 1 byte for its
// value instead of 8 (or 4), and a matrix of other values is told apart after
// a few hundred of them.  SpMV, FP64, 12 / 5 B per entry, one box: 100^3
// stencil renumbered 90 / 79 us, 90^3 in natural order 43 / 35, permuted 110^3
// 179 / 141, the 1000^2 Laplacian 14.5 / 11.8; below about 2M entries the gain
// is gone (the 256^2 Laplacian by single calls 6.6 / 6.3, in a graph 3.2 / 3.3).
bool value_table(const double *val, uint64_t n, bool f32, std::vector<double> &table, std::vector<uint8_t> &idx) {
    constexpr uint32_t SLOTS = 1024;  // open addressing over the values' bits
    std::vector<uint64_t> bits(SLOTS);
    std::vector<uint16_t> at(SLOTS, 0xffff);
    table.clear();
    auto find = [&](double d) {
        uint64_t u;
        std::memcpy(&u, &d, 8);
        uint32_t h = uint32_t((u * 0x9E3779B97F4A7C15ull) >> 54);
        while (at[h] != 0xffff && bits[h] != u) h = (h + 1) % SLOTS;
        bits[h] = u;
        return h;
    };
    for (uint64_t q = 0; q < n; ++q) {
        if (q && std::memcmp(val + q, val + q - 1, 8) == 0) continue;
        const double d = f32 ? double(float(val[q])) : val[q];
        const uint32_t h = find(d);
        if (at[h] != 0xffff) continue;
        if (table.size() == 256) return false;
        at[h] = uint16_t(table.size());
        table.push_back(d);
    }
    idx.resize(n);
#pragma omp parallel for schedule(static)
    for (uint64_t q = 0; q < n; ++q) {
        const double d = f32 ? double(float(val[q])) : val[q];
        uint64_t u;
        std::memcpy(&u, &d, 8);
        uint32_t h = uint32_t((u * 0x9E3779B97F4A7C15ull) >> 54);
        while (bits[h] != u || at[h] == 0xffff) h = (h + 1) % SLOTS;
        idx[q] = uint8_t(at[h]);
    }
    table.resize(256, 0.0);
    return true;
}

// RCT: row blocks of at most tile_rows rows and about equal nonzeros, column
// slices, entries of a tile sorted by (column, row).
int plan_rct(Plan &p, const axspmv_csr *a, hipStream_t s) {
    if (p.o.block > 1024 || p.o.block % 64)
        return fail(AXSPMV_E_INVALID, "RCT: block %u is not a multiple of 64 up to 1024", p.o.block);
    hipDeviceProp_t prop;
    size_t lds_max = 65536;
    uint64_t cus = 256;
    if (hipGetDeviceProperties(&prop, p.device) == hipSuccess) {
        if (prop.sharedMemPerBlock > 0) lds_max = prop.sharedMemPerBlock;
        if (prop.multiProcessorCount > 0) cus = uint64_t(prop.multiProcessorCount);
    }
    const uint32_t lds_rows = uint32_t(std::min<size_t>(65536, lds_max / p.lds_per_row));
    p.lds_max = lds_max;
    const uint32_t n = a->nrows;
    // Default tile height: as tall as the LDS allows (fewer row blocks, fewer
    // passes over x), but short enough that the tiles cover the 256 CUs.
    auto auto_rows = [&](uint32_t slices) {
        const uint64_t fill = ceil_div(ceil_div(uint64_t(n) * slices, 256), 64) * 64;
        return uint32_t(std::min<uint64_t>(std::min<uint32_t>(16384, lds_rows), std::max<uint64_t>(64, fill)));
    };
    // Default slicing: one slice when x fits 2 MB (one XCD's L2 share) or
    // the row blocks read narrow column bands anyway; else see below.
    constexpr uint64_t slice_cols = (2ull << 20) / 8;
    uint32_t S = p.o.slices;
    bool banded = false;
    if (S == 0) {
        S = 1;
        if (a->ncols > slice_cols) {
            banded = narrow_bands(a, p.o.tile_rows ? p.o.tile_rows : auto_rows(1), slice_cols);
            if (!banded) {
                uint32_t s2 = 1;  // slices of at most 2 MB of x
                while (s2 < 8 && ceil_div(a->ncols, s2) > slice_cols) s2 *= 2;
                if (p.lds_per_row > 8) {
                    // The plan of A^T behind a fused value gradient holds 16 B
                    // per tile row; 8192-row tiles with half the slices measured
                    // fastest for it (forward + adjoint on the 2^20-row
                    // power-law matrix 241 us against 269 us at 10240 rows and 4
                    // slices; 702 against 745 us on the permuted 27-point
                    // stencil on 128^3), and for the adjoint alone.
                    S = std::max(1u, s2 / 2);
                } else {
                    // Every slice adds each row's sum into y with an FP64
                    // atomic, so take the fewest slices that still give every
                    // CU a tile of full height (row blocks x slices >= CUs),
                    // but no more than the 2 MB rule asks and no fewer than
                    // slices of 8 MiB of x.  The permuted 27-point stencil on
                    // 128^3 (128 full-height row blocks): 2 slices 229.6 us,
                    // 4 slices 239.4 us, 8 slices 269.5 us; the 2^20-row
                    // power-law matrix (64 row blocks) keeps 4 slices (2: 121 us,
                    // half the CUs idle; 4: 74 us).
                    uint32_t s8 = 1;
                    while (s8 < 8 && ceil_div(a->ncols, s8) > (8ull << 20) / 8) s8 *= 2;
                    const uint64_t nrb_full = ceil_div(n, p.o.tile_rows ? p.o.tile_rows : std::min<uint32_t>(16384, lds_rows));
                    uint32_t sf = 1;
                    while (sf < 8 && nrb_full * sf < cus) sf *= 2;
                    S = std::max(s8, std::min(sf, s2));
                }
            }
        }
    }
    if (S != 1 && S != 2 && S != 4 && S != 8) return fail(AXSPMV_E_INVALID, "RCT: slices must be 1, 2, 4 or 8");
    // Narrow bands reuse x within a band whatever the tile height: 512-row
    // tiles (4 KB of LDS) let many workgroups share a CU and even out the
    // end of the launch, which pays on matrices mixing short and long rows
    // (256 banded matrices as one block-diagonal plan, row lengths varying
    // by 60 % of their mean, 16-bit keys: 985 us at 512 rows, 973 at 256,
    // 999 at 1024, 1035 at 2048; 32-bit keys: 1170 us at 512, 1227 at 2048,
    // 1390 at 16384).  Rows of one length (a mesh: the 128^3 stencil
    // renumbered by reverse Cuthill-McKee, 7 %) take the tallest tiles that
    // still cover the CUs: 168 against 180 us at 2048 rows, with the
    // non-temporal stream loads below.
    uint32_t Rt = p.o.tile_rows ? p.o.tile_rows : auto_rows(S);
    if (!p.o.tile_rows && banded) {
        double sum = 0.0, sq = 0.0;
#pragma omp parallel for schedule(static) reduction(+ : sum, sq)
        for (uint32_t i = 0; i < n; ++i) {
            const double l = double(a->row[i + 1] - a->row[i]);
            sum += l;
            sq += l * l;
        }
        const double mean = n ? sum / n : 0.0, var = n ? std::max(0.0, sq / n - mean * mean) : 0.0;
        if (!(mean > 0.0 && std::sqrt(var) < 0.25 * mean)) Rt = std::min<uint32_t>(512, auto_rows(1));
    }
    if (p.lds_per_row > 8)  // a transposed plan's tiles are cut to fit (8192 rows when automatic)
        Rt = std::min(Rt, p.o.tile_rows || banded ? lds_rows : std::min<uint32_t>(lds_rows, 8192));
    if (Rt == 0 || Rt > lds_rows)
        return fail(AXSPMV_E_UNSUPPORTED, "RCT: %u rows per tile do not fit %zu bytes of LDS", Rt, lds_max);
    const uint32_t nrb = uint32_t(ceil_div(n, Rt));
    // Blocks keep at most Rt rows (so the packed key keeps its bits); the
    // balancing uses whatever slack ceil(n / Rt) * Rt - n leaves.
    const std::vector<uint32_t> rbs = rct_row_blocks(a, nrb, Rt);
    uint32_t R = 1;  // rows of the largest block: the LDS accumulator size
    for (uint32_t k = 0; k < nrb; ++k) R = std::max(R, rbs[k + 1] - rbs[k]);
    const uint32_t C = uint32_t(std::max<uint64_t>(1, ceil_div(a->ncols, S)));
    // Heavy rows: blocks of their own, in column slices, their tiles after the
    // others.  Only in plans meant for SpMM (ktile or tile_rows given, tiles
    // short enough): SpMV and forward + adjoint of a default plan pay the clear
    // of the heavy rows, their adds and a residual pass of its own, and get
    // little for it (power-law, without / with, SpMV: 70,000 rows 11.1 / 13.1
    // us, 100,000 13.6 / 15.1, 200,000 21.5 / 22.5, 300,000 32.7 / 37.8; forward
    // + adjoint 23.0 / 26.6, 32.3 / 34.0, 59.6 / 58.4, 75.9 / 81.0; from 215,000
    // to 262,000 rows SpMV gains 6 to 12 % on changing matrices and loses 1 to 9
    // on one).  Not beside column slices that the plan chose itself, which do
    // the same for all rows (SpMM, k = 8, two slices: 270,000 rows 74.7 / 79.8
    // us, 350,000 97.9 / 107.2, 500,000 142.1 / 148.8; k = 4 60.7 / 69.8, 79.7 /
    // 91.4, 110.1 / 123.2).  Not in deterministic plans, which add no slice
    // atomically.
    std::vector<uint32_t> hrows, hbs(1, 0), hmask;
    if ((p.o.ktile || p.o.tile_rows) && (S == 1 || p.o.slices) && !(p.o.flags & AXSPMV_PLAN_DETERMINISTIC) && !p.keep_pos &&
        64ull * R <= lds_max)
        hrows = heavy_rows(a);
    // One slice per XCD, and blocks of few enough rows that their tiles reach
    // every CU: 100,000-row power-law matrix, k = 8, blocks as tall as the LDS
    // allows (64 tiles) 38 us, 256 tiles 26, 512 tiles 29.  4 slices lose where
    // X is large (k = 32, 400,003 rows: 252 against 237 us) and gain a little
    // elsewhere (k = 8, 600,000 rows: 144 against 149); 16 cost their adds (266).
    constexpr uint32_t HS = 8, HTILES = 256;
    const uint32_t HC = uint32_t(std::max<uint64_t>(1, ceil_div(a->ncols, HS)));
    const uint32_t nhb = uint32_t(std::max<uint64_t>(ceil_div(hrows.size(), R), std::min<uint64_t>(hrows.size(), HTILES / HS)));
    if (nhb) {
        hmask.assign(ceil_div(n, 32), 0);
        for (uint32_t r : hrows) hmask[r >> 5] |= 1u << (r & 31);
        for (uint32_t k = 1; k <= nhb; ++k) hbs.push_back(uint32_t(uint64_t(hrows.size()) * k / nhb));
    }
    auto heavy = [&](uint32_t r) { return nhb && (hmask[r >> 5] >> (r & 31) & 1); };
    const uint64_t ntile = uint64_t(nrb) * S, nall = ntile + uint64_t(nhb) * HS;
    // count entries per tile
    std::vector<uint64_t> cnt(nall + 1, 0);
#pragma omp parallel for schedule(dynamic, 1)
    for (uint32_t rb = 0; rb < nrb; ++rb)
        for (uint32_t r = rbs[rb]; r < rbs[rb + 1]; ++r) {
            if (heavy(r)) continue;
            for (uint32_t j = a->row[r]; j < a->row[r + 1]; ++j) cnt[uint64_t(rb) * S + a->col[j] / C + 1]++;
        }
#pragma omp parallel for schedule(dynamic, 1)
    for (uint32_t hb = 0; hb < nhb; ++hb)
        for (uint32_t i = hbs[hb]; i < hbs[hb + 1]; ++i)
            for (uint32_t j = a->row[hrows[i]]; j < a->row[hrows[i] + 1]; ++j)
                cnt[ntile + uint64_t(hb) * HS + a->col[j] / HC + 1]++;
    for (uint64_t t = 0; t < nall; ++t) cnt[t + 1] += cnt[t];
    const uint64_t nnz = a->nnz;
    std::vector<uint32_t> col(nnz ? nnz : 1);
    std::vector<uint16_t> lrow(nnz ? nnz : 1);
    std::vector<double> val(nnz ? nnz : 1);
    // the value gradient comes out in entry order: keep each entry's CSR position
    const bool keep_pos = p.keep_pos;
    std::vector<uint32_t> pos(keep_pos && nnz ? nnz : 1);
#pragma omp parallel
    {
        std::vector<std::pair<uint64_t, uint32_t>> key;  // (col << 16 | lrow, CSR position)
#pragma omp for schedule(dynamic, 1)
        for (uint32_t b = 0; b < nhb + nrb; ++b) {  // the heavy blocks, of the most entries, first
            key.clear();
            uint64_t q;
            if (b < nhb) {
                for (uint32_t i = hbs[b]; i < hbs[b + 1]; ++i)
                    for (uint32_t j = a->row[hrows[i]]; j < a->row[hrows[i] + 1]; ++j)
                        key.emplace_back((uint64_t(a->col[j]) << 16) | (i - hbs[b]), j);
                q = cnt[ntile + uint64_t(b) * HS];
            } else {
                const uint32_t rb = b - nhb, r0 = rbs[rb], r1 = rbs[rb + 1];
                for (uint32_t r = r0; r < r1; ++r) {
                    if (heavy(r)) continue;
                    for (uint32_t j = a->row[r]; j < a->row[r + 1]; ++j)
                        key.emplace_back((uint64_t(a->col[j]) << 16) | (r - r0), j);
                }
                q = cnt[uint64_t(rb) * S];
            }
            std::sort(key.begin(), key.end());
            // sorted by column, so the slices come out in order
            for (const auto &k : key) {
                col[q] = uint32_t(k.first >> 16);
                lrow[q] = uint16_t(k.first & 0xffff);
                val[q] = a->val[k.second];
                if (keep_pos) pos[q] = k.second;
                ++q;
            }
        }
    }
    // the kernel indexes entries in 32 bits with up to 2 * 8 * 1024 past the end
    if (cnt[nall] >= (1ull << 32) - (1u << 16)) return fail(AXSPMV_E_OVERFLOW, "RCT: too many entries");
    std::vector<uint32_t> tptr(nall + 1);
    for (uint64_t t = 0; t <= nall; ++t) tptr[t] = uint32_t(cnt[t]);
    const size_t vs = p.o.vtype == AXSPMV_F32 ? 4 : 8;
    // Pack (column offset, row within the tile) into one word when both fit
    // in 32 bits.  The offset is taken from a base column per run of 1024
    // entries, counting round from the last column to column 0: a run's
    // columns rise tile by tile, so they cover a short stretch of columns,
    // far shorter than a tile's.  The base is the run's smallest column, or,
    // where the run passes from the last slice of a row block into the first
    // of the next (its columns fall back towards 0), its first column.
    auto bits = [](uint64_t v) {  // bits to hold values 0 .. v-1
        uint32_t b = 1;
        while ((1ull << b) < v) ++b;
        return b;
    };
    constexpr uint32_t SEG_LOG = 10;  // entries per run: 1 << SEG_LOG
    const uint64_t nseg = std::max<uint64_t>(1, ceil_div(nnz + (nnz & 1), uint64_t(1) << SEG_LOG));
    std::vector<uint32_t> sbase(nseg, 0);
    const uint64_t nc = std::max<uint64_t>(1, a->ncols);
    uint64_t span = 1;
    // base of run g of 1 << log entries; returns the columns the run spans from it
    auto run_base = [&](uint64_t g, uint32_t log, uint32_t &base) -> uint64_t {
        const uint64_t q0 = g << log, q1 = std::min<uint64_t>(nnz, q0 + (uint64_t(1) << log));
        if (q0 >= nnz) return 1;
        const auto mm = std::minmax_element(col.begin() + q0, col.begin() + q1);
        const uint64_t lin = uint64_t(*mm.second) - *mm.first + 1;  // from the smallest column
        uint64_t cyc = 1;                                            // round from the first column
        for (uint64_t q = q0; q < q1; ++q) {
            const uint64_t off = col[q] >= col[q0] ? col[q] - col[q0] : col[q] + nc - col[q0];
            cyc = std::max(cyc, off + 1);
        }
        base = lin <= cyc ? *mm.first : col[q0];
        return std::min(lin, cyc);
    };
#pragma omp parallel for schedule(static) reduction(max : span)
    for (uint64_t g = 0; g < nseg; ++g) span = std::max(span, run_base(g, SEG_LOG, sbase[g]));
    const uint32_t rbits = bits(R), cbits = bits(span);
    const bool packed = rbits + cbits <= 32 && !(p.o.flags & AXSPMV_PLAN_RCT_SPLIT);
    // Narrow bands: one 16-bit key per entry, the column as an offset from
    // the smallest column of its run of 128 entries and, above it, the
    // entry's row minus its column less the smallest such difference, where
    // both fit 16 bits together -- 10 bytes per FP64 entry instead of 12.
    // Entries of a band lie within a few columns of the diagonal, and a run
    // of 128 of them covers few columns, also where it passes from one tile
    // to the next (its columns step back by about the band's width).
    constexpr uint32_t DSEG_LOG = 7;  // entries per run: 1 << DSEG_LOG
    const uint64_t nseg16 = std::max<uint64_t>(1, ceil_div(nnz + (nnz & 1), uint64_t(1) << DSEG_LOG));
    std::vector<uint32_t> sbase16;
    int64_t dlo = 0;
    uint32_t cbits16 = 0;
    bool diag = packed && nnz > 0 && !nhb && !(p.o.flags & AXSPMV_PLAN_RCT_WIDE_KEY);
    if (diag) {
        int64_t lo = INT64_MAX, hi = INT64_MIN;
#pragma omp parallel for schedule(dynamic, 1) reduction(min : lo) reduction(max : hi)
        for (uint32_t rb = 0; rb < nrb; ++rb)
            for (uint64_t q = cnt[uint64_t(rb) * S]; q < cnt[uint64_t(rb + 1) * S]; ++q) {
                const int64_t d = int64_t(rbs[rb]) + lrow[q] - int64_t(col[q]);
                lo = std::min(lo, d);
                hi = std::max(hi, d);
            }
        sbase16.assign(nseg16, 0);
        uint64_t span16 = 1;
#pragma omp parallel for schedule(static) reduction(max : span16)
        for (uint64_t g = 0; g < nseg16; ++g) {
            const uint64_t q0 = g << DSEG_LOG, q1 = std::min<uint64_t>(nnz, q0 + (uint64_t(1) << DSEG_LOG));
            if (q0 >= nnz) continue;
            const auto mm = std::minmax_element(col.begin() + q0, col.begin() + q1);
            sbase16[g] = *mm.first;
            span16 = std::max<uint64_t>(span16, uint64_t(*mm.second) - *mm.first + 1);
        }
        dlo = lo;
        cbits16 = bits(span16);
        diag = cbits16 + bits(uint64_t(hi - lo) + 1) <= 16;
    }
    std::vector<double> table;
    std::vector<uint8_t> vidx;
    const bool few = uint64_t(R) * p.lds_per_row + 2048 <= lds_max && nnz &&
                     value_table(val.data(), nnz, p.o.vtype == AXSPMV_F32, table, vidx);
    const size_t vbytes = few ? 1 : vs;
    // The packed key in 24 bits, with a base per run of 128 entries, where both
    // fields fit and the stream of 32-bit keys takes 64 to 256 MB.  Below, it
    // comes from the caches and the third load costs more than the bytes (FP64
    // power-law matrix, 32 / 24 bits: 50,000 rows 9.3 / 9.5 us; random rows,
    // 150,001, FP32 15.0 / 15.8); between, the bytes count, most of all where
    // they let the stream stay in the Infinity Cache (plans and vectors in
    // turn: power-law, 400,003 rows 42.6 / 42.5 us, 600,000 52.4 / 51.6, 2^20 rows
    // 86.8 / 85.9, FP32 78.0 / 75.1, forward + adjoint 212.8 / 209.5; random,
    // 450,007 rows, FP32 45.6 / 44.1; SpMM, k = 8, 150.4 / 149.5; 2^20 rows run
    // again and again 63.2 / 57.2); above, with non-temporal loads, it is level
    // or slightly behind (1.4M rows 160.0 / 161.0).
    const uint64_t stream32 = nnz * (4 + vbytes);
    std::vector<uint32_t> sbase24;
    bool key24 = packed && !diag && rbits < 24 && !(p.o.flags & AXSPMV_PLAN_RCT_WIDE_KEY) &&
                 stream32 >= (64ull << 20) && stream32 <= (256ull << 20);
    if (key24) {
        sbase24.assign(nseg16, 0);
        uint64_t span24 = 1;
#pragma omp parallel for schedule(static) reduction(max : span24)
        for (uint64_t g = 0; g < nseg16; ++g) span24 = std::max(span24, run_base(g, DSEG_LOG, sbase24[g]));
        key24 = rbits + bits(span24) <= 24;
    }
    const uint64_t kbytes = diag ? 2 : key24 ? 3 : packed ? 4 : 6;  // column and row per entry
    // one spare entry when nnz is odd: a kernel may load entries in aligned pairs
    const uint64_t nnz_pad = nnz + (nnz & 1);
    void *dv = p.dalloc(vbytes * nnz_pad);
    auto *dt = static_cast<uint32_t *>(p.dalloc(4 * tptr.size()));
    auto *drb = static_cast<uint32_t *>(p.dalloc(4 * rbs.size()));
    if (!dv || !dt || !drb) return AXSPMV_E_NOMEM;
    if (keep_pos) {
        pos.resize(nnz);
        p.rct_pos = std::move(pos);
    }
    AX_TRY(p.upload(drb, rbs.data(), 4 * rbs.size(), s));
    double *dpal = nullptr;
    if (few) {
        dpal = static_cast<double *>(p.dalloc(8 * table.size()));
        if (!dpal) return AXSPMV_E_NOMEM;
        AX_TRY(p.upload(dpal, table.data(), 8 * table.size(), s));
        AX_TRY(p.upload(dv, vidx.data(), nnz, s));
    } else if (p.o.vtype == AXSPMV_F32) {
        std::vector<float> v(val.begin(), val.begin() + nnz);
        AX_TRY(p.upload(dv, v.data(), 4 * nnz, s));
    } else {
        AX_TRY(p.upload(dv, val.data(), 8 * nnz, s));
    }
    AX_TRY(p.upload(dt, tptr.data(), 4 * tptr.size(), s));
    uint32_t *dc = nullptr, *dk = nullptr, *dcb = nullptr;
    uint16_t *dl = nullptr, *dk16 = nullptr, *dk24 = nullptr;
    uint8_t *dk8 = nullptr;
    if (diag) {
        std::vector<uint16_t> key(nnz);
#pragma omp parallel for schedule(dynamic, 1)
        for (uint32_t rb = 0; rb < nrb; ++rb)
            for (uint64_t q = cnt[uint64_t(rb) * S]; q < cnt[uint64_t(rb + 1) * S]; ++q) {
                const uint64_t d = uint64_t(int64_t(rbs[rb]) + lrow[q] - int64_t(col[q]) - dlo);
                key[q] = uint16_t(d << cbits16 | (col[q] - sbase16[q >> DSEG_LOG]));
            }
        dk16 = static_cast<uint16_t *>(p.dalloc(2 * nnz_pad));
        dcb = static_cast<uint32_t *>(p.dalloc(4 * nseg16));
        if (!dk16 || !dcb) return AXSPMV_E_NOMEM;
        AX_TRY(p.upload(dk16, key.data(), 2 * nnz, s));
        AX_TRY(p.upload(dcb, sbase16.data(), 4 * nseg16, s));
    } else if (key24) {
        std::vector<uint16_t> lo(nnz);
        std::vector<uint8_t> hi(nnz);
#pragma omp parallel for schedule(static)
        for (uint64_t q = 0; q < nnz; ++q) {
            const uint64_t b = sbase24[q >> DSEG_LOG], off = col[q] >= b ? col[q] - b : col[q] + nc - b;
            const uint32_t k = uint32_t(off << rbits) | lrow[q];
            lo[q] = uint16_t(k);
            hi[q] = uint8_t(k >> 16);
        }
        dk24 = static_cast<uint16_t *>(p.dalloc(2 * nnz_pad));
        dk8 = static_cast<uint8_t *>(p.dalloc(nnz_pad));
        dcb = static_cast<uint32_t *>(p.dalloc(4 * nseg16));
        if (!dk24 || !dk8 || !dcb) return AXSPMV_E_NOMEM;
        AX_TRY(p.upload(dk24, lo.data(), 2 * nnz, s));
        AX_TRY(p.upload(dk8, hi.data(), nnz, s));
        AX_TRY(p.upload(dcb, sbase24.data(), 4 * nseg16, s));
    } else if (packed) {
        std::vector<uint32_t> key(nnz ? nnz : 1);
#pragma omp parallel for schedule(static)
        for (uint64_t q = 0; q < nnz; ++q)
            key[q] = uint32_t(((col[q] + nc - sbase[q >> SEG_LOG]) % nc) << rbits) | lrow[q];
        dk = static_cast<uint32_t *>(p.dalloc(4 * nnz_pad));
        dcb = static_cast<uint32_t *>(p.dalloc(4 * nseg));
        if (!dk || !dcb) return AXSPMV_E_NOMEM;
        AX_TRY(p.upload(dk, key.data(), 4 * nnz, s));
        AX_TRY(p.upload(dcb, sbase.data(), 4 * nseg, s));
    } else {
        dc = static_cast<uint32_t *>(p.dalloc(4 * nnz_pad));
        dl = static_cast<uint16_t *>(p.dalloc(2 * nnz_pad));
        if (!dc || !dl) return AXSPMV_E_NOMEM;
        AX_TRY(p.upload(dc, col.data(), 4 * nnz, s));
        AX_TRY(p.upload(dl, lrow.data(), 2 * nnz, s));
    }
    uint32_t block = p.o.block;
    // 512 threads (8 waves, one workgroup per CU with R = 16384) measured
    // fastest on the 2^20-row power-law matrix (82K entries per tile; 1024 is
    // 2-3 % slower); tiles of few entries want fewer lanes (graph-timed: the
    // Laplacian on 256^2, 1.3K per tile, 3.69 -> 3.05 us at 128; a 2^16-row
    // power-law matrix, 5.1K per tile, 9.17 -> 7.83 us at 256).
    if (block == 0) {
        const uint64_t per_tile = nnz / std::max<uint64_t>(1, nall);
        block = per_tile < 2048 ? 128 : per_tile < 16384 ? 256 : 512;
    }

    // S > 1: every tile writes its rows' sums when its loop ends, and all
    // tiles end together.  Where that write-out is heavy against the loop
    // (S n row sums >= nnz / 6), storing them in slice partials and merging
    // those in a second kernel beats adding them into a cleared y with FP64
    // atomics; where it is light, the merge's extra pass over S + 1 vectors
    // costs more than the adds.  Measured on one box, whole SpMV: the 2^20-row
    // power-law matrix (nnz 21 M) with 4 slices 60 against 66 us, 8 slices
    // 74 against 88 us, 2 slices 87 against 83 us; the permuted 27-point
    // stencil on 128^3 (nnz 56 M) with 2 slices 231 against 224 us, 4 slices
    // 242 against 240 us, 8 slices 267 against 274 us (partials against
    // atomics).  The plan of A^T, which adds into x_bar from its fused
    // value-gradient sweep, keeps the atomic adds.
    double *dpart = nullptr;
    const size_t pstride = (size_t(n) + 1) & ~size_t(1);  // every partial 16-byte aligned: two rows per lane in the merge
    if (S > 1 && !nhb && p.lds_per_row == 8 && !(p.o.flags & AXSPMV_PLAN_RCT_ATOMIC) && 6ull * S * n >= nnz) {
        dpart = static_cast<double *>(p.dalloc(8ull * S * pstride));
        if (!dpart) return AXSPMV_E_NOMEM;
    }
    p.rct = launch::RctArgs{dv, dc, dl, dk, dcb, dt, drb, n, R, S, nrb, p.o.vtype, block, rbits, a->ncols, dpart, pstride};
    // A matrix stream larger than the 256 MB Infinity Cache comes from HBM
    // on every SpMV whatever the loads do: it is streamed with non-temporal
    // loads, whatever the tile height (permuted 100^3 stencil, renumbered, one
    // box: 3968-row tiles 98 -> 90 us per SpMV, 1024-row tiles 99 -> 97; the
    // same in natural order 62 -> 57; 48 banded matrices with 16-bit keys,
    // 512-row tiles 92.6 -> 90.5, 1.5M banded rows, 5888-row tiles 102 -> 97).
    // A smaller stream stays cached between SpMVs, and non-temporal loads
    // give that up (the 2^20-row power-law matrix, 252 MB, back to back: 58 ->
    // 89 us).  Plans with heavy rows, which are for SpMM, have no such kernel:
    // their SpMV loads the ordinary way.
    p.rct.pal = dpal;
    // The table's copy in LDS costs its fill and reads that queue behind the
    // LDS adds; small matrices, whose stream is cached anyway, read it from the
    // vector L1 (graph-timed, no table / copy in LDS / from L1: 256^2 Laplacian
    // 3.18 / 3.54 / 3.31 us, 1000^2 14.7 / 11.6 / 12.3, +-1 on power-law
    // patterns of 5,000 rows 6.2 / 7.3 / 6.3, of 50,000 7.2 / 7.6 / 7.3, of
    // 100,000 (2.05M entries) 12.0 / 9.9 / 9.8, of 400,000 30.4 / 26.5 / 28.0,
    // permuted 40^3 stencil (1.64M) 8.3 / 7.3 / 7.4).
    p.rct.pal_lds = nnz >= (1u << 21);
    p.rct.nt_stream = !nhb && (vbytes + kbytes) * nnz > (256ull << 20) ? 1 : 0;
    p.rct.key16 = dk16;
    p.rct.key24 = dk24;
    p.rct.key8 = dk8;
    p.rct.cbits16 = cbits16;
    p.rct.dmin = uint32_t(uint64_t(dlo));
    if (nhb) {
        auto *dh = static_cast<uint32_t *>(p.dalloc(4 * hrows.size()));
        auto *db = static_cast<uint32_t *>(p.dalloc(4 * hbs.size()));
        auto *dm = static_cast<uint32_t *>(p.dalloc(4 * hmask.size()));
        if (!dh || !db || !dm) return AXSPMV_E_NOMEM;
        AX_TRY(p.upload(dh, hrows.data(), 4 * hrows.size(), s));
        AX_TRY(p.upload(db, hbs.data(), 4 * hbs.size(), s));
        AX_TRY(p.upload(dm, hmask.data(), 4 * hmask.size(), s));
        p.rct.nhb = nhb;
        p.rct.hs = HS;
        p.rct.nheavy = uint32_t(hrows.size());
        p.rct.hrows = dh;
        p.rct.hb_start = db;
        p.rct.hmask = dm;
    }
    p.slots = nnz;
    // matrix stream; with S > 1 the partials written and read back and y
    // written by the merge, or the clear of y and S atomic adds per row
    p.stream_bytes = (vbytes + kbytes) * nnz + 4 * tptr.size() +
                     (S == 1 ? 0 : dpart ? 8ull * (2 * S + 1) * n : 8ull * (S + 1) * n) + 8ull * HS * hrows.size();
    p.launches = S > 1 || nhb ? 2 : 1;
    p.nblocks = uint32_t(nall);
    p.kind = Plan::RCT;
    std::snprintf(p.name, sizeof p.name, "rct_r%u_s%u%s%s", Rt, S, diag ? "_k16" : packed ? "" : "_split",
                  S > 1 && !dpart && p.lds_per_row == 8 ? "_atomic" : "");
    return AXSPMV_OK;
}

launch::SegArgs seg_args(const Plan &p, const uint32_t *rowsrc) {
    launch::SegArgs g{};
    g.vplane = p.d_vplane;
    g.cplane = p.d_cplane;
    g.rowsrc = rowsrc;
    g.blocks = p.d_blocks;
    g.nblocks = p.nblocks;
    g.empty = p.d_empty;
    g.nempty = p.nempty;
    g.thw = p.thw;
    g.th = p.th;
    g.vtype = p.o.vtype;
    g.block = p.o.block;
    g.win = p.d_win;
    g.nt = p.seg_nt;
    return g;
}

}  // namespace

extern "C" int axspmv_opts_default(uint32_t format, axspmv_opts *o) {
    if (!o) return fail(AXSPMV_E_INVALID, "opts_default: NULL");
    std::memset(o, 0, sizeof *o);
    o->format = format;
    o->kernel = AXSPMV_KER_DEFAULT;
    o->mode = AXSPMV_AXT_UNC;
    o->thw = 4;
    o->th = 1;
    o->bs = 256;
    o->hbs = format == AXSPMV_FMT_CSR || format == AXSPMV_FMT_AXC ? 0 : 64;  // picked from the mean row length
    o->chunk = 64;
    o->reorder = 1;
    o->vtype = AXSPMV_F64;
    o->block = format == AXSPMV_FMT_RCT ? 0 : 256;  // RCT: 512 for SpMV, 1024 for SpMM
    o->budget = 0;
    if (format > AXSPMV_FMT_RCT) return fail(AXSPMV_E_INVALID, "opts_default: unknown format %u", format);
    return AXSPMV_OK;
}

namespace {

int plan_create(const axspmv_csr *a, const axspmv_opts *o, void *stream, bool transposed, axspmv_plan **out);

// Mean |row - column| over the entries.
double mean_diagonal_distance(const axspmv_csr *a) {
    double sum = 0.0;
#pragma omp parallel for schedule(dynamic, 4096) reduction(+ : sum)
    for (uint32_t i = 0; i < a->nrows; ++i)
        for (uint32_t j = a->row[i]; j < a->row[i + 1]; ++j) sum += a->col[j] > i ? a->col[j] - i : i - a->col[j];
    return a->nnz ? sum / a->nnz : 0.0;
}

// dst[k] = src[perm[k]] in two passes of launch::permute_chunks through a
// staging vector t, in chunks of L = 8192 positions (64 KB of LDS).  t holds
// the values chunk of destinations by chunk (t[c L ..] feeds dst[c L ..]),
// inside a chunk by source block, then by destination.  Pass 1, workgroup s
// = source block s (src[s L ..]): reads the block, writes each value to its
// place in t (w1), the block's values for one destination chunk side by
// side (b1 = the value's offset in the block, in the order of w1).  Pass 2,
// workgroup c: reads t[c L ..] whole, dst[k] = that chunk's value b2[k].
// Measured on the permuted 128^3 stencil (2M entries, about 32 values per
// run; kernel trace): 11.3 + 8.3 us per vector, against 34 us for one plain
// gather (each 8-byte read pulls a whole line from the Infinity Cache), 29
// us for two XCD-segmented gathers (each XCD reading an L2-resident eighth
// of the source at random), 20.5 us with the runs on the reading side and
// 23.8 us with chunks of 4096.
//
// Vectors of up to 2^20 entries (8 MB) are gathered by one launch instead:
// while the source more or less fits an L2 (4 MB) the gather runs at the
// L2's rate, and the second launch costs more than the lines read twice.
// Permuted stencils, AXT UNC SpMV, gather / two passes: 60^3 24.9 / 37.6 us,
// 90^3 73.5 / 80.3, 116^3 (1.56M entries) 159.2 / 146.8; RCT on 100^3 97.7 /
// 102.7.
constexpr uint32_t PERM_DIRECT = 1u << 20;
int upload_perm(Plan &p, const std::vector<uint32_t> &perm, Plan::Perm &out, hipStream_t s) {
    const uint32_t n = uint32_t(perm.size());
    out.idx = static_cast<uint32_t *>(p.dalloc(4ull * n));
    if (!out.idx) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(out.idx, perm.data(), 4ull * n, s));
    if (n <= PERM_DIRECT) return AXSPMV_OK;
    const uint32_t L = 8192;
    const uint64_t nch = ceil_div(n, L);
    // t position of every destination: chunk by chunk, sorted by (source block, k)
    std::vector<uint32_t> tp(n ? n : 1);
    std::vector<uint16_t> b1(n ? n : 1), b2(n ? n : 1);
#pragma omp parallel for schedule(static)
    for (uint64_t c = 0; c < nch; ++c) {
        const uint32_t k0 = uint32_t(c * L), k1 = uint32_t(std::min<uint64_t>(n, k0 + uint64_t(L)));
        std::vector<std::pair<uint32_t, uint32_t>> v;  // (source block, destination)
        v.reserve(k1 - k0);
        for (uint32_t k = k0; k < k1; ++k) v.emplace_back(perm[k] / L, k);
        std::sort(v.begin(), v.end());
        for (uint32_t i = 0; i < k1 - k0; ++i) {
            tp[v[i].second] = k0 + i;
            b2[v[i].second] = uint16_t(i);
        }
    }
    // pass 1: each source block's values in order of their t positions (a
    // counting pass over t: destination k sits at t position tp[k])
    std::vector<uint32_t> kat(n ? n : 1), w1(n ? n : 1), next(nch);
    for (uint32_t k = 0; k < n; ++k) kat[tp[k]] = k;
    for (uint64_t c = 0; c < nch; ++c) next[c] = uint32_t(c * L);
    for (uint32_t t = 0; t < n; ++t) {
        const uint32_t k = kat[t], blk = perm[k] / L, j = next[blk]++;
        w1[j] = t;
        b1[j] = uint16_t(perm[k] - blk * L);
    }
    out.L = L;
    out.b1 = static_cast<uint16_t *>(p.dalloc(2ull * n));
    out.b2 = static_cast<uint16_t *>(p.dalloc(2ull * n));
    out.w1 = static_cast<uint32_t *>(p.dalloc(4ull * n));
    if (!out.b1 || !out.b2 || !out.w1) return AXSPMV_E_NOMEM;
    AX_TRY(p.upload(out.b1, b1.data(), 2ull * n, s));
    AX_TRY(p.upload(out.b2, b2.data(), 2ull * n, s));
    return p.upload(out.w1, w1.data(), 4ull * n, s);
}

// AXSPMV_PLAN_REORDER: Q = the reverse Cuthill-McKee order of A, the plan of
// B = Q A Q^T (every other option as given) in `inner`, the permutation and
// its inverse on the device, and the vectors the gathers go through.
int plan_reordered(const axspmv_csr *a, const axspmv_opts *o, void *stream, axspmv_plan **out) {
    if (a->nrows != a->ncols)
        return fail(AXSPMV_E_INVALID, "AXSPMV_PLAN_REORDER: the %u x %u matrix is not square", a->nrows, a->ncols);
    std::vector<uint32_t> q, pos;
    AX_TRY(rcm_order(a, q));
    axspmv_csr *b = nullptr;
    AX_TRY(csr_permute_sym(a, q, &b, &pos));
    axspmv_opts oi = *o;
    oi.flags &= ~AXSPMV_PLAN_REORDER;
    // Worth it only where the new order brings the entries at least twice
    // as close to the diagonal on average (a random matrix gains nothing, a
    // banded one is already close): else the plan of A itself.
    if (2.0 * mean_diagonal_distance(b) > mean_diagonal_distance(a)) {
        axspmv_csr_free(b);
        return plan_create(a, &oi, stream, false, out);
    }
    axspmv_plan *pi = nullptr;
    const int rc = plan_create(b, &oi, stream, false, &pi);
    axspmv_csr_free(b);
    if (rc) return rc;
    auto p = std::make_unique<Plan>();
    p->inner = pi;
    p->kind = Plan::REORDERED;
    p->o = pi->o;
    p->o.flags |= AXSPMV_PLAN_REORDER;
    p->device = pi->device;
    p->nrows = a->nrows;
    p->ncols = a->ncols;
    p->nnz = a->nnz;
    p->thw = pi->thw;
    p->th = pi->th;
    const uint32_t n = a->nrows;
    std::vector<uint32_t> qi(n);
    for (uint32_t k = 0; k < n; ++k) qi[q[k]] = k;
    hipStream_t s = static_cast<hipStream_t>(stream);
    AX_TRY(upload_perm(*p, q, p->to_b, s));
    AX_TRY(upload_perm(*p, qi, p->from_b, s));
    p->nscratch = pi->T ? 6 : 3;
    for (uint32_t k = 0; k < p->nscratch; ++k) {
        p->d_scr[k] = static_cast<double *>(p->dalloc(8ull * n));
        if (!p->d_scr[k]) return AXSPMV_E_NOMEM;
    }
    p->bpos = std::move(pos);
    std::snprintf(p->name, sizeof p->name, "%.59s_rcm", pi->name);
    p->slots = pi->slots;
    p->beta = pi->beta;
    p->device_bytes += pi->device_bytes;
    p->alg_bytes = pi->alg_bytes;
    // the inner plan's bytes, then per vector permuted (x into B's order
    // before the SpMV, y back after it) 8 B read and 8 B written, by one
    // gather with 4 B of index or by two passes with 2 + 6 B.  (RCT tiles
    // storing their rows straight into A's numbering, y[q[k]], measured slower
    // on the permuted 128^3 stencil: the tile kernel took 38 us more with
    // ordinary scattered stores, 56 us more with non-temporal ones, against 30
    // us for the two passes.)
    const bool direct = !p->to_b.L;
    p->stream_bytes = pi->stream_bytes + 2ull * (direct ? 20 : 40) * n;
    p->launches = pi->launches + (direct ? 2 : 4);
    p->nblocks = pi->by_slice ? pi->by_slice->nblocks : pi->nblocks;
    p->staged_blocks = pi->staged_blocks;
    p->rowwise = pi->rowwise;
    *out = p.release();
    return AXSPMV_OK;
}

// axspmv_plan_create; `transposed` marks the plan of A^T that a plan with
// AXSPMV_PLAN_TRANSPOSE builds (RCT: entry positions kept, 16 B of LDS per
// tile row for the fused value gradient).
int plan_create(const axspmv_csr *a, const axspmv_opts *o, void *stream, bool transposed, axspmv_plan **out) {
    if (!a || !o || !out) return fail(AXSPMV_E_INVALID, "plan_create: NULL argument");
    *out = nullptr;
    // Every kernel gathers x[col] without a bounds check: offsets and
    // columns are checked before anything is built.
    AX_TRY(check_csr_bounds(a, "plan_create"));
    if (o->vtype > AXSPMV_F32) return fail(AXSPMV_E_INVALID, "plan_create: unknown value type %u", o->vtype);
    // A group of lanes per row (CSR vector, AXC): the launch counts nrows x
    // lanes work-items, which must fit the 32-bit grid size of a dispatch.
    if ((o->format == AXSPMV_FMT_CSR && o->kernel == AXSPMV_KER_STREAM) ||
        (o->format == AXSPMV_FMT_AXC && !(o->flags & AXSPMV_PLAN_AX_LAYOUT))) {
        const uint64_t g = o->hbs ? o->hbs : lanes_for_mean(a);
        if (uint64_t(a->nrows) * g >= (1ull << 32))
            return fail(AXSPMV_E_OVERFLOW, "plan_create: %u rows x %llu lanes per row exceed a 32-bit grid", a->nrows,
                        (unsigned long long)g);
    }
    if (o->flags & AXSPMV_PLAN_REORDER) return plan_reordered(a, o, stream, out);
    auto p = std::make_unique<Plan>();
    p->o = *o;
    if (transposed) {
        p->keep_pos = true;
        p->lds_per_row = 16;
    }
    if (p->o.th == 0) p->o.th = 1;
    if (p->o.thw == 0) p->o.thw = p->o.th == 1 ? 4 : 64;
    if (p->o.hbs == 0 && p->o.format != AXSPMV_FMT_CSR && p->o.format != AXSPMV_FMT_AXC) p->o.hbs = 64;
    if (p->o.chunk == 0) p->o.chunk = 64;
    if (p->o.bs == 0) p->o.bs = 256;
    if (hipGetDevice(&p->device) != hipSuccess) return fail(AXSPMV_E_HIP, "plan_create: no HIP device");
    p->nrows = a->nrows;
    p->ncols = a->ncols;
    p->nnz = a->nnz;
    hipStream_t s = static_cast<hipStream_t>(stream);
    int rc = AXSPMV_OK;
    switch (o->format) {
        case AXSPMV_FMT_CSR: rc = plan_csr(*p, a, s); break;
        case AXSPMV_FMT_K1: rc = plan_k1(*p, a, s); break;
        case AXSPMV_FMT_AXC: rc = plan_axc(*p, a, s); break;
        case AXSPMV_FMT_AXT: rc = plan_axt(*p, a, s); break;
        case AXSPMV_FMT_RCT: rc = plan_rct(*p, a, s); break;
        default: rc = fail(AXSPMV_E_INVALID, "plan_create: unknown format %u", o->format);
    }
    if (rc) return rc;
    if (p->o.flags & AXSPMV_PLAN_TRANSPOSE) AX_TRY(plan_add_transpose(p.get(), a, s));
    const size_t vs = p->o.vtype == AXSPMV_F32 ? 4 : 8;
    p->alg_bytes = (vs + 4) * uint64_t(a->nnz) + 4ull * (a->nrows + 1) + 8ull * a->ncols + 8ull * a->nrows;
    p->stream_bytes += 8ull * a->ncols + 8ull * a->nrows;
    p->beta = p->slots ? double(a->nnz) / double(p->slots) : 0.0;
    *out = p.release();
    return AXSPMV_OK;
}

}  // namespace

extern "C" int axspmv_plan_create(const axspmv_csr *a, const axspmv_opts *o, void *stream, axspmv_plan **out) {
    return plan_create(a, o, stream, false, out);
}

extern "C" int axspmv_plan_destroy(axspmv_plan *p) {
    delete p;
    return AXSPMV_OK;
}

extern "C" int axspmv_plan_get_info(const axspmv_plan *p, axspmv_plan_info *info) {
    if (!p || !info) return fail(AXSPMV_E_INVALID, "plan_get_info: NULL argument");
    std::memset(info, 0, sizeof *info);
    std::snprintf(info->name, sizeof info->name, "%s", p->name);
    info->nrows = p->nrows;
    info->ncols = p->ncols;
    info->nnz = p->nnz;
    info->format = p->o.format;
    info->slots = p->slots;
    info->device_bytes = p->device_bytes;
    info->stream_bytes = p->stream_bytes;
    info->alg_bytes = p->alg_bytes;
    info->beta = p->beta;
    info->launches = p->launches;
    info->nblocks = p->by_slice ? p->by_slice->nblocks : p->nblocks;
    info->staged_blocks = p->staged_blocks;
    return AXSPMV_OK;
}

namespace axspmv {

// v.dst = v.src permuted by q, by a plain gather (q.L == 0) or in two passes,
// vector i staged in t[i] (no stage is another vector's source)
static hipError_t permute(const Plan *p, const Plan::Perm &q, const launch::PermVecs &v, double *const *t, hipStream_t s) {
    if (!q.L) {
        launch::GatherVecs g{};
        for (uint32_t i = 0; i < v.count; ++i) {
            g.idx[i] = q.idx;
            g.src[i] = v.src[i];
            g.dst[i] = v.dst[i];
        }
        g.count = v.count;
        g.rb = v.rb;
        g.res = v.res;
        return launch::gather_vecs(p->nrows, g, s);
    }
    launch::PermVecs one = v, two = v;
    one.res = nullptr;
    for (uint32_t i = 0; i < v.count; ++i) {
        one.dst[i] = t[i];
        two.src[i] = t[i];
    }
    hipError_t e = launch::permute_chunks(q.w1, q.b1, p->nrows, q.L, one, s);
    if (e == hipSuccess) e = launch::permute_chunks(nullptr, q.b2, p->nrows, q.L, two, s);
    return e;
}
static launch::PermVecs perm_vec(const double *src, double *dst) { return {{src}, {dst}, 1, nullptr, nullptr}; }
// One vector, staged in the plan's last scratch vector
static hipError_t permute(const Plan *p, const Plan::Perm &q, const double *src, double *dst, hipStream_t s) {
    return permute(p, q, perm_vec(src, dst), &p->d_scr[p->nscratch - 1], s);
}

hipError_t plan_launch(axspmv_plan *p, const double *x, double *y, hipStream_t s) {
    switch (p->kind) {
        case Plan::CSR_NAIVE:
            return launch::csr_naive(p->nrows, p->d_val, p->o.vtype, p->d_col, p->d_row, x, y, p->o.block, s);
        case Plan::CSR_VECTOR:
            return launch::csr_vector(p->nrows, p->d_val, p->o.vtype, p->d_col, p->d_row, p->lanes, p->spmm.long_slots,
                                      p->spmm.longrows, p->spmm.nlong, x, y, s, p->seg_nt);
        case Plan::AXT_UNC_H1:
            if (p->by_slice) return plan_launch(p->by_slice, x, y, s);
            return launch::axt_unc_h1(seg_args(*p, p->d_sec), x, y, s);
        case Plan::AXT_UNC_H1_SLICED: {
            launch::SegArgs g = seg_args(*p, p->d_sec);
            g.seq = p->seq.empty() ? nullptr : p->seq.data();
            g.nrows_add = p->nrows;
            g.mid = p->mid;
            g.part = p->d_part;
            g.S = p->slices;
            return launch::axt_unc_h1(g, x, y, s);
        }
        case Plan::AXT_UNC_H: return launch::axt_unc_h(seg_args(*p, p->d_sec), x, y, s);
        case Plan::AXT_COM: return launch::axt_com(p->com, x, y, s);
        case Plan::K1: return launch::k1(p->k1, x, y, s);
        case Plan::AXC: return launch::axc(p->axc, x, y, s);
        case Plan::RCT: return launch::rct(p->rct, x, y, s, p->mid);
        case Plan::REORDERED: {
            hipError_t e = permute(p, p->to_b, x, p->d_scr[0], s);
            if (e == hipSuccess) e = plan_launch(p->inner, p->d_scr[0], p->d_scr[1], s);
            if (e == hipSuccess) e = permute(p, p->from_b, p->d_scr[1], y, s);
            return e;
        }
        case Plan::AXT_UNC_H1_AX: {
            const hipError_t e = launch::x_refresh(p->d_axmap, p->slots, ilog2(p->thw), p->ncols, x, p->d_ax, s);
            if (e != hipSuccess) return e;
            launch::SegArgs g = seg_args(*p, p->d_sec);
            g.vplane = p->d_ax;
            g.win = nullptr;
            return launch::axt_unc_h1_ax(g, y, s);
        }
        default: return hipErrorInvalidValue;
    }
}

}  // namespace axspmv

extern "C" int axspmv_spmv(axspmv_plan *p, const double *d_x, double *d_y, void *stream) {
    if (!p || (!d_x && p->ncols) || (!d_y && p->nrows)) return fail(AXSPMV_E_INVALID, "spmv: NULL argument");
    const hipError_t e = plan_launch(p, d_x, d_y, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? AXSPMV_OK : hip_fail(e, "spmv launch");
}

// ---------------------------------------------------------------- adjoint
namespace {

launch::SegArgs fused_args(const Plan &p) {
    launch::SegArgs g = seg_args(p, p.d_sec);
    g.blocks = p.d_fblocks;
    g.nblocks = p.nfblocks;
    g.win = nullptr;  // windows belong to the SpMV blocks
    return g;
}

// u[0 .. nu) and v[0 .. nv) do not overlap
bool apart(const double *u, uint64_t nu, const double *v, uint64_t nv) { return u + nu <= v || v + nv <= u; }

hipError_t launch_vbar(Plan *p, const double *ybar, const double *x, double *vbar, hipStream_t s) {
    // RCT: over the plan of A^T (rows = columns of A), whose entry order is
    // the one the fused forward + adjoint writes: x rows in LDS, ybar gathered
    if (p->kind == Plan::RCT) return launch::rct_vbar(p->T->rct, x, ybar, vbar, s);
    if (p->kind == Plan::AXT_UNC_H1)
        return launch::axt_unc_h1_vbar(seg_args(*p, p->d_sec), p->nunits, x, ybar, vbar,
                                       launch::VbarArgs{p->d_rowptr, p->d_first}, s);
    return launch::csr_vbar(p->nrows, p->d_col, p->d_row, x, ybar, vbar, s);
}

hipError_t launch_fwd_adj(Plan *p, const double *x, const double *b, double *y, double *r, double *xbar,
                          double *vbar, bool fused, hipStream_t s) {
    hipError_t e;
    if (fused && p->kind != Plan::RCT) {  // RCT: r needs every slice's sums first
        if (p->kind == Plan::AXT_UNC_H1)
            e = launch::axt_unc_h1_fused(fused_args(*p), x, b, y, r, vbar, launch::VbarArgs{p->d_rowptr, p->d_first}, s);
        else
            e = launch::csr_fused(p->nrows, p->d_val, p->o.vtype, p->d_col, p->d_row, x, b, y, r, vbar, s);
        if (e != hipSuccess) return e;
        return plan_launch(p->T, r, xbar, s);
    }
    if (p->kind == Plan::RCT) {
        // r = y - b where y's rows are written (the slice merge, or the tile
        // kernel of one slice).  With the non-temporal v_bar stores of the
        // sweep over A^T, forward + adjoint on the 2^20-row power-law matrix,
        // one box: 232.6 -> 223.4 us.
        // The merge also clears x_bar where the sweep will add slices into it.
        const uint32_t nx = p->ncols;
        if (fused && p->T->rct.S > 1 && apart(xbar, nx, y, p->nrows) && apart(xbar, nx, b, p->nrows) &&
            apart(xbar, nx, r, p->nrows)) {
            e = launch::rct(p->rct, x, y, s, nullptr, nullptr, nullptr, b, r, xbar, nx);
            if (e == hipSuccess)
                e = launch::rct(p->T->rct, r, xbar, s, nullptr, x, vbar, nullptr, nullptr, nullptr, 0, true);
            return e;
        }
        e = launch::rct(p->rct, x, y, s, nullptr, nullptr, nullptr, b, r);
    } else {
        e = plan_launch(p, x, y, s);
        if (e == hipSuccess) e = launch::residual(p->nrows, y, b, r, s);
    }
    if (fused && p->kind == Plan::RCT) {
        // x_bar = A^T r and v_bar in one sweep over the plan of A^T
        if (e == hipSuccess) e = launch::rct(p->T->rct, r, xbar, s, nullptr, x, vbar);
        return e;
    }
    if (e == hipSuccess) e = plan_launch(p->T, r, xbar, s);
    if (e == hipSuccess) e = launch_vbar(p, r, x, vbar, s);
    return e;
}

// RCT tiles hold R x ktile sums in LDS: the default k-tile is also cut to
// what fits.
uint32_t pick_ktile(const Plan *p, uint32_t k) {
    if (p->o.ktile) return p->o.ktile;
    uint32_t kt = 8;
    while (kt < 64 && kt < k) kt *= 2;
    if (p->kind == Plan::RCT)
        while (kt > 8 && uint64_t(p->rct.R) * kt * 8 > p->lds_max) kt /= 2;
    return kt;
}

bool adjoint_kind(const Plan *p) {
    return p->kind == Plan::AXT_UNC_H1 || p->kind == Plan::CSR_NAIVE || p->kind == Plan::RCT;
}

}  // namespace

namespace axspmv {

int plan_add_transpose(Plan *p, const axspmv_csr *a, hipStream_t s) {
    axspmv_csr *t = nullptr;
    std::vector<uint32_t> perm;  // position in A^T -> position in A
    AX_TRY(csr_transpose_perm(a, &t, &perm));
    axspmv_opts o = p->o;
    o.flags &= ~AXSPMV_PLAN_TRANSPOSE;
    axspmv_plan *pt = nullptr;
    const int rc = plan_create(t, &o, s, true, &pt);
    if (rc) {
        axspmv_csr_free(t);
        return rc;
    }
    p->T = pt;
    if (pt->kind == Plan::RCT && (p->o.flags & AXSPMV_PLAN_DETERMINISTIC)) {
        // x_bar = A^T y_bar without atomics: the AXT layout of A^T in column
        // slices of at most 2 MB of y_bar (at most 8), slice partials summed
        // in slice order.  Two slots per tile: on the column-uniform rows of
        // a power-law matrix's transpose the least padding per slice.
        axspmv_opts od{};
        axspmv_opts_default(AXSPMV_FMT_AXT, &od);
        od.thw = 2;
        od.vtype = p->o.vtype;
        od.flags = AXSPMV_PLAN_DETERMINISTIC;
        uint32_t S = 1;
        while (S < 8 && 8ull * t->ncols > (2ull << 20) * S) S *= 2;
        od.slices = S;
        axspmv_plan *pd = nullptr;
        const int rd = plan_create(t, &od, s, false, &pd);
        if (rd) {
            axspmv_csr_free(t);
            return rd;
        }
        p->Tdet = pd;
    }
    axspmv_csr_free(t);
    if (pt->kind == Plan::RCT) {
        // v_bar comes out in the transposed plan's entry order: the position
        // in A of each of its entries
        p->rct_pos.resize(pt->rct_pos.size());
        for (size_t e = 0; e < pt->rct_pos.size(); ++e) p->rct_pos[e] = perm[pt->rct_pos[e]];
        std::vector<uint32_t>().swap(pt->rct_pos);
    }
    return AXSPMV_OK;
}

// A reordered plan: inputs gathered into B's numbering (x~ = Q x: x~[k] =
// x[perm[k]]), the operation on the plan of B, results gathered back (y =
// Q^T y~: y[i] = y~[iperm[i]]).  With B = Q A Q^T, A^T = Q^T B^T Q, so the
// adjoint takes the same two gathers; v_bar stays in the order of B's plan.
static hipError_t reordered_op(Plan *p, uint32_t op, const axspmv_operands &o, hipStream_t s) {
    double *const *w = p->d_scr;
    auto in = [&](const double *v, double *d) { return permute(p, p->to_b, v, d, s); };
    auto back = [&](const double *v, double *d) { return permute(p, p->from_b, v, d, s); };
    // two vectors into w[0] and w[1], together where there is a second stage
    auto in2 = [&](const double *u, const double *v) {
        if (p->nscratch < 4) {
            const hipError_t e = in(u, w[0]);
            return e == hipSuccess ? in(v, w[1]) : e;
        }
        double *const t[2] = {w[2], w[p->nscratch - 1]};
        return permute(p, p->to_b, launch::PermVecs{{u, v}, {w[0], w[1]}, 2, nullptr, nullptr}, t, s);
    };
    auto free_of_b = [&](const double *v) { return apart(o.b, p->nrows, v, p->nrows); };
    axspmv_operands io{};
    hipError_t e = hipSuccess;
    switch (op) {
        case AXSPMV_OP_SPMV: return plan_launch(p, o.x, o.y, s);
        case AXSPMV_OP_ADJOINT:
            io.ybar = w[0];
            io.xbar = w[1];
            e = in(o.ybar, w[0]);
            if (e == hipSuccess) e = plan_op(p->inner, op, io, s);
            if (e == hipSuccess) e = back(w[1], o.xbar);
            return e;
        case AXSPMV_OP_VBAR:
            io.ybar = w[0];
            io.x = w[1];
            io.vbar = o.vbar;
            e = in2(o.ybar, o.x);
            if (e == hipSuccess) e = plan_op(p->inner, op, io, s);
            return e;
        case AXSPMV_OP_FWD_ADJ:
        case AXSPMV_OP_FWD_ADJ_SPLIT:
            if (op == AXSPMV_OP_FWD_ADJ && p->inner->kind != Plan::RCT) {
                // the format's fused sweep takes b: x and b in together, y and
                // x_bar out together, r = y - b formed again on y's way out
                // (where an output lies over b: r out as the third vector)
                io.x = w[0];
                io.b = w[1];
                io.y = w[2];
                io.r = w[3];
                io.xbar = w[4];
                io.vbar = o.vbar;
                e = in2(o.x, o.b);
                if (e == hipSuccess) e = plan_op(p->inner, op, io, s);
                if (e != hipSuccess) return e;
                if (free_of_b(o.y) && free_of_b(o.xbar) && free_of_b(o.r))
                    return permute(p, p->from_b, launch::PermVecs{{w[2], w[4]}, {o.y, o.xbar}, 2, o.b, o.r}, w, s);
                double *const t[3] = {w[0], w[1], w[p->nscratch - 1]};
                return permute(p, p->from_b, launch::PermVecs{{w[2], w[3], w[4]}, {o.y, o.r, o.xbar}, 3, nullptr, nullptr}, t, s);
            }
            // x in, the product, y back and r in, then x_bar and v_bar from
            // B's plan of B^T (RCT: one sweep; otherwise the adjoint and the
            // value gradient), x_bar back.  y's way back and r's way in are
            // one launch of gathers, or, in two passes, meet in the same
            // chunks of A's numbering: one kernel does the second pass of the
            // one, the residual and the first pass of the other (y~'s vector,
            // spent by then, takes r's runs; with the non-temporal v_bar
            // stores of the RCT sweep, on one box: the permuted 128^3
            // stencil, RCT, 483.4 -> 470.0 us).
            e = in(o.x, w[0]);
            if (e == hipSuccess) e = plan_launch(p->inner, w[0], w[1], s);
            if (!p->to_b.L && !(free_of_b(o.y) && free_of_b(o.r))) {  // y or r over b: r from y, then r in
                if (e == hipSuccess)
                    e = permute(p, p->from_b, launch::PermVecs{{w[1]}, {o.y}, 1, o.b, o.r}, w, s);
                if (e == hipSuccess) e = in(o.r, w[2]);
            } else if (!p->to_b.L) {
                // one launch: y = y~ back, r = y - b, and r~ = y~ - (b in B's order)
                launch::GatherVecs g{};
                g.idx[0] = p->from_b.idx;
                g.src[0] = w[1];
                g.dst[0] = o.y;
                g.rb = o.b;
                g.res = o.r;
                g.idx[1] = p->to_b.idx;
                g.src[1] = o.b;
                g.from[1] = w[1];
                g.dst[1] = w[2];
                g.count = 2;
                if (e == hipSuccess) e = launch::gather_vecs(p->nrows, g, s);
            } else {
                double *t = p->d_scr[p->nscratch - 1];
                const Plan::Perm &f = p->from_b, &g = p->to_b;
                if (e == hipSuccess) e = launch::permute_chunks(f.w1, f.b1, p->nrows, f.L, perm_vec(w[1], t), s);
                if (e == hipSuccess)
                    e = launch::back_residual_in(f.b2, g.w1, g.b1, p->nrows, f.L, t, o.b, o.y, o.r, w[1], s);
                if (e == hipSuccess) e = launch::permute_chunks(nullptr, g.b2, p->nrows, g.L, perm_vec(w[1], w[2]), s);
            }
            if (e != hipSuccess) return e;
            if (op == AXSPMV_OP_FWD_ADJ) {  // RCT: x_bar = B^T r~ and v_bar in one sweep over the plan of B^T
                e = launch::rct(p->inner->T->rct, w[2], w[3], s, nullptr, w[0], o.vbar);
            } else {
                io.ybar = w[2];
                io.xbar = w[3];
                e = plan_op(p->inner, AXSPMV_OP_ADJOINT, io, s);
                io.x = w[0];
                io.vbar = o.vbar;
                if (e == hipSuccess) e = plan_op(p->inner, AXSPMV_OP_VBAR, io, s);
            }
            if (e == hipSuccess) e = back(w[3], o.xbar);
            return e;
        case AXSPMV_OP_SPMM: {  // rows of X into B's order, Y's rows back
            const uint64_t nk = uint64_t(p->nrows) * o.k;
            if (!p->d_mm || p->mm_cap < 2 * nk) return hipErrorInvalidValue;  // plan_op_prepare first
            io.k = o.k;
            io.X = p->d_mm;
            io.Y = p->d_mm + nk;
            e = launch::gather_rows(p->to_b.idx, p->nrows, o.k, o.X, p->d_mm, s);
            if (e == hipSuccess) e = plan_op(p->inner, op, io, s);
            if (e == hipSuccess) e = launch::gather_rows(p->from_b.idx, p->nrows, o.k, p->d_mm + nk, o.Y, s);
            return e;
        }
        case AXSPMV_OP_XREFRESH:
            io.x = w[0];
            e = in(o.x, w[0]);
            if (e == hipSuccess) e = plan_op(p->inner, op, io, s);
            return e;
        default: return hipErrorInvalidValue;
    }
}

hipError_t plan_op(Plan *p, uint32_t op, const axspmv_operands &o, hipStream_t s) {
    if (p->kind == Plan::REORDERED) return reordered_op(p, op, o, s);
    switch (op) {
        case AXSPMV_OP_SPMV: return plan_launch(p, o.x, o.y, s);
        case AXSPMV_OP_ADJOINT: return plan_launch(p->Tdet ? p->Tdet : p->T, o.ybar, o.xbar, s);
        case AXSPMV_OP_VBAR: return launch_vbar(p, o.ybar, o.x, o.vbar, s);
        case AXSPMV_OP_FWD_ADJ: return launch_fwd_adj(p, o.x, o.b, o.y, o.r, o.xbar, o.vbar, true, s);
        case AXSPMV_OP_FWD_ADJ_SPLIT: return launch_fwd_adj(p, o.x, o.b, o.y, o.r, o.xbar, o.vbar, false, s);
        case AXSPMV_OP_SPMM:
            if (p->kind == Plan::RCT) {
                // 1024-lane workgroups unless the plan sets the block: a tile
                // has ktile times the SpMV's LDS adds to hide
                launch::RctArgs a = p->rct;
                if (!p->o.block) a.block = 1024;
                return launch::rct_spmm(a, o.k, pick_ktile(p, o.k), o.X, o.Y, s);
            }
            return launch::spmm(p->spmm, o.k, pick_ktile(p, o.k), o.X, o.Y, s);
        case AXSPMV_OP_XREFRESH:
            return launch::x_refresh(p->d_axmap, p->slots, ilog2(p->thw), p->ncols, o.x, p->d_ax, s);
        default: return hipErrorInvalidValue;
    }
}

int plan_op_check(const Plan *p, uint32_t op, const axspmv_operands &o) {
    if (!p) return fail(AXSPMV_E_INVALID, "NULL plan");
    if (p->kind == Plan::REORDERED) {
        if (op > AXSPMV_OP_XREFRESH) return fail(AXSPMV_E_INVALID, "unknown operation %u", op);
        if (op == AXSPMV_OP_SPMM && uint64_t(p->nrows) * o.k >= (1ull << 40))
            return fail(AXSPMV_E_OVERFLOW, "SpMM: %u rows x k %u", p->nrows, o.k);
        if (op == AXSPMV_OP_SPMV && ((!o.x && p->ncols) || (!o.y && p->nrows)))
            return fail(AXSPMV_E_INVALID, "spmv: NULL argument");
        return plan_op_check(p->inner, op, o);  // the operation's own conditions, on the plan of B
    }
    const bool needT = op == AXSPMV_OP_ADJOINT || op == AXSPMV_OP_FWD_ADJ || op == AXSPMV_OP_FWD_ADJ_SPLIT ||
                       (op == AXSPMV_OP_VBAR && p->kind == Plan::RCT);
    if (needT && !p->T)
        return fail(AXSPMV_E_INVALID, "%s needs a plan created with AXSPMV_PLAN_TRANSPOSE",
                    op == AXSPMV_OP_VBAR ? "the RCT value gradient (it runs on the plan of A^T)" : "the adjoint");
    if ((op == AXSPMV_OP_VBAR || op == AXSPMV_OP_FWD_ADJ || op == AXSPMV_OP_FWD_ADJ_SPLIT) && !adjoint_kind(p))
        return fail(AXSPMV_E_UNSUPPORTED, "value gradient: plan %s is not CSR naive, AXT UNC th=1 or RCT", p->name);
    if (op == AXSPMV_OP_SPMM) {
        if (!p->rowwise && p->kind != Plan::RCT)
            return fail(AXSPMV_E_UNSUPPORTED, "SpMM: plan %s is not CSR, AXC, AXT UNC th=1 or RCT", p->name);
        if (o.k == 0) return fail(AXSPMV_E_INVALID, "SpMM: k must be > 0");
        const uint32_t kt = pick_ktile(p, o.k);
        if (kt != 8 && kt != 16 && kt != 32 && kt != 64) return fail(AXSPMV_E_INVALID, "SpMM: ktile %u not in 8/16/32/64", kt);
        if (p->kind != Plan::RCT && uint64_t(p->nrows) * kt >= (1ull << 32))
            return fail(AXSPMV_E_OVERFLOW, "SpMM: %u rows x ktile %u exceed a 32-bit grid", p->nrows, kt);
        if (p->kind == Plan::RCT && uint64_t(p->rct.R) * kt * 8 > p->lds_max)
            return fail(AXSPMV_E_UNSUPPORTED,
                        "SpMM: RCT tiles of %u rows x ktile %u need %llu bytes of LDS, %zu available (plan with "
                        "tile_rows <= %zu)",
                        p->rct.R, kt, (unsigned long long)(uint64_t(p->rct.R) * kt * 8), p->lds_max,
                        p->lds_max / (8 * size_t(kt)));
        if ((!o.X && p->ncols) || (!o.Y && p->nrows)) return fail(AXSPMV_E_INVALID, "SpMM: NULL operand");
    }
    if (op == AXSPMV_OP_XREFRESH) {
        if (p->kind != Plan::AXT_UNC_H1_AX)
            return fail(AXSPMV_E_UNSUPPORTED, "x refresh: plan %s was not created with AXSPMV_PLAN_AX_LAYOUT", p->name);
        if (!o.x && p->ncols) return fail(AXSPMV_E_INVALID, "x refresh: NULL x");
    }
    if (op > AXSPMV_OP_XREFRESH) return fail(AXSPMV_E_INVALID, "unknown operation %u", op);
    return AXSPMV_OK;
}

int plan_op_prepare(Plan *p, uint32_t op, const axspmv_operands &o) {
    if (p->kind != Plan::REORDERED || op != AXSPMV_OP_SPMM) return AXSPMV_OK;
    const uint64_t need = 2ull * p->nrows * o.k;
    if (p->d_mm && p->mm_cap >= need) return AXSPMV_OK;
    // A smaller buffer stays allocated until the plan goes: a graph captured
    // with it may still run.
    void *m = p->dalloc(8 * std::max<uint64_t>(need, 1));
    if (!m) return AXSPMV_E_NOMEM;
    p->d_mm = static_cast<double *>(m);
    p->mm_cap = need;
    return AXSPMV_OK;
}

}  // namespace axspmv

extern "C" int axspmv_adjoint(axspmv_plan *p, const double *d_ybar, double *d_xbar, void *stream) {
    axspmv_operands o{};
    o.ybar = d_ybar;
    o.xbar = d_xbar;
    AX_TRY(plan_op_check(p, AXSPMV_OP_ADJOINT, o));
    const hipError_t e = plan_op(p, AXSPMV_OP_ADJOINT, o, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? AXSPMV_OK : hip_fail(e, "adjoint launch");
}

extern "C" int axspmv_vbar(axspmv_plan *p, const double *d_ybar, const double *d_x, double *d_vbar, void *stream) {
    axspmv_operands o{};
    o.ybar = d_ybar;
    o.x = d_x;
    o.vbar = d_vbar;
    AX_TRY(plan_op_check(p, AXSPMV_OP_VBAR, o));
    const hipError_t e = plan_op(p, AXSPMV_OP_VBAR, o, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? AXSPMV_OK : hip_fail(e, "vbar launch");
}

extern "C" int axspmv_fwd_adj(axspmv_plan *p, const double *d_x, const double *d_b, double *d_y, double *d_r,
                              double *d_xbar, double *d_vbar, int fused, void *stream) {
    axspmv_operands o{};
    o.x = d_x;
    o.b = d_b;
    o.y = d_y;
    o.r = d_r;
    o.xbar = d_xbar;
    o.vbar = d_vbar;
    const uint32_t op = fused ? AXSPMV_OP_FWD_ADJ : AXSPMV_OP_FWD_ADJ_SPLIT;
    AX_TRY(plan_op_check(p, op, o));
    const hipError_t e = plan_op(p, op, o, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? AXSPMV_OK : hip_fail(e, "fwd_adj launch");
}

extern "C" int axspmv_spmm(axspmv_plan *p, uint32_t k, const double *d_X, double *d_Y, void *stream) {
    axspmv_operands o{};
    o.k = k;
    o.X = d_X;
    o.Y = d_Y;
    AX_TRY(plan_op_check(p, AXSPMV_OP_SPMM, o));
    AX_TRY(plan_op_prepare(p, AXSPMV_OP_SPMM, o));
    const hipError_t e = plan_op(p, AXSPMV_OP_SPMM, o, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? AXSPMV_OK : hip_fail(e, "spmm launch");
}

extern "C" int axspmv_plan_vbar_positions(const axspmv_plan *p, uint32_t *h_pos, uint64_t count) {
    if (!p || (count && !h_pos)) return fail(AXSPMV_E_INVALID, "vbar_positions: NULL argument");
    if (count != p->nnz) return fail(AXSPMV_E_INVALID, "vbar_positions: count %llu != nnz %u", (unsigned long long)count, p->nnz);
    if (p->kind == Plan::REORDERED) {  // positions in B, then in A
        AX_TRY(axspmv_plan_vbar_positions(p->inner, h_pos, count));
        for (uint64_t k = 0; k < count; ++k) h_pos[k] = p->bpos[h_pos[k]];
        return AXSPMV_OK;
    }
    if (p->kind == Plan::RCT) {
        if (!p->T)
            return fail(AXSPMV_E_UNSUPPORTED, "vbar_positions: RCT plan created without AXSPMV_PLAN_TRANSPOSE");
        std::copy(p->rct_pos.begin(), p->rct_pos.end(), h_pos);
        return AXSPMV_OK;
    }
    if (!adjoint_kind(p)) return fail(AXSPMV_E_UNSUPPORTED, "vbar_positions: plan %s has no value gradient", p->name);
    for (uint64_t k = 0; k < count; ++k) h_pos[k] = uint32_t(k);
    return AXSPMV_OK;
}
