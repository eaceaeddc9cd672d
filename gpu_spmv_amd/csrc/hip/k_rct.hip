// RCT: row-block x column-slice tiles with entries sorted by column.
//
// Random column indices make SpMV a gather problem: every nonzero costs one
// L2 request for x, and once x outgrows an XCD's 4 MB L2 the requests go to
// the Infinity Cache.  RCT attacks both:
//
//  * the matrix is cut into tiles of (at most) R rows x C columns (S = ncols /
//    C column slices); row blocks hold about equal numbers of nonzeros (the
//    host cuts them), and a workgroup owns one tile and accumulates its rows
//    in LDS;
//  * entries of a tile are stored sorted by column, so neighbouring lanes
//    gather neighbouring x entries -- one cache line serves several lanes;
//  * workgroups are dispatched round-robin to the 8 XCDs (workgroup w runs on
//    XCD w % 8), and tile w belongs to column slice (w % 8) % S: each XCD only
//    ever reads its own slice of x, which stays resident in its L2.
//
// With one slice a tile's sums are its rows' totals and are stored to y.
// With S slices either every tile stores its rows' sums in its slice's
// partial vector (S x n doubles held by the plan) and a merge kernel adds the
// S partials of each row in slice order, or y is cleared first and every
// tile adds its sums into it with FP64 atomics (global_atomic_add_f64).
// Every tile writes its rows when its loop ends and all tiles end together;
// the host picks partials where that burst is heavy against the loop.  The
// LDS adds (ds_add_f64) make the order of the additions inside a row
// nondeterministic; the result stays within the FP64 tolerance of the
// left-to-right CPU sum.
#include <type_traits>

#include "launch.hpp"
#include "wave64.hpp"

namespace {
using axspmv::launch::RctArgs;

// Entry e of a tile: value val[e] (VT double or float; uint8_t or SmallRef: the
// value's index in a table of at most 256, for matrices of few different
// values); its column and tile row stored one of four ways (KEY):
//  * KEY_SPLIT: col[e] and lrow[e];
//  * KEY_PACKED: one word key[e] = offset << rbits | row, the column being
//    (sbase[e >> 10] + offset) mod ncols: every run of 1024 entries has a
//    base column (its first entry's or its smallest), and its entries,
//    sorted by column tile by tile, lie a short way past it -- going round
//    from the last column to column 0 where a run passes from one row block
//    to the next;
//  * KEY_PACKED24: the same word in 24 bits, its low 16 in key24[e] and its
//    high 8 in key8[e], with a base per run of 128 entries;
//  * KEY_DIAG (narrow bands): a 16-bit key16[e] = d << cbits | offset, the
//    column being sbase[e >> 7] + offset (the smallest column of its run of
//    128 entries) and the row (global) column + d + dmin, where d + dmin is
//    the entry's row minus its column; the tile row is that row minus the
//    tile's first row (rofs = dmin - row0, all modulo 2^32).
// NT: the paired stream loads of load2 are non-temporal (the plan sets it
// when the matrix stream is too large to stay in the Infinity Cache from one
// SpMV to the next; there the L2 lines it would leave behind only crowd out
// x).
enum : int { KEY_SPLIT = 0, KEY_PACKED = 1, KEY_DIAG = 2, KEY_PACKED24 = 3 };

template <class VT, int KEY, bool NT = false>
struct RctEntries {
    const VT *__restrict__ val;
    const uint32_t *__restrict__ key;
    const uint32_t *__restrict__ col;
    const uint16_t *__restrict__ lrow;
    const uint16_t *__restrict__ key16;  // KEY_PACKED24: key24
    const uint8_t *__restrict__ key8;
    const uint32_t *__restrict__ sbase;
    uint32_t rbits, ncols, cbits, rofs;
    // the tile whose rows start at row0
    __device__ __forceinline__ RctEntries(const RctArgs &a, uint32_t row0)
        : val(static_cast<const VT *>(a.val)), key(a.key), col(a.col), lrow(a.lrow),
          key16(KEY == KEY_PACKED24 ? a.key24 : a.key16), key8(a.key8),
          sbase(a.sbase), rbits(a.rbits), ncols(a.ncols), cbits(a.cbits16), rofs(a.dmin - row0) {}
    __device__ __forceinline__ uint32_t column(uint32_t base, uint32_t off) const {
        const uint32_t room = ncols - base;  // columns from base to the end
        return off >= room ? off - room : base + off;
    }
    __device__ __forceinline__ void diag(uint32_t base, uint32_t k, uint32_t &c, uint32_t &r) const {
        c = base + (k & ((1u << cbits) - 1));
        r = c + (k >> cbits) + rofs;
    }
    // entries 2q and 2q + 1 with one 16-byte (8 for FP32 values, 2 for table
    // indices) and one 8-byte load (KEY_DIAG: 4 bytes; KEY_PACKED24: 4 and 2);
    // the plan pads the arrays to an even number of entries
    __device__ __forceinline__ void load2(uint32_t q, uint32_t (&c)[2], uint32_t (&r)[2], VT (&v)[2]) const {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        if constexpr (sizeof(VT) == 1) {
            const uint16_t *p = reinterpret_cast<const uint16_t *>(val) + q;
            const uint16_t vv = NT ? __builtin_nontemporal_load(p) : *p;
            v[0] = VT(vv & 0xff);
            v[1] = VT(vv >> 8);
        } else {
            typedef VT v2 __attribute__((ext_vector_type(2)));
            const v2 *p = reinterpret_cast<const v2 *>(val) + q;
            const v2 vv = NT ? __builtin_nontemporal_load(p) : *p;
            v[0] = vv.x;
            v[1] = vv.y;
        }
        if constexpr (KEY == KEY_DIAG) {
            const uint32_t *pk = reinterpret_cast<const uint32_t *>(key16) + q;
            const uint32_t k = NT ? __builtin_nontemporal_load(pk) : *pk;
            const uint32_t b = sbase[q >> 6];  // entries 2q, 2q + 1: one run of 128
            diag(b, k & 0xffffu, c[0], r[0]);
            diag(b, k >> 16, c[1], r[1]);
        } else if constexpr (KEY == KEY_PACKED24) {
            const uint32_t *pl = reinterpret_cast<const uint32_t *>(key16) + q;
            const uint16_t *ph = reinterpret_cast<const uint16_t *>(key8) + q;
            const uint32_t lo = NT ? __builtin_nontemporal_load(pl) : *pl;
            const uint32_t hi = NT ? __builtin_nontemporal_load(ph) : *ph;
            const uint32_t m = (1u << rbits) - 1, b = sbase[q >> 6];  // entries 2q, 2q + 1: one run of 128
            const uint32_t k0 = (lo & 0xffffu) | (hi & 0xffu) << 16, k1 = lo >> 16 | hi >> 8 << 16;
            c[0] = column(b, k0 >> rbits);
            r[0] = k0 & m;
            c[1] = column(b, k1 >> rbits);
            r[1] = k1 & m;
        } else if constexpr (KEY == KEY_PACKED) {
            const u32x2 *pk = reinterpret_cast<const u32x2 *>(key) + q;
            const u32x2 k = NT ? __builtin_nontemporal_load(pk) : *pk;
            const uint32_t m = (1u << rbits) - 1, b = sbase[q >> 9];  // entries 2q, 2q + 1: one segment
            c[0] = column(b, k.x >> rbits);
            r[0] = k.x & m;
            c[1] = column(b, k.y >> rbits);
            r[1] = k.y & m;
        } else {
            const u32x2 *pc = reinterpret_cast<const u32x2 *>(col) + q;
            const uint32_t *pr = reinterpret_cast<const uint32_t *>(lrow) + q;
            const u32x2 cc = NT ? __builtin_nontemporal_load(pc) : *pc;
            const uint32_t rr = NT ? __builtin_nontemporal_load(pr) : *pr;
            c[0] = cc.x;
            c[1] = cc.y;
            r[0] = rr & 0xffffu;
            r[1] = rr >> 16;
        }
    }
    // column and tile row only
    __device__ __forceinline__ void at(uint32_t e, uint32_t &c, uint32_t &r) const {
        if constexpr (KEY == KEY_DIAG) {
            diag(sbase[e >> 7], key16[e], c, r);
        } else if constexpr (KEY == KEY_PACKED24) {
            const uint32_t k = key16[e] | uint32_t(key8[e]) << 16;
            c = column(sbase[e >> 7], k >> rbits);
            r = k & ((1u << rbits) - 1);
        } else if constexpr (KEY == KEY_PACKED) {
            const uint32_t k = key[e];
            c = column(sbase[e >> 10], k >> rbits);
            r = k & ((1u << rbits) - 1);
        } else {
            c = col[e];
            r = lrow[e];
        }
    }
};

// uint8_t's form for small matrices: the tile kernel reads the table where it
// lies, in the vector L1, and not from a copy in LDS, where a read waits behind
// the LDS adds of the round before (see RctArgs::pal_lds).
enum class SmallRef : uint8_t {};

template <class VT>
__device__ __forceinline__ double entry_value(VT v, const double *table, const double *pal) {
    if constexpr (std::is_same_v<VT, SmallRef>) return pal[uint32_t(v)];
    else if constexpr (sizeof(VT) == 1) return table[v];
    else return double(v);
}

int key_mode(const RctArgs &a) {
    return a.key16 ? KEY_DIAG : a.key24 ? KEY_PACKED24 : a.key ? KEY_PACKED : KEY_SPLIT;
}

// Tile w of nb row blocks x S slices: XCD w % 8 takes slice (w % 8) % S; false
// for the workgroups past the last row block.
__device__ __forceinline__ bool tile_of(uint32_t w, uint32_t nb, uint32_t S, uint32_t &rb, uint32_t &s) {
    const uint32_t xcd = w % 8, i = w / 8;
    const uint32_t per = 8 / S;  // row-block groups per slice
    s = xcd % S;
    rb = i * per + xcd / S;
    return rb < nb;
}
__host__ __device__ constexpr uint32_t tile_groups(uint32_t nb, uint32_t S) { return (nb + 8 / S - 1) / (8 / S) * 8; }

// The tile of workgroup w.  HV: the heavy rows' tiles come first.
template <bool HV = false>
struct TileOf {
    uint32_t s, t;  // slice; index in storage order
    uint32_t row0, rows;
    bool heavy;
    __device__ __forceinline__ bool from(const RctArgs &a, uint32_t w) {
        uint32_t rb;
        heavy = false;
        if constexpr (HV) {
            const uint32_t nh = tile_groups(a.nhb, a.hs);
            if (w < nh) {
                heavy = true;
                if (!tile_of(w, a.nhb, a.hs, rb, s)) return false;
                t = a.nrb * a.S + rb * a.hs + s;
                row0 = a.hb_start[rb];
                rows = a.hb_start[rb + 1] - row0;
                return true;
            }
            w -= nh;
        }
        if (!tile_of(w, a.nrb, a.S, rb, s)) return false;
        t = rb * a.S + s;
        row0 = a.rb_start[rb];
        rows = a.rb_start[rb + 1] - row0;  // <= a.R
        return true;
    }
    // the row of y that the tile's row k adds to or is stored in; false: a
    // heavy row's place in a row block, nothing to write
    __device__ __forceinline__ bool out_row(const RctArgs &a, uint32_t k, uint32_t &r) const {
        r = row0 + k;
        if constexpr (HV) {
            if (heavy) r = a.hrows[r];
            else return !((a.hmask[r >> 5] >> (r & 31)) & 1);
        }
        return true;
    }
};

// Pairs of a lane per round of the value-gradient sweep: 4 with column slices
// (forward + adjoint, 2 / 3 / 4 pairs: 700,001-row power-law matrix 149.7 / 144.3 /
// 142.2 us, FP32 values 139.0 / 134.7 / 132.3), else 3 (random, 300,007 rows 85.9 /
// 82.1 / 79.9; permuted 60^3 stencil 73.6 / 70.8 / 68.6, but 80^3 renumbered 130.2 /
// 128.9 / 131.6), and 2 for the 128-lane workgroups of small tiles, which hardly fill
// one round (5,000-row power-law matrix 10.6 to 11.2 / 11.4 / 11.6).
int vb_pairs(const RctArgs &a) { return a.S > 1 ? 4 : a.block <= 128 ? 2 : 3; }

unsigned rct_grid(const RctArgs &a) { return tile_groups(a.nrb, a.S) + (a.nhb ? tile_groups(a.nhb, a.hs) : 0); }

// VB: the same product on the plan of A^T, fused with the value gradient of
// A: vb[e] = xr[row(e)] * x[col(e)] for every entry, in entry order (the
// tile's xr values sit in LDS after its sums).  With x = r and xr = the
// forward x, y = A^T r and vb holds r[i] * x[j] for every nonzero A(i, j).
//
// UP: pairs of a lane per round.  Two for the product alone (three and four:
// 2^20-row power-law matrix 85.8 / 86.3 / 87.4 us, 48 banded matrices 90.0 /
// 91.3 / 92.9).  The sweep with the value gradient has 8 bytes to store per
// entry as well and a chain of one more load, so it takes more at a time:
// see vb_pairs.
template <class VT, int KEY, bool VB, bool NT, bool HV = false, int UP = 2>
__global__ void __launch_bounds__(1024) rct_kernel(RctArgs a, const double *__restrict__ x, double *__restrict__ y,
                                                   const double *__restrict__ xr, double *__restrict__ vb,
                                                   const double *__restrict__ bvec, double *__restrict__ res) {
    extern __shared__ double yl[];
    TileOf<HV> tile;
    if (!tile.from(a, blockIdx.x)) return;  // the whole workgroup leaves together
    const uint32_t tid = threadIdx.x, nt = blockDim.x;
    const uint32_t row0 = tile.row0, rows = tile.rows;
    double *xs = yl + a.R;  // VB: xr of the tile's rows
    constexpr bool TABLE = std::is_same_v<VT, uint8_t>;
    __shared__ double table[TABLE ? 256 : 1];
    if constexpr (TABLE)
        for (uint32_t k = tid; k < 256; k += nt) table[k] = a.pal[k];
    for (uint32_t k = tid; k < rows; k += nt) {
        yl[k] = 0.0;
        if constexpr (VB) xs[k] = xr[row0 + k];
    }
    __syncthreads();
    const uint32_t beg = a.tile_ptr[tile.t], end = a.tile_ptr[tile.t + 1];
    const RctEntries<VT, KEY, NT> ent(a, row0);
    // Each lane takes entries in aligned pairs (2q, 2q + 1): a value load
    // moves 16 bytes and a key load 8, and the value gradient (VB) goes out
    // as one 16-byte store per pair.  Pairs pb .. pl cover the tile and each
    // holds at least one of its entries; an entry outside the tile borrows
    // its partner's column and row (both in the tile) and adds nothing.
    // Measured against one entry per lane: SpMV 1-4 % faster on the
    // power-law, stencil and banded matrices, forward + adjoint 2-4 %.
    //
    // Rounds of UP pairs per lane, in two register sets A and B: a round
    // issues its x gathers (and, for VB, its LDS reads of xr), then the loads
    // of the next round into the other set, then waits for the gathers only
    // and does its LDS adds.  Loads are never predicated (a lane past the end
    // re-reads the tile's last pair) and the products of such a lane are
    // zeroed.  The round count is the same for the whole workgroup, and the
    // last round (which fetches nothing) is peeled, so every fetch is used on
    // every path and the compiler has no reason to sink it behind the LDS
    // adds.
    //
    // VB stores are unpredicated too: a lane's two value gradients go to
    // entries of the tile (an entry outside it, or a lane past the end,
    // stores its partner's own value again), as one 16-byte store when every
    // lane of the wave holds a whole pair and vb is 16-byte aligned, else as
    // two 8-byte stores; non-temporal, as nothing here reads vb again (the
    // permuted 128^3 stencil's forward + adjoint, renumbered: 485.8 ->
    // 478.8 us; the 2^20-row power-law matrix's: 233.0 -> 229.2 us).
    struct PSet {
        uint32_t c[UP][2], r[UP][2];
        uint32_t at[UP][2];  // VB: the entries the two stores write
        VT v[UP][2];
        bool ok[UP][2];      // adds its product
    };
    if (beg < end) {
        const uint32_t pb = beg >> 1, pl = (end - 1) >> 1, span = UP * nt;
        const uint32_t nr = (pl - pb + span) / span;
        const bool vb16 = (reinterpret_cast<uintptr_t>(vb) & 15) == 0;
        auto fetch = [&](PSet &S, uint32_t q0) {
#pragma unroll
            for (int j = 0; j < UP; ++j) {
                const uint32_t q = q0 + j * nt, qc = min(q, pl);
                ent.load2(qc, S.c[j], S.r[j], S.v[j]);
                const bool in0 = 2 * qc >= beg, in1 = 2 * qc + 1 < end;
                const uint32_t c0 = S.c[j][0], r0 = S.r[j][0], c1 = S.c[j][1], r1 = S.r[j][1];
                S.c[j][0] = in0 ? c0 : c1;
                S.r[j][0] = in0 ? r0 : r1;
                S.c[j][1] = in1 ? c1 : c0;
                S.r[j][1] = in1 ? r1 : r0;
                S.ok[j][0] = q == qc && in0;  // a lane past the end adds nothing
                S.ok[j][1] = q == qc && in1;
                if constexpr (VB) {
                    S.at[j][0] = in0 ? 2 * qc : 2 * qc + 1;
                    S.at[j][1] = in1 ? 2 * qc + 1 : 2 * qc;
                }
            }
        };
        auto gather = [&](const PSet &S, double (&xv)[UP][2], double (&xl)[UP][2], double (&vv)[UP][2]) {
#pragma unroll
            for (int j = 0; j < UP; ++j) {
                xv[j][0] = x[S.c[j][0]];
                xv[j][1] = x[S.c[j][1]];
            }
            if constexpr (VB) {
#pragma unroll
                for (int j = 0; j < UP; ++j) {
                    xl[j][0] = xs[S.r[j][0]];
                    xl[j][1] = xs[S.r[j][1]];
                }
            }
#pragma unroll
            for (int j = 0; j < UP; ++j) {
                vv[j][0] = entry_value(S.v[j][0], table, a.pal);
                vv[j][1] = entry_value(S.v[j][1], table, a.pal);
            }
        };
        auto add = [&](const PSet &S, const double (&xv)[UP][2], const double (&xl)[UP][2], const double (&vv)[UP][2]) {
#pragma unroll
            for (int j = 0; j < UP; ++j) {
#pragma unroll
                for (int h = 0; h < 2; ++h) atomicAdd(&yl[S.r[j][h]], S.ok[j][h] ? vv[j][h] * xv[j][h] : 0.0);
                if constexpr (VB) {
                    const double p0 = xl[j][0] * xv[j][0], p1 = xl[j][1] * xv[j][1];
                    if (__all(vb16 && S.at[j][1] == S.at[j][0] + 1)) {  // whole pairs (at[j][0] even)
                        typedef double f64x2 __attribute__((ext_vector_type(2)));
                        __builtin_nontemporal_store(f64x2{p0, p1}, reinterpret_cast<f64x2 *>(vb) + (S.at[j][0] >> 1));
                    } else {
                        __builtin_nontemporal_store(p0, vb + S.at[j][0]);
                        __builtin_nontemporal_store(p1, vb + S.at[j][1]);
                    }
                }
            }
        };
        auto round = [&](const PSet &S, PSet &N, uint32_t q0) {
            double xv[UP][2], xl[UP][2], vv[UP][2];
            gather(S, xv, xl, vv);
            fetch(N, q0 + span);
            add(S, xv, xl, vv);
        };
        auto final_round = [&](const PSet &S) {
            double xv[UP][2], xl[UP][2], vv[UP][2];
            gather(S, xv, xl, vv);
            add(S, xv, xl, vv);
        };
        PSet A, B;
        uint32_t q = pb + tid;
        fetch(A, q);
        uint32_t k = 1;  // rounds k - 1 and k run in one pass; both have a successor
        for (; k + 1 < nr; k += 2) {
            round(A, B, q);
            round(B, A, q + span);
            q += 2 * span;
        }
        if (k < nr) {
            round(A, B, q);
            final_round(B);
        } else {
            final_round(A);
        }
    }
    __syncthreads();
    double *out = y + row0;
    if constexpr (HV) {
        // heavy rows add their slices' sums into y (cleared there, or
        // everywhere with S > 1); the others as below
        for (uint32_t k = tid; k < rows; k += nt) {
            uint32_t r;
            if (!tile.out_row(a, k, r)) continue;
            if (tile.heavy || a.S > 1) unsafeAtomicAdd(y + r, yl[k]);
            else __builtin_nontemporal_store(yl[k], y + r);
        }
    } else if (a.S == 1) {
        // non-temporal: y kept in the L2s would take room from the next
        // SpMV's x (the 1024^2 Laplacian: 14.6 -> 13.9 us)
        for (uint32_t k = tid; k < rows; k += nt) {
            __builtin_nontemporal_store(yl[k], out + k);
            if (res) res[row0 + k] = yl[k] - bvec[row0 + k];  // forward + adjoint: r = y - b, read next
        }
    } else if (a.part && !VB) {
        // the slice's partial vector, read once by the merge: non-temporal
        double *ps = a.part + tile.s * a.pstride + row0;
        for (uint32_t k = tid; k < rows; k += nt) __builtin_nontemporal_store(yl[k], ps + k);
    } else {
        for (uint32_t k = tid; k < rows; k += nt) unsafeAtomicAdd(out + k, yl[k]);
    }
}

// Value gradient in entry order: vbar[e] = ybar[row(e)] * x[col(e)].  The
// tile's ybar rows sit in LDS; x is gathered in the tile's column order;
// vbar goes out with non-temporal stores.
template <int KEY>
__global__ void __launch_bounds__(1024) rct_vbar_kernel(RctArgs a, const double *__restrict__ ybar,
                                                        const double *__restrict__ x, double *__restrict__ vbar) {
    extern __shared__ double yb[];
    TileOf<> tile;
    if (!tile.from(a, blockIdx.x)) return;
    const uint32_t tid = threadIdx.x, nt = blockDim.x;
    const uint32_t row0 = tile.row0, rows = tile.rows;
    for (uint32_t k = tid; k < rows; k += nt) yb[k] = ybar[row0 + k];
    __syncthreads();
    const uint32_t beg = a.tile_ptr[tile.t], end = a.tile_ptr[tile.t + 1];
    const RctEntries<double, KEY> ent(a, row0);  // columns and rows only
    constexpr int U = 4;
    uint32_t e = beg + tid;
    for (; e + (U - 1) * nt < end; e += U * nt) {
        uint32_t c[U], r[U];
#pragma unroll
        for (int j = 0; j < U; ++j) ent.at(e + j * nt, c[j], r[j]);
        double xv[U];
#pragma unroll
        for (int j = 0; j < U; ++j) xv[j] = x[c[j]];
#pragma unroll
        for (int j = 0; j < U; ++j) __builtin_nontemporal_store(yb[r[j]] * xv[j], vbar + e + j * nt);
    }
    for (; e < end; e += nt) {
        uint32_t c, r;
        ent.at(e, c, r);
        __builtin_nontemporal_store(yb[r] * x[c], vbar + e);
    }
}

// SpMM: Y[:, k0 .. k0 + KT) (+)= A X[:, k0 .. k0 + KT) over one tile.  A
// group of GL lanes serves one entry at a time, V neighbouring right-hand
// sides per lane (KT = GL * V; one contiguous KT x 8-byte read of the entry's
// X row); the tile's rows x KT sums stay in LDS (ds_add_f64) and go to Y at
// the end: stored with one slice, added with FP64 atomics (Y cleared first)
// with several.
//
// Values and keys are loaded and decoded a batch at a time, one entry per
// lane, and handed to the group by DPP: with every lane of a group loading
// its entry's value, key and base, the vector L1 spent three of its four
// requests per entry on them.  Power-law matrices, FP64: 600,000 rows, k = 8,
// 1024-row tiles 259 -> 222 us (4 slices 209 -> 184); 400,003 rows, k = 32,
// 256-row tiles 468 -> 323 us; the 64^3 stencil, k = 16, 512-row tiles 169 ->
// 57 us.  What is left on the power-law ones are the X rows that miss L2 (one
// 128-byte line per entry, 5.5 TB/s from the Infinity Cache).  A batch's X
// loads go out together; the next batch's values and keys are in flight
// behind them.  X rows are addressed by 32-bit byte offsets, or (WIDE: X of
// 4 GB and more) by their column.
//
// LDS layout: sum (row, right-hand side l V + v) sits at row KT + l + GL (v
// xor the row's parity), so the groups of one ds_add_f64 spread over both
// halves of their rows' banks.
template <class VT, int KEY, int GL, int V, bool WIDE>
struct SpmmBatch {
    static constexpr int KT = GL * V;
    static constexpr int ROW = GL < 16 ? GL : 16;  // lanes that share a batch: wider groups load it once per 16
    static constexpr int E = ROW == 4 ? 2 : 1;     // entries per lane
    static constexpr int B = ROW * E;
    VT v[E];
    uint32_t c[E], r[E];  // X row (byte offset, or column), tile row's first sum
    __device__ __forceinline__ void load(const RctEntries<VT, KEY> &ent, uint32_t e0, uint32_t end, uint32_t k) {
        const uint32_t i = e0 + threadIdx.x % ROW;
#pragma unroll
        for (int u = 0; u < E; ++u)
            if (i + u * ROW < end) {
                v[u] = ent.val[i + u * ROW];
                uint32_t cc, rr;
                ent.at(i + u * ROW, cc, rr);
                c[u] = WIDE ? cc : cc * k * 8;
                r[u] = rr * KT + (V == 2 ? (rr & 1) * GL : 0);
            } else if constexpr (sizeof(VT) == 1) {
                v[u] = 0;  // the table is read for every lane
            }
    }
};

template <class VT, int KEY, int GL, int V, bool WIDE, bool HV>
__global__ void __launch_bounds__(1024) rct_spmm_kernel(RctArgs a, uint32_t k, uint32_t k0,
                                                        const double *__restrict__ X, double *__restrict__ Y) {
    using namespace axspmv::dev;
    using Batch = SpmmBatch<VT, KEY, GL, V, WIDE>;
    typedef double vec __attribute__((ext_vector_type(V)));
    using XV = std::conditional_t<V == 1, double, vec>;
    constexpr uint32_t KT = GL * V, B = Batch::B, ROW = Batch::ROW, STEP = 8;
    extern __shared__ double acc[];
    TileOf<HV> tile;
    if (!tile.from(a, blockIdx.x)) return;
    const uint32_t tid = threadIdx.x, nt = blockDim.x;
    const uint32_t row0 = tile.row0, rows = tile.rows;
    for (uint32_t q = tid; q < rows * KT; q += nt) acc[q] = 0.0;
    __syncthreads();
    const uint32_t beg = a.tile_ptr[tile.t], end = a.tile_ptr[tile.t + 1];
    const RctEntries<VT, KEY> ent(a, row0);
    const uint32_t l = tid % GL, g = tid / GL, chunk = nt / GL * B;  // nt is a multiple of 64
    // a lane past the last right-hand side (a partial k-tile) works on the
    // k-tile's first X and on sums of its own that are not stored
    const uint32_t kx = k0 + l * V < k ? k0 + l * V : k0;
    double *const al = acc + l;
    auto work = [&](const Batch &b, uint32_t left) {
        // a table index becomes its value before it is handed round
        using BV = std::conditional_t<sizeof(VT) == 1, double, VT>;
        BV bv[Batch::E];
#pragma unroll
        for (int u = 0; u < Batch::E; ++u) {
            if constexpr (sizeof(VT) == 1) bv[u] = a.pal[b.v[u]];
            else bv[u] = b.v[u];
        }
        static_for<B / STEP ? B / STEP : 1>([&](auto H) {
            constexpr int N = B < STEP ? B : STEP, j0 = H.value * N;
            XV xv[N];
            static_for<N>([&](auto J) {
                constexpr int j = j0 + J.value;
                const uint32_t c = group_bcast_u32<ROW, j % ROW>(b.c[j / ROW]);
                if (uint32_t(j) < left) {
                    if constexpr (WIDE) xv[J.value] = *reinterpret_cast<const XV *>(X + size_t(c) * k + kx);
                    else xv[J.value] = *reinterpret_cast<const XV *>(reinterpret_cast<const char *>(X) + (c + kx * 8));
                }
            });
            __builtin_amdgcn_sched_barrier(0);
            static_for<N>([&](auto J) {
                constexpr int j = j0 + J.value;
                const double v = double(group_bcast<ROW, j % ROW>(bv[j / ROW]));
                const uint32_t r = group_bcast_u32<ROW, j % ROW>(b.r[j / ROW]);
                if (uint32_t(j) < left) {
                    if constexpr (V == 1) {
                        atomicAdd(al + r, v * xv[J.value]);
                    } else {
                        atomicAdd(al + r, v * xv[J.value].x);
                        atomicAdd(al + (r ^ GL), v * xv[J.value].y);
                    }
                }
            });
        });
    };
    uint32_t e = beg + g * B;
    if (e < end) {
        Batch b;
        b.load(ent, e, end, k);
        for (; e + chunk < end; e += chunk) {
            Batch n;
            n.load(ent, e + chunk, end, k);
            work(b, B);  // every batch but a group's last is whole
            b = n;
        }
        work(b, end - e);
    }
    __syncthreads();
    if (a.S == 1 && !tile.heavy) {
        for (uint32_t q = tid; q < rows * GL; q += nt) {
            const uint32_t rr = q / GL, ll = q % GL;
            uint32_t r;
            if (k0 + ll * V >= k || !tile.out_row(a, rr, r)) continue;
            const uint32_t i = rr * KT + ll + (V == 2 ? (rr & 1) * GL : 0);
            double *out = Y + size_t(r) * k + k0 + ll * V;
            if constexpr (V == 1) *out = acc[i];
            else *reinterpret_cast<XV *>(out) = XV{acc[i], acc[rr * KT + ll + (~rr & 1) * GL]};
        }
    } else {
        // one sum per lane, so that the lanes' atomics fall side by side (two
        // per lane made 4 slices 25 % slower)
        for (uint32_t q = tid; q < rows * KT; q += nt) {
            const uint32_t rr = q / KT, jj = q % KT;
            uint32_t r;
            if (k0 + jj < k && tile.out_row(a, rr, r))
                unsafeAtomicAdd(Y + size_t(r) * k + k0 + jj,
                                acc[rr * KT + jj / V + (V == 2 ? ((jj ^ rr) & 1) * GL : 0)]);
        }
    }
}

// Y[rows[i], :] = 0: the heavy rows' place before their slices' adds
__global__ void __launch_bounds__(256) clear_rows_kernel(const uint32_t *__restrict__ rows, uint64_t total, uint32_t k,
                                                         double *__restrict__ Y) {
    const uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < total) Y[size_t(rows[t / k]) * k + t % k] = 0.0;
}

template <class VT, int KEY, int V, bool WIDE, bool HV>
hipError_t rct_spmm_run(const RctArgs &a, uint32_t k, uint32_t kt, const double *X, double *Y, hipStream_t s) {
    const unsigned grid = rct_grid(a);
    for (uint32_t k0 = 0; k0 < k; k0 += kt) {
        while (kt > 8 && k - k0 <= kt / 2) kt /= 2;  // the last right-hand sides: no wider than they need
        const size_t lds = size_t(a.R) * kt * sizeof(double);
        switch (kt) {
            case 8: rct_spmm_kernel<VT, KEY, 8 / V, V, WIDE, HV><<<grid, a.block, lds, s>>>(a, k, k0, X, Y); break;
            case 16: rct_spmm_kernel<VT, KEY, 16 / V, V, WIDE, HV><<<grid, a.block, lds, s>>>(a, k, k0, X, Y); break;
            case 32: rct_spmm_kernel<VT, KEY, 32 / V, V, WIDE, HV><<<grid, a.block, lds, s>>>(a, k, k0, X, Y); break;
            case 64: rct_spmm_kernel<VT, KEY, 64 / V, V, WIDE, HV><<<grid, a.block, lds, s>>>(a, k, k0, X, Y); break;
            default: return hipErrorInvalidValue;
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Two right-hand sides per lane where every 16-byte access is aligned: k
// even, X and Y 16-byte aligned (k0 is a multiple of 8).
template <class VT, int KEY, bool HV>
hipError_t rct_spmm_hv(const RctArgs &a, uint32_t k, uint32_t kt, const double *X, double *Y, hipStream_t s) {
    const bool two = k % 2 == 0 && (reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y)) % 16 == 0;
    const bool wide = uint64_t(a.ncols) * k * 8 >= (1ull << 32);
    if (wide)
        return two ? rct_spmm_run<VT, KEY, 2, true, HV>(a, k, kt, X, Y, s)
                   : rct_spmm_run<VT, KEY, 1, true, HV>(a, k, kt, X, Y, s);
    return two ? rct_spmm_run<VT, KEY, 2, false, HV>(a, k, kt, X, Y, s)
               : rct_spmm_run<VT, KEY, 1, false, HV>(a, k, kt, X, Y, s);
}
template <class VT, int KEY>
hipError_t rct_spmm_vt(const RctArgs &a, uint32_t k, uint32_t kt, const double *X, double *Y, hipStream_t s) {
    if constexpr (KEY != KEY_DIAG)
        if (a.nhb) return rct_spmm_hv<VT, KEY, true>(a, k, kt, X, Y, s);
    return rct_spmm_hv<VT, KEY, false>(a, k, kt, X, Y, s);
}

}  // namespace

namespace axspmv {
namespace launch {

hipError_t rct_spmm(const RctArgs &a, uint32_t k, uint32_t kt, const double *X, double *Y, hipStream_t s) {
    if (!a.nrows || !k) return hipSuccess;
    if (a.S > 1) {
        const hipError_t e = clear_f64(Y, size_t(a.nrows) * k, s);
        if (e != hipSuccess) return e;
    } else if (a.nhb) {
        const uint64_t total = uint64_t(a.nheavy) * k;
        clear_rows_kernel<<<unsigned((total + 255) / 256), 256, 0, s>>>(a.hrows, total, k, Y);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    const int km = key_mode(a);
    auto with = [&](auto vt) {
        using VT = decltype(vt);
        return km == KEY_DIAG       ? rct_spmm_vt<VT, KEY_DIAG>(a, k, kt, X, Y, s)
               : km == KEY_PACKED24 ? rct_spmm_vt<VT, KEY_PACKED24>(a, k, kt, X, Y, s)
               : km == KEY_PACKED   ? rct_spmm_vt<VT, KEY_PACKED>(a, k, kt, X, Y, s)
                                    : rct_spmm_vt<VT, KEY_SPLIT>(a, k, kt, X, Y, s);
    };
    return a.pal ? with(uint8_t()) : a.vtype == 1 ? with(float()) : with(double());
}

hipError_t rct_vbar(const RctArgs &a, const double *ybar, const double *x, double *vbar, hipStream_t s) {
    if (!a.nrows) return hipSuccess;
    const unsigned grid = rct_grid(a);
    const size_t lds = size_t(a.R) * sizeof(double);
    switch (key_mode(a)) {
        case KEY_DIAG: rct_vbar_kernel<KEY_DIAG><<<grid, a.block, lds, s>>>(a, ybar, x, vbar); break;
        case KEY_PACKED24: rct_vbar_kernel<KEY_PACKED24><<<grid, a.block, lds, s>>>(a, ybar, x, vbar); break;
        case KEY_PACKED: rct_vbar_kernel<KEY_PACKED><<<grid, a.block, lds, s>>>(a, ybar, x, vbar); break;
        default: rct_vbar_kernel<KEY_SPLIT><<<grid, a.block, lds, s>>>(a, ybar, x, vbar);
    }
    return hipGetLastError();
}

hipError_t rct(const RctArgs &a, const double *x, double *y, hipStream_t s, hipEvent_t mid, const double *xr,
               double *vbar, const double *rb, double *res, double *clear, size_t nclear, bool cleared) {
    if (!a.nrows) return clear ? clear_f64(clear, nclear, s) : hipSuccess;
    if (vbar) rb = res = nullptr;  // the residual belongs to a forward pass
    const unsigned grid = rct_grid(a);
    const bool vb = vbar != nullptr;
    const size_t lds = size_t(a.R) * sizeof(double) * (vb ? 2 : 1);
    const bool partials = a.S > 1 && a.part && !vb;
    if (a.S > 1 && !partials) {
        if (!cleared) {
            const hipError_t e = clear_f64(y, a.nrows, s);
            if (e != hipSuccess) return e;
        }
        if (mid) {
            const hipError_t e = hipEventRecord(mid, s);
            if (e != hipSuccess) return e;
        }
    } else if (a.nhb) {
        const hipError_t e = fill_rows(a.hrows, a.nheavy, y, s);
        if (e != hipSuccess) return e;
    }
    const int km = key_mode(a);
    // the value-gradient sweep too streams with non-temporal loads where the
    // plan asks for them (its v_bar stores are non-temporal anyway): the
    // permuted 128^3 stencil's forward + adjoint, renumbered, 472.8 -> 467.7
    // us, one box
    // (24-bit keys are for streams that are loaded the ordinary way)
#define AX_RCT_VB(VT, P, nt, UP)                                                                                  \
    do {                                                                                                          \
        if (nt && a.nt_stream)                                                                                    \
            rct_kernel<VT, P, true, nt, false, UP><<<grid, a.block, lds, s>>>(a, x, y, xr, vbar, rb, res);        \
        else                                                                                                      \
            rct_kernel<VT, P, true, false, false, UP><<<grid, a.block, lds, s>>>(a, x, y, xr, vbar, rb, res);     \
    } while (0)
    // (small matrices have neither 24-bit keys nor non-temporal loads, and
    // their plans with heavy rows take the table in LDS)
#define AX_RCT_LAUNCH(T, P)                                                                               \
    do {                                                                                                  \
        constexpr bool small = std::is_same_v<T, SmallRef>, nt = P != KEY_PACKED24 && !small;             \
        using HVT = std::conditional_t<small, uint8_t, T>;                                                \
        using VT = std::conditional_t<P == KEY_PACKED24, HVT, T>;                                         \
        if (P != KEY_DIAG && a.nhb)                                                                       \
            rct_kernel<HVT, P == KEY_DIAG ? KEY_SPLIT : P, false, false, true><<<grid, a.block, lds, s>>>( \
                a, x, y, xr, vbar, rb, res);                                                              \
        else if (vb && vb_pairs(a) == 2)                                                                  \
            AX_RCT_VB(VT, P, nt, 2);                                                                      \
        else if (vb && vb_pairs(a) == 3)                                                                  \
            AX_RCT_VB(VT, P, nt, 3);                                                                      \
        else if (vb)                                                                                      \
            AX_RCT_VB(VT, P, nt, 4);                                                                      \
        else if (nt && a.nt_stream)                                                                       \
            rct_kernel<VT, P, false, nt><<<grid, a.block, lds, s>>>(a, x, y, xr, vbar, rb, res);          \
        else                                                                                              \
            rct_kernel<VT, P, false, false><<<grid, a.block, lds, s>>>(a, x, y, xr, vbar, rb, res);       \
    } while (0)
    auto with = [&](auto vt) {
        using V = decltype(vt);
        if (km == KEY_DIAG)
            AX_RCT_LAUNCH(V, KEY_DIAG);
        else if (km == KEY_PACKED24)
            AX_RCT_LAUNCH(V, KEY_PACKED24);
        else if (km == KEY_PACKED)
            AX_RCT_LAUNCH(V, KEY_PACKED);
        else
            AX_RCT_LAUNCH(V, KEY_SPLIT);
    };
    if (a.pal && a.pal_lds)
        with(uint8_t());
    else if (a.pal)
        with(SmallRef());
    else if (a.vtype == 1)
        with(float());
    else
        with(double());
#undef AX_RCT_LAUNCH
#undef AX_RCT_VB
    hipError_t e = hipGetLastError();
    if (partials) {
        if (e == hipSuccess && mid) e = hipEventRecord(mid, s);
        if (e == hipSuccess) e = part_merge(a.part, a.S, a.nrows, a.pstride, y, s, rb, res, clear, nclear);
        return e;
    }
    if (clear && e == hipSuccess) e = clear_f64(clear, nclear, s);
    if (res && (a.S > 1 || a.nhb) && e == hipSuccess) {
        e = residual(a.nrows, y, rb, res, s);  // after the slices' adds
    }
    return e;
}

}  // namespace launch
}  // namespace axspmv
