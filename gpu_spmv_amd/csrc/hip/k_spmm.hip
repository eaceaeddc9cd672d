// SpMM: Y = A X with k right-hand sides stored interleaved (X[c*k + j],
// Y[r*k + j]).  Works on any layout whose rows are contiguous runs of slots
// (CSR, the AXT UNC th == 1 planes, AXC): row r's entries sit at plane slots
// first[r] .. first[r] + rl - 1.
//
// A group of GL lanes owns one row and KT = GL * V right-hand sides (the
// k-tile: 8, 16, 32 or 64), V neighbouring ones per lane.  What bounds this
// path is the vector L1's request rate: a lane-uniform load costs a request
// per group, so values and columns are loaded a batch at a time, one entry
// per lane, and handed to the group's lanes by DPP; the only loads left per
// entry are the KT * 8 contiguous bytes of its X row, 16 bytes a lane with V
// = 2.  The 27-point stencil on 64^3 in natural order, 6.9M nonzeros, FP64,
// k = 16: 64M L1 requests and 139 us with every lane loading value and column,
// 18M and 58 us so (64 us with 64-bit X offsets per lane); the 200,000-row
// power-law matrix, k = 32: 746 -> 166 us.  Rows longer than `long_slots` are listed on the host and taken by a
// whole wave, whose groups split the row's batches and combine with
// cross-group DPP/swizzle sums.
#include "launch.hpp"
#include "wave64.hpp"

namespace {
using namespace axspmv::dev;

template <int V>
struct XVec {
    typedef double type __attribute__((ext_vector_type(V)));
};
template <>
struct XVec<1> {
    typedef double type;
};

// One batch: entries [t, t + B) of the group's row (m of them inside it, m <=
// B), loaded E per lane; lanes past the row hold nothing.  c is the entry's
// X row as a byte offset, or (WIDE: X of 4 GB and more) its column.
template <class VT, int GL, bool WIDE>
struct Batch {
    static constexpr int ROW = GL < 16 ? GL : 16;    // lanes that share a batch: wider groups load it once per 16
    static constexpr int E = ROW == 4 ? 2 : 1;       // entries per lane
    static constexpr int B = ROW * E;
    VT v[E];
    uint32_t c[E];
    __device__ __forceinline__ void load(const VT *__restrict__ val, const uint32_t *__restrict__ col, uint32_t q,
                                         uint32_t left, uint32_t k) {
        const uint32_t i = threadIdx.x % ROW;
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (e * ROW + i < left) {
                v[e] = val[q + e * ROW + i];
                const uint32_t cc = col[q + e * ROW + i];
                c[e] = WIDE ? cc : cc * k * 8;
            }
    }
};

// acc += the first m entries of b times their X rows (from the lane's
// right-hand side kc on); FULL: m is the whole batch.  The X loads go out
// together before the first product.
template <class VT, int GL, int V, bool WIDE, bool FULL>
__device__ __forceinline__ void batch_fma(const Batch<VT, GL, WIDE> &b, uint32_t m, uint32_t k, uint32_t kc,
                                          const double *__restrict__ X, typename XVec<V>::type &acc) {
    using XV = typename XVec<V>::type;
    constexpr int B = Batch<VT, GL, WIDE>::B, ROW = Batch<VT, GL, WIDE>::ROW;
    XV xv[B];
    static_for<B>([&](auto J) {
        constexpr int j = J.value;
        const uint32_t c = group_bcast_u32<ROW, j % ROW>(b.c[j / ROW]);
        if (FULL || uint32_t(j) < m) {
            if constexpr (WIDE) xv[j] = *reinterpret_cast<const XV *>(X + size_t(c) * k + kc);
            else xv[j] = *reinterpret_cast<const XV *>(reinterpret_cast<const char *>(X) + (c + kc * 8));
        }
    });
    __builtin_amdgcn_sched_barrier(0);
    static_for<B>([&](auto J) {
        constexpr int j = J.value;
        const double v = double(group_bcast<ROW, j % ROW>(b.v[j / ROW]));
        if (FULL || uint32_t(j) < m) {
            if constexpr (V == 1) {
                acc = fma(v, xv[j], acc);
            } else {
                acc.x = fma(v, xv[j].x, acc.x);
                acc.y = fma(v, xv[j].y, acc.y);
            }
        }
    });
}

// XCD: the rows are cut into 8 contiguous parts and workgroup w, which runs
// on XCD w % 8, takes the next rows of part w % 8, so that neighbouring rows'
// X rows meet in one L2 (gridDim.x is a multiple of 8).
template <class VT, int GL, int V, bool WIDE>
__global__ void __launch_bounds__(256) spmm_rows_kernel(uint32_t nrows, const uint32_t *__restrict__ first,
                                                        const uint32_t *__restrict__ rowptr, const VT *__restrict__ val,
                                                        const uint32_t *__restrict__ col, uint32_t k,
                                                        uint32_t long_slots, uint32_t xcd,
                                                        const double *__restrict__ X, double *__restrict__ Y) {
    using XV = typename XVec<V>::type;
    constexpr uint32_t PER = 256 / GL;
    constexpr uint32_t B = Batch<VT, GL, WIDE>::B;
    const uint32_t w = xcd ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
    const uint64_t rr = uint64_t(w) * PER + threadIdx.x / GL;
    if (rr >= nrows) return;  // whole groups leave together
    const uint32_t r = uint32_t(rr), kc = blockIdx.y * (GL * V) + threadIdx.x % GL * V;
    const uint32_t len = rowptr[r + 1] - rowptr[r];
    if (len > long_slots) return;
    const bool on = kc < k;
    const uint32_t kx = on ? kc : blockIdx.y * (GL * V);  // past the last right-hand side: a live lane's X, nothing stored
    uint32_t q = first[r], left = len;
    XV acc = XV(0.0);
    Batch<VT, GL, WIDE> b;
    b.load(val, col, q, left, k);
    while (left >= B) {
        Batch<VT, GL, WIDE> n;
        n.load(val, col, q + B, left - B, k);
        batch_fma<VT, GL, V, WIDE, true>(b, B, k, kx, X, acc);
        b = n;
        q += B;
        left -= B;
    }
    if (left) batch_fma<VT, GL, V, WIDE, false>(b, left, k, kx, X, acc);
    if (on) *reinterpret_cast<XV *>(Y + size_t(r) * k + kc) = acc;
}

// Sum over the 64/GL groups of a wave (lanes with equal lane % GL).
template <int GL>
__device__ __forceinline__ double cross_group_sum(double v) {
    if constexpr (GL <= 4) v += __shfl_xor(v, 4);
    if constexpr (GL <= 8) v += __shfl_xor(v, 8);
    if constexpr (GL <= 16) v += __shfl_xor(v, 16);
    if constexpr (GL <= 32) v += __shfl_xor(v, 32);
    return v;
}

template <class VT, int GL, int V, bool WIDE>
__global__ void __launch_bounds__(256) spmm_long_kernel(const uint32_t *__restrict__ rows, uint32_t nlong,
                                                        const uint32_t *__restrict__ first,
                                                        const uint32_t *__restrict__ rowptr, const VT *__restrict__ val,
                                                        const uint32_t *__restrict__ col, uint32_t k,
                                                        const double *__restrict__ X, double *__restrict__ Y) {
    using XV = typename XVec<V>::type;
    constexpr uint32_t B = Batch<VT, GL, WIDE>::B, G = 64 / GL;
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (wave >= nlong) return;
    const uint32_t r = rows[wave], g = lane / GL;
    const uint32_t kc = blockIdx.y * (GL * V) + lane % GL * V;
    const bool on = kc < k;
    const uint32_t kx = on ? kc : blockIdx.y * (GL * V);  // past the last right-hand side: a live lane's X, nothing stored
    const uint32_t q0 = first[r], len = rowptr[r + 1] - rowptr[r];
    XV acc = XV(0.0);
    uint32_t t = g * B;  // group g takes batches g, g + G, ...
    Batch<VT, GL, WIDE> b;
    if (t < len) b.load(val, col, q0 + t, len - t, k);
    for (; t + B <= len; t += G * B) {
        Batch<VT, GL, WIDE> n;
        if (t + G * B < len) n.load(val, col, q0 + t + G * B, len - t - G * B, k);
        batch_fma<VT, GL, V, WIDE, true>(b, B, k, kx, X, acc);
        b = n;
    }
    if (t < len) batch_fma<VT, GL, V, WIDE, false>(b, len - t, k, kx, X, acc);
    if constexpr (V == 1) {
        acc = cross_group_sum<GL>(acc);
    } else {
        acc.x = cross_group_sum<GL>(acc.x);
        acc.y = cross_group_sum<GL>(acc.y);
    }
    if (g == 0 && on) *reinterpret_cast<XV *>(Y + size_t(r) * k + kc) = acc;
}

template <class VT, int KT, int V, bool WIDE>
hipError_t run_kt(const axspmv::launch::SpmmArgs &a, uint32_t k, const double *X, double *Y, hipStream_t s) {
    constexpr int GL = KT / V;
    const VT *val = static_cast<const VT *>(a.val);
    const uint32_t ktiles = (k + KT - 1) / KT;
    if (a.nrows) {
        const uint64_t wgs = (uint64_t(a.nrows) * GL + 255) / 256;
        dim3 grid(unsigned(a.xcd ? (wgs + 7) / 8 * 8 : wgs), ktiles);
        spmm_rows_kernel<VT, GL, V, WIDE><<<grid, 256, 0, s>>>(a.nrows, a.first, a.rowptr, val, a.col, k, a.long_slots,
                                                               a.xcd, X, Y);
    }
    if (a.nlong) {
        dim3 grid((a.nlong + 3) / 4, ktiles);
        spmm_long_kernel<VT, GL, V, WIDE><<<grid, 256, 0, s>>>(a.longrows, a.nlong, a.first, a.rowptr, val, a.col, k, X,
                                                               Y);
    }
    return hipGetLastError();
}

// Two right-hand sides per lane where every 16-byte access is aligned: k
// even, X and Y 16-byte aligned.  X rows by 32-bit byte offsets where X is
// under 4 GB.  Not at k-tile 8 where X rows are read without locality and
// every row is short (a.far: the k-tile's part of X, 64 bytes a row whatever k
// is, over 4 MB): groups of 4 lanes then keep 16 rows of a wave waiting for the
// slowest line, against 8.  One / two per lane, k = 8: permuted 66^3 stencil 133 / 149 us, 110^3 731 / 808,
// 300,007 random rows 115 / 130; but natural 66^3 53.1 / 51.7, 200,000-row
// power-law matrix (long rows) 98.6 / 92.4, permuted 40^3 (X of 4 MB) 17.7 / 16.9.
template <class VT, int KT>
hipError_t run_v(const axspmv::launch::SpmmArgs &a, uint32_t k, const double *X, double *Y, hipStream_t s) {
    const bool two = !(KT == 8 && a.far) && k % 2 == 0 && (reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y)) % 16 == 0;
    const bool wide = uint64_t(a.ncols) * k * 8 >= (1ull << 32);
    if (wide) return two ? run_kt<VT, KT, 2, true>(a, k, X, Y, s) : run_kt<VT, KT, 1, true>(a, k, X, Y, s);
    return two ? run_kt<VT, KT, 2, false>(a, k, X, Y, s) : run_kt<VT, KT, 1, false>(a, k, X, Y, s);
}

template <class VT>
hipError_t run_vt(const axspmv::launch::SpmmArgs &a, uint32_t k, uint32_t kt, const double *X, double *Y, hipStream_t s) {
    switch (kt) {
        case 8: return run_v<VT, 8>(a, k, X, Y, s);
        case 16: return run_v<VT, 16>(a, k, X, Y, s);
        case 32: return run_v<VT, 32>(a, k, X, Y, s);
        case 64: return run_v<VT, 64>(a, k, X, Y, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

namespace axspmv {
namespace launch {

hipError_t spmm(const SpmmArgs &a, uint32_t k, uint32_t kt, const double *X, double *Y, hipStream_t s) {
    return a.vtype == 1 ? run_vt<float>(a, k, kt, X, Y, s) : run_vt<double>(a, k, kt, X, Y, s);
}

}  // namespace launch
}  // namespace axspmv
