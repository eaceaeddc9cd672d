// K1 and AXC kernels.
//
// K1 (reference gk1, cudaSpmv.cu:851-867): a chunk of C rows stored column
// major (element j of row r of chunk c at chp[c] + j*C + r), one lane per
// row, so every step of the 64 lanes reads 64 neighbouring values.  Here a
// 64-row chunk is one wavefront.  Rows sorted by length put the longest rows
// together; a chunk whose nmc exceeds the per-wave step limit is split over
// several waves (work items) whose partial sums a second kernel adds in a
// fixed order -- the reference instead runs one thread for the whole row.
// The reference's first step is unconditional and reads past an all-empty
// chunk (nmc = 0); here the loop simply does not run.
//
// AXC (reference gaxc, cudaSpmv.cu:1072-1096): each row is a run of bricks
// of hbs slots (value plane slot brp[r]/2 + k, column in mapx).  A group of
// G = hbs lanes walks one row brick by brick and reduces with DPP; rows
// longer than 64 bricks are taken by a whole wave (listed on the host), so a
// few long rows do not serialise on G lanes.
#include "launch.hpp"
#include "wave64.hpp"

namespace {
using namespace axspmv::dev;
using axspmv::launch::K1Item;

// NT: val and col are streamed with non-temporal loads.  MODE (launch::K1Mode):
//
//  * K1_LONG: steps 8 at a time, the values and columns of the next 8 in
//    flight while the x gathers of these are waited for (a chunk is one chain
//    of steps, and a small matrix has few chunks per SIMD to hide it behind).
//    Steps past the end re-read the item's last one and add nothing.  Against
//    K1_FAR's way: random rows of 4 to 40 entries, 20,001 rows 8.3 -> 7.2 us
//    in a graph, 300,007 rows, FP32 values, 41.3 -> 37.4; 100,001-row
//    power-law matrix 36.4 -> 28.5; 400,001 banded rows of 10 22.7 -> 18.4;
//    permuted 90^3 stencil renumbered 84 -> 71.
//  * K1_SHORT, rows of up to 6 entries on average: 4 at a time, none loaded
//    past the end (8 at a time take 8 steps' loads and 66 to 80 registers for
//    5 steps).  K1_FAR / K1_LONG / this: 700^2 Laplacian, FP32 values, in a
//    graph 6.5 / 7.4 / 6.3 us, 1400^2 35.6 / 33.6 / 31.9, 400,001 banded rows of
//    5 14.4 / 12.6 / 12.8, of 2.7 10.2 / 9.5 / 9.2.
//  * K1_FAR, rows of up to 12 entries that gather without locality from an x
//    larger than an L2: 4 at a time, the next 4 not before these are added.
//    More loads in flight gain nothing there.  Random, this / K1_LONG: 540,001
//    rows of 0 to 9 21.6 / 23.4 us, 700,001 30.7 / 34.0 (K1_SHORT 33.6), of 0 to
//    16 45.1 / 50.9, 900,001 of 4 to 12 74.4 / 79.4, 1,200,001 of 9 to 13 146.8 /
//    155.0, 600,001 of 10 to 14 66.2 / 62.4 (in a graph 52.9 / 55.4), 700,001 of 8
//    to 24 95.4 / 93.3, FP32 values in a graph 75.4 / 80.9.
using axspmv::launch::K1Mode;
template <class VT, bool NT, K1Mode MODE>
__global__ void __launch_bounds__(256) k1_kernel(const K1Item *__restrict__ items, uint32_t nitems, uint32_t chunk,
                                                 const VT *__restrict__ val, const uint32_t *__restrict__ col,
                                                 const uint32_t *__restrict__ permi, uint32_t nrows,
                                                 const double *__restrict__ x, double *__restrict__ y,
                                                 double *__restrict__ part) {
    const uint32_t gl = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t per_wave = 64 / chunk;  // chunks per wave (1 for chunk 64)
    const uint32_t wave = gl >> 6, lane = gl & 63;
    const uint32_t it = wave * per_wave + lane / chunk;
    if (it >= nitems) return;
    const K1Item w = items[it];
    const uint32_t r = lane % chunk;
    const uint32_t gid = w.chunk * chunk + r;
    const uint64_t base = uint64_t(w.chp) + r;
    double acc = 0.0;
    if constexpr (MODE == K1Mode::K1_FAR) {
        uint32_t j = w.j0;
        for (; j + 4 <= w.j1; j += 4) {
            const uint64_t q = base + uint64_t(j) * chunk;
            VT v[4];
            double xv[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v[u] = stream_load<NT>(val + q + u * chunk);
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) xv[u] = xpad(x, stream_load<NT>(col + q + u * chunk));
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) acc = fma(double(v[u]), xv[u], acc);
        }
        for (; j < w.j1; ++j) {
            const uint64_t q = base + uint64_t(j) * chunk;
            acc = fma(double(stream_load<NT>(val + q)), xpad(x, stream_load<NT>(col + q)), acc);
        }
    } else if (w.j0 < w.j1) {
        constexpr uint32_t U = MODE == K1Mode::K1_LONG ? 8 : 4;
        VT v[U];
        uint32_t c[U];
        auto step = [&](uint32_t j, uint32_t u) {
            const uint64_t q = base + uint64_t(j) * chunk;
            v[u] = stream_load<NT>(val + q);
            c[u] = stream_load<NT>(col + q);
        };
        auto half = [&](uint32_t j, uint32_t u0) {
#pragma unroll
            for (uint32_t u = u0; u < u0 + U / 2; ++u) step(min(j + u, w.j1 - 1), u);
        };
        auto fetch = [&](uint32_t j) {
            if constexpr (MODE == K1Mode::K1_LONG) {
                half(j, 0);
                if (j + U / 2 < w.j1) half(j, U / 2);
            } else {
#pragma unroll
                for (uint32_t u = 0; u < U; ++u)
                    if (j + u < w.j1) step(j + u, u);
            }
        };
        fetch(w.j0);
        for (uint32_t j = w.j0; j < w.j1; j += U) {
            double xv[U], vv[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                xv[u] = j + u < w.j1 ? xpad(x, c[u]) : 0.0;
                vv[u] = j + u < w.j1 ? double(v[u]) : 0.0;
            }
            if (j + U < w.j1) fetch(j + U);
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) acc = fma(vv[u], xv[u], acc);
        }
    }
    if (w.slot == NOROW) {
        if (gid < nrows) y[permi[gid]] = acc;
    } else {
        part[uint64_t(w.slot) * chunk + r] = acc;
    }
}

// Sum of the partial results of one split chunk, in item order.
__global__ void __launch_bounds__(256) k1_fixup(const uint32_t *__restrict__ split, uint32_t nsplit, uint32_t chunk,
                                                const uint32_t *__restrict__ permi, uint32_t nrows,
                                                const double *__restrict__ part, double *__restrict__ y) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t s = g / chunk, r = g % chunk;
    if (s >= nsplit) return;
    const uint32_t c = split[3 * s], slot0 = split[3 * s + 1], ns = split[3 * s + 2];
    const uint32_t gid = c * chunk + r;
    double acc = 0.0;
    for (uint32_t k = 0; k < ns; ++k) acc += part[uint64_t(slot0 + k) * chunk + r];
    if (gid < nrows) y[permi[gid]] = acc;
}

// AXC: G lanes per row; rows listed in `longrows` are skipped here and done
// by axc_long (one wave per row).
template <class VT, int G, bool NT, uint32_t R>
__global__ void __launch_bounds__(256) axc_kernel(uint32_t nrows, const uint32_t *__restrict__ brp,
                                                  const VT *__restrict__ vp, const uint32_t *__restrict__ mapx,
                                                  uint32_t long_slots, const double *__restrict__ x,
                                                  double *__restrict__ y) {
    const size_t gl = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gl / G * R >= nrows) return;  // whole groups leave together (G divides 64)
    const uint32_t r = uint32_t(gl / G) * R, g = uint32_t(gl % G);
    if constexpr (R == 1) {
        const uint32_t b = brp[r] >> 1, e = brp[r + 1] >> 1;
        if (e - b > long_slots) return;
        double acc = strided_dot<NT, true, G <= 16 ? 4 : 1>(vp, mapx, b + g, e, G, x);
        acc = group_sum_f64<G>(acc);
        if (g == 0) y[r] = acc;
    } else {
        uint32_t b[R], e[R];
        double acc[R];
#pragma unroll
        for (uint32_t i = 0; i < R; ++i) {
            b[i] = brp[min(r + i, nrows)] >> 1;
            e[i] = brp[min(r + i + 1, nrows)] >> 1;
        }
        bool mine[R];  // not axc_long's row, not past the last
#pragma unroll
        for (uint32_t i = 0; i < R; ++i) {
            mine[i] = r + i < nrows && e[i] - b[i] <= long_slots;
            if (!mine[i]) e[i] = b[i];
        }
        strided_dots<NT, true, R>(vp, mapx, b, e, g, G, x, acc);
#pragma unroll
        for (uint32_t i = 0; i < R; ++i) {
            acc[i] = group_sum_f64<G>(acc[i]);
            if (g == 0 && mine[i]) y[r + i] = acc[i];
        }
    }
}

template <class VT, bool NT>
__global__ void __launch_bounds__(256) axc_long(const uint32_t *__restrict__ rows, uint32_t nlong,
                                                const uint32_t *__restrict__ brp, const VT *__restrict__ vp,
                                                const uint32_t *__restrict__ mapx, const double *__restrict__ x,
                                                double *__restrict__ y) {
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (wave >= nlong) return;
    const uint32_t r = rows[wave];
    const uint32_t b = brp[r] >> 1, e = brp[r + 1] >> 1;
    double acc = strided_dot<NT, true, 4>(vp, mapx, b + lane, e, 64, x);
    acc = group_sum_f64<64>(acc);
    if (lane == 0) y[r] = acc;
}

template <class VT>
hipError_t k1_vt(const axspmv::launch::K1Args &a, const double *x, double *y, hipStream_t s) {
    const uint32_t per_wave = 64 / a.chunk;
    const uint32_t waves = (a.nitems + per_wave - 1) / per_wave;
    auto run = [&](auto kernel) {
        kernel<<<(waves + 3) / 4, 256, 0, s>>>(a.items, a.nitems, a.chunk, static_cast<const VT *>(a.val), a.col, a.permi,
                                               a.nrows, x, y, a.part);
    };
    if (waves) switch (a.mode) {
        case K1Mode::K1_LONG: a.nt ? run(k1_kernel<VT, true, K1Mode::K1_LONG>) : run(k1_kernel<VT, false, K1Mode::K1_LONG>); break;
        case K1Mode::K1_SHORT: a.nt ? run(k1_kernel<VT, true, K1Mode::K1_SHORT>) : run(k1_kernel<VT, false, K1Mode::K1_SHORT>); break;
        case K1Mode::K1_FAR: a.nt ? run(k1_kernel<VT, true, K1Mode::K1_FAR>) : run(k1_kernel<VT, false, K1Mode::K1_FAR>); break;
    }
    if (a.nsplit) {
        const uint32_t th = a.nsplit * a.chunk;
        k1_fixup<<<(th + 255) / 256, 256, 0, s>>>(a.split, a.nsplit, a.chunk, a.permi, a.nrows, a.part, y);
    }
    return hipGetLastError();
}

template <class VT, bool NT>
hipError_t axc_vt(const axspmv::launch::AxcArgs &a, const double *x, double *y, hipStream_t s) {
    const VT *vp = static_cast<const VT *>(a.vplane);
    const uint32_t rows = rows_per_group(a.hbs, a.nrows);
    const unsigned grid = unsigned(((uint64_t(a.nrows) + rows - 1) / rows * a.hbs + 255) / 256);
    if (a.nrows) switch (a.hbs) {
#define AX_G(G) \
    case G: axc_kernel<VT, G, NT, 1><<<grid, 256, 0, s>>>(a.nrows, a.brp, vp, a.mapx, a.long_slots, x, y); break;
        AX_G(1)
        AX_G(2)
        AX_G(4)
        AX_G(8)
        AX_G(16)
        AX_G(64)
        case 32:
            if (rows == 2)
                axc_kernel<VT, 32, NT, 2><<<grid, 256, 0, s>>>(a.nrows, a.brp, vp, a.mapx, a.long_slots, x, y);
            else
                axc_kernel<VT, 32, NT, 1><<<grid, 256, 0, s>>>(a.nrows, a.brp, vp, a.mapx, a.long_slots, x, y);
            break;
#undef AX_G
        default: return hipErrorInvalidValue;
    }
    if (a.nlong) axc_long<VT, NT><<<(a.nlong + 3) / 4, 256, 0, s>>>(a.longrows, a.nlong, a.brp, vp, a.mapx, x, y);
    return hipGetLastError();
}

}  // namespace

namespace axspmv {
namespace launch {

hipError_t k1(const K1Args &a, const double *x, double *y, hipStream_t s) {
    return a.vtype == 1 ? k1_vt<float>(a, x, y, s) : k1_vt<double>(a, x, y, s);
}

hipError_t axc(const AxcArgs &a, const double *x, double *y, hipStream_t s) {
    if (a.nt) return a.vtype == 1 ? axc_vt<float, true>(a, x, y, s) : axc_vt<double, true>(a, x, y, s);
    return a.vtype == 1 ? axc_vt<float, false>(a, x, y, s) : axc_vt<double, false>(a, x, y, s);
}

}  // namespace launch
}  // namespace axspmv
