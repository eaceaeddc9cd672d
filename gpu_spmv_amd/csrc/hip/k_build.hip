// Format builders on the device: CSR (device arrays) -> AXC / AXT arrays in
// the reference's layouts, equal bit for bit to the host builders.
//
// Each layout is a count, an exclusive scan and a fill:
//   count : per row, the units it occupies (AXC / AXT UNC th == 1: tiles of
//           hw slots, ceil(rl / hw); AXT UNC th > 1: tile columns,
//           ceil(rl / th); COM layouts are packed by CSR position and need
//           no count);
//   scan  : rocPRIM's device exclusive scan over the counts (64-bit, so the
//           host can reject layouts whose lengths overflow 32 bits);
//   fill  : one lane per value slot writes the slot's value, x value and
//           column, or the padding's zeros, so the arrays are written once
//           and need no clearing (row starts and the UNC headers come from
//           a kernel over the rows before it).
#include <rocprim/device/device_scan.hpp>

#include "launch.hpp"

namespace {
using axspmv::launch::BuildGeo;
using axspmv::launch::BuildOut;
using axspmv::launch::DevCsr;

constexpr uint32_t GROUP = 8;      // lanes per row in heads_kernel
constexpr uint32_t SLOTS = 4;      // value slots per lane in fill_kernel

// The device CSR's offsets and columns, checked before the fill reads col /
// val through them: bit 1 offsets decrease, 2 row[0] != 0, 4 row[nrows] !=
// nnz, 8 a column >= ncols; and, with cnt, every row's units (cnt[nrows] = 0,
// the scan's last input).  One thread per row and per four entries (VEC: col
// 16-byte aligned); reads only row[0 .. nrows] and col[0 .. nnz).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <bool VEC>
__global__ void __launch_bounds__(256) check_kernel(DevCsr a, uint32_t div, uint64_t *__restrict__ cnt,
                                                    uint32_t *__restrict__ flag) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    uint32_t bad = 0;
    if (i < a.nrows) {
        const uint32_t b = a.row[i], e = a.row[i + 1];
        if (e < b) bad |= 1u;
        if (cnt) cnt[i] = (e - b + uint64_t(div) - 1) / div;
    }
    if (i == 0) {
        if (a.row[0] != 0) bad |= 2u;
        if (a.row[a.nrows] != a.nnz) bad |= 4u;
        if (cnt) cnt[a.nrows] = 0;
    }
    if (VEC && 4 * i + 4 <= a.nnz) {
        const u32x4 c = reinterpret_cast<const u32x4 *>(a.col)[i];
        if (max(max(c.x, c.y), max(c.z, c.w)) >= a.ncols) bad |= 8u;
    } else {
        for (uint64_t k = 4 * i; k < a.nnz && k < 4 * i + 4; ++k)
            if (a.col[k] >= a.ncols) bad |= 8u;
    }
    if (bad) atomicOr(flag, bad);
}

// Row starts (con) and, with sec, the row of every tile (KIND 0) or tile
// column (KIND 1; 0 in the columns past the last row's) of the UNC layouts,
// GROUP lanes per row.
template <int KIND>
__global__ void __launch_bounds__(256) heads_kernel(DevCsr a, const uint64_t *__restrict__ start, BuildGeo g,
                                                    uint64_t nsec, BuildOut o) {
    const uint64_t gid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const uint32_t j = uint32_t(gid % GROUP), hw = g.hw;
    if (gid == 0) o.con[KIND == 0 ? 0 : a.nrows] = 0;
    if (KIND == 1 && o.sec) {
        const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
        for (uint64_t c = start[a.nrows] + gid; c < nsec; c += stride) o.sec[c] = 0;
    }
    if (gid / GROUP >= a.nrows) return;
    const uint32_t r = uint32_t(gid / GROUP);
    const uint64_t c0 = start[r], c1 = start[r + 1];
    if (j == 0) {
        if constexpr (KIND == 0) o.con[r + 1] = uint32_t(c1 * 2 * hw);
        else o.con[r] = uint32_t((c0 / hw) * 2 * hw * g.th + c0 % hw);
    }
    if (o.sec)
        for (uint64_t t = c0 + j; t < c1; t += GROUP) o.sec[t] = r;
}

// The row of a position: the r in [lo, hi) with at[r] <= key < at[r + 1],
// given at[lo] <= key < at[hi].  By the whole wave (the same key in every
// lane, 64 probes a step), and lane by lane.
template <class T>
__device__ __forceinline__ uint32_t wave_row_of(const T *__restrict__ at, uint32_t lo, uint32_t hi, uint64_t key) {
    const uint32_t lane = threadIdx.x & 63;
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint64_t i = uint64_t(lo) + uint64_t(step) * (lane + 1);
        const uint32_t c = uint32_t(__popcll(__ballot(i < hi && at[i < hi ? i : lo] <= key)));
        hi = uint32_t(min(uint64_t(hi), uint64_t(lo) + uint64_t(step) * (c + 1)));
        lo += step * c;
    }
    return lo;
}
template <class T>
__device__ __forceinline__ uint32_t row_of(const T *__restrict__ at, uint32_t lo, uint32_t hi, uint64_t key) {
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (at[mid] <= key) lo = mid;
        else hi = mid;
    }
    return lo;
}

// KIND 0: AXC / AXT UNC th == 1; 1: AXT UNC th > 1; 2: COM th == 1; 3: COM th
// > 1.  A wave takes 64 * SLOTS consecutive value slots, a lane SLOTS of them
// 64 apart, so val, col, plane and ax go in whole lines whatever the row
// lengths; a row's length does not decide how long its lanes run (with 8
// lanes per row and cleared arrays the 2^18-row power-law matrix, rows of up
// to 2048 entries, hw 4, took 269 us in the fill and 26 us in the clears; one
// slot per lane takes 70 us).  The
// slot's row: from sec (UNC, written by heads_kernel), or by a search of the
// row starts (AXC, which has no sec, and COM), narrowed by the wave to the
// rows of its slots first.  nslots value slots; plane has nplane >= nslots
// entries (AXC: 8 spare zeros).  SHIFT: hw and th are powers of two.
template <int KIND, bool SHIFT>
__global__ void __launch_bounds__(256) fill_kernel(DevCsr a, const uint64_t *__restrict__ start, BuildGeo g,
                                                   uint32_t nslots, uint32_t nplane, const double *__restrict__ x,
                                                   BuildOut o) {
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t q0 = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x - lane) * SLOTS;
    if (q0 >= nplane) return;  // whole waves leave together
    const uint32_t hw = g.hw, th = g.th, ths = hw * th;
    const uint32_t hs = SHIFT ? __builtin_ctz(hw) : 0, ts = SHIFT ? __builtin_ctz(th) : 0;
    auto div_hw = [&](uint32_t v) { return SHIFT ? v >> hs : v / hw; };
    auto div_ths = [&](uint32_t v) { return SHIFT ? v >> (hs + ts) : v / ths; };
    const bool find = KIND >= 2 || !o.sec;
    uint32_t lo = 0, hi = 0;  // rows of this wave's slots: [lo, hi)
    if (find && q0 < nslots) {
        const uint32_t qe = uint32_t(min(q0 + 64 * SLOTS, uint64_t(nslots))) - 1;
        uint64_t k0, k1;  // smallest and largest position looked up
        if constexpr (KIND == 0) {
            k0 = div_hw(uint32_t(q0));
            k1 = div_hw(qe);
        } else if constexpr (KIND == 2) {
            k0 = q0;
            k1 = qe;
        } else {
            k0 = uint64_t(div_ths(uint32_t(q0))) * ths;
            k1 = uint64_t(div_ths(qe)) * ths + ths - 1;
        }
        if constexpr (KIND == 0) {
            lo = wave_row_of(start, 0, a.nrows, k0);
            hi = wave_row_of(start, lo, a.nrows, k1) + 1;
        } else if (k0 < a.nnz) {
            lo = wave_row_of(a.row, 0, a.nrows, k0);
            hi = wave_row_of(a.row, lo, a.nrows, min(k1, uint64_t(a.nnz) - 1)) + 1;
        }
    }
    // the SLOTS slots step by step, so their loads go out together
    uint32_t q[SLOTS], t[SLOTS], f[SLOTS], r[SLOTS], p[SLOTS], c[SLOTS], head[SLOTS];
    bool slot[SLOTS], in[SLOTS];  // a value slot; one that holds an entry
    double v[SLOTS], xv[SLOTS];
#pragma unroll
    for (uint32_t u = 0; u < SLOTS; ++u) {
        const uint64_t qq = q0 + u * 64 + lane;
        slot[u] = qq < nslots;
        q[u] = slot[u] ? uint32_t(qq) : 0;
        if (!slot[u] && qq < nplane) o.plane[qq] = 0;
        t[u] = div_hw(q[u]);
        f[u] = q[u] - t[u] * hw;
        in[u] = slot[u];
        r[u] = 0;
        if constexpr (KIND == 0) {
            if (slot[u]) r[u] = o.sec ? o.sec[t[u]] : row_of(start, lo, hi, t[u]);
        } else if constexpr (KIND == 1) {
            const uint32_t T = div_ths(q[u]);
            p[u] = T * hw + f[u];        // tile column
            head[u] = t[u] - T * th;     // level
            in[u] = slot[u] && p[u] < uint32_t(start[a.nrows]);
            if (in[u]) r[u] = o.sec[p[u]];
        } else {
            const uint32_t T = div_ths(q[u]), lvl = t[u] - T * th;
            const uint64_t pp = KIND == 2 ? uint64_t(q[u]) : uint64_t(T) * ths + uint64_t(f[u]) * th + lvl;
            in[u] = slot[u] && pp < a.nnz;
            p[u] = uint32_t(pp);
            if (in[u]) r[u] = row_of(a.row, lo, hi, pp);
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < SLOTS; ++u) {
        if (!in[u]) continue;
        const uint32_t b = a.row[r[u]], e = a.row[r[u] + 1];
        if constexpr (KIND <= 1) {
            const uint32_t s0 = uint32_t(start[r[u]]);
            const uint32_t k = KIND == 0 ? q[u] - s0 * hw : (p[u] - s0) * th + head[u];
            in[u] = k < e - b;
            p[u] = b + k;
        } else {
            const uint32_t at = KIND == 2 ? p[u] % g.bs : t[u] - div_ths(q[u]) * th;
            const uint32_t last = (KIND == 2 ? g.bs : th) - 1 - at;
            head[u] = p[u] == b || at == 0 ? (r[u] << g.log) | min(e - p[u] - 1, last) : 0;
        }
    }
#pragma unroll
    for (uint32_t u = 0; u < SLOTS; ++u) {
        v[u] = 0.0;
        c[u] = 0;
        if (!in[u]) continue;
        v[u] = a.val[p[u]];
        c[u] = a.col[p[u]];
    }
#pragma unroll
    for (uint32_t u = 0; u < SLOTS; ++u) {
        xv[u] = 0.0;
        if (x && in[u]) xv[u] = x[c[u]];
    }
#pragma unroll
    for (uint32_t u = 0; u < SLOTS; ++u) {
        if (!slot[u]) continue;
        const uint64_t s = uint64_t(t[u]) * 2 * hw + f[u];  // groups of hw values followed by hw x values
        o.ax[s] = v[u];
        o.ax[s + hw] = xv[u];
        o.plane[q[u]] = c[u];
        if constexpr (KIND >= 2) o.sec[q[u]] = in[u] ? head[u] : 0;
    }
}

// AXT UNC th == 1 with hw 4 to 256, a power of two, and ax and plane 16-byte
// aligned: a lane takes four neighbouring slots of a tile, so the tile's row
// is looked up once for the four.  The requests to L2 bound this kernel (one
// per entry for x is the least), so a wave's 256 slots -- whole tiles, 4 KB of
// ax -- pass through LDS and leave as 1 KB runs: stored from the lanes'
// registers, each 16-byte piece was a request of its own (the 2^18-row
// power-law matrix, 5.2M entries, hw 4: 64 us, against 73 us from registers,
// 82 with non-temporal stores there, and 70 us one slot per lane), and now
// whole lines, non-temporal, so that they leave the L2s to x: 37 us.
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x2_at8 __attribute__((ext_vector_type(2), aligned(8)));
typedef uint32_t u32x4_at4 __attribute__((ext_vector_type(4), aligned(4)));
__global__ void __launch_bounds__(256) fill_quads_kernel(DevCsr a, const uint64_t *__restrict__ start, uint32_t hw_log,
                                                         uint32_t nquads, const double *__restrict__ x, BuildOut o) {
    __shared__ f64x2 buf[4][256];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
    f64x2 v0 = {0.0, 0.0}, v1 = {0.0, 0.0}, x0 = {0.0, 0.0}, x1 = {0.0, 0.0};
    u32x4 c = {0, 0, 0, 0};
    uint32_t k = 0, len = 0, p = 0;
    if (i < nquads) {
        const uint32_t q = i * 4, t = q >> hw_log, r = o.sec[t], b = a.row[r];
        len = a.row[r + 1] - b;
        k = q - (uint32_t(start[r]) << hw_log);
        p = b + k;
    }
    if (k < len && len - k >= 4) {
        c = *reinterpret_cast<const u32x4_at4 *>(a.col + p);
        v0 = *reinterpret_cast<const f64x2_at8 *>(a.val + p);
        v1 = *reinterpret_cast<const f64x2_at8 *>(a.val + p + 2);
        if (x) {
            x0 = f64x2{x[c.x], x[c.y]};
            x1 = f64x2{x[c.z], x[c.w]};
        }
    } else if (k < len) {  // 1 to 3 entries, then padding
        const uint32_t m = len - k;
        c.x = a.col[p];
        v0.x = a.val[p];
        if (m > 1) {
            c.y = a.col[p + 1];
            v0.y = a.val[p + 1];
        }
        if (m > 2) {
            c.z = a.col[p + 2];
            v1.x = a.val[p + 2];
        }
        if (x) {
            x0.x = x[c.x];
            if (m > 1) x0.y = x[c.y];
            if (m > 2) x1.x = x[c.z];
        }
    }
    if (i < nquads) __builtin_nontemporal_store(c, reinterpret_cast<u32x4 *>(o.plane) + i);
    // slots 4 lane .. 4 lane + 3 of the wave's 256, as pairs of doubles of ax
    f64x2 *w = buf[threadIdx.x >> 6];
    const uint32_t sl = lane * 4, pr = (((sl >> hw_log) << (hw_log + 1)) + (sl & ((1u << hw_log) - 1))) / 2;
    w[pr] = v0;
    w[pr + 1] = v1;
    w[pr + (1u << hw_log) / 2] = x0;
    w[pr + (1u << hw_log) / 2 + 1] = x1;
    __syncthreads();
    const uint32_t first = i - lane;  // the wave's first quad; 4 pairs of ax per quad
    f64x2 *s = reinterpret_cast<f64x2 *>(o.ax) + uint64_t(first) * 4;
    const uint32_t pairs = first < nquads ? min(nquads - first, 64u) * 4 : 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
        if (j * 64 + lane < pairs) __builtin_nontemporal_store(w[j * 64 + lane], s + j * 64 + lane);
}

}  // namespace

namespace axspmv {
namespace launch {

hipError_t build_check(const DevCsr &a, uint32_t div, uint64_t *cnt, uint32_t *flag, hipStream_t s) {
    const uint64_t threads = std::max<uint64_t>(1, std::max<uint64_t>(a.nrows, (uint64_t(a.nnz) + 3) / 4));
    const unsigned grid = unsigned((threads + 255) / 256);
    if (reinterpret_cast<uintptr_t>(a.col) % 16 == 0)
        check_kernel<true><<<grid, 256, 0, s>>>(a, div, cnt, flag);
    else
        check_kernel<false><<<grid, 256, 0, s>>>(a, div, cnt, flag);
    return hipGetLastError();
}

hipError_t build_scan(const uint64_t *in, uint64_t *out, size_t n, void *tmp, size_t &tmp_bytes, hipStream_t s) {
    return rocprim::exclusive_scan(tmp, tmp_bytes, in, out, uint64_t(0), n, rocprim::plus<uint64_t>(), s);
}

hipError_t build_fill(const DevCsr &a, int kind, const uint64_t *start, const BuildGeo &g, const double *x,
                      const BuildOut &o, uint32_t nslots, uint32_t nplane, uint32_t nsec, hipStream_t s) {
    hipError_t e;
    if (kind <= 1) {
        const uint64_t threads = std::max<uint64_t>(1, uint64_t(a.nrows) * GROUP);
        const unsigned grid = unsigned((threads + 255) / 256);
        if (kind == 0)
            heads_kernel<0><<<grid, 256, 0, s>>>(a, start, g, nsec, o);
        else
            heads_kernel<1><<<grid, 256, 0, s>>>(a, start, g, nsec, o);
        e = hipGetLastError();
    } else {
        e = fill_u32(o.con, size_t(a.nrows) + 1, 0u, s);
    }
    if (e != hipSuccess || !nplane) return e;
    const bool shift = (g.hw & (g.hw - 1)) == 0 && (g.th & (g.th - 1)) == 0;
    if (kind == 0 && o.sec && shift && g.hw >= 4 && g.hw <= 256 &&
        (reinterpret_cast<uintptr_t>(o.ax) | reinterpret_cast<uintptr_t>(o.plane)) % 16 == 0) {
        const uint32_t quads = nslots / 4;
        fill_quads_kernel<<<(quads + 255) / 256, 256, 0, s>>>(a, start, __builtin_ctz(g.hw), quads, x, o);
        return hipGetLastError();
    }
    const unsigned grid = unsigned((uint64_t(nplane) + 256 * SLOTS - 1) / (256 * SLOTS));
#define AX_FILL(K)                                                                      \
    do {                                                                                \
        if (shift)                                                                      \
            fill_kernel<K, true><<<grid, 256, 0, s>>>(a, start, g, nslots, nplane, x, o);  \
        else                                                                            \
            fill_kernel<K, false><<<grid, 256, 0, s>>>(a, start, g, nslots, nplane, x, o); \
    } while (0)
    switch (kind) {
        case 0: AX_FILL(0); break;
        case 1: AX_FILL(1); break;
        case 2: AX_FILL(2); break;
        default: AX_FILL(3); break;
    }
#undef AX_FILL
    return hipGetLastError();
}

}  // namespace launch
}  // namespace axspmv
