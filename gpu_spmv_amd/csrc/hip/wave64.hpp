// Wave64 cross-lane primitives for gfx950 built on DPP (data-parallel
// primitives: row_shr, row_bcast15/31, wave_shr/shl, mirrors) and readlane.
//
// They replace the 32-lane __shfl_* trees and Hillis-Steele scans of the
// reference (cudaSpmv.cu:1086-1090, 1586-1594, 2061-2086; scan.cu:239-414).
// A 64-bit value moves as two 32-bit DPP movs with the same control.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace axspmv {
namespace dev {

constexpr uint32_t NOROW = 0xffffffffu;

// x[c] for a slot of a padded layout: the plans mark padding slots with the
// column 0xffffffff (AXSPMV_PAD_COL), which reads 0.0, so a non-finite x
// entry cannot reach a row through a padding slot (0 * inf = NaN).
__device__ __forceinline__ double xpad(const double *__restrict__ x, uint32_t c) {
    return c == 0xffffffffu ? 0.0 : x[c];
}

// One load of a matrix stream; NT: non-temporal (the plans ask for it where
// the stream passes through the Infinity Cache without staying, so its
// lines need not evict the x lines the gathers reuse).
template <bool NT, class T>
__device__ __forceinline__ T stream_load(const T *p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// Sum of val[j] x[col[j]] over j = first, first + stride, ... < end, U terms in
// flight at a time (PAD: columns may be padding), in the order of j.  The row
// kernels take U = 4 with up to 16 lanes per row and for the long rows' waves,
// where one term at a time made a chain of load pairs: CSR vector / AXC on the
// 50,000-row power-law matrix 25.8 -> 15.6 / 42.8 -> 25.8 us, on 10^6 rows
// 250 -> 240 / 277 -> 253, the 1000^2 Laplacian 22.1 -> 18.3 / 29.4 -> 25.9; U
// = 1 with 32 and 64 lanes per row, which a row seldom fills twice (the 80^3
// stencil, 32 lanes: 67.6 us, 71.7 with U = 4).
template <bool NT, bool PAD, uint32_t U, class VT>
__device__ __forceinline__ double strided_dot(const VT *__restrict__ val, const uint32_t *__restrict__ col,
                                              uint32_t first, uint32_t end, uint32_t stride,
                                              const double *__restrict__ x) {
    double acc = 0.0;
    for (uint32_t j = first; j < end; j += U * stride) {
        // (CSR positions reach 2^32, where j + u stride would wrap; padded
        // layouts stay under 2^31, and the plain test is the faster one)
        const uint32_t left = end - j;
        auto in = [&](uint32_t u) { return PAD ? j + u * stride < end : u * stride < left; };
        VT v[U];
        uint32_t c[U];
        double xv[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (in(u)) {
                v[u] = stream_load<NT>(val + j + u * stride);
                c[u] = stream_load<NT>(col + j + u * stride);
            }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (in(u)) xv[u] = PAD ? xpad(x, c[u]) : x[c[u]];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (in(u)) acc = fma(double(v[u]), xv[u], acc);
        if (!PAD && left <= U * stride) break;
    }
    return acc;
}

// Rows a group of G lanes takes at once in the row-per-group kernels (CSR
// vector, AXC): two with 32 lanes, where most rows are one short round each
// and the waves' own cost shows (the 80^3 stencil in natural order, CSR / AXC
// 67.3 -> 52.6 / 71.7 -> 56.1 us; four rows take 48.5 / 50.9 there but lose 4 %
// on random rows of 20 to 46 entries); with 64 lanes two lost 8 % on rows of
// 60 to 90 entries, with fewer a group has four terms in flight already.  One
// on matrices of under 32,768 rows, where the second row halves the waves of a
// chip that two rows a wave fill once or twice (CSR vector, graph-timed, one /
// two rows: banded rows of 38 entries, 5,001 rows 2.49 / 2.90 us, 10,001 2.79 /
// 3.17, 20,001 3.84 / 4.04, 30,001 4.85 / 4.86, 60,001 9.64 / 8.56; random rows
// of 20 to 46, 10,001 rows 3.31 / 3.61, 100,001 21.4 / 20.9).
inline uint32_t rows_per_group(uint32_t G, uint32_t nrows) { return G == 32 && nrows >= 32768 ? 2 : 1; }

// R rows at once: acc[i] = the sum of val[j] x[col[j]] over j = b[i] + g, b[i] +
// g + stride, ... < e[i], term by term with the R rows' loads in flight
// together.
template <bool NT, bool PAD, uint32_t R, class VT>
__device__ __forceinline__ void strided_dots(const VT *__restrict__ val, const uint32_t *__restrict__ col,
                                             const uint32_t *b, const uint32_t *e, uint32_t g, uint32_t stride,
                                             const double *__restrict__ x, double *acc) {
    uint32_t most = 0;  // the longest row
#pragma unroll
    for (uint32_t i = 0; i < R; ++i) {
        acc[i] = 0.0;
        most = max(most, e[i] - b[i]);
    }
    for (uint32_t k = g; k < most; k += stride) {
        VT v[R];
        uint32_t c[R];
        double xv[R];
#pragma unroll
        for (uint32_t i = 0; i < R; ++i)
            if (k < e[i] - b[i]) {
                v[i] = stream_load<NT>(val + b[i] + k);
                c[i] = stream_load<NT>(col + b[i] + k);
            }
#pragma unroll
        for (uint32_t i = 0; i < R; ++i)
            if (k < e[i] - b[i]) xv[i] = PAD ? xpad(x, c[i]) : x[c[i]];
#pragma unroll
        for (uint32_t i = 0; i < R; ++i)
            if (k < e[i] - b[i]) acc[i] = fma(double(v[i]), xv[i], acc[i]);
    }
}

// DPP control words (GFX9 encoding).
enum : int {
    DPP_ROW_SHR1 = 0x111,
    DPP_ROW_SHR2 = 0x112,
    DPP_ROW_SHR4 = 0x114,
    DPP_ROW_SHR8 = 0x118,
    DPP_ROW_BCAST15 = 0x142,
    DPP_ROW_BCAST31 = 0x143,
    DPP_WAVE_SHL1 = 0x130,
    DPP_WAVE_SHR1 = 0x138,
    DPP_ROW_MIRROR = 0x140,
    DPP_ROW_HALF_MIRROR = 0x141,
    DPP_QUAD_1032 = 0xB1,  // quad_perm [1,0,3,2]
    DPP_QUAD_2301 = 0x4E,  // quad_perm [2,3,0,1]
    DPP_QUAD_BCAST0 = 0x00,  // quad_perm [j,j,j,j] = j * 0x55
    DPP_ROW_NEWBCAST0 = 0x150,  // lane j of each 16-lane row = 0x150 + j
};

// Lanes whose DPP source is out of range or whose row is masked keep `old`.
template <int CTRL, int ROWMASK = 0xf>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t old, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWMASK, 0xf, false);
}

template <int CTRL, int ROWMASK = 0xf>
__device__ __forceinline__ double dpp_f64(double old, double v) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, ROWMASK, 0xf, false);
    return __hiloint2double(hi, lo);
}

// f(integral constant 0), ..., f(integral constant N - 1): the DPP control of
// step j is a constant
template <int J>
struct StaticInt {
    static constexpr int value = J;
};
template <int N, int J = 0, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (J < N) {
        f(StaticInt<J>{});
        static_for<N, J + 1>(f);
    }
}

// The value of lane J of the lane's aligned group of G lanes (G = 4, 8 or
// 16), in every lane of the group.
template <int G, int J>
__device__ __forceinline__ uint32_t group_bcast_u32(uint32_t v) {
    static_assert((G == 4 || G == 8 || G == 16) && J < G, "group_bcast");
    const int x = int(v);
    if constexpr (G == 4) return uint32_t(__builtin_amdgcn_update_dpp(x, x, DPP_QUAD_BCAST0 + J * 0x55, 0xf, 0xf, false));
    else if constexpr (G == 16) return uint32_t(__builtin_amdgcn_update_dpp(x, x, DPP_ROW_NEWBCAST0 + J, 0xf, 0xf, false));
    else {  // lanes 0-7 of a row (banks 0, 1) take lane J, lanes 8-15 lane 8 + J
        const int lo = __builtin_amdgcn_update_dpp(x, x, DPP_ROW_NEWBCAST0 + J, 0xf, 0x3, false);
        return uint32_t(__builtin_amdgcn_update_dpp(lo, x, DPP_ROW_NEWBCAST0 + 8 + J, 0xf, 0xc, false));
    }
}
template <int G, int J>
__device__ __forceinline__ float group_bcast(float v) {
    return __uint_as_float(group_bcast_u32<G, J>(__float_as_uint(v)));
}
template <int G, int J>
__device__ __forceinline__ double group_bcast(double v) {
    return __hiloint2double(int(group_bcast_u32<G, J>(uint32_t(__double2hiint(v)))),
                            int(group_bcast_u32<G, J>(uint32_t(__double2loint(v)))));
}

__device__ __forceinline__ uint32_t lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ __forceinline__ uint32_t readlane_u32(uint32_t v, int lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ uint32_t readfirst_u32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// Lane i receives lane i-1's value; lane 0 receives `fill`.
__device__ __forceinline__ uint32_t shift_up_u32(uint32_t v, uint32_t fill) { return dpp_u32<DPP_WAVE_SHR1>(fill, v); }
__device__ __forceinline__ double shift_up_f64(double v, double fill) { return dpp_f64<DPP_WAVE_SHR1>(fill, v); }
// Lane i receives lane i+1's value; lane 63 receives `fill`.
__device__ __forceinline__ uint32_t shift_down_u32(uint32_t v, uint32_t fill) { return dpp_u32<DPP_WAVE_SHL1>(fill, v); }

// Segmented inclusive sum over the wave.  On entry `head` is nonzero on the
// lanes that start a segment; on exit v is the sum from the lane's segment
// head (or lane 0) to the lane, and `head` is nonzero iff a head lies in
// [0, lane].  Hillis-Steele inside 16-lane rows, then row_bcast15/31.
__device__ __forceinline__ double seg_scan_f64(double v, uint32_t &head) {
#define AX_SEG_STEP(CTRL, RM)                          \
    {                                                  \
        const double sv = dpp_f64<CTRL, RM>(0.0, v);   \
        const uint32_t sf = dpp_u32<CTRL, RM>(0u, head); \
        v = head ? v : v + sv;                         \
        head |= sf;                                    \
    }
    AX_SEG_STEP(DPP_ROW_SHR1, 0xf)
    AX_SEG_STEP(DPP_ROW_SHR2, 0xf)
    AX_SEG_STEP(DPP_ROW_SHR4, 0xf)
    AX_SEG_STEP(DPP_ROW_SHR8, 0xf)
    AX_SEG_STEP(DPP_ROW_BCAST15, 0xa)
    AX_SEG_STEP(DPP_ROW_BCAST31, 0xc)
#undef AX_SEG_STEP
    return v;
}

// Inclusive max over the wave of unsigned values (used to propagate the
// current row id forward: rows are nondecreasing in slot order).
__device__ __forceinline__ uint32_t scan_max_u32(uint32_t v) {
    v = max(v, dpp_u32<DPP_ROW_SHR1>(0u, v));
    v = max(v, dpp_u32<DPP_ROW_SHR2>(0u, v));
    v = max(v, dpp_u32<DPP_ROW_SHR4>(0u, v));
    v = max(v, dpp_u32<DPP_ROW_SHR8>(0u, v));
    v = max(v, dpp_u32<DPP_ROW_BCAST15, 0xa>(0u, v));
    v = max(v, dpp_u32<DPP_ROW_BCAST31, 0xc>(0u, v));
    return v;
}

// Sum over aligned groups of G lanes (G in 1,2,4,8,16,32,64); every lane of
// a group ends with the group total.
template <int G>
__device__ __forceinline__ double group_sum_f64(double v) {
    if constexpr (G >= 2) v += dpp_f64<DPP_QUAD_1032>(0.0, v);
    if constexpr (G >= 4) v += dpp_f64<DPP_QUAD_2301>(0.0, v);
    if constexpr (G >= 8) v += dpp_f64<DPP_ROW_HALF_MIRROR>(0.0, v);
    if constexpr (G >= 16) v += dpp_f64<DPP_ROW_MIRROR>(0.0, v);
    if constexpr (G >= 32) {
        const int lo = __builtin_amdgcn_ds_swizzle(__double2loint(v), 0x401F);  // xor 16 (bitmask mode)
        const int hi = __builtin_amdgcn_ds_swizzle(__double2hiint(v), 0x401F);
        v += __hiloint2double(hi, lo);
    }
    if constexpr (G >= 64) {
        const double lo_half = readlane_f64(v, 0), hi_half = readlane_f64(v, 32);
        v = lo_half + hi_half;
    }
    return v;
}

}  // namespace dev
}  // namespace axspmv
