// In-place transform kernels of the FP64 Poisson solve on the register-direct FFT
// (fft_reg.h), for the lengths 16..768 with prime factors up to 13 that have no
// kernels in poisson_ct.h.  Element of x row a, z index j, plane k of a field
// (the caller's array): k nz nx + j nx + a.
//
// Bound: HBM (one read and one write of the field).  Measured on one MI355X,
// x forward / z forward / z inverse / x inverse in us (mean of 12 solves under
// the profiler), against the runtime-sized kernels of poisson.hip, which these
// lengths ran before (they divide per element, load 8 bytes at a time under
// branches and gather their twiddles): 560 x 280 x 280 (0.70 GB a kernel) 170 /
// 152 / 138 / 164 against 560 / 618 / 432 / 409 (4.1-5.1 TB/s); 624 x 312 x 770
// (2.4 GB) 502 / 426 / 415 / 539, x forward against 1990.  At the lengths of
// poisson_ct.h they were within 5% of the best variant there on either side
// (in the blocked layouts, 768 x 384 x 384: 376 / 353 / 315 / 323), so those
// lengths keep their tuned variants and have no kernels here.
#pragma once

#include <hip/hip_runtime.h>

#include "fft_reg.h"
#include "poisson_ct_launch.h"

namespace dnsp {

__device__ __forceinline__ double rg_ld(const double* base, unsigned off) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
}
__device__ __forceinline__ double2 rg_ld2(const double* base, unsigned off) {
    return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(base) + off);
}
__device__ __forceinline__ void rg_st(double* base, unsigned off, double v) {
    *reinterpret_cast<double*>(reinterpret_cast<char*>(base) + off) = v;
}
__device__ __forceinline__ void rg_st2(double* base, unsigned off, double2 v) {
    *reinterpret_cast<double2*>(reinterpret_cast<char*>(base) + off) = v;
}

// Tile shapes.  x: G pairs of lines per workgroup, about 1536 complex values
// (28 KB of LDS: four or five workgroups per CU, whose loads, exchanges and
// stores overlap); z: the 8 pairs of one 16-row block (128-byte rows).  Threads:
// one per 12 complex values, so that a radix-8..16 butterfly per thread covers
// the tile.
constexpr int rg_x_lines(int n) { return 1536 / n > 0 ? 1536 / n : 1; }
constexpr int rg_threads(int elems) {
    const int t = (elems / 12 + 63) / 64 * 64;
    return t < 64 ? 64 : (t > 512 ? 512 : t);
}
constexpr int kRgCols = 8;
// LDS pitch of a z column: = 2 mod 16 complex values, so that the 8 columns
// (fastest over lanes) and two neighbouring elements fall on different banks.
constexpr int rg_col_pitch(int n) { return ct_pitch(n) + (18 - ct_pitch(n) % 16) % 16; }

// x forward, lines -> lines (in place allowed).
template <int N, int G, int NT>
__global__ __launch_bounds__(NT) void kr_xfwd(const double* P, double* S, long nlines, const double2* __restrict__ tw) {
    constexpr int LP = ct_pitch(N);
    __shared__ double2 buf[G * LP];
    __shared__ double2 stw[N];
    ct_stage_twiddles<N, NT>(stw, tw);
    const long l0 = (long)xcd_tile(blockIdx.x, gridDim.x) * 2 * G;
    const int left = nlines - l0 < 2 * G ? (int)(nlines - l0) : 2 * G;  // valid lines of this tile
    const double* src = P + l0 * N;
    double* dst = S + l0 * N;
    auto ld = [&](int g, int j, int m, auto& v) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        const int la = 2 * g < left ? 2 * g : 0;
        const bool vb = 2 * g + 1 < left;
        const unsigned oa = (unsigned)(la * N + j) * 8u, ob = vb ? oa + N * 8u : oa;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            v[r].x = rg_ld(src, oa + (unsigned)(r * m) * 8u);
            v[r].y = rg_ld(src, ob + (unsigned)(r * m) * 8u);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) v[r].y = vb ? v[r].y : 0.0;
    };
    auto st = [&](int g, int lo, int hi, bool both, double2 L, double2 H) {
        if (2 * g >= left) return;
        const unsigned oa = (unsigned)(2 * g * N) * 8u, ob = oa + N * 8u;
        const bool vb = 2 * g + 1 < left;
        rg_st(dst, oa + (unsigned)lo * 8u, L.x);
        if (vb) rg_st(dst, ob + (unsigned)lo * 8u, L.y);
        if (both) {
            rg_st(dst, oa + (unsigned)hi * 8u, H.x);
            if (vb) rg_st(dst, ob + (unsigned)hi * 8u, H.y);
        }
    };
    rg_forward<N, G, NT, LP, false>(buf, stw, ld, st);
}

// x inverse, lines -> lines (in place allowed), times scale.
template <int N, int G, int NT>
__global__ __launch_bounds__(NT) void kr_xbwd(const double* S, double* P, long nlines, double scale,
                                              const double2* __restrict__ tw) {
    constexpr int LP = ct_pitch(N);
    __shared__ double2 buf[G * LP];
    __shared__ double2 stw[N];
    ct_stage_twiddles<N, NT>(stw, tw);
    const long l0 = (long)xcd_tile(blockIdx.x, gridDim.x) * 2 * G;
    const int left = nlines - l0 < 2 * G ? (int)(nlines - l0) : 2 * G;
    const double* src = S + l0 * N;
    double* dst = P + l0 * N;
    auto ld = [&](int g, int lo, int hi, double2& A, double2& B) {
        const int la = 2 * g < left ? 2 * g : 0;
        const bool vb = 2 * g + 1 < left;
        const unsigned oa = (unsigned)(la * N) * 8u, ob = vb ? oa + N * 8u : oa;
        A = make_double2(rg_ld(src, oa + lo * 8u), rg_ld(src, ob + lo * 8u));
        B = make_double2(rg_ld(src, oa + hi * 8u), rg_ld(src, ob + hi * 8u));
        A.y = vb ? A.y : 0.0;
        B.y = vb ? B.y : 0.0;
    };
    auto st = [&](int g, int j, int m, auto& v) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        if (2 * g >= left) return;
        const unsigned oa = (unsigned)(2 * g * N + j) * 8u, ob = oa + N * 8u;
#pragma unroll
        for (int r = 0; r < R; ++r) rg_st(dst, oa + (unsigned)(r * m) * 8u, v[r].x * scale);
        if (2 * g + 1 < left) {
#pragma unroll
            for (int r = 0; r < R; ++r) rg_st(dst, ob + (unsigned)(r * m) * 8u, v[r].y * scale);
        }
    };
    rg_inverse<N, G, NT, LP, false>(buf, stw, ld, st);
}

// z kernels, in place: one workgroup per (plane k, block c of 16 x rows); complex
// column g pairs rows 16c + 2g and 16c + 2g + 1 (the last row of an odd nx is
// paired with zero).  A pair is one 16-byte access where all pairs are 16-byte
// aligned (even nx, aligned array; uniform over the grid), else two 8-byte ones.
__device__ __forceinline__ double2 rg_ldp(const double* base, unsigned off, bool al, bool two) {
    if (al) return rg_ld2(base, off);
    const double a = rg_ld(base, off), b = rg_ld(base, two ? off + 8u : off);
    return make_double2(a, two ? b : 0.0);
}
__device__ __forceinline__ void rg_stp(double* base, unsigned off, bool al, bool two, double2 v) {
    if (al) {
        rg_st2(base, off, v);
    } else {
        rg_st(base, off, v.x);
        if (two) rg_st(base, off + 8u, v.y);
    }
}
__device__ __forceinline__ bool rg_pairs_aligned(const void* p, int nx) { return ((size_t)p & 15) == 0 && nx % 2 == 0; }

template <int N, int NT>
__global__ __launch_bounds__(NT) void kr_zfwd(double* S, int nx, const double2* __restrict__ tw) {
    constexpr int G = kRgCols, LP = rg_col_pitch(N);
    __shared__ double2 buf[G * LP];
    __shared__ double2 stw[N];
    ct_stage_twiddles<N, NT>(stw, tw);
    const int nab = (nx + 15) / 16;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int k = tile / nab, c = tile - k * nab;
    const int w = nx - 16 * c < 16 ? nx - 16 * c : 16;  // rows of the block
    const bool al = rg_pairs_aligned(S, nx);
    double* s = S + (long)k * nx * N + 16 * c;
    const unsigned nxb = (unsigned)nx * 8u;
    auto ld = [&](int g, int j, int m, auto& v) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        const int gg = 2 * g < w ? g : 0;
        const unsigned o = (unsigned)j * nxb + (unsigned)gg * 16u, ms = (unsigned)m * nxb;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = rg_ldp(s, o + (unsigned)r * ms, al, 2 * gg + 1 < w);
    };
    auto st = [&](int g, int lo, int hi, bool both, double2 L, double2 H) {
        if (2 * g >= w) return;
        rg_stp(s, (unsigned)lo * nxb + (unsigned)g * 16u, al, 2 * g + 1 < w, L);
        if (both) rg_stp(s, (unsigned)hi * nxb + (unsigned)g * 16u, al, 2 * g + 1 < w, H);
    };
    rg_forward<N, G, NT, LP, true>(buf, stw, ld, st);
}

template <int N, int NT>
__global__ __launch_bounds__(NT) void kr_zbwd(double* S, int nx, const double2* __restrict__ tw) {
    constexpr int G = kRgCols, LP = rg_col_pitch(N);
    __shared__ double2 buf[G * LP];
    __shared__ double2 stw[N];
    ct_stage_twiddles<N, NT>(stw, tw);
    const int nab = (nx + 15) / 16;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int k = tile / nab, c = tile - k * nab;
    const int w = nx - 16 * c < 16 ? nx - 16 * c : 16;
    const bool al = rg_pairs_aligned(S, nx);
    double* s = S + (long)k * nx * N + 16 * c;
    const unsigned nxb = (unsigned)nx * 8u;
    auto ld = [&](int g, int lo, int hi, double2& A, double2& B) {
        const int gg = 2 * g < w ? g : 0;
        A = rg_ldp(s, (unsigned)lo * nxb + (unsigned)gg * 16u, al, 2 * gg + 1 < w);
        B = rg_ldp(s, (unsigned)hi * nxb + (unsigned)gg * 16u, al, 2 * gg + 1 < w);
    };
    auto st = [&](int g, int j, int m, auto& v) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        if (2 * g >= w) return;
        const unsigned o = (unsigned)j * nxb + (unsigned)g * 16u, ms = (unsigned)m * nxb;
#pragma unroll
        for (int r = 0; r < R; ++r) rg_stp(s, o + (unsigned)r * ms, al, 2 * g + 1 < w, v[r]);
    };
    rg_inverse<N, G, NT, LP, true>(buf, stw, ld, st);
}

}  // namespace dnsp
