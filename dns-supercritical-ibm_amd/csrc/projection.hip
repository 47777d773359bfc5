// Projection stencils around the Poisson solve (FP64, gfx950): halos and
// wall planes, the Poisson right-hand side, the rho_min reduction and the
// gradient correction, on the reference's halo arrays.
//
// Halo arrays are the reference's (-1:nx, -1:nz, -1:ny) fields, x fastest:
// element (i,j,k) at (i+1) + (nx+2)*((j+1) + (nz+2)*(k+1)).  P without halo
// is (0:nx-1, 0:nz-1, 0:ny-1).  Every kernel keeps the reference's
// evaluation order with contraction off, so results are bit-identical to a
// serial FP64 evaluation of the same expressions.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>
#include <vector>

#include "common.h"
#include "halo_set.h"
#include "stencil_grid.h"

namespace dnsp {

struct Halo {
    int nx, nz, ny;
    __host__ __device__ long sx() const { return 1; }
    __host__ __device__ long sz() const { return nx + 2; }
    __host__ __device__ long sy() const { return (long)(nx + 2) * (nz + 2); }
    __host__ __device__ long at(int i, int j, int k) const {
        return (long)(i + 1) + (long)(nx + 2) * ((long)(j + 1) + (long)(nz + 2) * (k + 1));
    }
    __host__ __device__ long total() const { return (long)(nx + 2) * (nz + 2) * (ny + 2); }
};

constexpr int kStencilThreads = 256;

static inline int blocks_for(long n, int t = kStencilThreads) { return (int)((n + t - 1) / t); }

// ---------------------------------------------------------------------------
// halos and wall planes
// ---------------------------------------------------------------------------

// Periodic x and z halos over the whole padded array (every k, ghosts
// included): the one-rank effect of the x pass followed by the z pass, i.e.
// A(i,j,k) = A(wrap(i), wrap(j), k) on the halo shell.
__global__ void k_halo_xz(double* A, Halo h) {
    const long per_plane = 2L * (h.nz + 2) + 2L * h.nx;
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= per_plane * (h.ny + 2)) return;
    const int k = (int)(idx / per_plane) - 1;
    const long s = idx % per_plane;
    int i, j;
    if (s < 2L * (h.nz + 2)) {
        i = (s < h.nz + 2) ? -1 : h.nx;
        j = (int)(s % (h.nz + 2)) - 1;
    } else {
        const long t = s - 2L * (h.nz + 2);
        i = (int)(t % h.nx);
        j = (t < h.nx) ? -1 : h.nz;
    }
    const int wi = i < 0 ? h.nx - 1 : (i >= h.nx ? 0 : i);
    const int wj = j < 0 ? h.nz - 1 : (j >= h.nz ? 0 : j);
    A[h.at(i, j, k)] = A[h.at(wi, wj, k)];
}

// set_val_slice: padded planes kp0..kp1 (0 = the k = -1 ghost) set to val
__global__ void k_set_planes(double* A, long plane_elems, long first, long count, double val) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < count) A[first * plane_elems + idx] = val;
}

// Neumann ghosts in y: A(:,:,-1) = A(:,:,0), A(:,:,ny) = A(:,:,ny-1) over the padded plane
__global__ void k_neumann_y(double* A, Halo h) {
    const long pe = h.sy();
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= 2 * pe) return;
    if (idx < pe) A[idx] = A[pe + idx];
    else A[(long)(h.ny + 1) * pe + (idx - pe)] = A[(long)h.ny * pe + (idx - pe)];
}

// ---------------------------------------------------------------------------
// Poisson right-hand side (mod_cfd_subroutines.f90:527-574)
// ---------------------------------------------------------------------------

__global__ void k_rhs_incomp(double* P, const double* __restrict__ Uh, const double* __restrict__ Wh,
                             const double* __restrict__ Vh, const double* __restrict__ inv_dy_p, Halo h,
                             BandGrid bg, double inv_dtmax, double inv_dx, double inv_dz) {
#pragma clang fp contract(off)
    int i, j, k;
    if (!band_point(bg, i, j, k)) return;
    const long idx = (long)i + (long)h.nx * ((long)j + (long)h.nz * k);
    const long c = h.at(i, j, k);
    P[idx] = inv_dtmax * (((Uh[c + 1] - Uh[c]) * inv_dx + (Wh[c + h.sz()] - Wh[c]) * inv_dz) +
                          (Vh[c + h.sy()] - Vh[c]) * inv_dy_p[k]);
}

__device__ __forceinline__ double rfac(double rho_min, double nb, double rc) {
#pragma clang fp contract(off)
    return 1.0 - rho_min * (0.5 / nb + 0.5 / rc);
}

// Variable-density right-hand side.  P_now, P_old and rho are read at seven
// points each, so they are staged in LDS: a workgroup owns a 64 x 4 (i, j)
// tile and marches through a run of planes, keeping planes k-1, k,
// k+1 of the three fields (tile plus one halo point in x and z) in a ring of
// LDS slots and loading one new plane per step (issued before the
// step's arithmetic), so each of their values is read about once instead
// of by every neighbouring thread (0.36 -> 0.28 ms at 384x256x192; the
// per-thread version made 6.3 L1 requests per point).
__global__ __launch_bounds__(kTileX * kTileZ) void k_rhs_varprop(
    double* P, const double* __restrict__ Uh, const double* __restrict__ Wh, const double* __restrict__ Vh,
    const double* __restrict__ Pn, const double* __restrict__ Po, const double* __restrict__ rho,
    const double* __restrict__ div_now, const double* __restrict__ inv_dy_p, const double* __restrict__ inv_dy_p_pad,
    const double* __restrict__ rho_min_p, Halo h, BandGrid bg, double inv_dtmax, double inv_dx, double inv_dz,
    double inv_dx2, double inv_dz2) {
#pragma clang fp contract(off)
    __shared__ double sF[3][kRingSlots][kRingP];  // P_now, P_old, rho
    int i0, j0, k0, k1;
    if (!ring_tile(bg, h.ny, i0, j0, k0, k1)) return;
    const double* fields[3] = {Pn, Po, rho};
    PlaneRing<3> ring(sF, fields, i0, j0, h.nx, h.nz);
    ring.prime(k0);
    // lanes past the last column repeat its point (same loads, same stores)
    const int row = tile_row(), j = j0 + row;
    if (j >= h.nz) {
        ring.stage(k0, k1);
        return;
    }
    const int i = min(i0 + (int)threadIdx.x, h.nx - 1);
    const int e0 = (row + 1) * kRingX + (i - i0) + 1;
    const long sz = h.sz(), sy = h.sy();
    // the point's velocities and div_now, loaded a plane ahead; V_hat(k + 1) is
    // the next step's V_hat(k)
    struct Ahead {
        double u, ux, w, wz, vy, d;
    };
    auto ahead = [&](int k) {
        const long c = h.at(i, j, k);
        return Ahead{Uh[c], Uh[c + 1], Wh[c], Wh[c + sz], Vh[c + sy], div_now[c]};
    };
    double v = Vh[h.at(i, j, k0)];
    Ahead nxt = ahead(k0);
    const double rho_min = *rho_min_p;
    for (int k = k0; k < k1; ++k) {
        ring.put(k + 1);
        const Ahead a = nxt;
        __syncthreads();
        // in flight during this step's arithmetic
        ring.fetch(min(k + 2, k1));
        nxt = ahead(min(k + 1, k1 - 1));
        const int sm = ring_slot(k - 1), s0 = ring_slot(k), sp = ring_slot(k + 1);
        auto ps = [&](int slot, int e) { return 2 * sF[0][slot][e] - sF[1][slot][e]; };
        auto rh = [&](int slot, int e) { return sF[2][slot][e]; };
        const double Ps_00 = ps(s0, e0);
        const double Ps_xp = ps(s0, e0 + 1), Ps_xm = ps(s0, e0 - 1);
        const double Ps_zp = ps(s0, e0 + kRingX), Ps_zm = ps(s0, e0 - kRingX);
        const double Ps_yp = ps(sp, e0), Ps_ym = ps(sm, e0);
        const double rc = rh(s0, e0);
        const double rho_xp = rfac(rho_min, rh(s0, e0 + 1), rc), rho_xm = rfac(rho_min, rh(s0, e0 - 1), rc);
        const double rho_zp = rfac(rho_min, rh(s0, e0 + kRingX), rc);
        const double rho_zm = rfac(rho_min, rh(s0, e0 - kRingX), rc);
        const double rho_yp = rfac(rho_min, rh(sp, e0), rc), rho_ym = rfac(rho_min, rh(sm, e0), rc);
        const double idy = uniform_load(inv_dy_p, k);
        const double t1 =
            inv_dtmax * (((a.ux - a.u) * inv_dx + (a.wz - a.w) * inv_dz) + (a.vy - v) * idy) * rho_min;
        const double t2 = inv_dtmax * rho_min * a.d;
        const double t3 = ((rho_xp * (Ps_xp - Ps_00) - rho_xm * (Ps_00 - Ps_xm)) * inv_dx2 +
                           (rho_zp * (Ps_zp - Ps_00) - rho_zm * (Ps_00 - Ps_zm)) * inv_dz2) +
                          (rho_yp * (Ps_yp - Ps_00) * uniform_load(inv_dy_p_pad, k + 1) -
                           rho_ym * (Ps_00 - Ps_ym) * uniform_load(inv_dy_p_pad, k)) * idy;
        P[(long)i + (long)h.nx * ((long)j + (long)h.nz * k)] = (t1 - t2) + t3;
        v = a.vy;
    }
}

// ---------------------------------------------------------------------------
// rho_min over the interior (mod_cfd_subroutines.f90:470-499): an ordered
// 64-bit key per double so a global atomicMin gives the minimum.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long dkey(double v) {
    unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double dunkey(unsigned long long k) {
    unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)b);
}

__global__ void k_min_init(double* out) {
    if (threadIdx.x == 0 && blockIdx.x == 0)
        *reinterpret_cast<unsigned long long*>(out) = 0xffffffffffffffffull;
}

// Minimum key of this thread's share of the interior: the grid strides over the
// padded planes 0..ny-1 (workgroups side by side on adjacent memory), kMinLoads
// coalesced loads in flight per thread; halo points are masked by their row
// and column, which advance by additions (one division per thread and stride,
// none per point).
constexpr int kMinLoads = 8;
__device__ __forceinline__ unsigned long long min_key_range(const double* __restrict__ A, const Halo& h) {
    const unsigned px = (unsigned)h.nx + 2, pz = (unsigned)h.nz + 2;
    const long n = (long)h.ny * h.sy();  // plane 0 starts at element sy
    constexpr int per = kMinLoads * kStencilThreads;
    const double* src = A + h.sy();
    // column and row advance of one load, and of the rest of a grid stride
    const unsigned dr = kStencilThreads / px, dc = kStencilThreads - dr * px, drz = dr % pz;
    const unsigned skip = (gridDim.x - 1) * (unsigned)per, sr = skip / px, sc = skip - sr * px, srz = sr % pz;
    long e = (long)blockIdx.x * per + (long)threadIdx.x;
    const long row = e / px;
    unsigned c = (unsigned)(e - row * px), r = (unsigned)(row % pz);
    auto advance = [&](unsigned ac, unsigned ar) {
        c += ac;
        r += ar;
        if (c >= px) {
            c -= px;
            ++r;
        }
        r = r >= pz ? r - pz : r;
    };
    unsigned long long best = 0xffffffffffffffffull;
    for (; e < n; e += (long)gridDim.x * per) {
        double v[kMinLoads];
#pragma unroll
        for (int u = 0; u < kMinLoads; ++u) {
            const long at = e + (long)u * kStencilThreads;
            v[u] = src[at < n ? at : e];
        }
#pragma unroll
        for (int u = 0; u < kMinLoads; ++u) {
            const bool in = e + (long)u * kStencilThreads < n && c >= 1 && c <= (unsigned)h.nx && r >= 1 &&
                            r <= (unsigned)h.nz;
            const unsigned long long key = dkey(v[u]);
            best = in && key < best ? key : best;
            advance(dc, drz);
        }
        advance(sc, srz);
    }
    return best;
}

// Minimum over the workgroup, in thread 0.
__device__ __forceinline__ unsigned long long min_key_block(unsigned long long best, unsigned long long* red) {
    red[threadIdx.x] = best;
    __syncthreads();
    for (int s = kStencilThreads / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s && red[threadIdx.x + s] < red[threadIdx.x]) red[threadIdx.x] = red[threadIdx.x + s];
        __syncthreads();
    }
    return red[0];
}

__global__ __launch_bounds__(kStencilThreads) void k_min_interior(const double* __restrict__ A, Halo h, double* out) {
    __shared__ unsigned long long red[kStencilThreads];
    const unsigned long long m = min_key_block(min_key_range(A, h), red);
    if (threadIdx.x == 0) atomicMin(reinterpret_cast<unsigned long long*>(out), m);
}

// The same with one key per workgroup in part, then one workgroup over them.
__global__ __launch_bounds__(kStencilThreads) void k_min_partial(const double* __restrict__ A, Halo h,
                                                                 unsigned long long* __restrict__ part) {
    __shared__ unsigned long long red[kStencilThreads];
    const unsigned long long m = min_key_block(min_key_range(A, h), red);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}
__global__ __launch_bounds__(kStencilThreads) void k_min_final(const unsigned long long* __restrict__ part, int n,
                                                               double* out) {
    __shared__ unsigned long long red[kStencilThreads];
    unsigned long long best = 0xffffffffffffffffull;
    for (int i = (int)threadIdx.x; i < n; i += kStencilThreads) best = part[i] < best ? part[i] : best;
    const unsigned long long m = min_key_block(best, red);
    if (threadIdx.x == 0) *out = dunkey(m);
}

__global__ void k_min_decode(double* out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *out = dunkey(*reinterpret_cast<unsigned long long*>(out));
}

// ---------------------------------------------------------------------------
// gradient correction (mod_cfd_subroutines.f90:1087-1216)
// P_per is the periodic/Neumann extension of P: P_per(i,j,k) = P(wrap i, wrap j, clamp k).
// ---------------------------------------------------------------------------
__device__ __forceinline__ long pidx(const Halo& h, int i, int j, int k) {
    i = i < 0 ? h.nx - 1 : (i >= h.nx ? 0 : i);
    j = j < 0 ? h.nz - 1 : (j >= h.nz ? 0 : j);
    k = k < 0 ? 0 : (k >= h.ny ? h.ny - 1 : k);
    return (long)i + (long)h.nx * ((long)j + (long)h.nz * k);
}

__global__ void k_update_incomp(const double* __restrict__ P, double* U, double* V, double* W,
                                const double* __restrict__ Uh, const double* __restrict__ Vh,
                                const double* __restrict__ Wh, const double* __restrict__ hi,
                                const double* __restrict__ lo, Halo h, BandGrid bg, int kmin_Vhat, double dtmax,
                                double inv_dx, double inv_dz) {
#pragma clang fp contract(off)
    int i, j, k;
    if (!band_point(bg, i, j, k)) return;
    const long idx = (long)i + (long)h.nx * ((long)j + (long)h.nz * k);
    const long c = h.at(i, j, k);
    const double p = P[idx];
    U[c] = Uh[c] - dtmax * (p - P[pidx(h, i - 1, j, k)]) * inv_dx;
    W[c] = Wh[c] - dtmax * (p - P[pidx(h, i, j - 1, k)]) * inv_dz;
    if (k >= kmin_Vhat) V[c] = Vh[c] - dtmax * (hi[k] * p + lo[k] * P[pidx(h, i, j, k - 1)]);
}

__global__ void k_update_varprop(const double* __restrict__ P, double* U, double* V, double* W,
                                 const double* __restrict__ Uh, const double* __restrict__ Vh,
                                 const double* __restrict__ Wh, const double* __restrict__ Pn,
                                 const double* __restrict__ Po, const double* __restrict__ rho,
                                 const double* __restrict__ hi, const double* __restrict__ lo,
                                 const double* __restrict__ rho_min_p, Halo h, BandGrid bg, int kmin_Vhat,
                                 double dtmax, double inv_dx, double inv_dz) {
#pragma clang fp contract(off)
    int i, j, k;
    if (!band_point(bg, i, j, k)) return;
    const long idx = (long)i + (long)h.nx * ((long)j + (long)h.nz * k);
    const long c = h.at(i, j, k);
    const double inv_rho_min = 1.0 / *rho_min_p;
    const double p = P[idx];
    const double ps_c = 2 * Pn[c] - Po[c];
    const double rc = rho[c];
    auto flux = [&](long cb, double pb) {
        const double inv_rho_now = 0.5 / rc + 0.5 / rho[cb];
        const double P_fwd = p * inv_rho_min + (inv_rho_now - inv_rho_min) * ps_c;
        const double P_bwd = pb * inv_rho_min + (inv_rho_now - inv_rho_min) * (2 * Pn[cb] - Po[cb]);
        return make_double2(P_fwd, P_bwd);
    };
    double2 f = flux(c - 1, P[pidx(h, i - 1, j, k)]);
    U[c] = Uh[c] - dtmax * (f.x - f.y) * inv_dx;
    f = flux(c - h.sz(), P[pidx(h, i, j - 1, k)]);
    W[c] = Wh[c] - dtmax * (f.x - f.y) * inv_dz;
    if (k >= kmin_Vhat) {
        f = flux(c - h.sy(), P[pidx(h, i, j, k - 1)]);
        V[c] = Vh[c] - dtmax * (hi[k] * f.x + lo[k] * f.y);
    }
}

// The variable-density correction reads P, P_now, P_old and rho at the point and
// at (-1, 0, 0), (0, -1, 0), (0, 0, -1).  A workgroup owns a 64 x 4 tile and
// marches through a run of planes: a thread loads its own point's values a plane
// ahead, keeps those of the plane below in registers and hands them to its x
// and z neighbours through LDS (two slots, one barrier a plane); wave w loads
// the halo row j0 - 1 of field w and every wave the four fields of its row's
// x - 1 point.  That is 12 vector memory instructions a point against 22 when
// every thread read its neighbours itself, which kept the address units 85% busy:
// at 384x192x256 345 -> 327 us (5.3 TB/s over 67 + 25 B/pt).  On grids that get
// shorter runs than 16 planes a point per thread is faster, whose loads are all in
// flight at once (96x48x65: 7.9 against 9.0 us).
// Loads are unconditional, as PlaneRing's.
__global__ __launch_bounds__(kTileX * kTileZ) void k_update_varprop_march(
    const double* __restrict__ P, double* U, double* V, double* W, const double* Uh, const double* Vh,
    const double* Wh, const double* __restrict__ Pn, const double* __restrict__ Po, const double* __restrict__ rho,
    const double* __restrict__ hi, const double* __restrict__ lo, const double* __restrict__ rho_min_p, Halo h,
    BandGrid bg, int kmin_Vhat, double dtmax, double inv_dx, double inv_dz) {
#pragma clang fp contract(off)
    constexpr int X = kTileX + 1;  // point (i, j) of the tile at (j + 1) * X + i + 1
    __shared__ double sF[4][2][X * (kTileZ + 1)];
    int i0, j0, k0, k1;
    if (!ring_tile(bg, h.ny, i0, j0, k0, k1)) return;
    const long sy = h.sy(), sp = (long)h.nx * h.nz;
    const int row = tile_row(), j = j0 + row;
    // lanes past the last column repeat its point (same loads, same stores)
    const int i = min(i0 + (int)threadIdx.x, h.nx - 1);
    const int x = i - i0 + 1;
    // field q at (ii, jj) and a plane apart; P has no halo and wraps
    auto column = [&](int q, int ii, int jj) -> const double* {
        return q == 0 ? P + pidx(h, ii, jj, 0) : (q == 1 ? Pn : (q == 2 ? Po : rho)) + h.at(ii, jj, 0);
    };
    const double* zrow = column(row, i, j0 - 1);
    const long zs = row == 0 ? sp : sy;
    if (j >= h.nz) {  // a wave without a row: the halo row of its field
        for (int k = k0; k < k1; ++k) {
            sF[row][k & 1][x] = zrow[k * zs];
            __syncthreads();
        }
        return;
    }
    const int xq = min((int)threadIdx.x, 3);
    const double* xcol = column(xq, i0 - 1, j);
    const long xs = xq == 0 ? sp : sy;
    struct Ahead {
        double f[4], z, x, u, v, w;
    };
    auto load = [&](int k) {
        const long c = h.at(i, j, k);
        return Ahead{{P[pidx(h, i, j, k)], Pn[c], Po[c], rho[c]}, zrow[k * zs], xcol[k * xs], Uh[c], Vh[c], Wh[c]};
    };
    const double inv_rho_min = 1.0 / uniform_load(rho_min_p, 0);
    // the plane below
    const long cm = h.at(i, j, k0 - 1);
    double pm = P[pidx(h, i, j, k0 - 1)], psm = 2 * Pn[cm] - Po[cm], rm = rho[cm];
    Ahead buf[2];
    buf[0] = load(k0);
    auto step = [&](auto B, int k) {
#pragma clang fp contract(off)
        const Ahead& a = buf[B];
        const int slot = k & 1, e = (row + 1) * X + x;
#pragma unroll
        for (int q = 0; q < 4; ++q) sF[q][slot][e] = a.f[q];
        sF[row][slot][x] = a.z;
        sF[xq][slot][(row + 1) * X] = a.x;
        __syncthreads();
        buf[B ^ 1] = load(min(k + 1, k1 - 1));
        const double p = a.f[0], ps_c = 2 * a.f[1] - a.f[2], rc = a.f[3];
        auto flux = [&](double pb, double ps_b, double rb) {
            const double inv_rho_now = 0.5 / rc + 0.5 / rb;
            const double P_fwd = p * inv_rho_min + (inv_rho_now - inv_rho_min) * ps_c;
            const double P_bwd = pb * inv_rho_min + (inv_rho_now - inv_rho_min) * ps_b;
            return make_double2(P_fwd, P_bwd);
        };
        auto at = [&](int n) { return flux(sF[0][slot][n], 2 * sF[1][slot][n] - sF[2][slot][n], sF[3][slot][n]); };
        const long c = h.at(i, j, k);
        double2 f = at(e - 1);
        U[c] = a.u - dtmax * (f.x - f.y) * inv_dx;
        f = at(e - X);
        W[c] = a.w - dtmax * (f.x - f.y) * inv_dz;
        f = flux(pm, psm, rm);
        const double v = a.v - dtmax * (uniform_load(hi, k) * f.x + uniform_load(lo, k) * f.y);
        if (k >= kmin_Vhat) V[c] = v;
        pm = p;
        psm = ps_c;
        rm = rc;
    };
    for (int k = k0;;) {
        step(std::integral_constant<int, 0>(), k);
        if (++k >= k1) break;
        step(std::integral_constant<int, 1>(), k);
        if (++k >= k1) break;
    }
}

// P_per over the whole padded array, and (varprop) P_old <- P_now, P_now <- P_per
// One thread per padded point, x fastest (a pure stream: no tiles, so no
// idle lanes on the nx + 2 wide rows); IDX32: the padded array has fewer
// than 2^31 points (32-bit index split).
template <bool IDX32>
__global__ void k_pper_rotate(const double* __restrict__ P, double* P_per, double* Pn, double* Po, Halo h,
                              int rotate) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= h.total()) return;
    int i, j, k;
    if constexpr (IDX32) {
        const unsigned px = (unsigned)(h.nx + 2), pe = (unsigned)h.sy(), x = (unsigned)idx;
        const unsigned kp = x / pe, r = x - kp * pe, jp = r / px;
        i = (int)(r - jp * px) - 1;
        j = (int)jp - 1;
        k = (int)kp - 1;
    } else {
        i = (int)(idx % (h.nx + 2)) - 1;
        j = (int)((idx / (h.nx + 2)) % (h.nz + 2)) - 1;
        k = (int)(idx / h.sy()) - 1;
    }
    const double v = P[pidx(h, i, j, k)];
    if (P_per) P_per[idx] = v;
    if (rotate) {
        Po[idx] = Pn[idx];
        Pn[idx] = v;
    }
}

// Columns, periodic halos and wall planes of a HaloSet.  Blocks are numbered per
// field: CB over the columns, ny PB over the halo points of planes 0..ny-1, then
// 3 WB over the wall planes -1, ny and (V) 0; the block's part and plane are
// workgroup-uniform.  Every point has one writer: columns leave the wall
// planes out, and a halo point whose image lies in a column takes the column's
// value instead of reading it.
constexpr int kWallElems = 4 * kStencilThreads;  // wall-plane points per block
struct SetGrid {
    int CB, PB, WB;
    __host__ __device__ int per_field(int ny) const { return CB + ny * PB + 3 * WB; }
};

__global__ __launch_bounds__(kStencilThreads) void k_halo_set(HaloSet s, Halo h, SetGrid sg) {
    const int per = sg.per_field(h.ny);
    const int f = (int)blockIdx.x / per;
    int b = (int)blockIdx.x - f * per;
    double* A = s.A[f];
    const int* bot = s.bot[f];
    const int* top = s.top[f];
    const double wb = s.dw ? s.dw[f] : s.wb[f], wt = s.dw ? s.dw[s.n + f] : s.wt[f];
    const int k0 = f == s.v ? 1 : 0;  // first plane that is not a wall plane
    const int tid = (int)threadIdx.x;
    if (b < sg.CB) {
        const int col = b * kStencilThreads + tid;
        if (bot == nullptr || col >= h.nx * h.nz) return;
        const int j = col / h.nx, i = col - j * h.nx;
        const int cb = bot[col], ct = top[col];
        const int t0 = ct > k0 ? ct : k0;
        double* c = A + h.at(i, j, 0);
        for (int k = k0; k <= cb && k < t0 && k < h.ny; ++k) c[k * h.sy()] = wb;
        for (int k = t0; k < h.ny; ++k) c[k * h.sy()] = wt;
        return;
    }
    b -= sg.CB;
    if (b < h.ny * sg.PB) {
        const int k = b / sg.PB;
        const int e = (b - k * sg.PB) * kStencilThreads + tid;
        const int pz = h.nz + 2;
        if (k < k0 || e >= 2 * pz + 2 * h.nx) return;
        int i, j;
        if (e < 2 * pz) {
            i = e < pz ? -1 : h.nx;
            j = (e < pz ? e : e - pz) - 1;
        } else {
            const int t = e - 2 * pz;
            i = t < h.nx ? t : t - h.nx;
            j = t < h.nx ? -1 : h.nz;
        }
        const int wi = i < 0 ? h.nx - 1 : (i >= h.nx ? 0 : i);
        const int wj = j < 0 ? h.nz - 1 : (j >= h.nz ? 0 : j);
        double v;
        bool column = false;
        if (bot != nullptr) {
            const int col = wi + h.nx * wj;
            const bool up = k >= top[col];
            column = up || k <= bot[col];
            v = up ? wt : wb;
        }
        if (!column) v = A[h.at(wi, wj, k)];
        A[h.at(i, j, k)] = v;
        return;
    }
    b -= h.ny * sg.PB;
    const int w = b / sg.WB;  // 0: plane -1, 1: plane ny, 2: plane 0 (V)
    if (w == 2 && f != s.v) return;
    const int pe = (int)h.sy();
    double* pl = A + (long)(w == 0 ? 0 : (w == 1 ? h.ny + 1 : 1)) * pe;
    const double val = w == 1 ? wt : wb;
    for (int u = 0; u < 4; ++u) {
        const int o = (b - w * sg.WB) * kWallElems + u * kStencilThreads + tid;
        if (o < pe) pl[o] = val;
    }
}

static int launch_halo_set(const HaloSet& s, const Halo& h, hipStream_t st) {
    bool columns = false;
    for (int f = 0; f < s.n; ++f) columns = columns || s.bot[f];
    SetGrid sg;
    sg.CB = columns ? blocks_for((long)h.nx * h.nz) : 0;
    sg.PB = blocks_for(2L * (h.nz + 2) + 2L * h.nx);
    sg.WB = blocks_for(h.sy(), kWallElems);
    k_halo_set<<<s.n * sg.per_field(h.ny), kStencilThreads, 0, st>>>(s, h, sg);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

// Workgroups of the minimum: one range of kMinLoads loads per thread at least,
// at most kMinBlocks (four per CU).
static int min_blocks(const Halo& h) {
    const long n = (long)h.ny * h.sy(), per = (long)kMinLoads * kStencilThreads;
    return (int)std::min((long)kMinBlocks, (n + per - 1) / per);
}

static bool halo_ok(int nx, int nz, int ny) {
    return nx >= 1 && nz >= 1 && ny >= 1 && (double)(nx + 2) * (nz + 2) * (ny + 2) < 4e12;
}

int halo_columns_periodicity(const HaloSet& s, int nx, int nz, int ny, hipStream_t st) {
    return launch_halo_set(s, Halo{nx, nz, ny}, st);
}

int rho_min_scratch(const double* rho, int nx, int nz, int ny, double* out, double* scratch, hipStream_t st) {
    const Halo h{nx, nz, ny};
    const int nb = min_blocks(h);
    auto* part = reinterpret_cast<unsigned long long*>(scratch);
    k_min_partial<<<nb, kStencilThreads, 0, st>>>(rho, h, part);
    k_min_final<<<1, kStencilThreads, 0, st>>>(part, nb, out);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int update_vars_interior(const double* P, double* P_per, double* P_now, double* P_old, double* U, double* V, double* W,
                         const double* U_hat, const double* V_hat, const double* W_hat, const double* rho,
                         const double* hi, const double* lo, const double* rho_min, int nx, int nz, int ny,
                         int kmin_Vhat, double dtmax, double inv_dx, double inv_dz, int use_incompressible,
                         hipStream_t st) {
    const Halo h{nx, nz, ny};
    const BandGrid bg = band_grid(nx, nz, ny), br = ring_grid(nx, nz, ny);
    if (use_incompressible)
        k_update_incomp<<<bg.blocks(), band_block(), 0, st>>>(P, U, V, W, U_hat, V_hat, W_hat, hi, lo, h, bg,
                                                              kmin_Vhat, dtmax, inv_dx, inv_dz);
    else if (br.run == kRunK)
        k_update_varprop_march<<<br.blocks(), band_block(), 0, st>>>(P, U, V, W, U_hat, V_hat, W_hat, P_now, P_old, rho,
                                                                     hi, lo, rho_min, h, br, kmin_Vhat, dtmax, inv_dx,
                                                                     inv_dz);
    else
        k_update_varprop<<<bg.blocks(), band_block(), 0, st>>>(P, U, V, W, U_hat, V_hat, W_hat, P_now, P_old, rho, hi,
                                                               lo, rho_min, h, bg, kmin_Vhat, dtmax, inv_dx, inv_dz);
    DNSP_LAUNCH_CHECK();
    if (P_per || !use_incompressible) {
        auto kr = h.total() < (1L << 31) ? k_pper_rotate<true> : k_pper_rotate<false>;
        kr<<<blocks_for(h.total()), kStencilThreads, 0, st>>>(P, P_per, P_now, P_old, h, use_incompressible ? 0 : 1);
        DNSP_LAUNCH_CHECK();
    }
    return DNSP_OK;
}

}  // namespace dnsp

using namespace dnsp;

extern "C" {

int dnsp_halo_periodic_xz(double* A, int nx, int nz, int ny, void* stream) {
    clear_error();
    DNSP_ARG_CHECK(A && halo_ok(nx, nz, ny), "invalid halo array arguments");
    Halo h{nx, nz, ny};
    const long n = (2L * (nz + 2) + 2L * nx) * (ny + 2);
    k_halo_xz<<<blocks_for(n), kStencilThreads, 0, as_stream(stream)>>>(A, h);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int dnsp_set_val_slice(double* A, int nx, int nz, int ny, int k0, int k1, double val, void* stream) {
    clear_error();
    DNSP_ARG_CHECK(A && halo_ok(nx, nz, ny), "invalid halo array arguments");
    const int n2 = ny + 2;
    if (k0 < 0) k0 += n2;
    if (k1 < 0) k1 += n2;
    DNSP_ARG_CHECK(k0 >= 0 && k0 < n2 && k1 >= 0 && k1 < n2, "plane index out of range");
    const int kmin = k0 < k1 ? k0 : k1, kmax = k0 < k1 ? k1 : k0;
    Halo h{nx, nz, ny};
    const long count = (long)(kmax - kmin + 1) * h.sy();
    k_set_planes<<<blocks_for(count), kStencilThreads, 0, as_stream(stream)>>>(A, h.sy(), kmin, count, val);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int dnsp_neumann_ghosts_y(double* A, int nx, int nz, int ny, void* stream) {
    clear_error();
    DNSP_ARG_CHECK(A && halo_ok(nx, nz, ny), "invalid halo array arguments");
    Halo h{nx, nz, ny};
    k_neumann_y<<<blocks_for(2 * h.sy()), kStencilThreads, 0, as_stream(stream)>>>(A, h);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int dnsp_build_p_rhs(double* P, const double* U_hat, const double* W_hat, const double* V_hat,
                     const double* inv_dy_p, int nx, int nz, int ny, double inv_dtmax, double inv_dx, double inv_dz,
                     void* stream) {
    clear_error();
    DNSP_ARG_CHECK(P && U_hat && W_hat && V_hat && inv_dy_p && halo_ok(nx, nz, ny), "invalid arguments");
    Halo h{nx, nz, ny};
    const BandGrid bg = band_grid(nx, nz, ny);
    k_rhs_incomp<<<bg.blocks(), band_block(), 0, as_stream(stream)>>>(P, U_hat, W_hat, V_hat, inv_dy_p, h, bg,
                                                                      inv_dtmax, inv_dx, inv_dz);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int dnsp_build_p_rhs_varprop(double* P, const double* U_hat, const double* W_hat, const double* V_hat,
                             const double* P_now, const double* P_old, const double* rho, const double* div_now,
                             const double* inv_dy_p, const double* inv_dy_p_pad, const double* rho_min, int nx,
                             int nz, int ny, double inv_dtmax, double inv_dx, double inv_dz, double inv_dx2,
                             double inv_dz2, void* stream) {
    clear_error();
    DNSP_ARG_CHECK(P && U_hat && W_hat && V_hat && P_now && P_old && rho && div_now && inv_dy_p && inv_dy_p_pad &&
                       rho_min && halo_ok(nx, nz, ny),
                   "invalid arguments");
    Halo h{nx, nz, ny};
    const BandGrid bg = ring_grid(nx, nz, ny);
    k_rhs_varprop<<<bg.blocks(), band_block(), 0, as_stream(stream)>>>(
        P, U_hat, W_hat, V_hat, P_now, P_old, rho, div_now, inv_dy_p, inv_dy_p_pad, rho_min, h, bg, inv_dtmax, inv_dx,
        inv_dz, inv_dx2, inv_dz2);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int dnsp_rho_min(const double* rho, int nx, int nz, int ny, double* out, void* stream) {
    clear_error();
    DNSP_ARG_CHECK(rho && out && halo_ok(nx, nz, ny), "invalid arguments");
    Halo h{nx, nz, ny};
    hipStream_t st = as_stream(stream);
    const int nb = min_blocks(h);
    k_min_init<<<1, 1, 0, st>>>(out);
    k_min_interior<<<nb, kStencilThreads, 0, st>>>(rho, h, out);
    k_min_decode<<<1, 1, 0, st>>>(out);
    DNSP_LAUNCH_CHECK();
    return DNSP_OK;
}

int dnsp_update_vars(const double* P, double* P_per, double* P_now, double* P_old, double* U, double* V, double* W,
                     const double* U_hat, const double* V_hat, const double* W_hat, const double* rho,
                     const double* dPdy_ddy_hi, const double* dPdy_ddy_lo, const double* rho_min,
                     const double* wall_bc, int nx, int nz, int ny, int kmin_Vhat, double dtmax, double inv_dx,
                     double inv_dz, int use_incompressible, void* stream) {
    clear_error();
    DNSP_ARG_CHECK(P && U && V && W && U_hat && V_hat && W_hat && dPdy_ddy_hi && dPdy_ddy_lo && wall_bc &&
                       halo_ok(nx, nz, ny),
                   "invalid arguments");
    DNSP_ARG_CHECK(kmin_Vhat >= 0 && kmin_Vhat <= ny, "kmin_Vhat=%d", kmin_Vhat);
    DNSP_ARG_CHECK(use_incompressible || (P_now && P_old && rho && rho_min),
                   "variable-density correction needs P_now, P_old, rho and rho_min");
    const int rc = update_vars_interior(P, P_per, P_now, P_old, U, V, W, U_hat, V_hat, W_hat, rho, dPdy_ddy_hi,
                                        dPdy_ddy_lo, rho_min, nx, nz, ny, kmin_Vhat, dtmax, inv_dx, inv_dz,
                                        use_incompressible, as_stream(stream));
    if (rc) return rc;
    HaloSet hs;
    hs.n = 3;
    hs.v = 1;
    double* const A[3] = {U, V, W};
    for (int f = 0; f < 3; ++f) hs.A[f] = A[f];
    hs.dw = wall_bc;
    return halo_columns_periodicity(hs, nx, nz, ny, as_stream(stream));
}

// calc_bands.py:272-277 and :336-343 (rows 0..ny-1 of dPdy_ddy_lh, as read at
// inc_set_alloc_arrays.f90:51-52).  Host only.
int dnsp_geom_coeffs(int ny, const double* yu, double* inv_dy_p, double* inv_dy_u, double* inv_dy_p_pad,
                     double* dPdy_ddy_lo, double* dPdy_ddy_hi) {
    clear_error();
    DNSP_ARG_CHECK(ny >= 1 && yu, "invalid arguments");
    std::vector<double> yp((size_t)ny), ext((size_t)ny + 2), pad((size_t)ny + 2);
    for (int i = 0; i < ny; ++i) yp[(size_t)i] = (yu[i] + yu[i + 1]) / 2;
    ext[0] = yu[0];
    pad[0] = 2 * yu[0] - yp[0];
    for (int i = 0; i < ny; ++i) ext[(size_t)i + 1] = pad[(size_t)i + 1] = yp[(size_t)i];
    ext[(size_t)ny + 1] = yu[ny];
    pad[(size_t)ny + 1] = 2 * yu[ny] - yp[(size_t)ny - 1];
    for (int i = 0; i < ny; ++i)
        if (inv_dy_p) inv_dy_p[i] = 1. / (yu[i + 1] - yu[i]);
    for (int i = 0; i <= ny; ++i) {
        if (inv_dy_u) inv_dy_u[i] = 1. / (ext[(size_t)i + 1] - ext[(size_t)i]);
        if (inv_dy_p_pad) inv_dy_p_pad[i] = 1. / (pad[(size_t)i + 1] - pad[(size_t)i]);
    }
    for (int i = 0; i < ny; ++i) {
        double lo = 0.0, hi = 0.0;
        if (i != 0) {
            const double dy = yp[(size_t)i] - yp[(size_t)i - 1];
            lo = -1 / dy;
            hi = 1 / dy;
        }
        if (dPdy_ddy_lo) dPdy_ddy_lo[i] = lo;
        if (dPdy_ddy_hi) dPdy_ddy_hi[i] = hi;
    }
    return DNSP_OK;
}

}  // extern "C"
