// Block order of the point-wise and stencil kernels on (nx, nz, ny) grids.
//
// Blocks of 64 x 4 threads cover 64 x 4 (i, j) points of one plane k.  The
// tile rows of a plane are split into bands, one per XCD (each XCD has its
// own L2 and receives every 8th workgroup), and an XCD walks its band plane
// by plane: the blocks it holds at once cover a few consecutive planes of
// one band, so the k +- 1 planes and the halo rows a stencil reads are
// shared in its L2.  Dispatching plane by plane instead spreads each plane's
// tiles over all XCDs (the predictor's momentum kernel then read 177 B/pt
// from beyond L2 against 80 algorithmic).  The point of a block comes from
// a few workgroup-uniform 32-bit divisions, not per-point 64-bit ones.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fft_ct.h"

namespace dnsp {

constexpr int kTileX = 64, kTileZ = 4;

struct BandGrid {
    int nx, nz, nbx, hb, nbands, ny;
    int run = 1;  // planes per workgroup
    __host__ __device__ int per_band() const { return nbx * hb * ny; }
    __host__ __device__ int blocks() const { return per_band() * nbands; }
};

// Grid of nx x nz x ny points (a padded grid passes its padded sizes).
inline BandGrid band_grid(int nx, int nz, int ny) {
    BandGrid b;
    b.nx = nx;
    b.nz = nz;
    b.ny = ny;
    b.nbx = (nx + kTileX - 1) / kTileX;
    const int nbz = (nz + kTileZ - 1) / kTileZ;
    b.hb = (nbz + 7) / 8;
    b.nbands = (nbz + b.hb - 1) / b.hb;
    return b;
}

inline dim3 band_block() { return dim3(kTileX, kTileZ, 1); }

// This workgroup's tile (bx, bz) and plane (or run of planes) k.  Launch:
// band_grid(..).blocks() workgroups of band_block().
__device__ __forceinline__ void band_tile(const BandGrid& b, int& bx, int& bz, int& k) {
    const int L = xcd_tile((int)blockIdx.x, (int)gridDim.x);
    const int band = L / b.per_band();
    const int r = L - band * b.per_band();
    const int tb = b.nbx * b.hb;
    k = r / tb;
    const int t = r - k * tb;
    bz = band * b.hb + t / b.nbx;
    bx = t - (t / b.nbx) * b.nbx;
}

// This thread's point (i, j, k), 0-based; false outside the grid (rows of
// the last band past nz, columns past nx).
__device__ __forceinline__ bool band_point(const BandGrid& b, int& i, int& j, int& k) {
    int bx, bz;
    band_tile(b, bx, bz, k);
    i = bx * kTileX + (int)threadIdx.x;
    j = bz * kTileZ + (int)threadIdx.y;
    return i < b.nx && j < b.nz;
}

// Ring of four planes of NF halo fields in LDS, for a workgroup of
// kTileX x kTileZ threads that owns one (i, j) tile and marches through a run
// of planes in k.  A slot holds one plane of the tile plus one halo point on
// each side in x and z (kRingX x kRingZ values, point (i, j) of the tile at
// (j + 1) * kRingX + i + 1); plane kp (-1..ny) lives in slot kp & 3.
// Each thread stages halo-tile points tid and tid + 256: fetch(kp) loads
// plane kp into registers, put(kp) stores them to the slot, so the loads of
// the next plane can be issued before a step's arithmetic.  Fields are the
// reference's halo arrays ((nx+2)(nz+2)(ny+2), x fastest).
//
// Four slots, so that a step needs one barrier: plane k + 2 goes to the slot
// of plane k - 2, which nobody reads once the barrier of step k - 1 is passed.
//
// No load here is conditional.  Vector memory returns in order and the compiler
// counts what was issued since, over all paths: behind a branch that might skip
// a load it waits for everything outstanding, the step's prefetches and the last
// step's stores included.  Threads past the halo tile and points past the grid's
// halo repeat a valid address instead (and the value stored with it).
constexpr int kRingX = kTileX + 2, kRingZ = kTileZ + 2, kRingP = kRingX * kRingZ;

// Band order over tiles and runs of planes (an XCD walks the tiles of its band
// one run at a time, so neighbouring tiles' halo rows meet in its L2): launch
// ring_grid(nx, nz, ny).blocks() workgroups of band_block().  A run is 16
// planes (it reads two more than it owns) where that leaves kRingBlocks
// workgroups, else shorter: on a small grid a few long runs leave most of the
// chip idle, each waiting for its own loads plane after plane.
// (about three workgroups per CU are resident: 768 at once.  At 96 x 48 x 65 the
// momentum, right-hand side and energy kernels took 45, 20 and 20 us in 120
// workgroups of 16 planes; runs of 2 took the whole time step from 177 to 126
// us.  Bounds of 1024 to 4096 differ by 1%.)
constexpr int kRunK = 16, kRunMin = 2, kRingBlocks = 2048;
inline BandGrid ring_grid(int nx, int nz, int ny) {
    const BandGrid one = band_grid(nx, nz, 1);
    int run = kRunK;
    while (run > kRunMin && (long)one.blocks() * ((ny + run - 1) / run) < kRingBlocks) run /= 2;
    BandGrid b = band_grid(nx, nz, (ny + run - 1) / run);
    b.run = run;
    return b;
}

// This workgroup's tile origin (i0, j0) and planes [k0, k1); false for a
// workgroup past the last band's rows (uniform, before any barrier).
__device__ __forceinline__ bool ring_tile(const BandGrid& b, int ny, int& i0, int& j0, int& k0, int& k1) {
    int bx, bz, run;
    band_tile(b, bx, bz, run);
    i0 = bx * kTileX;
    j0 = bz * kTileZ;
    k0 = run * b.run;
    k1 = k0 + b.run < ny ? k0 + b.run : ny;
    return j0 < b.nz;
}

constexpr int kRingSlots = 4;
__device__ __forceinline__ int ring_slot(int kp) { return kp & (kRingSlots - 1); }

template <int NF>
struct PlaneRing {
    static constexpr int kNT = kTileX * kTileZ;
    static_assert(kRingP <= 2 * kNT, "two staged points per thread");
    double (*lds)[kRingSlots][kRingP];
    const double* f[NF];
    long go[2], sy;
    int le[2];
    double r[NF][2];

    // Tile at (i0, j0) of an nx x nz x ny grid; lds points to NF x 4 slots.
    __device__ __forceinline__ PlaneRing(double (*lds_)[kRingSlots][kRingP], const double* const* fields, int i0,
                                         int j0, int nx, int nz)
        : lds(lds_) {
        for (int q = 0; q < NF; ++q) f[q] = fields[q];
        const int tid = (int)threadIdx.y * kTileX + (int)threadIdx.x;
        const long sz = nx + 2;
        sy = sz * (nz + 2);
        for (int u = 0; u < 2; ++u) {
            const int e = min(tid + u * kNT, kRingP - 1);
            const int rr = e / kRingX, qq = e - rr * kRingX;
            const int gi = min(i0 - 1 + qq, nx), gj = min(j0 - 1 + rr, nz);
            le[u] = e;
            go[u] = (long)(gi + 1) + sz * (long)(gj + 1) + sy;  // plane 0
        }
    }
    __device__ __forceinline__ void fetch(int kp) {
        for (int u = 0; u < 2; ++u)
            for (int q = 0; q < NF; ++q) r[q][u] = f[q][go[u] + (long)kp * sy];
    }
    __device__ __forceinline__ void put(int kp) {
        const int slot = ring_slot(kp);
        for (int u = 0; u < 2; ++u)
            for (int q = 0; q < NF; ++q) lds[q][slot][le[u]] = r[q][u];
    }
    // Planes k0 - 1 and k0 into their slots and k0 + 1 into the registers, the
    // loads of all three in flight together.
    __device__ __forceinline__ void prime(int k0) {
        double a[2][NF][2];
        for (int h = 0; h < 2; ++h)
            for (int u = 0; u < 2; ++u)
                for (int q = 0; q < NF; ++q) a[h][q][u] = f[q][go[u] + (long)(k0 - 1 + h) * sy];
        fetch(k0 + 1);
        for (int h = 0; h < 2; ++h) {
            const int slot = ring_slot(k0 - 1 + h);
            for (int u = 0; u < 2; ++u)
                for (int q = 0; q < NF; ++q) lds[q][slot][le[u]] = a[h][q][u];
        }
    }
    // The march of a wave that owns no row of the grid: it only stages.
    __device__ __forceinline__ void stage(int k0, int k1) {
        for (int k = k0; k < k1; ++k) {
            put(k + 1);
            __syncthreads();
            fetch(min(k + 2, k1));
        }
    }
};

// Store past the caches (NT) or through them.  A kernel that writes several
// fields whose next reader is a whole pass away only evicts with them what
// others will read: at 384x192x256 (155 MB a field), through / past: eight
// streams of a copy 302 / 225 us, the property kernel 352 / 310, momentum 568 /
// 555, and the next kernels gain what stays cached (the minimum of rho 42 / 30).
// Where a kernel's outputs fit the cache they are read back from it: at 96x48x65
// the whole time step takes 120.5 / 124.5.
template <bool NT>
__device__ __forceinline__ void stream_store(double* p, double v) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}
template <bool NT>
__device__ __forceinline__ void stream_store(double2* p, double2 v) {
    if constexpr (NT) {
        typedef double Pair __attribute__((ext_vector_type(2)));
        __builtin_nontemporal_store(Pair{v.x, v.y}, reinterpret_cast<Pair*>(p));
    } else {
        *p = v;
    }
}
// The load of a value that only this thread reads, in the same kernels (at
// 384x192x256: the old R's of momentum 577 / 563 us, divjac of the energy right-hand
// side 184 / 167).
template <bool NT>
__device__ __forceinline__ double stream_load(const double* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
// Whether a kernel that writes nout fields of `points` values stores past the
// caches: more than the 256 MB of the last one.
inline bool streams_past(long points, int nout) { return points * nout * (long)sizeof(double) > (256L << 20); }

// This wave's row of the tile (a wave is one row), as a uniform value.
__device__ __forceinline__ int tile_row() { return __builtin_amdgcn_readfirstlane((int)threadIdx.y); }

// p[i] for a uniform i of data no kernel in flight writes, as a scalar load: a
// vector load would be waited for in order behind the step's prefetches.
__device__ __forceinline__ double uniform_load(const double* p, int i) {
    typedef const double __attribute__((address_space(4))) * ConstPtr;
    return ((ConstPtr)(uintptr_t)p)[i];
}

}  // namespace dnsp
