// Launchers of the compile-time-sized kernels (poisson_ct_x.hip,
// poisson_ct_z.hip, poisson_tri.hip, poisson_mixed_x.hip).  FFT `variant` in
// [0, kCtVariants) selects the (tile, threads) pair of ct_xvar_tile /
// ct_xvar_threads (x) or ct_zvar_tile / ct_zvar_threads (z).
#pragma once

#include <hip/hip_runtime.h>

namespace dnsp {

// The lengths with compile-time-sized kernels.
constexpr bool ct_fft_supported(int n) {
    for (int m : {32, 64, 96, 128, 192, 256, 384, 512, 768})
        if (n == m) return true;
    return false;
}
// at (inverse only; device, NULL: src and dst): the place of the address of the
// array to transform in place, read when the kernel runs (array_at).
void ct_x_launch(int n, int variant, bool inv, const double* src, double* dst, long nlines, const double2* tw,
                 double scale, hipStream_t st, double* const* at = nullptr);
void ct_z_launch(int n, int variant, bool inv, double* S, int nx, int ny, const double2* tw, hipStream_t st);
// The blocked FP64 solve (poisson_ct.h): the x forward transform from lines
// to the x-blocked layout (variants as ct_x_launch); the z transforms from
// x-blocked to mode-major (forward) and from x-blocked to halfcomplex lines
// (inverse), variant 0: 256 threads, 1: 512.  at: the place of the address of
// the caller's array (src of xb_x_launch, dst of mm_z_launch), as ct_x_launch.
void xb_x_launch(int n, int variant, const double* src, double* dst, long nlines, int nz, const double2* tw,
                 hipStream_t st, const double* const* at = nullptr);
void mm_z_launch(int n, int variant, bool inv, const double* src, double* dst, int nx, int ny, const double2* tw,
                 hipStream_t st, double* const* at = nullptr);
// The in-place FP64 transforms of the other lengths 16..768 with prime factors up
// to 13 (poisson_reg.h).
constexpr int kRgMin = 16, kRgMax = 768;
constexpr bool rg_supported(int n) {
    if (n < kRgMin || n > kRgMax || ct_fft_supported(n)) return false;
    for (int p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n == 1;
}
struct RgOps {
    void (*xfwd)(const double* P, double* S, long nlines, const double2* tw, hipStream_t st);
    void (*xbwd)(const double* S, double* P, long nlines, double scale, const double2* tw, hipStream_t st);
    void (*zfwd)(double* S, int nx, int ny, const double2* tw, hipStream_t st);
    void (*zbwd)(double* S, int nx, int ny, const double2* tw, hipStream_t st);
};
const RgOps* rg_ops(int n);  // NULL where not supported
// The x variants the blocked solve starts with (us).  Forward: 1536 complex
// elements a workgroup where the field outgrows the 256 MB cache (768x384x384
// 354 against 368 for 768, 256x256x256 43 against 46), else 768 (512x128x192 35
// against 39).  Inverse: 768 at 384 and 512 points (384x384x256 100 against
// 105), else 1536 (256x256x256 39 against 41, 768x384x384 316 against 321):
// measured by length, without a known cause.
constexpr int blk_xfwd_variant(size_t points) { return points >= ((size_t)1 << 24) ? 2 : 0; }
constexpr int blk_xbwd_variant(int nx) { return nx == 384 || nx == 512 ? 0 : 2; }
constexpr int kBlkZVariant = 1;
// FP32 z transforms; the forward one also turns the FP64 line sums lsum (if
// not NULL) into the FP64 plane sums msum.
void ct_z_launch(int n, int variant, bool inv, float* S, int nx, int ny, const float2* tw, const double* lsum,
                 double* msum, hipStream_t st);

// Partitioned tridiagonal solve, ny <= 32 * kPartChunks.  Variants (P chunks
// per mode of up to 32 rows, M modes per workgroup), FP64 spectra: 0 = P 32, M
// 16, registers capped for 4 resident waves per SIMD; 1 = P 32, M 8; 2 = the
// shape part_shape gives ny, with exactly ceil(ny / P) rows a chunk; 3 = P 16, M
// 16 (ny <= 512, else P 64, M 8); 4, 5, 7 = 0, 1, 3 with two-pass chunks; 6 = 2.
constexpr int kPartChunks = 32;
constexpr int kPartVariants = 8;
// tuner table: first slot of the x, z and tridiagonal variants of one form
constexpr int kTuneSlot[3] = {0, 4, 8};
constexpr int kTuneFormSlots = 16;
int part_rows_for(int ny);  // rows per chunk at kPartChunks chunks (0: ny too large)
// Chunks per mode by ny.  Fewer chunks shorten the reduced system (its
// log2(P) barrier steps, and the serial sweep of the low modes) and move less
// through LDS; more rows a chunk take more registers (about 6 VGPRs a row), hence
// fewer resident waves.  us per launch, one pass, 576 x 288 modes in mode-major
// blocks, by P:
//   ny  33  P 4  17.7  P 8  18.9  P 16 31.0
//   ny  65  P 8  29.2  P 4  29.7  P 16 35.5
//   ny 129  P 16 68.8  P 8  69.5  P 12 70.4
//   ny 280  P 16 146   P 32 150   P 24 183
//   ny 384  P 16 206   P 32 206   P 24 297
//   ny 770  P 32, M 8 477   M 16 555   P 24, M 8 461   P 16 959
// Inside the library, the shape against (32, 16) with its rows rounded up to {2,
// 3, 4, 6, 8, 12, 16, 24, 32}, in place at 576 x 288 modes and in the blocked layouts
// at 768 x 192: ny 33 18 / 67 and 16 / 58, 65 31 / 69 and 28 / 62, 129 57 / 95 and 64 /
// 100, 280 159 / 218 and 138 / 192, 384 236 / 254 and 196 / 227, 512 301 / 314 and
// 242 / 272, 770 584 / 1620 (3.5 TB/s) and 504 / 1403.
// Above 512 rows two workgroups of 16 modes no longer fit a CU's registers, so
// a workgroup holds 8, whose rows are half a cache line.  FP32 spectra take twice
// the modes: 32 make 128-byte rows.
struct PartShape {
    int P, M, MR;
};
constexpr PartShape part_shape(int ny, bool fp32 = false) {
    const int P = ny <= 48 ? 4 : (ny <= 128 ? 8 : (ny <= 512 ? 16 : 32));
    const int mr = (ny + P - 1) / P;
    return {P, (P == 32 ? 8 : 16) * (fp32 ? 2 : 1), mr < 2 ? 2 : mr};
}
// The variant a handle starts with, FP32 or FP64 spectra: part_shape's, one-pass.
// Two passes save registers but solve a chunk's interior again, and were 2-11%
// slower (us, one / two passes; in place at 576 x 288 modes: ny 65 31 / 32, 280 159 /
// 167, 384 236 / 244, 512 301 / 308, 770 584 / 645; blocked at 768 x 192: 65 27.5 / 28.7,
// 129 64 / 63, 280 138 / 143, 384 196 / 213, 512 242 / 254, 770 504 / 561; a whole
// mixed solve of 512x256x256 692 / 702, 384x192x600 1139 / 1215), so the shape has no
// two-pass form and variant 6 runs the same kernels.
constexpr int kPartDefault = 2;
// The group lists of an FP32-spectrum variant (the mixed form launches the
// well-conditioned groups in FP32 arithmetic and the rest in FP64): 0 = groups
// of 8 modes, 1 = of 16, 2 and 3 = 32-mode workgroups whose lists hold pairs of
// 16-mode groups, paired where all 32 modes qualify (2) or 16 by 16 (3).
enum PartList { PL_8 = 0, PL_16 = 1, PL_32 = 2, PL_PAIRS = 3 };
int part_list_kind(int variant, int ny);
// Ar: arithmetic type (double, or float for FP32 spectra); glist (device,
// nlist entries): solve only the listed mode groups (NULL: all of them);
// MM: S in the mode-major blocks of the blocked solve, the solution written
// to So in its x-blocked layout.
// The arguments of a rule-shaped launch (poisson_tri_rule_*.hip).
template <typename T>
struct PartArgs {
    T* S;
    const double *ax, *az, *bands;
    int nx, nz, ny;
    double pcr_min;
    const double* msum;
    double* pbar;
    double inv_nxnz;
    const int* glist;
    int nlist;
    T* So;
    T* const* at = nullptr;  // MM: the place of S's address, as ct_x_launch
};
template <typename T, typename Ar, bool MM>
void part_launch_rule(const PartArgs<T>& a, hipStream_t st);
template <typename T, typename Ar = double, bool MM = false>
void part_launch(int variant, T* S, const double* ax, const double* az, const double* bands, int nx, int nz,
                 int ny, double pcr_min, const double* msum, double* pbar, double inv_nxnz, hipStream_t st,
                 const int* glist = nullptr, int nlist = 0, T* So = nullptr);

// Mixed-precision x kernels (poisson_mixed.h).
enum MxKind { MX_FWD = 0, MX_RES_F32 = 1, MX_RES_F64 = 2, MX_BWD = 3, MX_ACC_F32 = 4, MX_ACC_F64 = 5 };
struct MxArgs {
    const void* src = nullptr;      // f (FWD), iterate p (RES), FP32 spectrum (BWD, ACC)
    const double* f = nullptr;      // RES: right-hand side
    const double* q = nullptr;      // RES: per-plane constants
    const double* bands = nullptr;  // RES: plain a, b, c
    const void* base = nullptr;     // ACC: FP32 field or FP64 iterate (NULL = 0)
    const double* pbar0 = nullptr;  // ACC
    const double* pbar1 = nullptr;  // ACC
    void* dst = nullptr;            // FP32 spectrum (FWD, RES), FP32 field (BWD), FP64 P (ACC)
    double* lsum = nullptr;         // FP64 line sums of the input (FWD), of r (RES), of the output
    int nz = 0, ny = 0;
    double ix2 = 0, iz2 = 0;
    long nlines = 0;
    const float2* tw = nullptr;
    double scale = 1.0;
};
void mx_x_launch(int kind, int n, int variant, const MxArgs& a, hipStream_t st);

}  // namespace dnsp
