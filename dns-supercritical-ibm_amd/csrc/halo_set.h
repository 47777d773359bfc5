// Periodic halos, wall planes, rough-wall columns and IBM forcing of the
// velocity (and temperature) fields of one grid, one launch for all fields
// (projection.hip, ibm.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace dnsp {

// Up to four halo fields ((nx+2)(nz+2)(ny+2), x fastest) with their wall
// values; v: the index of V (-1: none), whose bottom wall lies on plane k = 0
// too.  bot / top: column slabs (nx nz ints each) or NULL.
struct HaloSet {
    int n = 0, v = -1;
    double* A[4] = {};
    double wb[4] = {}, wt[4] = {};
    const double* dw = nullptr;  // when set: n bottom and n top values on the device, used instead
    const int* bot[4] = {};
    const int* top[4] = {};
};

// ibm_part_2 where a field has slabs (mod_cfd_ibm.f90:47-141), then
// cfd_periodicity (mod_cfd_subroutines.f90:860-899): periodic x/z halos of
// planes 0..ny-1 and the wall values over the
// whole padded planes -1 and ny (V: 0 too).
int halo_columns_periodicity(const HaloSet& s, int nx, int nz, int ny, hipStream_t st);

// ibm_part_1 (mod_cfd_ibm.f90:10-45): the forcing of every field with a handle
// (h[c] or NULL), then planes -1 and ny of all fields.
int ibm_force_walls(dnsp_ibm* const* h, const HaloSet& s, int nx, int nz, int ny, hipStream_t st);

// Minimum of the interior of rho into *out; scratch: one double per workgroup,
// at most kMinBlocks and never more than nx nz ny.
constexpr int kMinBlocks = 1024;
int rho_min_scratch(const double* rho, int nx, int nz, int ny, double* out, double* scratch, hipStream_t st);

// update_vars without its halos and wall planes.
int update_vars_interior(const double* P, double* P_per, double* P_now, double* P_old, double* U, double* V, double* W,
                         const double* U_hat, const double* V_hat, const double* W_hat, const double* rho,
                         const double* hi, const double* lo, const double* rho_min, int nx, int nz, int ny,
                         int kmin_Vhat, double dtmax, double inv_dx, double inv_dz, int use_incompressible,
                         hipStream_t st);

}  // namespace dnsp
