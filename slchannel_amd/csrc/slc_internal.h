// slc_internal.h -- host-side declarations shared by the library's sources.
#pragma once

#include <hip/hip_runtime.h>

#include "slc_device.h"

namespace slc {

// Poisson coefficient tables (projection.py:47-103, on the fly per mode).
struct PoissonTabs {
    int nx, ny, nz, nky;
    const double* kxsq;   // nx      modified wavenumber squared
    const double* kysq;   // nky
    const double* cl;     // nz      1/(dz_c[k]   dz_f[k])
    const double* cr;     // nz      1/(dz_c[k+1] dz_f[k])
    const double* cs;     // nz      cl + cr
};

// semi-Lagrangian kernels (slc_sl.hip)
// layout 0: ghost-shaped trajectory fields a; 1: packed node buffers.  ncl
// non-null: z clamped and the clamped feet counted.
struct ArrivalTabs;
hipError_t run_departure(const Grid& g, int comp, const ArrivalTabs& A, const double* const a[3],
                         int layout, double dt, double* xd, double* yd, double* zd,
                         unsigned long long* ncl, hipStream_t s);
hipError_t run_gather(const Grid& g, int comp, const double* F, long fsx, long fsy, int fox,
                      int foy, const double* xd, const double* yd, const double* zd, double* out,
                      unsigned long long* ncl, hipStream_t s);
hipError_t run_gather_tiled(const Grid& g, int comp, int shape, const double* F,
                            const double* xd, const double* yd, const double* zd, double* out,
                            unsigned long long* ncl, hipStream_t s);
hipError_t run_locate(const Grid& g, int comp, const double* z, long n, int* exact, int* fast,
                      hipStream_t s);
hipError_t run_stencil(const Grid& g, int comp, const double* xd, const double* yd,
                       const double* zd, int* ix, int* iy, int* k0, unsigned long long* ncl,
                       hipStream_t s);
hipError_t run_advect(const Grid& g, int comp, const TrajVel& V, const double* F, double dt,
                      double* out, unsigned long long* ncl, hipStream_t s);
hipError_t run_bdf1(const Grid& g, int comp, const TrajVel& V, const double* F, double dt,
                    double* out, unsigned long long* ncl, hipStream_t s);
hipError_t run_bdf2(const Grid& g, int comp, int pass, const TrajVel& V, const double* Fn,
                    const double* Fm, double dt, double* out, unsigned long long* ncl,
                    hipStream_t s);

// Per-component arrival table: per arrival z (nzi) 2 * its face cell + (z >=
// the cell's centre split).
struct ArrivalTabs {
    const int* csel;
};

// Whether the tile kernels address this grid's fields in 64 bits with 32-bit
// index products (BIG): a field of 4 GiB or more, or a row, plane or index of
// 2^24 or more.  All other grids take 32-bit byte offsets and 24-bit products.
inline bool big_index(const Grid& g) {
    const double pl = (double)(g.ny + 2) * (g.nz + 2);
    return pl * (g.nx + 2) >= 536870912.0 || pl >= 16777216.0 || g.nx + 2 >= (1 << 24);
}

// Compute units of the current device (cached per device).
int device_cus();

// LDS-tiled step kernels (slc_step.hip) of one component; mode: 0 advect,
// 1 bdf1, 2 far, 3 near, 4 gather (feet given), 5 far + near in one pass (no
// feet arrays)
// Fn32 / Fm32: float copies of F / Fm to gather from (FP32 storage), or null.
// defer (mode 4 only): (tiles of the component) unsigned of device scratch,
// one flag per tile; when given, tiles whose box exceeds the LDS budget are
// gathered by a second pass with a larger budget instead of by direct loads.
hipError_t run_tile_step(const Grid& g, int comp, int mode, const ArrivalTabs& A,
                         const TrajVel& V, const double* F, const double* Fm, const float* Fn32,
                         const float* Fm32, double dt, double* out, double* fx, double* fy,
                         double* fz, unsigned long long* ncl, hipStream_t s,
                         unsigned* defer = nullptr);
// Modes 0, 1 and 5 for the three components in one launch (slc_step3.hip).
hipError_t run_tile_step3(const Grid& g, int mode, const ArrivalTabs A[3], const TrajVel& V,
                          const double* const F[3], const double* const Fm[3],
                          const float* const Fn32[3], const float* const Fm32[3], double dt,
                          double* const out[3], unsigned long long* ncl, hipStream_t s);
// Tiles of the step kernels for component comp (the defer flags' count).
long step_tiles(const Grid& g, int comp);
// Tiles of a component up to which the three components share a launch, which
// saves two launches and drained tails (10-25 us).  BDF2 predictor, one launch
// against three, order 6: 1024 tiles 106 and 121 us, 8192 562 and 587, 12288
// 833 and 858, 27648 1.89 and 1.91 ms, 65536 the same 4.46 ms; order 4: 62 and
// 71 us, 386 and 400, 580 and 598, 1.40 and 1.41 ms, 3.32 ms.  Past the line the
// saving is 3% and falling.
constexpr long kMergeTiles = 8192;
hipError_t run_arrival_tabs(const Grid& g, int comp, int* cell, hipStream_t s);
hipError_t run_ustar(const Grid& g, double* const o[3], const double* const a[3],
                     const double* const b[3], float* const fa[3], float* const fb[3],
                     hipStream_t s);
hipError_t run_to_f32(const Grid& g, float* const o[3], const double* const a[3],
                      hipStream_t s);

// field operators (slc_ops.hip)
hipError_t run_fill_u64(unsigned long long* p, long n, unsigned long long v, hipStream_t s);
hipError_t run_fill_f64(double* p, long n, double v, hipStream_t s);
hipError_t run_bc(const Grid& g, double* u, double* v, double* w, hipStream_t s);
hipError_t run_zfactor(const Grid& g, int comp, double dt, double theta, const double* dz_c,
                       const double* dz_f, double* tab, hipStream_t s);
// Whether run_zsolve takes a column of component comp (nz up to about 6000).
bool zsolve_fits(int comp, int nz);
// src to f: the same array, or another one where theta < 1
hipError_t run_zsolve(const Grid& g, int comp, const double* src, double* f, double dt,
                      double theta, const double* dz_c, const double* dz_f, double* tab,
                      bool refactor, hipStream_t s);
// the three components' z-solves (tab, refactor: per component) in one launch
hipError_t run_zsolve3(const Grid& g, const double* const src[3], double* const f[3], double dt,
                       double theta, const double* dz_c, const double* dz_f,
                       double* const tab[3], const bool refactor[3], hipStream_t s);
// wrap: read no ghost entry (the fields' ghosts need not be filled)
hipError_t run_div_planes(const Grid& g, const double* u, const double* v, const double* w,
                          const double* dz_f, double scale, double* planes, bool wrap,
                          hipStream_t s);
hipError_t run_div_field(const Grid& g, const double* u, const double* v, const double* w,
                         const double* dz_f, double* div, hipStream_t s);
hipError_t run_field_to_planes(const Grid& g, const double* f, double scale, double* planes,
                               hipStream_t s);
hipError_t run_poisson_thomas(const PoissonTabs& t, double* dhat, double* cp, hipStream_t s);
// writes the ghosts of u, v, w and p too
hipError_t run_project_planes(const Grid& g, double* u, double* v, double* w,
                              const double* planes, double inv_n, double dt,
                              const double* dz_c, double* p, hipStream_t s);
hipError_t run_project_p(const Grid& g, double* u, double* v, double* w, const double* p,
                         double dt, const double* dz_c, hipStream_t s);
// Doubles of scratch of the bulk constraint over np partial sums: the sums
// before and after the shift, and the ticket of the blocks that have finished.
constexpr int bulk_scratch(int np) { return 2 * np + 1; }
// partials: bulk_scratch(bulk_partials_needed(g)) doubles; scal: [0] correction,
// [1] forcing, [2] mean after the shift, [3] before it
hipError_t run_bulk(const Grid& g, double* u, const double* cv, double total_volume,
                    double U_bulk, double dt, double* partials, double* scal, hipStream_t s);
// the mean to out[3]
hipError_t run_bulk_velocity(const Grid& g, const double* u, const double* cv,
                             double total_volume, double* partials, double* out, hipStream_t s);
hipError_t run_axpby(double* out, const double* a, const double* b, double alpha, double beta,
                     long n, hipStream_t s);
int bulk_partials_needed(const Grid& g);

}  // namespace slc
