// slc_ens_kernels.hip -- batched persistent kernels of the ensemble step.
//
// Each kernel walks the concatenated work units of one kind (slc_ens.h) in
// contiguous chunks: logical workgroup l (XCD-aware order, so neighbouring
// chunks share an XCD's L2) owns units [l*T/G, (l+1)*T/G) and finds its first
// member by bisection of the prefix table, then steps through members as
// the units cross their boundaries.  The unit bodies are the single-channel
// ones.
#include "slc_ens_dev.h"
#include "slc_ops_dev.h"

namespace slc {


// ---------------------------------------------------------------------------
// ghost fill of V^n
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void ens_bc3_kernel(ENS_PARAMS) {
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        const int set = ens_a(*M.state);
        const unsigned b0 = ublocks(M.nghost[0]), b1 = ublocks(M.nghost[1]);
        int c;
        unsigned lb;
        if (u < b0) { c = 0; lb = u; }
        else if (u < b0 + b1) { c = 1; lb = u - b0; }
        else { c = 2; lb = u - b0 - b1; }
        bc_body(M.g, M.fld[set][c], c, (long)lb * 256 + threadIdx.x);
    });
}

hipError_t run_ens_bc3(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_bc3_kernel, dim3(grid), dim3(256), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// U* (BDF2) or the V^{n-1} copy (BDF1), plus the FP32-storage copies
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void ens_ustar_kernel(ENS_PARAMS) {
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        const int st = *M.state;
        const int a = ens_a(st), b = ens_b(st);
        const Grid& g = M.g;
        const long n[3] = {(long)(g.nx + 1) * (g.ny + 2) * (g.nz + 2),
                           (long)(g.nx + 2) * (g.ny + 1) * (g.nz + 2),
                           (long)(g.nx + 2) * (g.ny + 2) * (g.nz + 1)};
        const long i = (long)u * 256 + threadIdx.x;
        const bool f32 = M.f32n[0] != nullptr;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (i >= n[c]) continue;
            const double va = M.fld[a][c][i];
            if (ens_bdf2(st)) {
                const double vb = M.fld[b][c][i];
                M.us[c][i] = 2.0 * va - vb;
                if (f32) {
                    M.f32n[c][i] = (float)va;
                    M.f32m[c][i] = (float)vb;
                }
            } else {
                M.fld[b][c][i] = va;
                if (f32) M.f32n[c][i] = (float)va;
            }
        }
    });
}

hipError_t run_ens_ustar(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_ustar_kernel, dim3(grid), dim3(256), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// SL tiles (slc_ens_tile.h, instantiated per storage type and order in
// slc_ens_tile_{d4,d6,f4,f6}.hip so they compile in parallel)
// ---------------------------------------------------------------------------

hipError_t run_ens_tile(const EnsMember* mem, const EnsTiles& t, int pass, int order, int f32,
                        int shape, hipStream_t s) {
    if (t.n[0] + t.n[1] + t.n[2] == 0) return hipSuccess;
    if (f32) {
        if (order == 4) run_ens_tile_f4(mem, t, pass, shape, s);
        else run_ens_tile_f6(mem, t, pass, shape, s);
    } else {
        if (order == 4) run_ens_tile_d4(mem, t, pass, shape, s);
        else run_ens_tile_d6(mem, t, pass, shape, s);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// implicit z-diffusion (theta = 1) of the predictor, BDF1 or BDF2 factor
// ---------------------------------------------------------------------------

// One kernel per longest column of the ensemble, so that its registers (and
// the wavefronts that they leave) are those of the columns it solves: at most
// 2 unknowns per lane, at most 4 or 8, or any (MAXCH 0: the LDS path as well).
// The three components in one launch (workgroups of u, then v, then w): a
// component's columns of small members are one generation of workgroups.
template <int C, int MAXCH>
__device__ inline void ens_zsolve_units(const EnsMember* __restrict__ mem, const EnsColumns& z,
                                        int nmem, unsigned blk, double* lds, long* cbase) {
    ens_for(z.start[C], nmem, z.n[C], blk, z.grid[C], [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        const int st = *M.state;
        const int nz = M.g.nz;
        const double* tab = M.ztab + (ens_bdf2(st) ? 9 : 0) * (long)(nz + 2) + C * 3L * (nz + 2);
        if (MAXCH > 0 || M.zch[C] > 0) {
            const unsigned col0 = u * kEnsZCols, ncols = (unsigned)(M.g.nx * M.g.ny);
            zsolve_run_any<C, (MAXCH > 0 ? MAXCH : kZScanMaxCh)>(
                M.g, M.fld[ens_c(st)][C], tab, col0 + (threadIdx.x >> 6), kZScanCols,
                min(col0 + kEnsZCols, ncols), M.zch[C]);
        } else {
            double* f = M.fld[ens_c(st)][C];
            zsolve_body<C>(M.g, f, f, tab, 0.0, M.dzc, M.dzf, M.zcols[C], u, lds, cbase);
        }
    });
}

template <int MAXCH>
__global__ __launch_bounds__(256, MAXCH == 2 ? 5 : MAXCH == 4 ? 4 : MAXCH == 8 ? 2 : 1)
void ens_zsolve_kernel(const EnsMember* __restrict__ mem, EnsColumns z, int nmem) {
    extern __shared__ double lds[];
    __shared__ long cbase[kZColsMax];
    const unsigned b = blockIdx.x;
    if (b < z.grid[0])
        ens_zsolve_units<0, MAXCH>(mem, z, nmem, b, lds, cbase);
    else if (b < z.grid[0] + z.grid[1])
        ens_zsolve_units<1, MAXCH>(mem, z, nmem, b - z.grid[0], lds, cbase);
    else
        ens_zsolve_units<2, MAXCH>(mem, z, nmem, b - z.grid[0] - z.grid[1], lds, cbase);
}

hipError_t run_ens_zsolve(const EnsMember* mem, int nmem, const EnsColumns& z, size_t lds_bytes,
                          int max_ch, hipStream_t s) {
    if (z.n[0] + z.n[1] + z.n[2] == 0) return hipSuccess;
    const dim3 grid(z.grid[0] + z.grid[1] + z.grid[2]);
#define SLC_ENS_ZS(MAXCH) \
    hipLaunchKernelGGL(ens_zsolve_kernel<MAXCH>, grid, dim3(256), lds_bytes, s, mem, z, nmem)
    if (max_ch == 2) SLC_ENS_ZS(2);
    else if (max_ch == 4) SLC_ENS_ZS(4);
    else if (max_ch == 8) SLC_ENS_ZS(8);
    else SLC_ENS_ZS(0);
#undef SLC_ENS_ZS
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// projection: divergence -> planes, Thomas, gradient update with the ghosts
// ---------------------------------------------------------------------------

__device__ inline double ens_dt_eff(const EnsMember& M, int st) {
    return ens_bdf2(st) ? (2.0 / 3.0) * M.dt : M.dt;
}

__global__ __launch_bounds__(256) void ens_div_planes_kernel(ENS_PARAMS) {
    __shared__ double tile[kT][kT + 1];
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        const int st = *M.state;
        const int c = ens_c(st);
        int i, j0, k0;
        plane_tile(M.g, u, i, j0, k0);
        div_planes_body<true>(M.g, M.fld[c][0], M.fld[c][1], M.fld[c][2], M.dzf, ens_dt_eff(M, st),
                              M.planes, i, j0, k0, tile);
    });
}

hipError_t run_ens_div_planes(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_div_planes_kernel, dim3(grid), dim3(256), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

// one unit = one block of the single-run solve (the partition solve of
// spike_modes(nz) modes, or 256 modes of the sequential sweep), so members
// get the single run's doubles
__global__ __launch_bounds__(256) void ens_thomas_kernel(ENS_PARAMS) {
    __shared__ double lds[256 * 8];
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        if (spike_ok(M.pt.nz))
            poisson_spike_body(M.pt, reinterpret_cast<double2*>(M.dhat), (long)u, lds);
        else
            poisson_thomas_body(M.pt, reinterpret_cast<double2*>(M.dhat), M.cpw,
                                (long)u * 256 + threadIdx.x);
    });
}

hipError_t run_ens_thomas(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_thomas_kernel, dim3(grid), dim3(256), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void ens_project_kernel(ENS_PARAMS) {
    __shared__ double t0[kT + 1][kT + 2];
    __shared__ double t1[kT][kT + 1];
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        const int st = *M.state;
        const int c = ens_c(st);
        int i, j0, k0;
        plane_tile(M.g, u, i, j0, k0);
        project_planes_body(M.g, M.fld[c][0], M.fld[c][1], M.fld[c][2], M.planes, M.inv_n,
                            ens_dt_eff(M, st), M.dzc, M.p, i, j0, k0, t0, t1);
    });
}

hipError_t run_ens_project(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_project_kernel, dim3(grid), dim3(256), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// bulk constraint and the end-of-step state advance
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(kRedBlock) void ens_bulk_before_kernel(ENS_PARAMS) {
    __shared__ double red[kRedBlock];
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        bulk_before_body(M.g, M.fld[ens_c(*M.state)][0], M.cv, M.partials, (int)u, M.npart, red);
    });
}

hipError_t run_ens_bulk_before(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_bulk_before_kernel, dim3(grid), dim3(kRedBlock), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

// The member's last block also publishes the step's statistics, clears the
// clamp counter and rotates the buffer sets (its other blocks have read the
// state by then).
__global__ __launch_bounds__(kRedBlock) void ens_bulk_shift_kernel(ENS_PARAMS) {
    __shared__ double red[kRedBlock];
    __shared__ bool last;
    ens_for(start, nmem, total, [&](int m, unsigned u) {
        const EnsMember& M = mem[m];
        const int st = *M.state;
        const bool done =
            bulk_shift_body(M.g, M.fld[ens_c(st)][0], M.cv, M.partials, (int)u, M.npart,
                            M.total_volume, M.U_bulk, M.dt, M.scal, red, &last);
        if (!done || threadIdx.x != 0) return;
        double* S = M.stats;
        S[ES_UBULK] = M.scal[2];
        S[ES_FORCING] = M.scal[1];
        S[ES_NCLAMP] = (double)*M.ncl;
        S[ES_STEPS] = S[ES_STEPS] + 1.0;
        S[ES_UBULK_PRE] = M.scal[3];
        *M.ncl = 0ull;
        *M.state = ens_next(st);
    });
}

hipError_t run_ens_bulk_shift(const EnsLaunch& L, unsigned grid, hipStream_t s) {
    if (L.total == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_bulk_shift_kernel, dim3(grid), dim3(kRedBlock), 0, s, ENS_ARGS(L));
    return hipGetLastError();
}

__global__ void ens_clear_ncl_kernel(const EnsMember* __restrict__ mem, int nmem) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < nmem) *mem[m].ncl = 0ull;
}

hipError_t run_ens_clear_ncl(const EnsLaunch& L, hipStream_t s) {
    if (L.nmem == 0) return hipSuccess;
    hipLaunchKernelGGL(ens_clear_ncl_kernel, dim3((L.nmem + 63) / 64), dim3(64), 0, s, L.mem,
                       L.nmem);
    return hipGetLastError();
}

__global__ void ens_set_int_kernel(int* p, int v) { *p = v; }

hipError_t run_ens_set_int(int* p, int v, hipStream_t s) {
    hipLaunchKernelGGL(ens_set_int_kernel, dim3(1), dim3(1), 0, s, p, v);
    return hipGetLastError();
}

}  // namespace slc
