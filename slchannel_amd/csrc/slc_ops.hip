// slc_ops.hip -- field operators of the SL-BDF2 step for gfx950:
//   ghost/boundary fill            solver.py:70-107, projection.py:180-195
//   theta-method z-diffusion       operators.py:382-630 (Thomas, shared factor)
//   divergence (+transpose)        utils.py:166-180
//   per-wavenumber Poisson Thomas  projection.py:133-247 (coefficients on the fly)
//   gradient projection            projection.py:250-272
//   bulk-flux constraint           solver.py:694-723, utils.py:147-163
// (device bodies in slc_ops_dev.h)
//
// All of these are HBM-bound (well under one flop per byte); they are written
// for coalesced 64-lane access: z-contiguous fields are read/written along z,
// the spectral data lives plane-major (k, i, j) so rocFFT transforms contiguous
// x-y planes and the Thomas sweep over k reads consecutive modes per lane.
// Every pass is deterministic (fixed partition, fixed reduction trees).
#include "slc_ops_dev.h"

namespace slc {

// ---------------------------------------------------------------------------
// fills (graph-capture friendly replacements for memset)
// ---------------------------------------------------------------------------

__global__ void fill_u64_kernel(unsigned long long* p, long n, unsigned long long v) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void fill_f64_kernel(double* p, long n, double v) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t run_fill_u64(unsigned long long* p, long n, unsigned long long v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_u64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n,
                       v);
    return hipGetLastError();
}

hipError_t run_fill_f64(double* p, long n, double v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(fill_f64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n,
                       v);
    return hipGetLastError();
}

__global__ void axpby_kernel(double* out, const double* a, const double* b, double alpha,
                             double beta, long n) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = alpha * a[i] + beta * b[i];
}

hipError_t run_axpby(double* out, const double* a, const double* b, double alpha, double beta,
                     long n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(axpby_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, out, a, b,
                       alpha, beta, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// ghost fill
// ---------------------------------------------------------------------------

__global__ void bc_kernel(Grid g, double* u, double* v, double* w) {
    const int kind = (int)blockIdx.y;
    double* F = kind == 0 ? u : kind == 1 ? v : w;
    if (!F) return;
    bc_body(g, F, kind, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

hipError_t run_bc(const Grid& g, double* u, double* v, double* w, hipStream_t st) {
    long nmax = 0;
    for (int k = 0; k < 3; ++k) {
        long n = ghost_count(k, g.nx, g.ny, g.nz);
        if (n > nmax) nmax = n;
    }
    hipLaunchKernelGGL(bc_kernel, dim3((unsigned)((nmax + 255) / 256), 3), dim3(256), 0, st, g, u,
                       v, w);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// implicit z-diffusion
// ---------------------------------------------------------------------------
// The shared factorisation is built by one thread (n is at most a few
// thousand).

__global__ void zfactor_kernel(Grid g, int comp, double dt, double theta, const double* dz_c,
                               const double* dz_f, double* tab) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const int nz = g.nz;
    const int n = comp == 2 ? nz - 1 : nz;
    double* A = tab;
    double* CP = tab + n;
    double* INV = tab + 2 * n;
    const double alpha = theta * dt * g.nu;
    double cprev = 0.0;
    for (int k = 0; k < n; ++k) {
        double dzl, dzr, dzc;
        if (comp < 2) { dzl = dz_c[k]; dzr = dz_c[k + 1]; dzc = dz_f[k]; }
        else { dzl = dz_f[k]; dzr = dz_f[k + 1]; dzc = dz_c[k + 1]; }
        double lower = -alpha / (dzl * dzc);
        double center = 1.0 + alpha * (1.0 / dzl + 1.0 / dzr) / dzc;
        double upper = -alpha / (dzr * dzc);
        double a = lower, b = center, c = upper;
        if (k == 0) {
            a = 0.0;
            if (comp < 2) b = center - lower;
        }
        if (k == n - 1) {
            if (comp < 2) b = g.top_neumann ? center + upper : center - upper;
            c = 0.0;
        }
        // (k == 0 and k == n-1 coincide only for n == 1)
        double den = (k == 0) ? b : b - a * cprev;
        double cp = c / den;
        A[k] = a;
        CP[k] = cp;
        INV[k] = 1.0 / den;
        cprev = cp;
    }
}

hipError_t run_zfactor(const Grid& g, int comp, double dt, double theta, const double* dz_c,
                       const double* dz_f, double* tab, hipStream_t s) {
    hipLaunchKernelGGL(zfactor_kernel, dim3(1), dim3(64), 0, s, g, comp, dt, theta, dz_c, dz_f,
                       tab);
    return hipGetLastError();
}

template <int C>
__global__ __launch_bounds__(256) void zsolve_kernel(Grid g, const double* S, double* F,
                                                     const double* __restrict__ tab, double beta,
                                                     const double* __restrict__ dz_c,
                                                     const double* __restrict__ dz_f,
                                                     int kZCols) {
    extern __shared__ double lds[];
    __shared__ long cbase[kZColsMax];
    zsolve_body<C>(g, S, F, tab, beta, dz_c, dz_f, kZCols, blockIdx.x, lds, cbase);
}

// Columns of 8 or more unknowns per lane move through LDS (coalesced), the
// shorter ones straight to the lanes.  Measured: 1024x1024x512 (8 per lane)
// 4.1 -> 2.8 ms per component; 256^3 (4 per lane) 0.0825 -> 0.0845 ms.
#ifndef SLC_ZSCAN_LDS_MIN_CH
#define SLC_ZSCAN_LDS_MIN_CH 8
#endif

// The components' column solves in one launch: nb[c] blocks of component c
// walk its columns with a stride of all its wavefronts.
struct ZSolve3 {
    const double* s[3];
    double* f[3];
    const double* tab[3];
    const double* dz_c;
    const double* dz_f;
    double beta;
    unsigned nb[3];
};

// Wavefronts per SIMD that the columns' registers leave.
constexpr int zwaves(int ch, bool expl) {
    return ch <= 1 ? (expl ? 5 : 8) : ch <= 2 ? (expl ? 4 : 6) : ch <= 4 ? (expl ? 3 : 4)
           : ch <= 8 ? 2 : 1;
}

template <int CHU, int CHW, bool EXPL>
__global__ __launch_bounds__(256, zwaves(CHU, EXPL)) void zsolve3_kernel(Grid g, ZSolve3 a) {
    constexpr bool XU = CHU >= SLC_ZSCAN_LDS_MIN_CH, XW = CHW >= SLC_ZSCAN_LDS_MIN_CH;
    __shared__ double xl[kZScanCols][XU ? zscan_lds<CHU>() : 1];
    unsigned b = blockIdx.x;
    const int c = b < a.nb[0] ? 0 : b < a.nb[0] + a.nb[1] ? 1 : 2;
    if (c > 0) b -= a.nb[0];
    if (c > 1) b -= a.nb[1];
    const unsigned ncols = (unsigned)(g.nx * g.ny);
    const unsigned wave = threadIdx.x >> 6;
    const unsigned col = b * kZScanCols + wave, stride = a.nb[c] * kZScanCols;
    double* xu = XU ? xl[wave] : nullptr;
    double* xw = XW ? xl[wave] : nullptr;
    if (c == 0)
        zsolve_run<0, CHU, EXPL>(g, a.s[0], a.f[0], a.tab[0], col, stride, ncols, a.beta,
                                  a.dz_c, a.dz_f, xu);
    else if (c == 1)
        zsolve_run<1, CHU, EXPL>(g, a.s[1], a.f[1], a.tab[1], col, stride, ncols, a.beta,
                                  a.dz_c, a.dz_f, xu);
    else
        zsolve_run<2, CHW, EXPL>(g, a.s[2], a.f[2], a.tab[2], col, stride, ncols, a.beta,
                                  a.dz_c, a.dz_f, xw);
}

// Arguments of `comps` components in one launch: a block per 4 columns, and
// where those are more than the chip holds at once, as many as it holds.
static ZSolve3 zsolve3(const Grid& g, double beta, const double* dz_c, const double* dz_f,
                       int comps) {
    ZSolve3 a{};
    a.dz_c = dz_c;
    a.dz_f = dz_f;
    a.beta = beta;
    const long ncols = (long)g.nx * g.ny;
    const long most = std::max<long>(
        1, (long)device_cus() * zwaves(zsolve_scan_ch(0, g.nz), beta != 0.0) / comps);
    for (int c = 0; c < 3; ++c)
        a.nb[c] = (unsigned)std::min<long>((ncols + kZScanCols - 1) / kZScanCols, most);
    return a;
}

static hipError_t launch_zsolve3(const Grid& g, const ZSolve3& a, hipStream_t s) {
    const int cu = zsolve_scan_ch(0, g.nz), cw = zsolve_scan_ch(2, g.nz);
    const dim3 grid(a.nb[0] + a.nb[1] + a.nb[2]), blk(256);
    bool expl = a.beta != 0.0;
    for (int c = 0; c < 3; ++c) expl = expl || a.s[c] != a.f[c];
#define SLC_ZS3(CU, CW)                                                              \
    if (expl)                                                                        \
        hipLaunchKernelGGL((zsolve3_kernel<CU, CW, true>), grid, blk, 0, s, g, a);   \
    else                                                                             \
        hipLaunchKernelGGL((zsolve3_kernel<CU, CW, false>), grid, blk, 0, s, g, a)
    // w's columns are one unknown shorter: a class below where u's just
    // spill over
    switch (cu) {
        case 1: SLC_ZS3(1, 1); break;
        case 2: if (cw == 2) { SLC_ZS3(2, 2); } else { SLC_ZS3(2, 1); } break;
        case 4: if (cw == 4) { SLC_ZS3(4, 4); } else { SLC_ZS3(4, 2); } break;
        case 8: if (cw == 8) { SLC_ZS3(8, 8); } else { SLC_ZS3(8, 4); } break;
        case 16: if (cw == 16) { SLC_ZS3(16, 16); } else { SLC_ZS3(16, 8); } break;
        default: SLC_ZS3(16, 16);  // w alone: u's columns are too long
    }
#undef SLC_ZS3
    return hipGetLastError();
}

bool zsolve_fits(int comp, int nz) {
    return zsolve_scan_ch(comp, nz) > 0 || zsolve_cols(comp, nz) > 0;
}

hipError_t run_zsolve(const Grid& g, int comp, const double* src, double* f, double dt,
                      double theta, const double* dz_c, const double* dz_f, double* tab,
                      bool refactor, hipStream_t s) {
    if (refactor)
        hipLaunchKernelGGL(zfactor_kernel, dim3(1), dim3(64), 0, s, g, comp, dt, theta, dz_c,
                           dz_f, tab);
    double beta = theta < 1.0 ? (1.0 - theta) * dt * g.nu : 0.0;
    const int ch = zsolve_scan_ch(comp, g.nz);
    if (ch > 0) {
        ZSolve3 a = zsolve3(g, beta, dz_c, dz_f, 1);
        a.s[comp] = src;
        a.f[comp] = f;
        a.tab[comp] = tab;
        for (int c = 0; c < 3; ++c) a.nb[c] = c == comp ? a.nb[c] : 0u;
        return launch_zsolve3(g, a, s);
    }
    long ncols = (long)g.nx * g.ny;
    const int cols = zsolve_cols(comp, g.nz);
    if (cols < 1) return hipErrorInvalidValue;  // nz beyond ~6000: column does not fit LDS
    dim3 grid((unsigned)((ncols + cols - 1) / cols));
    size_t shm = (size_t)cols * zsolve_ld(comp, g.nz) * sizeof(double);
    if (comp == 0)
        hipLaunchKernelGGL(zsolve_kernel<0>, grid, dim3(256), shm, s, g, src, f, tab, beta, dz_c,
                           dz_f, cols);
    else if (comp == 1)
        hipLaunchKernelGGL(zsolve_kernel<1>, grid, dim3(256), shm, s, g, src, f, tab, beta, dz_c,
                           dz_f, cols);
    else
        hipLaunchKernelGGL(zsolve_kernel<2>, grid, dim3(256), shm, s, g, src, f, tab, beta, dz_c,
                           dz_f, cols);
    return hipGetLastError();
}

// The three components' solves, in one launch where the columns fit the lanes.
hipError_t run_zsolve3(const Grid& g, const double* const src[3], double* const f[3], double dt,
                       double theta, const double* dz_c, const double* dz_f,
                       double* const tab[3], const bool refactor[3], hipStream_t s) {
    if (zsolve_scan_ch(0, g.nz) == 0 || zsolve_scan_ch(2, g.nz) == 0) {
        for (int c = 0; c < 3; ++c) {
            hipError_t e =
                run_zsolve(g, c, src[c], f[c], dt, theta, dz_c, dz_f, tab[c], refactor[c], s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    ZSolve3 a = zsolve3(g, theta < 1.0 ? (1.0 - theta) * dt * g.nu : 0.0, dz_c, dz_f, 3);
    for (int c = 0; c < 3; ++c) {
        if (refactor[c])
            hipLaunchKernelGGL(zfactor_kernel, dim3(1), dim3(64), 0, s, g, c, dt, theta, dz_c, dz_f,
                               tab[c]);
        a.s[c] = src[c];
        a.f[c] = f[c];
        a.tab[c] = tab[c];
    }
    return launch_zsolve3(g, a, s);
}

// ---------------------------------------------------------------------------
// divergence -> plane-major (k, i, j) Poisson right-hand side
// ---------------------------------------------------------------------------

template <bool WRAP>
__global__ __launch_bounds__(256) void div_planes_kernel(Grid g, const double* __restrict__ u,
                                                         const double* __restrict__ v,
                                                         const double* __restrict__ w,
                                                         const double* __restrict__ dz_f,
                                                         double scale,
                                                         double* __restrict__ planes) {
    __shared__ double tile[kT][kT + 1];
    div_planes_body<WRAP>(g, u, v, w, dz_f, scale, planes, blockIdx.z, blockIdx.y * kT,
                          blockIdx.x * kT, tile);
}

hipError_t run_div_planes(const Grid& g, const double* u, const double* v, const double* w,
                          const double* dz_f, double scale, double* planes, bool wrap,
                          hipStream_t s) {
    dim3 grid((g.nz + kT - 1) / kT, (g.ny + kT - 1) / kT, g.nx);
    if (wrap)
        hipLaunchKernelGGL(div_planes_kernel<true>, grid, dim3(256), 0, s, g, u, v, w, dz_f, scale,
                           planes);
    else
        hipLaunchKernelGGL(div_planes_kernel<false>, grid, dim3(256), 0, s, g, u, v, w, dz_f, scale,
                           planes);
    return hipGetLastError();
}

__global__ void div_field_kernel(Grid g, const double* __restrict__ u,
                                 const double* __restrict__ v, const double* __restrict__ w,
                                 const double* __restrict__ dz_f, double* __restrict__ div) {
    long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long N = (long)g.nx * g.ny * g.nz;
    if (n >= N) return;
    const unsigned un = (unsigned)n;
    int k = (int)(un % (unsigned)g.nz);
    unsigned r = un / (unsigned)g.nz;
    int j = (int)(r % (unsigned)g.ny), i = (int)(r / (unsigned)g.ny);
    div[n] = divergence_at<false>(g, u, v, w, dz_f, i + 1, j + 1, k + 1);
}

hipError_t run_div_field(const Grid& g, const double* u, const double* v, const double* w,
                         const double* dz_f, double* div, hipStream_t s) {
    long N = (long)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL(div_field_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, g, u,
                       v, w, dz_f, div);
    return hipGetLastError();
}

// (nx, ny, nz) z-contiguous -> plane-major, divided by `scale`
__global__ __launch_bounds__(256) void to_planes_kernel(Grid g, const double* __restrict__ f,
                                                        double scale,
                                                        double* __restrict__ planes) {
    __shared__ double tile[kT][kT + 1];
    const int i = blockIdx.z;
    const int j0 = blockIdx.y * kT, k0 = blockIdx.x * kT;
    const int t = threadIdx.x;
    {
        const int kk = t % kT;
        for (int jj = t / kT; jj < kT; jj += 256 / kT) {
            int j = j0 + jj, k = k0 + kk;
            if (j < g.ny && k < g.nz) tile[jj][kk] = f[((long)i * g.ny + j) * g.nz + k] / scale;
        }
    }
    __syncthreads();
    {
        const int jj = t % kT;
        for (int kk = t / kT; kk < kT; kk += 256 / kT) {
            int j = j0 + jj, k = k0 + kk;
            if (j < g.ny && k < g.nz) planes[((long)k * g.nx + i) * g.ny + j] = tile[jj][kk];
        }
    }
}

hipError_t run_field_to_planes(const Grid& g, const double* f, double scale, double* planes,
                               hipStream_t s) {
    dim3 grid((g.nz + kT - 1) / kT, (g.ny + kT - 1) / kT, g.nx);
    hipLaunchKernelGGL(to_planes_kernel, grid, dim3(256), 0, s, g, f, scale, planes);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// per-wavenumber Thomas
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void poisson_thomas_kernel(PoissonTabs t,
                                                             double2* __restrict__ d,
                                                             double* __restrict__ cpw) {
    poisson_thomas_body(t, d, cpw, (long)blockIdx.x * blockDim.x + threadIdx.x);
}

template <int NT>
__global__ __launch_bounds__(NT) void poisson_spike_kernel(PoissonTabs t,
                                                           double2* __restrict__ d) {
    __shared__ double lds[NT * 8];
    poisson_spike_body<NT>(t, d, (long)blockIdx.x, lds);
}

// Segments from which the partition solve runs 512-thread workgroups: at 64
// or more segments a 256-thread workgroup holds 4 modes or fewer, i.e. plane
// rows of 64 bytes or less.
#ifndef SLC_SPIKE_WIDE_SEGS
#define SLC_SPIKE_WIDE_SEGS 64
#endif

// The partition solve (32 B per unknown) where nz allows it, else the
// sequential sweep with c' through the cp scratch.
hipError_t run_poisson_thomas(const PoissonTabs& t, double* dhat, double* cp, hipStream_t s) {
    long M = (long)t.nx * t.nky;
    if (spike_ok(t.nz)) {
        double2* d = reinterpret_cast<double2*>(dhat);
        if (spike_segs(t.nz) >= SLC_SPIKE_WIDE_SEGS) {
            const long MB = spike_modes(t.nz, 512);
            hipLaunchKernelGGL(poisson_spike_kernel<512>, dim3((unsigned)((M + MB - 1) / MB)),
                               dim3(512), 0, s, t, d);
        } else {
            const long MB = spike_modes(t.nz);
            hipLaunchKernelGGL(poisson_spike_kernel<256>, dim3((unsigned)((M + MB - 1) / MB)),
                               dim3(256), 0, s, t, d);
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL(poisson_thomas_kernel, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, s,
                       t, reinterpret_cast<double2*>(dhat), cp);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// projection
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void project_planes_kernel(
    Grid g, double* __restrict__ u, double* __restrict__ v, double* __restrict__ w,
    const double* __restrict__ P, double inv_n, double dt, const double* __restrict__ dz_c,
    double* __restrict__ p) {
    __shared__ double t0[kT + 1][kT + 2];  // plane i   rows j0..j0+kT, k0..k0+kT
    __shared__ double t1[kT][kT + 1];      // plane i+1 rows j0..j0+kT-1
    project_planes_body(g, u, v, w, P, inv_n, dt, dz_c, p, blockIdx.z, blockIdx.y * kT,
                        blockIdx.x * kT, t0, t1);
}

hipError_t run_project_planes(const Grid& g, double* u, double* v, double* w,
                              const double* planes, double inv_n, double dt,
                              const double* dz_c, double* p, hipStream_t s) {
    dim3 grid((g.nz + kT - 1) / kT, (g.ny + kT - 1) / kT, g.nx);
    hipLaunchKernelGGL(project_planes_kernel, grid, dim3(256), 0, s, g, u, v, w, planes, inv_n, dt,
                       dz_c, p);
    return hipGetLastError();
}

// u -= dt grad p with a ghost-shaped p (projection.py:250-272)
__global__ void project_p_kernel(Grid g, double* __restrict__ u, double* __restrict__ v,
                                 double* __restrict__ w, const double* __restrict__ p, double dt,
                                 const double* __restrict__ dz_c) {
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= (long)nx * ny * nz) return;
    const unsigned un = (unsigned)n;
    const int k = (int)(un % (unsigned)nz);
    const unsigned r = un / (unsigned)nz;
    const int j = (int)(r % (unsigned)ny), i = (int)(r / (unsigned)ny);
    const int I = i + 1, J = j + 1, K = k + 1;
    const long PSY = ny + 2, PSZ = nz + 2;
    const long pc = ((long)I * PSY + J) * PSZ + K;
    const double p0 = p[pc];
    long ui = ((long)I * (ny + 2) + J) * (nz + 2) + K;
    u[ui] = u[ui] - dt * ((p[pc + PSY * PSZ] - p0) / g.dx);
    long vi = ((long)I * (ny + 1) + J) * (nz + 2) + K;
    v[vi] = v[vi] - dt * ((p[pc + PSZ] - p0) / g.dy);
    if (K <= nz - 1) {
        long wi = ((long)I * (ny + 2) + J) * (nz + 1) + K;
        w[wi] = w[wi] - dt * ((p[pc + 1] - p0) / dz_c[K]);
    }
}

hipError_t run_project_p(const Grid& g, double* u, double* v, double* w, const double* p,
                         double dt, const double* dz_c, hipStream_t s) {
    long N = (long)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL(project_p_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, g, u,
                       v, w, p, dt, dz_c);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// bulk velocity and the exact flux shift
// ---------------------------------------------------------------------------

int bulk_partials_needed(const Grid& g) { return bulk_blocks(g.nx, g.ny, g.nz); }

__global__ __launch_bounds__(kRedBlock) void bulk_before_kernel(Grid g, const double* u,
                                                                const double* __restrict__ cv,
                                                                double* partials) {
    __shared__ double red[kRedBlock];
    bulk_before_body(g, u, cv, partials, blockIdx.x, gridDim.x, red);
}

__global__ __launch_bounds__(kRedBlock) void bulk_shift_kernel(Grid g, double* __restrict__ u,
                                                               const double* __restrict__ cv,
                                                               double* partials,
                                                               double total_volume, double U_bulk,
                                                               double dt,
                                                               double* __restrict__ scal) {
    __shared__ double red[kRedBlock];
    __shared__ bool last;
    bulk_shift_body(g, u, cv, partials, blockIdx.x, gridDim.x, total_volume, U_bulk, dt, scal, red,
                    &last);
}

__global__ __launch_bounds__(kRedBlock) void bulk_mean_kernel(const double* __restrict__ partials,
                                                              int np, double total_volume,
                                                              double* __restrict__ out) {
    __shared__ double red[kRedBlock];
    const double ub = bulk_mean(partials, np, total_volume, red);
    if (threadIdx.x == 0) *out = ub;
}

// u's ghosts follow the shifted interior (solver.py:720; v, w unchanged).
hipError_t run_bulk(const Grid& g, double* u, const double* cv, double total_volume,
                    double U_bulk, double dt, double* partials, double* scal, hipStream_t s) {
    const int np = bulk_partials_needed(g);
    hipLaunchKernelGGL(bulk_before_kernel, dim3(np), dim3(kRedBlock), 0, s, g, u, cv, partials);
    hipLaunchKernelGGL(bulk_shift_kernel, dim3(np), dim3(kRedBlock), 0, s, g, u, cv, partials,
                       total_volume, U_bulk, dt, scal);
    return hipGetLastError();
}

hipError_t run_bulk_velocity(const Grid& g, const double* u, const double* cv,
                             double total_volume, double* partials, double* out, hipStream_t s) {
    const int np = bulk_partials_needed(g);
    hipLaunchKernelGGL(bulk_before_kernel, dim3(np), dim3(kRedBlock), 0, s, g, u, cv, partials);
    hipLaunchKernelGGL(bulk_mean_kernel, dim3(1), dim3(kRedBlock), 0, s, partials, np,
                       total_volume, out + 3);
    return hipGetLastError();
}

}  // namespace slc
