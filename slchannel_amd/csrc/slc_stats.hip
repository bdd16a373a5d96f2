// slc_stats.hip -- on-device turbulence statistics (include/slc_stats.h).
//
// One snapshot of TurbulenceStats.accumulate_statistics
// (slchannel/turbstats.py:156-361) as four launches plus, with spectra
// planes, two more:
//
//   shift    a provisional mean of u, v and w per z level, from 64 columns;
//   pass     sums of the cell-centred u and v, of the u / v nodes and w
//            faces and of their squares, and of the cell-centred u w, all of
//            values less the provisional means, per z level, as column-chunk
//            partials, and the planes of the spectra pairs into a contiguous
//            batch;
//   reduce   partials -> plane averages (fixed order);
//   final    means and central moments of the averages (the squares' average
//            less the square of the average of the same shifted values),
//            running sums += this snapshot's profiles (w'w' faces averaged
//            to centres, turbstats.py:229-231);
//   rocFFT   batched real-forward 2-D transforms (torch.fft.rfft2 layout);
//   fold     auto / cross spectra, both walls averaged, folded onto
//            kx > 0, ky > 0, added to the running sums
//            (turbstats.py:256-351).
//
// One read of the fields in place of two (a pass of means, then one of
// fluctuations about them; 86 + 82 us at 256^3, each at the rate of memory).
// What the shift costs in precision: with m the provisional mean's error and s2
// the variance, the last subtraction takes m^2 from s2 + m^2, so rounding of
// the sums weighs up to 1 + 2 m^2 / s2 times as much as in sums about the mean
// itself.  For fields whose columns are samples of one distribution m^2 is
// about s2 / 64.  The columns are a regular 8 x 8 lattice: a pattern whose
// wavenumbers are multiples of 8 in x and y may be met at one phase only
// (m^2 = 4 s2 for a product of two cosines), and values that stand out on those
// very columns have m^2 up to N / 64 s2, N the plane's columns, the most that
// any field can have.  A variance below zero, which the final kernel sets to
// zero, is at most such rounding.
//
// Layout of the pass: a workgroup is 64 z lanes x 4 column groups.  The z
// lanes make every load a coalesced 512-byte row segment; each thread walks
// an x-run of 16 cells for 4 y-rows (shorter on small grids), carrying the
// previous u face in a register so the cell-centred u costs one load.  Partials go to
// part[(chunk * NQ + q) * (nz + 1) + k] and are summed in chunk order by the
// reduce kernel, so the result does not depend on scheduling.
#include <rocfft/rocfft.h>

#include <cstring>
#include <vector>

#include "../../include/slc_stats.h"
#include "slc_plan.h"

using namespace slc;

namespace {

constexpr int kLanes = 64;  // z lanes per workgroup
constexpr int kSub = 4;     // column groups per workgroup
constexpr int kRun = 16;    // most x cells of a thread's run, and y rows of a workgroup
constexpr int kSide = 8;    // shift: kSide x kSide columns
// sums of shifted values: u, v at centres; u node and square; v node and
// square; w face and square; u w at centres
enum { kUc = 0, kVc, kUn, kUU, kVn, kVV, kWf, kWW, kUW, kNQ };

// ib x cells per thread run, jb y rows per workgroup (jb / kSub per thread);
// nbx x nby chunks of columns
struct Dims {
    int nx, ny, nz, ib, jb, nbx, nby;
};

// shift[c * (nz + 1) + k]: the average of component c at level k (w: face k)
// over kSide x kSide columns spread over the plane.
constexpr int kRSub = 16;

__global__ __launch_bounds__(kLanes * kRSub) void stats_shift_kernel(
    Dims d, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ w, double* __restrict__ shift) {
    __shared__ double red[3][kRSub][kLanes];
    const int lane = threadIdx.x % kLanes, sub = threadIdx.x / kLanes;
    const int k = blockIdx.x * kLanes + lane, nz = d.nz;
    constexpr int kPer = kSide * kSide / kRSub;
    double s[3] = {0.0, 0.0, 0.0};
    if (k <= nz) {
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            const int c = sub * kPer + t;
            const size_t I = (size_t)((long)(c / kSide) * d.nx / kSide) + 1;
            const size_t J = (size_t)((long)(c % kSide) * d.ny / kSide) + 1;
            if (k < nz) {
                s[0] += u[(I * (d.ny + 2) + J) * (nz + 2) + k + 1];
                s[1] += v[(I * (d.ny + 1) + J) * (nz + 2) + k + 1];
            }
            s[2] += w[(I * (d.ny + 2) + J) * (nz + 1) + k];
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) red[q][sub][lane] = s[q];
    __syncthreads();
    if (sub < 3 && k <= nz) {
        double t = red[sub][0][lane];
        for (int g = 1; g < kRSub; ++g) t += red[sub][g][lane];
        shift[sub * (nz + 1) + k] = t * (1.0 / (kSide * kSide));
    }
}

// Plane sums over one workgroup's columns for z lane k (0..nz-1); lane
// nz-1 also sums the top w face (index nz), which it loads anyway.
//
// Lanes at a level of a spectra pair also write its planes, batch index
// 6 * pair + c: c = 0, 1, 2 bottom u node, v node, cell-centred w; 3, 4, 5
// the same at the top with w negated (turbstats.py:256-276).  Planes are
// (nx, ny), y fastest, of the shifted values: what those lack to the
// fluctuations is a constant, which only the mean mode sees, and no spectrum
// holds it (kx > 0, ky > 0).  Read back from the fields, a level at a time,
// the planes of 4 pairs cost 37 us at 256^3 (a cache line per value).
__global__ __launch_bounds__(kLanes * kSub) void stats_pass_kernel(
    Dims d, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ w, const double* __restrict__ shift, double* __restrict__ part,
    const int* __restrict__ kp, int nsides, double* __restrict__ planes) {
    __shared__ double red[kSub][kNQ][kLanes];
    __shared__ double red_top[2][kSub];
    const int lane = threadIdx.x % kLanes, sub = threadIdx.x / kLanes;
    const int k = blockIdx.x * kLanes + lane;
    const int nx = d.nx, ny = d.ny, nz = d.nz, nzf = nz + 1;
    const int i0 = blockIdx.y * d.ib, i1 = min(nx, i0 + d.ib);
    const int j0 = blockIdx.z * d.jb, j1 = min(ny, j0 + d.jb);
    const size_t su = (size_t)(ny + 2) * (nz + 2), sv = (size_t)(ny + 1) * (nz + 2),
                 sw = (size_t)(ny + 2) * (nz + 1);
    double s[kNQ];
#pragma unroll
    for (int q = 0; q < kNQ; ++q) s[q] = 0.0;
    double top = 0.0, top2 = 0.0;  // lane nz-1: sums of the top face
    double pu = 0.0, pv = 0.0, pw = 0.0, pt = 0.0;
    if (k < nz) {
        pu = shift[k];
        pv = shift[nzf + k];
        pw = shift[2 * nzf + k];
        pt = shift[2 * nzf + k + 1];
    }
    // sides whose plane is this level: bits of the first 64
    unsigned long long sides = 0ull;
    for (int q = 0; q < min(nsides, 64); ++q)
        if (kp[q] - 1 == k) sides |= 1ull << q;
    const size_t plane = (size_t)nx * ny;
    for (int j = j0 + sub; j < j1; j += kSub) {
        // u[i0, j+1, k+1], v[i0+1, j, k+1], w[i0+1, j+1, k]
        const double* ur = u + ((size_t)i0 * (ny + 2) + (j + 1)) * (nz + 2) + (k + 1);
        const double* vr = v + ((size_t)(i0 + 1) * (ny + 1) + j) * (nz + 2) + (k + 1);
        const double* wr = w + ((size_t)(i0 + 1) * (ny + 2) + (j + 1)) * (nz + 1) + k;
        if (k < nz) {
            double up = ur[0] - pu;
            for (int i = i0; i < i1; ++i) {
                const size_t o = (size_t)(i - i0);
                const double un = ur[(o + 1) * su] - pu;
                const double v0 = vr[o * sv] - pv, v1 = vr[o * sv + (nz + 2)] - pv;
                const double w0 = wr[o * sw] - pw, w1 = wr[o * sw + 1] - pt;
                const double ucc = 0.5 * (up + un);
                s[kUc] += ucc;
                s[kVc] += 0.5 * (v0 + v1);
                s[kUn] += un;
                s[kUU] += un * un;
                s[kVn] += v1;
                s[kVV] += v1 * v1;
                s[kWf] += w0;
                s[kWW] += w0 * w0;
                s[kUW] += ucc * (0.5 * (w0 + w1));
                if (k == nz - 1) {
                    top += w1;
                    top2 += w1 * w1;
                }
                auto put = [&](int side) {
                    double* o3 = planes + (size_t)side * 3 * plane + ((size_t)i * ny + j);
                    o3[0] = un;
                    o3[plane] = v1;
                    o3[2 * plane] = (side & 1) ? -(0.5 * (w0 + w1)) : 0.5 * (w0 + w1);
                };
                for (unsigned long long m = sides; m; m &= m - 1) put(__ffsll(m) - 1);
                for (int q = 64; q < nsides; ++q)
                    if (kp[q] - 1 == k) put(q);
                up = un;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < kNQ; ++q) red[sub][q][lane] = s[q];
    if (k == nz - 1) {
        red_top[0][sub] = top;
        red_top[1][sub] = top2;
    }
    __syncthreads();
    if (sub == 0 && k < nz) {
        const size_t chunk = (size_t)blockIdx.z * d.nbx + blockIdx.y;
#pragma unroll
        for (int q = 0; q < kNQ; ++q) {
            double r = red[0][q][lane];
#pragma unroll
            for (int t = 1; t < kSub; ++t) r += red[t][q][lane];
            part[(chunk * kNQ + q) * nzf + k] = r;
        }
        if (k == nz - 1) {
            // the other quantities have no entry at the top face (zero)
#pragma unroll
            for (int q = 0; q < kNQ; ++q) {
                double r = 0.0;
                if (q == kWf || q == kWW)
                    for (int t = 0; t < kSub; ++t) r += red_top[q == kWW][t];
                part[(chunk * kNQ + q) * nzf + nz] = r;
            }
        }
    }
}

// Sums the partials of quantity q = blockIdx.y at lane k in chunk order
// (column group t of kRSub takes chunks t, t + kRSub, ...; groups combined in
// order) and divides by the plane size: out[q * (nz + 1) + k].
__global__ __launch_bounds__(kLanes * kRSub) void stats_reduce_kernel(
    const double* __restrict__ part, int nchunks, int nz, double plane,
    double* __restrict__ out) {
    __shared__ double red[kRSub][kLanes];
    const int lane = threadIdx.x % kLanes, sub = threadIdx.x / kLanes;
    const int k = blockIdx.x * kLanes + lane, q = blockIdx.y, nzf = nz + 1;
    double r = 0.0;
    if (k <= nz)
        for (int c = sub; c < nchunks; c += kRSub) r += part[((size_t)c * kNQ + q) * nzf + k];
    red[sub][lane] = r;
    __syncthreads();
    if (sub == 0 && k <= nz) {
        double t = red[0][lane];
        for (int g = 1; g < kRSub; ++g) t += red[g][lane];
        out[(size_t)q * nzf + k] = t / plane;
    }
}

// Means and central moments from the shifted averages; running sums += this
// snapshot (turbstats.py:177, 195-200, 239-242).
__global__ __launch_bounds__(256) void stats_final_kernel(int nz, const double* __restrict__ avg,
                                                           const double* __restrict__ shift,
                                                           double* __restrict__ prof) {
    const int nzf = nz + 1;
    // a variance of rounding size may come out below zero
    auto var = [&](int sq, int av, int k) {
        const double m = avg[av * nzf + k], x = avg[sq * nzf + k] - m * m;
        return x < 0.0 ? 0.0 : x;
    };
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nz; k += gridDim.x * blockDim.x) {
        const double pu = shift[k], pv = shift[nzf + k];
        const double pw = shift[2 * nzf + k], pt = shift[2 * nzf + k + 1];
        const double dU = avg[kUc * nzf + k];
        const double dw = avg[kWf * nzf + k], dt = avg[kWf * nzf + k + 1];
        const double U = pu + dU, V = pv + avg[kVc * nzf + k];
        const double W = 0.5 * ((pw + dw) + (pt + dt));
        prof[0 * nz + k] += U;
        prof[1 * nz + k] += var(kUU, kUn, k);
        prof[2 * nz + k] += var(kVV, kVn, k);
        prof[3 * nz + k] += 0.5 * (var(kWW, kWf, k) + var(kWW, kWf, k + 1));
        prof[4 * nz + k] += avg[kUW * nzf + k] - dU * (0.5 * (dw + dt));
        prof[5 * nz + k] += V;
        prof[6 * nz + k] += W;
        prof[7 * nz + k] += U * U;
        prof[8 * nz + k] += V * V;
        prof[9 * nz + k] += W * W;
        prof[10 * nz + k] += U * W;
    }
}

__device__ inline double auto_spec(double2 f, double norm) {
    return (f.x * f.x + f.y * f.y) / norm;
}
__device__ inline double cross_spec(double2 f, double2 g, double norm) {
    return (f.x * g.x + f.y * g.y) / norm;
}

// spec[pair][c][a][b] += fold(0.5 (E_bot + E_top)) with
// fold(E)[a, b] = E[a + 1, b + 1] + E[nx - 1 - a, b + 1] (turbstats.py:278-351).
__global__ __launch_bounds__(256) void stats_fold_kernel(Dims d, const double2* __restrict__ F,
                                                         double norm, double* __restrict__ spec) {
    const int nx = d.nx, ny = d.ny, nkx = nx / 2, nky = ny / 2, nyc = ny / 2 + 1;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nkx * nky) return;
    const int a = t / nky, b = t % nky, pair = blockIdx.y;
    const size_t plane = (size_t)nx * nyc;
    const double2* Fp = F + (size_t)pair * 6 * plane;
    const size_t pos = (size_t)(a + 1) * nyc + (b + 1), neg = (size_t)(nx - 1 - a) * nyc + (b + 1);
    double* out = spec + (size_t)pair * 4 * nkx * nky + t;
    const size_t cs = (size_t)nkx * nky;
    double e[4][2];
    for (int side = 0; side < 2; ++side) {
        const size_t o = side == 0 ? pos : neg;
        const double2 ub = Fp[0 * plane + o], vb = Fp[1 * plane + o], wb = Fp[2 * plane + o];
        const double2 ut = Fp[3 * plane + o], vt = Fp[4 * plane + o], wt = Fp[5 * plane + o];
        e[0][side] = 0.5 * (auto_spec(ub, norm) + auto_spec(ut, norm));
        e[1][side] = 0.5 * (auto_spec(vb, norm) + auto_spec(vt, norm));
        e[2][side] = 0.5 * (auto_spec(wb, norm) + auto_spec(wt, norm));
        e[3][side] = 0.5 * (cross_spec(ub, wb, norm) + cross_spec(ut, wt, norm));
    }
    for (int c = 0; c < 4; ++c) out[c * cs] += e[c][0] + e[c][1];
}

}  // namespace

struct slc_stats {
    int device = 0;
    Dims d{};
    int nzc = 0, nzr = 0, nchunks = 0, nplanes = 0;
    double* part = nullptr;    // nchunks x kNQ x (nz + 1)
    double* shift = nullptr;   // 3 x (nz + 1)
    double* avg = nullptr;     // kNQ x (nz + 1)
    int* kp = nullptr;         // 2 x nplanes (k_bot, k_top)
    double* planes = nullptr;  // 6 nplanes x nx x ny
    double2* fhat = nullptr;   // 6 nplanes x nx x (ny/2 + 1)
    rocfft_plan fwd = nullptr;
    rocfft_execution_info info = nullptr;
    void* work = nullptr;
    std::vector<void*> allocs;
    int64_t bytes = 0;
};

namespace {

int stats_alloc(slc_stats* st, size_t bytes, void** out) {
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes ? bytes : 8);
    if (e != hipSuccess)
        return fail(SLC_ENOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    st->allocs.push_back(p);
    st->bytes += (int64_t)bytes;
    *out = p;
    return SLC_OK;
}

}  // namespace

extern "C" {

int slc_stats_destroy(slc_stats* st) {
    if (!st) return SLC_OK;
    DeviceGuard dg(st->device);
    (void)hipDeviceSynchronize();
    if (st->fwd) rocfft_plan_destroy(st->fwd);
    if (st->info) rocfft_execution_info_destroy(st->info);
    for (void* p : st->allocs) (void)hipFree(p);
    delete st;
    return SLC_OK;
}

int slc_stats_create(int device, int nx, int ny, int nz, int nplanes, const int* k_bot,
                     const int* k_top, slc_stats** out) {
    if (!out) return fail(SLC_EINVAL, "null argument");
    *out = nullptr;
    if (nx < 1 || ny < 1 || nz < 1)
        return fail(SLC_EINVAL, "grid too small (nx=%d ny=%d nz=%d)", nx, ny, nz);
    if ((double)(nx + 2) * (ny + 2) * (nz + 2) >= 2147483647.0)
        return fail(SLC_EINVAL, "grid too large ((nx+2)(ny+2)(nz+2) >= 2^31)");
    if (nplanes < 0) return fail(SLC_EINVAL, "nplanes must be >= 0");
    if (nplanes > 0) {
        if (!k_bot || !k_top) return fail(SLC_EINVAL, "null plane index arrays");
        if (nx < 2 || ny < 2) return fail(SLC_EINVAL, "spectra need nx, ny >= 2");
        for (int i = 0; i < nplanes; ++i)
            if (k_bot[i] < 1 || k_bot[i] > nz || k_top[i] < 1 || k_top[i] > nz)
                return fail(SLC_EINVAL, "plane %d: k_bot=%d k_top=%d outside 1..%d", i, k_bot[i],
                            k_top[i], nz);
    }
    DeviceGuard dg(device);
    slc_stats* st = new slc_stats();
    st->device = device;
    st->nzc = (nz + kLanes - 1) / kLanes;        // pass workgroups along z
    // 16 x 16 columns a workgroup; smaller chunks while the workgroups do not
    // fill the chip, since a thread's walk is a chain of loads (30x20x40:
    // 53 us a snapshot with 16 x 16, 30 with 4 x 4; 128^3: 49)
    int ib = kRun, jb = kRun;
    auto cover = [](int n, int m) { return (n + m - 1) / m; };
    while (jb > kSub && (long)st->nzc * cover(nx, ib) * cover(ny, jb) < 512) {
        jb /= 2;
        ib /= 2;
    }
    st->d = Dims{nx, ny, nz, ib, jb, cover(nx, ib), cover(ny, jb)};
    st->nzr = (nz + 1 + kLanes - 1) / kLanes;    // reduce workgroups along z (faces)
    st->nchunks = st->d.nbx * st->d.nby;
    st->nplanes = nplanes;
    const size_t nzf = (size_t)nz + 1;
    void* p = nullptr;
    int rc;
    if ((rc = stats_alloc(st, sizeof(double) * st->nchunks * kNQ * nzf, &p))) goto bad;
    st->part = (double*)p;
    if ((rc = stats_alloc(st, sizeof(double) * (3 + kNQ) * nzf, &p))) goto bad;
    st->shift = (double*)p;
    st->avg = st->shift + 3 * nzf;
    if (nplanes > 0) {
        std::vector<int> kp(2 * (size_t)nplanes);
        for (int i = 0; i < nplanes; ++i) {
            kp[2 * i] = k_bot[i];
            kp[2 * i + 1] = k_top[i];
        }
        if ((rc = stats_alloc(st, sizeof(int) * kp.size(), &p))) goto bad;
        st->kp = (int*)p;
        hipError_t e = hipMemcpy(st->kp, kp.data(), sizeof(int) * kp.size(), hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            rc = fail(SLC_EHIP, "plane table upload: %s", hipGetErrorString(e));
            goto bad;
        }
        const size_t nb = 6 * (size_t)nplanes;
        if ((rc = stats_alloc(st, sizeof(double) * nb * nx * ny, &p))) goto bad;
        st->planes = (double*)p;
        if ((rc = stats_alloc(st, sizeof(double2) * nb * nx * (ny / 2 + 1), &p))) goto bad;
        st->fhat = (double2*)p;
        rocfft_setup();
        // torch.fft.rfft2 over (x, y): y is the halved dimension (fastest first)
        size_t lengths[2] = {(size_t)ny, (size_t)nx};
        if (rocfft_plan_create(&st->fwd, rocfft_placement_notinplace,
                               rocfft_transform_type_real_forward, rocfft_precision_double, 2,
                               lengths, nb, nullptr) != rocfft_status_success) {
            rc = fail(SLC_EFFT, "rocfft_plan_create(spectra, batch %zu) failed", nb);
            goto bad;
        }
        if (rocfft_execution_info_create(&st->info) != rocfft_status_success) {
            rc = fail(SLC_EFFT, "rocfft_execution_info_create failed");
            goto bad;
        }
        size_t wb = 0;
        rocfft_plan_get_work_buffer_size(st->fwd, &wb);
        if (wb) {
            if ((rc = stats_alloc(st, wb, &p))) goto bad;
            st->work = p;
            rocfft_execution_info_set_work_buffer(st->info, st->work, wb);
        }
    }
    *out = st;
    return SLC_OK;
bad:
    slc_stats_destroy(st);
    return rc;
}

int slc_stats_workspace_bytes(const slc_stats* st, int64_t* bytes) {
    if (!st || !bytes) return fail(SLC_EINVAL, "null argument");
    *bytes = st->bytes;
    return SLC_OK;
}

int slc_stats_accumulate(slc_stats* st, const double* u, const double* v, const double* w,
                         double* prof, double* spec, void* stream) {
    if (!st) return fail(SLC_EINVAL, "null stats");
    if (!u || !v || !w || !prof) return fail(SLC_EINVAL, "null array");
    if (st->nplanes > 0 && !spec) return fail(SLC_EINVAL, "spec required with %d planes",
                                              st->nplanes);
    DeviceGuard dg(st->device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const Dims d = st->d;
    const dim3 grid(st->nzc, d.nbx, d.nby), blk(kLanes * kSub);
    const double plane = (double)d.nx * (double)d.ny;
    hipLaunchKernelGGL(stats_shift_kernel, dim3(st->nzr), dim3(kLanes * kRSub), 0, s, d, u, v, w,
                       st->shift);
    HIP_OK(hipGetLastError());
    hipLaunchKernelGGL(stats_pass_kernel, grid, blk, 0, s, d, u, v, w, st->shift, st->part,
                       st->kp, 2 * st->nplanes, st->planes);
    hipLaunchKernelGGL(stats_reduce_kernel, dim3(st->nzr, kNQ), dim3(kLanes * kRSub), 0, s,
                       st->part, st->nchunks, d.nz, plane, st->avg);
    hipLaunchKernelGGL(stats_final_kernel, dim3((d.nz + 255) / 256), dim3(256), 0, s, d.nz,
                       st->avg, st->shift, prof);
    HIP_OK(hipGetLastError());
    if (st->nplanes == 0) return SLC_OK;
    FFT_OK(rocfft_execution_info_set_stream(st->info, s));
    void* in[1] = {st->planes};
    void* outp[1] = {st->fhat};
    FFT_OK(rocfft_execute(st->fwd, in, outp, st->info));
    const int nfold = (d.nx / 2) * (d.ny / 2);
    if (nfold > 0) {
        hipLaunchKernelGGL(stats_fold_kernel, dim3((nfold + 255) / 256, st->nplanes), dim3(256), 0,
                           s, d, st->fhat, plane * plane, spec);
        HIP_OK(hipGetLastError());
    }
    return SLC_OK;
}

}  // extern "C"
