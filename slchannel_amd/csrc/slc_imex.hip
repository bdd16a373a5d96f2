// slc_imex.hip -- the Eulerian IMEX explicit terms (slc_imex_rhs,
// slc_ab2_update, slc_imex_advance) and the step's part up to the projection
// (slc_imex_step).
//
// compute_momentum_rhs_fused_imex (operators.py:639-835; the Triton kernel of
// eulerian_triton.py:31-193 computes the same): divergence-form advection on
// the MAC grid and the xy Laplacian, rhs = diffusion_xy - advection on each
// component's interior and 0 on every other entry of its ghost-shaped array.
// The three components in one launch; each output element uses the
// reference's operation order (no contraction), so it is the same double the
// eager path computes.
//
// slc_ab2_update: u += dt (1.5 r - 0.5 r_prev) (forward Euler, u += dt r,
// without a previous rhs) over the whole arrays (solver.py:1074-1081).
// slc_imex_advance: both in one pass, the new fields to other arrays (a
// point's neighbours still read the old ones).
#include <algorithm>

#include "slc_plan.h"

using namespace slc;

namespace {

struct Rhs3 {
    double *u, *v, *w;
};

struct ImexK {
    double dx_inv, dy_inv, nu_dx2, nu_dy2;
};

// The AB2 update joined to the rhs: f = V + dt (1.5 r - 0.5 prev), or V + dt r
// where prev is null.
struct Ab2 {
    Rhs3 f, prev;
    double dt;
};

// One thread per (j, k) of a plane (z fastest) and run of `chunk` planes i of
// x: walking x, the values of planes i - 1 and i stay in registers, so a point
// costs 17 loads in place of the 60 its three stencils name, and HBM sees the
// fields once (the neighbours in y and z come from L1/L2).  ADVANCE: the
// update as well, on interior entries only; otherwise the rest of the rhs
// arrays is cleared.  At 256x192x192 a thread per point and the update in a
// launch of its own took 272 + 162 us; this pass 257 us, 3.5 TB/s of its twelve
// arrays' bytes.  512 and 1024 threads a block: 267 and 278 us; runs of 4 and
// 16 planes: no better.
constexpr int kImexBlock = 256;
constexpr int kImexChunk = 8;
constexpr int kImexFill = 2048;  // blocks below which a run is shortened

template <bool ADVANCE>
__global__ __launch_bounds__(kImexBlock) void imex_rhs_kernel(
    Grid g, const double* __restrict__ u, const double* __restrict__ v,
    const double* __restrict__ w, const double* __restrict__ dzfi, const double* __restrict__ dzc,
    ImexK c, Rhs3 out, Ab2 ab, unsigned nplane, int chunk) {
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const unsigned blk = (unsigned)xcd_block(gridDim.x);
    const unsigned t = blk % nplane * kImexBlock + threadIdx.x;
    if (t >= (unsigned)((ny + 2) * (nz + 2))) return;
    const int k = (int)(t % (unsigned)(nz + 2)), j = (int)(t / (unsigned)(nz + 2));
    const int i0 = 1 + (int)(blk / nplane) * chunk, i1 = min(i0 + chunk, nx + 1);
    // strides of the three arrays (z fastest)
    const int uz = nz + 2, uy = (ny + 2) * uz;  // u: (nx+1, ny+2, nz+2)
    const int vz = nz + 2, vy = (ny + 1) * vz;  // v: (nx+2, ny+1, nz+2)
    const int wz = nz + 1, wy = (ny + 2) * wz;  // w: (nx+2, ny+2, nz+1)
    const bool inner = j >= 1 && j <= ny && k >= 1 && k <= nz;
    auto clear = [&](int i) {
        if (i <= nx) out.u[i * uy + j * uz + k] = 0.0;
        if (j <= ny) out.v[i * vy + j * vz + k] = 0.0;
        if (k <= nz) out.w[i * wy + j * wz + k] = 0.0;
    };
    if (!ADVANCE) {
        if (i0 == 1) clear(0);
        if (i1 == nx + 1) clear(nx + 1);
        if (!inner)
            for (int i = i0; i < i1; ++i) clear(i);
    }
    if (!inner) return;
    const double dzi = dzfi[k - 1];
    const bool wface = k < nz;  // w's interior faces
    const double dzw = wface ? dzc[k] : 1.0;
    const int vjp = j == ny ? -(ny - 1) * vz : vz;  // v[j+1], periodic at j = ny
    const int wkp = wface ? 1 : 0;                  // w's row ends at the top face
    const double* pu = u + ((i0 - 1) * uy + j * uz + k);
    const double* pv = v + ((i0 - 1) * vy + j * vz + k);
    const double* pw = w + ((i0 - 1) * wy + j * wz + k);
    // plane i - 1: m; plane i: the point and its row and level neighbours
    double u_m = pu[0], uj_m = pu[uz], uk_m = pu[1], v_m = pv[0], w_m = pw[0];
    double u_c = pu[uy], v_c = pv[vy], vj_c = pv[vy - vz], w_c = pw[wy], wk_c = pw[wy - 1];
#pragma unroll 1
    for (int i = i0; i < i1; ++i) {
        pu += uy;
        pv += vy;
        pw += wy;
        const double u_jp = pu[uz], u_jm = pu[-uz], u_kp = pu[1], u_km = pu[-1];
        const double v_jp = pv[vjp], v_kp = pv[1], v_km = pv[-1], v_jmkp = pv[1 - vz];
        const double w_jp = pw[wz], w_jm = pw[-wz], w_kp = pw[wkp], w_jpkm = pw[wz - 1];
        // plane i + 1; U(i+1) at i = nx is the periodic u[1]
        const double u_p = i == nx ? pu[-(nx - 1) * uy] : pu[uy];
        const double v_p = pv[vy], vj_p = pv[vy - vz], w_p = pw[wy], wk_p = pw[wy - 1];
        const int uo = i * uy + j * uz + k, vo = i * vy + j * vz + k, wo = i * wy + j * wz + k;
        double qu = 0.0, qv = 0.0, qw = 0.0;
        if (ADVANCE && ab.prev.u) {
            qu = ab.prev.u[uo];
            qv = ab.prev.v[vo];
            if (wface) qw = ab.prev.w[wo];
        }
        double ru, rv, rw;
        {
            // ---- u (operators.py:679-728)
            const double a = 0.5 * (u_c + u_p);
            const double b = 0.5 * (u_m + u_c);
            const double duudx = (a * a - b * b) * c.dx_inv;
            double vi = 0.5 * (v_c + v_p);
            double ui = 0.5 * (u_c + u_jp);
            const double vu_top = vi * ui;
            vi = 0.5 * (vj_c + vj_p);
            ui = 0.5 * (u_jm + u_c);
            const double dvudy = (vu_top - vi * ui) * c.dy_inv;
            double wi = 0.5 * (w_c + w_p);
            ui = 0.5 * (u_c + u_kp);
            const double wu_top = wi * ui;
            wi = 0.5 * (wk_c + wk_p);
            ui = 0.5 * (u_km + u_c);
            const double dwudz = (wu_top - wi * ui) * dzi;
            const double adv = duudx + dvudy + dwudz;
            const double d2x = (u_p - 2.0 * u_c + u_m) * c.nu_dx2;
            const double d2y = (u_jp - 2.0 * u_c + u_jm) * c.nu_dy2;
            ru = (d2x + d2y) - adv;
        }
        {
            // ---- v (operators.py:734-781); V(j+1) at j = ny is the periodic v[:, 1]
            double ui = 0.5 * (u_c + u_jp);
            double vi = 0.5 * (v_c + v_p);
            const double uv_right = ui * vi;
            ui = 0.5 * (u_m + uj_m);
            vi = 0.5 * (v_m + v_c);
            const double duvdx = (uv_right - ui * vi) * c.dx_inv;
            const double a = 0.5 * (v_c + v_jp);
            const double b = 0.5 * (vj_c + v_c);
            const double dvvdy = (a * a - b * b) * c.dy_inv;
            double wi = 0.5 * (w_c + w_jp);
            vi = 0.5 * (v_c + v_kp);
            const double wv_top = wi * vi;
            wi = 0.5 * (wk_c + w_jpkm);
            vi = 0.5 * (v_km + v_c);
            const double dwvdz = (wv_top - wi * vi) * dzi;
            const double adv = duvdx + dvvdy + dwvdz;
            const double d2x = (v_p - 2.0 * v_c + v_m) * c.nu_dx2;
            const double d2y = (v_jp - 2.0 * v_c + vj_c) * c.nu_dy2;
            rv = (d2x + d2y) - adv;
        }
        {
            // ---- w (operators.py:787-833), interior faces k = 1..nz-1
            double ui = 0.5 * (u_c + u_kp);
            double wi = 0.5 * (w_c + w_p);
            const double uw_right = ui * wi;
            ui = 0.5 * (u_m + uk_m);
            wi = 0.5 * (w_m + w_c);
            const double duwdx = (uw_right - ui * wi) * c.dx_inv;
            double vi = 0.5 * (v_c + v_kp);
            wi = 0.5 * (w_c + w_jp);
            const double vw_top = vi * wi;
            vi = 0.5 * (vj_c + v_jmkp);
            wi = 0.5 * (w_jm + w_c);
            const double dvwdy = (vw_top - vi * wi) * c.dy_inv;
            const double a = 0.5 * (w_c + w_kp);
            const double b = 0.5 * (wk_c + w_c);
            const double dwwdz = (a * a - b * b) / dzw;
            const double adv = duwdx + dvwdy + dwwdz;
            const double d2x = (w_p - 2.0 * w_c + w_m) * c.nu_dx2;
            const double d2y = (w_jp - 2.0 * w_c + w_jm) * c.nu_dy2;
            rw = (d2x + d2y) - adv;
        }
        out.u[uo] = ru;
        out.v[vo] = rv;
        if (wface) out.w[wo] = rw;
        else if (!ADVANCE) out.w[wo] = 0.0;
        if (ADVANCE) {
            if (ab.prev.u) {
                ab.f.u[uo] = u_c + ab.dt * (1.5 * ru - 0.5 * qu);
                ab.f.v[vo] = v_c + ab.dt * (1.5 * rv - 0.5 * qv);
                if (wface) ab.f.w[wo] = w_c + ab.dt * (1.5 * rw - 0.5 * qw);
            } else {
                ab.f.u[uo] = u_c + ab.dt * ru;
                ab.f.v[vo] = v_c + ab.dt * rv;
                if (wface) ab.f.w[wo] = w_c + ab.dt * rw;
            }
        }
        u_m = u_c; uj_m = u_jp; uk_m = u_kp; u_c = u_p;
        v_m = v_c; v_c = v_p; vj_c = vj_p;
        w_m = w_c; w_c = w_p; wk_c = wk_p;
    }
}

// Runs of up to kImexChunk planes, shorter on grids whose blocks would
// otherwise leave compute units idle.
template <bool ADVANCE>
hipError_t run_imex(const slc_plan* p, const double* u, const double* v, const double* w,
                    const Rhs3& out, const Ab2& ab, hipStream_t s) {
    const Grid& g = p->g;
    // operators.py:662-672: reciprocals and nu-scaled squares as the reference forms them
    ImexK c;
    c.dx_inv = 1.0 / g.dx;
    c.dy_inv = 1.0 / g.dy;
    c.nu_dx2 = g.nu * (1.0 / (g.dx * g.dx));
    c.nu_dy2 = g.nu * (1.0 / (g.dy * g.dy));
    const unsigned nplane =
        (unsigned)(((long)(g.ny + 2) * (g.nz + 2) + kImexBlock - 1) / kImexBlock);
    const long most = (long)nplane * g.nx / kImexFill;
    const int chunk = (int)std::min<long>(kImexChunk, std::max<long>(1, most));
    const unsigned nrun = (unsigned)((g.nx + chunk - 1) / chunk);
    hipLaunchKernelGGL(imex_rhs_kernel<ADVANCE>, dim3(nplane * nrun), dim3(kImexBlock), 0, s, g, u,
                       v, w, p->d_dzf_inv, p->d_dzc, c, out, ab, nplane, chunk);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void ab2_update_kernel(double* __restrict__ u,
                                                         double* __restrict__ v,
                                                         double* __restrict__ w, Rhs3 r,
                                                         Rhs3 rp, double dt, unsigned nu_,
                                                         unsigned nv, unsigned nw) {
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    double* f[3] = {u, v, w};
    const double* a[3] = {r.u, r.v, r.w};
    const double* b[3] = {rp.u, rp.v, rp.w};
    const unsigned n[3] = {nu_, nv, nw};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (t >= n[c]) continue;
        if (b[c]) f[c][t] = f[c][t] + dt * (1.5 * a[c][t] - 0.5 * b[c][t]);
        else f[c][t] = f[c][t] + dt * a[c][t];
    }
}

}  // namespace

extern "C" int slc_imex_rhs(slc_plan* p, const double* u, const double* v, const double* w,
                            double* ru, double* rv, double* rw, void* stream) {
    if (!p) return fail(SLC_EINVAL, "null plan");
    if (!u || !v || !w || !ru || !rv || !rw) return fail(SLC_EINVAL, "null array");
    DeviceGuard dg(p->device);
    Timed tm(p, "imex_rhs", stream);
    HIP_OK(run_imex<false>(p, u, v, w, Rhs3{ru, rv, rw}, Ab2{}, static_cast<hipStream_t>(stream)));
    return SLC_OK;
}

extern "C" int slc_imex_advance(slc_plan* p, const double* u, const double* v, const double* w,
                                double* un, double* vn, double* wn, double* ru, double* rv,
                                double* rw, const double* ru_prev, const double* rv_prev,
                                const double* rw_prev, double dt, void* stream) {
    if (!p) return fail(SLC_EINVAL, "null plan");
    if (!u || !v || !w || !un || !vn || !wn || !ru || !rv || !rw)
        return fail(SLC_EINVAL, "null array");
    // neighbours read the old fields while others are written
    const double* const in[3] = {u, v, w};
    const double* const out[6] = {un, vn, wn, ru, rv, rw};
    for (int i = 0; i < 6; ++i) {
        if (std::find(in, in + 3, out[i]) != in + 3 || std::find(out, out + i, out[i]) != out + i)
            return fail(SLC_EINVAL, "the new fields and the rhs need arrays of their own");
    }
    const bool prev = ru_prev || rv_prev || rw_prev;
    if (prev && !(ru_prev && rv_prev && rw_prev))
        return fail(SLC_EINVAL, "previous rhs: all three components or none");
    DeviceGuard dg(p->device);
    Timed tm(p, "imex_rhs", stream);
    const Ab2 ab{{un, vn, wn}, {(double*)ru_prev, (double*)rv_prev, (double*)rw_prev}, dt};
    HIP_OK(run_imex<true>(p, u, v, w, Rhs3{ru, rv, rw}, ab, static_cast<hipStream_t>(stream)));
    return SLC_OK;
}

extern "C" int slc_imex_step(slc_plan* p, double* u, double* v, double* w, double* ru, double* rv,
                             double* rw, const double* ru_prev, const double* rv_prev,
                             const double* rw_prev, double dt, double theta, double* pr,
                             void* stream) {
    if (!p) return fail(SLC_EINVAL, "null plan");
    if (!(theta > 0.0 && theta < 1.0)) return fail(SLC_EINVAL, "theta must be in (0, 1)");
    if (int rc = check_zsolves(p)) return rc;
    // the advanced fields wait in the plan's U* arrays for the z-solves, which
    // write u, v and w: as many bytes as solves in place, no copy
    if (int rc = slc_imex_advance(p, u, v, w, p->us[0], p->us[1], p->us[2], ru, rv, rw, ru_prev,
                                  rv_prev, rw_prev, dt, stream))
        return rc;
    DeviceGuard dg(p->device);
    double* const f[3] = {u, v, w};
    return implicit_project(p, p->us, f, dt, theta, dt, dt, pr, stream);
}

extern "C" int slc_ab2_update(slc_plan* p, double* u, double* v, double* w, const double* ru,
                              const double* rv, const double* rw, const double* ru_prev,
                              const double* rv_prev, const double* rw_prev, double dt,
                              void* stream) {
    if (!p) return fail(SLC_EINVAL, "null plan");
    if (!u || !v || !w || !ru || !rv || !rw) return fail(SLC_EINVAL, "null array");
    const bool prev = ru_prev || rv_prev || rw_prev;
    if (prev && !(ru_prev && rv_prev && rw_prev))
        return fail(SLC_EINVAL, "previous rhs: all three components or none");
    DeviceGuard dg(p->device);
    const Grid& g = p->g;
    const unsigned n[3] = {(unsigned)((g.nx + 1) * (g.ny + 2) * (g.nz + 2)),
                           (unsigned)((g.nx + 2) * (g.ny + 1) * (g.nz + 2)),
                           (unsigned)((g.nx + 2) * (g.ny + 2) * (g.nz + 1))};
    const unsigned nmax = n[0] > n[1] ? (n[0] > n[2] ? n[0] : n[2]) : (n[1] > n[2] ? n[1] : n[2]);
    Timed tm(p, "ab2_update", stream);
    hipLaunchKernelGGL(ab2_update_kernel, dim3((nmax + 255) / 256), dim3(256), 0,
                       static_cast<hipStream_t>(stream), u, v, w,
                       Rhs3{(double*)ru, (double*)rv, (double*)rw},
                       Rhs3{(double*)ru_prev, (double*)rv_prev, (double*)rw_prev}, dt, n[0],
                       n[1], n[2]);
    HIP_OK(hipGetLastError());
    return SLC_OK;
}
