// slc_ops_dev.h -- device bodies of the step's field operators, shared by the
// single-run kernels (slc_ops.hip) and the batched ensemble kernels
// (slc_ens_kernels.hip), so both compute the very same arithmetic:
//   ghost/boundary fill            solver.py:70-107, projection.py:180-195
//   theta-method z-diffusion       operators.py:382-630 (Thomas, shared factor)
//   divergence (+transpose)        utils.py:166-180
//   per-wavenumber Poisson Thomas  projection.py:133-247 (coefficients on the fly)
//   gradient projection            projection.py:250-272
//   bulk-flux constraint           solver.py:694-723, utils.py:147-163
// Each body takes its work coordinates explicitly (block or thread index
// within one channel) instead of reading blockIdx.
#pragma once

#include <type_traits>

#include "slc_internal.h"

namespace slc {

// ---------------------------------------------------------------------------
// ghost fill
// ---------------------------------------------------------------------------
// The reference assigns ghost slabs in a fixed order (x, then y, then z), so
// every ghost's final value is +-(one interior value).  Each thread writes one
// ghost entry from its interior source; interiors are only read, so there is
// no ordering hazard.  Entries are enumerated as
//   S1: whole x-ghost planes          (contiguous)
//   S2: y-ghost rows of interior x    (contiguous along z)
//   S3: the two z ends of interior columns.
// Field kinds: 0 u, 1 v, 2 w, 3 p.

struct GhostShape {
    int NI, NJ, NK;
    int nxg, xg0, xg1;  // x-ghost planes
    int nyg, yg0, yg1;  // y-ghost rows
    long S1, S2, S3;
};

__host__ __device__ inline GhostShape ghost_shape(int kind, int nx, int ny, int nz) {
    GhostShape s;
    s.NI = (kind == 0) ? nx + 1 : nx + 2;
    s.NJ = (kind == 1) ? ny + 1 : ny + 2;
    s.NK = (kind == 2) ? nz + 1 : nz + 2;
    if (kind == 0) { s.nxg = 1; s.xg0 = 0; s.xg1 = 0; }
    else { s.nxg = 2; s.xg0 = 0; s.xg1 = nx + 1; }
    if (kind == 1) { s.nyg = 1; s.yg0 = 0; s.yg1 = 0; }
    else { s.nyg = 2; s.yg0 = 0; s.yg1 = ny + 1; }
    s.S1 = (long)s.nxg * s.NJ * s.NK;
    s.S2 = (long)nx * s.nyg * s.NK;
    s.S3 = (long)nx * ny * 2;
    return s;
}

__host__ __device__ inline long ghost_count(int kind, int nx, int ny, int nz) {
    const GhostShape s = ghost_shape(kind, nx, ny, nz);
    return s.S1 + s.S2 + s.S3;
}

__device__ inline void ghost_value(int kind, const Grid& g, const double* F, const GhostShape& s,
                                   int I, int J, int K, double* out_val) {
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    int is = I, js = J, ks = K;
    double sg = 1.0;
    bool zero = false;
    if (I == 0) is = nx;
    else if (kind != 0 && I == nx + 1) is = 1;
    if (J == 0) js = ny;
    else if (kind != 1 && J == ny + 1) js = 1;
    if (kind == 2) {
        if (K == 0 || K == nz) zero = true;
    } else if (kind == 3) {
        if (K == 0) ks = 1;
        else if (K == nz + 1) ks = nz;
    } else {
        if (K == 0) { ks = 1; sg = -1.0; }
        else if (K == nz + 1) { ks = nz; sg = g.top_neumann ? 1.0 : -1.0; }
    }
    double v = zero ? 0.0 : F[((long)is * s.NJ + js) * s.NK + ks];
    *out_val = (sg < 0.0) ? -v : v;
}

// Ghost entry t (0 <= t < ghost_count) of field F of the given kind.
__device__ inline void bc_body(const Grid& g, double* F, int kind, long t) {
    const GhostShape s = ghost_shape(kind, g.nx, g.ny, g.nz);
    int I, J, K;
    if (t < s.S1) {
        long pl = (long)s.NJ * s.NK;
        int p = (int)(t / pl);
        long r = t % pl;
        I = p == 0 ? s.xg0 : s.xg1;
        J = (int)(r / s.NK);
        K = (int)(r % s.NK);
    } else if (t < s.S1 + s.S2) {
        long t2 = t - s.S1;
        long row = t2 / s.NK;
        K = (int)(t2 % s.NK);
        I = 1 + (int)(row / s.nyg);
        J = (row % s.nyg) == 0 ? s.yg0 : s.yg1;
    } else if (t < s.S1 + s.S2 + s.S3) {
        long t3 = t - s.S1 - s.S2;
        long col = t3 >> 1;
        I = 1 + (int)(col / g.ny);
        J = 1 + (int)(col % g.ny);
        K = (t3 & 1) ? s.NK - 1 : 0;
    } else {
        return;
    }
    double v;
    ghost_value(kind, g, F, s, I, J, K, &v);
    F[((long)I * s.NJ + J) * s.NK + K] = v;
}

// Every ghost entry that takes its value from interior point (I, J, K), whose
// value is v (for w at K = nz, which has no interior face: the top wall face):
// with a call per interior point, the ghost fill of bc_body.  The wall entries
// of the own column are two predicated stores; the images of the column in x
// and y are for a few columns of a field.  A fill of its own costs a launch
// and a pass of strided reads per set of fields: with the projection writing
// the ghosts of u, v, w and p, its kernel went from 11.6 to 14.9 us at 64^3
// and from 242 to 274 us at 256^3, and the two fills (2 x 4.8 and 2 x 13 us
// and their launch gaps) went.
__device__ inline void put_ghosts(const Grid& g, double* __restrict__ F, int kind, int I, int J,
                                  int K, double v) {
    const int NJ = kind == 1 ? g.ny + 1 : g.ny + 2, NK = kind == 2 ? g.nz + 1 : g.nz + 2;
    const double lo = kind == 2 ? 0.0 : kind == 3 ? v : -v;
    const double hi = kind == 2 ? 0.0 : kind == 3 || g.top_neumann ? v : -v;
    double* col = F + ((long)I * NJ + J) * NK;
    if (K == 1) col[0] = lo;
    if (K == g.nz) col[NK - 1] = hi;
    const bool x0 = I == g.nx, x1 = kind != 0 && I == 1;
    const bool y0 = J == g.ny, y1 = kind != 1 && J == 1;
    if (!(x0 || x1 || y0 || y1)) return;
    auto image = [&](int X, int Y) {
        double* img = F + ((long)X * NJ + Y) * NK;
        if (kind != 2 || K < g.nz) img[K] = v;
        if (K == 1) img[0] = lo;
        if (K == g.nz) img[NK - 1] = hi;
    };
    if (x0) image(0, J);
    if (x1) image(g.nx + 1, J);
    if (y0) image(I, 0);
    if (y1) image(I, g.ny + 1);
    if ((x0 || x1) && (y0 || y1)) {
        if (x0 && y0) image(0, 0);
        if (x0 && y1) image(0, g.ny + 1);
        if (x1 && y0) image(g.nx + 1, 0);
        if (x1 && y1) image(g.nx + 1, g.ny + 1);
    }
}

// ---------------------------------------------------------------------------
// implicit z-diffusion: (I - theta dt nu Dzz) x = d + (1-theta) dt nu Dzz d
// ---------------------------------------------------------------------------
// The matrix is the same for every (i, j) column, so it is factored once
// (tab = [a | c' | 1/den], n entries each) and every column only runs
// forward/back substitution.  Columns are staged through LDS so the HBM
// traffic is one coalesced read and one coalesced write per unknown.

constexpr int kZColsMax = 16;
constexpr int kZLdsBytes = 48 * 1024;  // dynamic LDS budget per workgroup

__host__ __device__ inline int zsolve_ld(int comp, int nz) {
    const int SZ = comp == 2 ? nz + 1 : nz + 2;
    return SZ + ((SZ & 1) ? 0 : 1);  // odd stride: conflict-free column walk
}

// columns per workgroup (0: a column does not fit the LDS budget)
__host__ __device__ inline int zsolve_cols(int comp, int nz) {
    int cols = kZLdsBytes / (zsolve_ld(comp, nz) * (int)sizeof(double));
    return cols > kZColsMax ? kZColsMax : cols;
}

// Column block cb (kZCols columns) of component C, of S into F (the same array
// or another).  lds: kZCols * ld doubles; cbase: kZColsMax longs.  Ends with a
// barrier-free write-back; the caller synchronises before reusing lds.
template <int C>
__device__ inline void zsolve_body(const Grid& g, const double* S, double* F,
                                   const double* __restrict__ tab, double beta,
                                   const double* __restrict__ dz_c,
                                   const double* __restrict__ dz_f, int kZCols, long cb,
                                   double* __restrict__ lds, long* cbase) {
    const int SZ = (int)Comp<C>::SZ(g);
    const long SY = Comp<C>::SY(g);
    const int ld = zsolve_ld(C, g.nz);
    const int n = (C == 2) ? g.nz - 1 : g.nz;
    const long ncols = (long)g.nx * g.ny;
    const long col0 = cb * kZCols;
    const int tid = threadIdx.x;

    // column base addresses (one 32-bit division per column, not per element)
    if (tid < kZCols) {
        const long gc = col0 + tid;
        long a = -1;
        if (gc < ncols) {
            const unsigned ug = (unsigned)gc;
            const int I = 1 + (int)(ug / (unsigned)g.ny), J = 1 + (int)(ug % (unsigned)g.ny);
            a = ((long)I * SY + J) * SZ;
        }
        cbase[tid] = a;
    }
    __syncthreads();
    // coalesced load of kZCols whole columns (ghost ends included)
    for (int e = tid; e < kZCols * SZ; e += blockDim.x) {
        const int c = e / SZ, k = e - (e / SZ) * SZ;
        const long a = cbase[c];
        if (a >= 0) lds[c * ld + k] = S[a + k];
    }
    __syncthreads();

    if (tid < kZCols && col0 + tid < ncols) {
        double* s = lds + tid * ld;
        if (beta != 0.0) {
            // explicit part, operators.py:446-466 (u, v) and 609-623 (w)
            if (C < 2) {
                double lo = s[0], mid = s[1];
                for (int k = 0; k < n; ++k) {
                    double hi = s[k + 2];
                    double dzl = dz_c[k], dzr = dz_c[k + 1], dzc = dz_f[k];
                    double d2;
                    if (k == 0) {
                        d2 = ((hi - mid) / dzr - 2.0 * mid / dzl) / dzc;
                    } else if (k == n - 1) {
                        if (g.top_neumann) d2 = (-(mid - lo) / dzl) / dzc;
                        else d2 = (-2.0 * mid / dzr - (mid - lo) / dzl) / dzc;
                    } else {
                        d2 = ((hi - mid) / dzr - (mid - lo) / dzl) / dzc;
                    }
                    s[k + 1] = mid + beta * d2;
                    lo = mid;
                    mid = hi;
                }
            } else {
                // the reference's w stencil is centred on face m (not m+1)
                double a = 0.0, b = s[0], c = s[1];
                for (int m = 0; m < n; ++m) {
                    double dzl = dz_f[m], dzr = dz_f[m + 1], dzc = dz_c[m + 1];
                    double d2;
                    if (m == 0) d2 = ((c - b) / dzr - b / dzl) / dzc;
                    else if (m == n - 1) d2 = (-b / dzr - (b - a) / dzl) / dzc;
                    else d2 = ((c - b) / dzr - (b - a) / dzl) / dzc;
                    double nxt = s[m + 2];
                    s[m + 1] = c + beta * d2;
                    a = b;
                    b = c;
                    c = nxt;
                }
            }
        }
        const double* A = tab;
        const double* CP = tab + n;
        const double* INV = tab + 2 * n;
        double dp = s[1] * INV[0];
        s[1] = dp;
        for (int k = 1; k < n; ++k) {
            dp = (s[k + 1] - A[k] * dp) * INV[k];
            s[k + 1] = dp;
        }
        double x = dp;
        for (int k = n - 2; k >= 0; --k) {
            x = s[k + 1] - CP[k] * x;
            s[k + 1] = x;
        }
    }
    __syncthreads();

    for (int e = tid; e < kZCols * SZ; e += blockDim.x) {
        const int c = e / SZ, k = e - (e / SZ) * SZ;
        const long a = cbase[c];
        if (a >= 0 && k >= 1 && k <= n) F[a + k] = lds[c * ld + k];
    }
}

// z-solve of the theta-method, a column at a time per wavefront.  Lane
// l holds unknowns [l CH, (l+1) CH) in registers.  Forward and back
// substitution of the shared factorisation are first-order linear
// recurrences: each lane runs its stretch as an affine map of the value
// entering it (the same operations as the sequential sweep where that value
// is known: lane 0 forward, the lane holding the last unknown backward), the
// 64 maps are composed with a Kogge-Stone scan (6 shuffle steps), and each
// lane applies its entering value.  Every unknown is read and written once;
// a wavefront's loads and stores cover its column's n contiguous doubles.
// Differs from the sequential sweep by rounding only (tridiagonal solves
// carry the 1e-13 tolerance, not bit-exactness).
constexpr int kZScanMaxCh = 16;
constexpr int kZScanCols = 4;  // columns (wavefronts) per 256-thread workgroup

// unknowns per lane (power of two), 0 when the column is too long for the
// register path (n > 64 kZScanMaxCh)
__host__ __device__ inline int zsolve_scan_ch(int comp, int nz) {
    const int n = comp == 2 ? nz - 1 : nz;
    int ch = 1;
    while (ch * 64 < n) ch *= 2;
    return ch <= kZScanMaxCh ? ch : 0;
}

// The level distances of a lane's unknowns, with their reciprocals as pairs
// (quotient) on lanes of up to 4: a wavefront's columns share them.
// Correctly rounded either way; 12 general divisions a column made the
// theta < 1 solve of 256x192x192 60 us where theta = 1 takes 31 (now 45; 256^3
// 98 -> 61).  Longer columns' pairs would not fit the registers.
template <int C, int CH>
struct ZDist {
    static constexpr bool kPairs = CH <= 4;
    double d[CH + 1], m[CH];  // below and above the unknowns, around them
    double dh[kPairs ? CH + 1 : 1], dl[kPairs ? CH + 1 : 1];
    double mh[kPairs ? CH : 1], ml[kPairs ? CH : 1];

    __device__ ZDist(int j0, int n, const double* __restrict__ dz_c,
                     const double* __restrict__ dz_f) {
#pragma unroll
        for (int i = 0; i <= CH; ++i) {
            const int j = j0 + i < n ? j0 + i : n;
            d[i] = C < 2 ? dz_c[j] : dz_f[j];
            if (kPairs) {
                dh[i] = 1.0 / d[i];
                dl[i] = fma(-d[i], dh[i], 1.0) * dh[i];
            }
            if (i == CH) break;
            const int jm = j0 + i < n ? j0 + i : n - 1;
            m[i] = C < 2 ? dz_f[jm] : dz_c[jm + 1];
            if (kPairs) {
                mh[i] = 1.0 / m[i];
                ml[i] = fma(-m[i], mh[i], 1.0) * mh[i];
            }
        }
    }
    __device__ double by_d(double x, int i) const {
        return kPairs ? quotient(x, d[i], dh[i], dl[i]) : x / d[i];
    }
    __device__ double by_m(double x, int i) const {
        return kPairs ? quotient(x, m[i], mh[i], ml[i]) : x / m[i];
    }
};

// Explicit part of the theta-method right-hand side, x_j + beta Dzz x_j, on
// the lane's unknowns (the formulas and operation order of zsolve_body, from
// operators.py:446-466 for u, v and 609-623 for w).  p[i] holds unknown
// j0 + i and, for j0 + i == n, the entry just above the last unknown (the
// top ghost of u, v; the top wall face of w); s0 is the bottom ghost / wall
// face.  Neighbours across lanes come by shuffles (all lanes take part).
template <int C, int CH>
__device__ inline void zsolve_explicit(const Grid& g, double* p, int j0, int n, double beta,
                                       const ZDist<C, CH>& z, double s0) {
    double ext[CH + 3];  // unknowns j0-2 .. j0+CH
    ext[1] = __shfl_up(p[CH - 1], 1);
    ext[0] = CH >= 2 ? __shfl_up(p[CH >= 2 ? CH - 2 : 0], 1) : __shfl_up(p[0], 2);
    ext[CH + 2] = __shfl_down(p[0], 1);
#pragma unroll
    for (int i = 0; i < CH; ++i) ext[i + 2] = p[i];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int j = j0 + i;
        if (j >= n) continue;
        // (x / dzr - y / dzl) / dzc, the walls' cases by x and y
        double x, y, at;
        if (C < 2) {
            const double lo = ext[i + 1], mid = ext[i + 2], hi = ext[i + 3];
            x = hi - mid;
            y = mid - lo;
            if (j == 0) y = 2.0 * mid;
            else if (j == n - 1) x = g.top_neumann ? -0.0 : -2.0 * mid;
            at = mid;
        } else {
            // centred on face j (value b), stored to face j + 1 (value c)
            const double c = ext[i + 2];
            const double b = (j == 0) ? s0 : ext[i + 1];
            const double a = (j == 1) ? s0 : ext[i];
            x = c - b;
            y = b - a;
            if (j == 0) y = b;
            else if (j == n - 1) x = -b;
            at = c;
        }
        const double d2 = z.by_m(z.by_d(x, i + 1) - z.by_d(y, i), i);
        p[i] = at + beta * d2;
    }
}

// Orders the wavefront's LDS accesses (a wavefront executes them in order;
// this keeps the compiler from moving them across).
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS doubles per column of the transposed z-solve (zsolve_run): one
// pad after every CH unknowns, so that lane-contiguous reads of CH values
// spread over the banks.
template <int CH>
__host__ __device__ constexpr int zscan_lds() {
    return 64 * (CH + 1);
}

// The lane's part of the factorisation and of both scans' multipliers: the
// same for every column, so a wavefront that solves several keeps it in
// registers.  a = 0 at unknown 0 and c = 0 at unknown n - 1 end the
// recurrences there.
template <int CH>
struct ZFactor {
    double a[CH], r[CH], c[CH];  // the three tables
    double q[CH], t[CH];         // the affine maps' factors
    double Q[6], T[6];           // their products before each scan step
};

template <int CH>
__device__ inline void zfactor_load(ZFactor<CH>& z, const double* __restrict__ tab, int n,
                                    int lane) {
    const int j0 = lane * CH;
    double qr = 1.0, tr = 1.0;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int j = j0 + i, jl = j < n ? j : n - 1;
        z.a[i] = j == 0 ? 0.0 : tab[jl];
        z.c[i] = j == n - 1 ? 0.0 : tab[n + jl];
        z.r[i] = tab[2 * n + jl];
        if (j < n) qr = j == 0 ? 0.0 : -(z.a[i] * qr) * z.r[i];
        z.q[i] = qr;
    }
#pragma unroll
    for (int i = CH - 1; i >= 0; --i) {
        const int j = j0 + i;
        if (j < n) tr = j == n - 1 ? 0.0 : -(z.c[i] * tr);
        z.t[i] = tr;
    }
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        const int off = 1 << s;
        z.Q[s] = qr;
        z.T[s] = tr;
        const double Qp = __shfl_up(qr, off), Tn = __shfl_down(tr, off);
        if (lane >= off) qr = qr * Qp;
        if (lane + off < 64) tr = tr * Tn;
    }
}

struct ZNoDist {
    __device__ ZNoDist(int, int, const double*, const double*) {}
};

// The columns col, col + stride, .. below end of F, one at a time, the next
// one's loads ahead of the solve.  EXPL: theta < 1, and the columns come from S
// (F or another array; without EXPL S is not read: a second address spilled
// the eight waves of one unknown per lane).  With X (zscan_lds<CH> doubles
// of the wavefront's own LDS) a column moves between HBM and the registers
// through LDS in wavefront-contiguous pieces (each load instruction touches
// 512 consecutive bytes) instead of each lane reading its CH consecutive
// unknowns (an instruction touches every cache line of the column).
// The factorisation's part done once for many columns halves the arithmetic
// and the shuffles of a column and leaves its own bytes as its only loads.
// One column per wavefront and all of it per column: 52 us a component at
// 256x192x192, 88 at 256^3, 707 at 512^3, 578 at 256x256x1000 (2.9, 3.1,
// 3.0, 1.8 TB/s); so 31, 61, 427 and 226 us (4.8, 4.4, 5.0, 4.6 TB/s).
template <int C, int CH, bool EXPL>
__device__ inline void zsolve_run(const Grid& g, const double* S, double* F,
                                  const double* __restrict__ tab, unsigned col, unsigned stride,
                                  unsigned end, double beta = 0.0,
                                  const double* __restrict__ dz_c = nullptr,
                                  const double* __restrict__ dz_f = nullptr,
                                  double* __restrict__ X = nullptr) {
    typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
    const int lane = threadIdx.x & 63;
    const int n = (C == 2) ? g.nz - 1 : g.nz;
    const int j0 = lane * CH;
    const unsigned ny = (unsigned)g.ny;
    unsigned I = col / ny, J = col % ny;
    const unsigned dI = stride / ny, dJ = stride % ny;
    auto column = [&] {
        return F + (((long)(I + 1) * Comp<C>::SY(g) + (J + 1)) * Comp<C>::SZ(g) + 1);
    };
    auto source = [&](const double* Fc) { return EXPL ? S + (Fc - F) : Fc; };
    // raw: through LDS the wavefront's coalesced pieces of the column, else
    // the lane's own unknowns (and the entry above the last one)
    auto load = [&](const double* Fc, double* raw) {
        if (X) {
#pragma unroll
            for (int m = 0; m < CH; ++m) raw[m] = 64 * m + lane <= n ? Fc[64 * m + lane] : 0.0;
        } else if (CH > 1 && j0 + CH - 1 <= n) {
#pragma unroll
            for (int i = 0; i < CH / 2; ++i) {
                const Two d = *reinterpret_cast<const Two*>(Fc + j0 + 2 * i);
                raw[2 * i] = d.x;
                raw[2 * i + 1] = d.y;
            }
        } else {
#pragma unroll
            for (int i = 0; i < CH; ++i) raw[i] = j0 + i <= n ? Fc[j0 + i] : 0.0;
        }
    };
    if (col >= end) return;
    double next[CH];
    double* Fn = column();
    load(source(Fn), next);
    double sn = EXPL ? source(Fn)[-1] : 0.0;
    ZFactor<CH> z;
    zfactor_load(z, tab, n, lane);
    const std::conditional_t<EXPL, ZDist<C, CH>, ZNoDist> dist(j0, n, dz_c, dz_f);
#pragma unroll 1
    while (true) {
        double p[CH];
        double* Fc = Fn;
        const double s0 = sn;
        if (X) {
#pragma unroll
            for (int m = 0; m < CH; ++m) {
                const int e = 64 * m + lane;
                X[e + e / CH] = next[m];
            }
            wave_sync();
#pragma unroll
            for (int i = 0; i < CH; ++i) p[i] = X[lane * (CH + 1) + i];
            wave_sync();
        } else {
#pragma unroll
            for (int i = 0; i < CH; ++i) p[i] = next[i];
        }
        const bool more = col + stride < end;
        if (more) {
            col += stride;
            J += dJ;
            I += dI;
            if (J >= ny) {
                J -= ny;
                ++I;
            }
            Fn = column();
            load(source(Fn), next);
            if (EXPL) sn = source(Fn)[-1];
        }
        if constexpr (EXPL) zsolve_explicit<C, CH>(g, p, j0, n, beta, dist, s0);
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (j0 + i < n) v = (p[i] - z.a[i] * v) * z.r[i];
            p[i] = v;
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            const double Pp = __shfl_up(v, 1 << s);
            if (lane >= 1 << s) v = v + z.Q[s] * Pp;
        }
        double y = __shfl_up(v, 1);
        if (lane == 0) y = 0.0;
        v = 0.0;
#pragma unroll
        for (int i = CH - 1; i >= 0; --i) {
            if (j0 + i < n) v = (p[i] + z.q[i] * y) - z.c[i] * v;
            p[i] = v;
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) {
            const double Rn = __shfl_down(v, 1 << s);
            if (lane + (1 << s) < 64) v = v + z.T[s] * Rn;
        }
        double x = __shfl_down(v, 1);
        if (lane == 63) x = 0.0;
#pragma unroll
        for (int i = 0; i < CH; ++i) p[i] = p[i] + z.t[i] * x;
        if (X) {
#pragma unroll
            for (int i = 0; i < CH; ++i) X[lane * (CH + 1) + i] = p[i];
            wave_sync();
#pragma unroll
            for (int m = 0; m < CH; ++m) {
                const int e = 64 * m + lane;
                if (e < n) Fc[e] = X[e + e / CH];
            }
            wave_sync();
        } else if (CH > 1 && j0 + CH <= n) {
#pragma unroll
            for (int i = 0; i < CH / 2; ++i) {
                Two d;
                d.x = p[2 * i];
                d.y = p[2 * i + 1];
                *reinterpret_cast<Two*>(Fc + j0 + 2 * i) = d;
            }
        } else {
#pragma unroll
            for (int i = 0; i < CH; ++i)
                if (j0 + i < n) Fc[j0 + i] = p[i];
        }
        if (!more) break;
    }
}

// Runtime dispatch of ch (from zsolve_scan_ch, at most MAXCH), theta = 1.
template <int C, int MAXCH>
__device__ inline void zsolve_run_any(const Grid& g, double* F,
                                      const double* __restrict__ tab, unsigned col,
                                      unsigned stride, unsigned end, int ch) {
    switch (ch) {
        case 1: zsolve_run<C, 1, false>(g, F, F, tab, col, stride, end); break;
        case 2: zsolve_run<C, 2, false>(g, F, F, tab, col, stride, end); break;
        case 4:
            if constexpr (MAXCH >= 4) zsolve_run<C, 4, false>(g, F, F, tab, col, stride, end);
            break;
        case 8:
            if constexpr (MAXCH >= 8) zsolve_run<C, 8, false>(g, F, F, tab, col, stride, end);
            break;
        default:
            if constexpr (MAXCH >= 16) zsolve_run<C, 16, false>(g, F, F, tab, col, stride, end);
    }
}

// ---------------------------------------------------------------------------
// divergence -> plane-major (k, i, j) Poisson right-hand side
// ---------------------------------------------------------------------------

constexpr int kT = 32;  // transpose tile edge

// tiles of the (i; j, k) transposes: nx * ceil(ny/kT) * ceil(nz/kT)
__host__ __device__ inline long plane_tiles(int nx, int ny, int nz) {
    return (long)nx * ((ny + kT - 1) / kT) * ((nz + kT - 1) / kT);
}

// tile index -> (i, j0, k0), k-tiles fastest
__device__ inline void plane_tile(const Grid& g, long t, int& i, int& j0, int& k0) {
    const int ntk = (g.nz + kT - 1) / kT, ntj = (g.ny + kT - 1) / kT;
    k0 = (int)(t % ntk) * kT;
    const long r = t / ntk;
    j0 = (int)(r % ntj) * kT;
    i = (int)(r / ntj);
}

// WRAP: the ghost columns and the wall faces of w are not read but taken from
// where a ghost fill takes them (the same values without the fill).
template <bool WRAP>
__device__ inline double divergence_at(const Grid& g, const double* __restrict__ u,
                                       const double* __restrict__ v,
                                       const double* __restrict__ w,
                                       const double* __restrict__ dz_f, int I, int J, int K) {
    const long uSY = g.ny + 2, uSZ = g.nz + 2;
    const long vSY = g.ny + 1, vSZ = g.nz + 2;
    const long wSY = g.ny + 2, wSZ = g.nz + 1;
    const int Im = WRAP && I == 1 ? g.nx : I - 1, Jm = WRAP && J == 1 ? g.ny : J - 1;
    double du = (u[((long)I * uSY + J) * uSZ + K] - u[((long)Im * uSY + J) * uSZ + K]) / g.dx;
    double dv = (v[((long)I * vSY + J) * vSZ + K] - v[((long)I * vSY + Jm) * vSZ + K]) / g.dy;
    long wb = ((long)I * wSY + J) * wSZ;
    const double wt = WRAP && K == g.nz ? 0.0 : w[wb + K];
    const double wl = WRAP && K == 1 ? 0.0 : w[wb + K - 1];
    double dw = (wt - wl) / dz_f[K - 1];
    return du + dv + dw;
}

// tile: kT x (kT+1) doubles of LDS
template <bool WRAP>
__device__ inline void div_planes_body(const Grid& g, const double* __restrict__ u,
                                       const double* __restrict__ v,
                                       const double* __restrict__ w,
                                       const double* __restrict__ dz_f, double scale,
                                       double* __restrict__ planes, int i, int j0, int k0,
                                       double (*tile)[kT + 1]) {
    const int t = threadIdx.x;
    {
        const int kk = t % kT;
        for (int jj = t / kT; jj < kT; jj += 256 / kT) {
            int j = j0 + jj, k = k0 + kk;
            if (j < g.ny && k < g.nz) {
                double d = divergence_at<WRAP>(g, u, v, w, dz_f, i + 1, j + 1, k + 1);
                tile[jj][kk] = d / scale;
            }
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

// ---------------------------------------------------------------------------
// per-wavenumber Thomas (projection.py:199-247 with the matrices of 47-114)
// ---------------------------------------------------------------------------
// dhat: (nz, nx, nky) complex, plane-major; one lane per mode walks k, so a
// wavefront reads 64 consecutive modes (1 KiB) per plane.  c' is kept in a
// real scratch of the same (nz, modes) shape.

__device__ inline void poisson_thomas_body(const PoissonTabs& t, double2* __restrict__ d,
                                           double* __restrict__ cpw, long m) {
    const long M = (long)t.nx * t.nky;
    if (m >= M) return;
    const int nz = t.nz;
    const int i = (int)(m / t.nky), jc = (int)(m % t.nky);
    const double khsq = t.kxsq[i] + t.kysq[jc];
    // row 0 (Neumann bottom; identity row for the (0,0) mode)
    double b = -(t.cs[0] + khsq);
    b += t.cl[0];
    if (nz == 1) b += t.cr[0];
    double c = nz > 1 ? t.cr[0] : 0.0;
    if (m == 0) {
        b = 1.0;
        c = 0.0;
    }
    double cp = c / b;
    double2 dk = d[m];
    double dr = dk.x / b, di = dk.y / b;
    d[m] = make_double2(dr, di);
    cpw[m] = cp;
    for (int k = 1; k < nz; ++k) {
        const double a = t.cl[k];
        double bk = -(t.cs[k] + khsq);
        double ck = 0.0;
        if (k == nz - 1) bk += t.cr[nz - 1];
        else ck = t.cr[k];
        double den = bk - a * cp;
        if (k < nz - 1) cp = ck / den;
        long idx = (long)k * M + m;
        dk = d[idx];
        dr = (dk.x - a * dr) / den;
        di = (dk.y - a * di) / den;
        d[idx] = make_double2(dr, di);
        cpw[idx] = cp;
    }
    double xr = dr, xi = di;
    for (int k = nz - 2; k >= 0; --k) {
        long idx = (long)k * M + m;
        double cpk = cpw[idx];
        dk = d[idx];
        xr = dk.x - cpk * xr;
        xi = dk.y - cpk * xi;
        d[idx] = make_double2(xr, xi);
    }
}

// ---------------------------------------------------------------------------
// per-wavenumber tridiagonal solve by partition (the system of
// poisson_thomas_body, solved in another order: 32 B of memory traffic per
// complex unknown instead of 80)
// ---------------------------------------------------------------------------
// A 256-thread block takes spike_modes(nz) consecutive modes; its threads
// split each mode's nz levels into spike_segs(nz) segments of at most
// kSpikeR levels (thread t: mode t % MB, segment t / MB), so each plane row
// of the block is one contiguous run of MB complex values.  Per segment the
// thread solves, in registers, the segment's rows with the couplings to its
// neighbours removed, for the right-hand side (y) and for the two couplings
// (alpha: unit value one level below the segment, beta: one level above):
//   x = y + alpha L_prev + beta F_next,
// L_prev the last level of the segment below and F_next the first of the
// one above.  One thread per mode then solves the reduced system of the
// segments' first and last levels (a scalar two-term recurrence across the
// segments, forward then back), and every thread forms its levels.  Rows,
// the bottom Neumann row and the (0,0) mode's identity row are those of
// poisson_thomas_body (projection.py:47-114); the partition is exact
// algebra, so the solution agrees to rounding.  Needs nz <= 8 * 256; LDS:
// 256 x 8 doubles.
constexpr int kSpikeR = 8;

__host__ __device__ inline int spike_segs(int nz) {
    int s = 32;
    while (s * kSpikeR < nz) s *= 2;
    return s;
}

// modes per workgroup of NT threads
__host__ __device__ inline int spike_modes(int nz, int NT = 256) { return NT / spike_segs(nz); }

#ifndef SLC_SPIKE_MAX_NZ
#define SLC_SPIKE_MAX_NZ (kSpikeR * 256)
#endif
__host__ __device__ inline bool spike_ok(int nz) { return nz <= SLC_SPIKE_MAX_NZ; }

// row k of the Poisson system of mode m (khsq = kx^2 + ky^2): a (below),
// b (diagonal), c (above), as poisson_thomas_body builds them
__device__ inline void poisson_row(const PoissonTabs& t, long m, double khsq, int k, double& a,
                                   double& b, double& c) {
    const int nz = t.nz;
    if (k == 0) {
        a = 0.0;
        b = -(t.cs[0] + khsq);
        b += t.cl[0];
        if (nz == 1) b += t.cr[0];
        c = nz > 1 ? t.cr[0] : 0.0;
        if (m == 0) {
            b = 1.0;
            c = 0.0;
        }
        return;
    }
    a = t.cl[k];
    b = -(t.cs[k] + khsq);
    c = 0.0;
    if (k == nz - 1) b += t.cr[nz - 1];
    else c = t.cr[k];
}

// NT threads per workgroup (lds: NT * 8 doubles).
template <int NT = 256>
__device__ inline void poisson_spike_body(const PoissonTabs& t, double2* __restrict__ d,
                                          long unit, double* __restrict__ lds) {
    const int nz = t.nz;
    const long M = (long)t.nx * t.nky;
    const int S = spike_segs(nz), MB = NT / S;
    const int R = (nz + S - 1) / S;          // levels per segment (<= kSpikeR)
    const int nseg = (nz + R - 1) / R;       // segments holding levels
    const int ml = threadIdx.x % MB, seg = threadIdx.x / MB;
    const long m = unit * MB + ml;
    const bool live = m < M && seg < nseg;
    const int k0 = seg * R;
    const int nr = live ? min(R, nz - k0) : 0;
    double khsq = 0.0;
    if (live) khsq = t.kxsq[m / t.nky] + t.kysq[m % t.nky];
    double yr[kSpikeR], yi[kSpikeR], al[kSpikeR], be[kSpikeR], cp[kSpikeR];
    // forward elimination of the segment (couplings to the neighbours moved
    // to the alpha / beta right-hand sides)
#pragma unroll
    for (int i = 0; i < kSpikeR; ++i) {
        if (i < nr) {
            const int k = k0 + i;
            double a, b, c;
            poisson_row(t, m, khsq, k, a, b, c);
            const double2 dk = d[(long)k * M + m];
            const double ra = (i == 0) ? -a : 0.0;           // coupling below
            const double rb = (i == nr - 1) ? -c : 0.0;      // coupling above
            if (i == 0) {
                yr[0] = dk.x / b;
                yi[0] = dk.y / b;
                al[0] = ra / b;
                be[0] = rb / b;
                cp[0] = (nr > 1) ? c / b : 0.0;
            } else {
                const double den = b - a * cp[i - 1];
                yr[i] = (dk.x - a * yr[i - 1]) / den;
                yi[i] = (dk.y - a * yi[i - 1]) / den;
                al[i] = (0.0 - a * al[i - 1]) / den;
                be[i] = (rb - a * be[i - 1]) / den;
                cp[i] = (i < nr - 1) ? c / den : 0.0;
            }
        }
    }
#pragma unroll
    for (int i = kSpikeR - 2; i >= 0; --i) {
        if (i < nr - 1) {
            yr[i] -= cp[i] * yr[i + 1];
            yi[i] -= cp[i] * yi[i + 1];
            al[i] -= cp[i] * al[i + 1];
            be[i] -= cp[i] * be[i + 1];
        }
    }
    // the segment's first and last levels for the reduced system
    double* slot = lds + (seg * MB + ml) * 8;
    if (live) {
        slot[0] = yr[0];
        slot[1] = yi[0];
        slot[2] = al[0];
        slot[3] = be[0];
        slot[4] = yr[nr - 1];
        slot[5] = yi[nr - 1];
        slot[6] = al[nr - 1];
        slot[7] = be[nr - 1];
    }
    __syncthreads();
    // reduced system, one thread per mode: with L_{s-1} = P + Q F_s,
    // F_s = U_s + V_s F_{s+1} and L_s = P_s + Q_s F_{s+1}
    if (seg == 0 && m < M) {
        double Pr = 0.0, Pi = 0.0, Q = 0.0;
        for (int s = 0; s < nseg; ++s) {
            double* q = lds + (s * MB + ml) * 8;
            const double y0r = q[0], y0i = q[1], a0 = q[2], b0 = q[3];
            const double y1r = q[4], y1i = q[5], a1 = q[6], b1 = q[7];
            const double D = 1.0 - a0 * Q;
            const double Ur = (y0r + a0 * Pr) / D, Ui = (y0i + a0 * Pi) / D, V = b0 / D;
            const double nPr = y1r + a1 * Pr + a1 * Q * Ur, nPi = y1i + a1 * Pi + a1 * Q * Ui;
            const double nQ = a1 * Q * V + b1;
            q[0] = Ur;
            q[1] = Ui;
            q[2] = V;
            q[4] = nPr;
            q[5] = nPi;
            q[6] = nQ;
            Pr = nPr;
            Pi = nPi;
            Q = nQ;
        }
        double Fr = 0.0, Fi = 0.0;  // F_{s+1}
        for (int s = nseg - 1; s >= 0; --s) {
            double* q = lds + (s * MB + ml) * 8;
            const double Lr = q[4] + q[6] * Fr, Li = q[5] + q[6] * Fi;
            const double nFr = q[0] + q[2] * Fr, nFi = q[1] + q[2] * Fi;
            q[0] = nFr;  // F_s
            q[1] = nFi;
            q[4] = Lr;   // L_s
            q[5] = Li;
            Fr = nFr;
            Fi = nFi;
        }
    }
    __syncthreads();
    if (!live) return;
    double Lr = 0.0, Li = 0.0, Fr = 0.0, Fi = 0.0;
    if (seg > 0) {
        const double* q = lds + ((seg - 1) * MB + ml) * 8;
        Lr = q[4];
        Li = q[5];
    }
    if (seg < nseg - 1) {
        const double* q = lds + ((seg + 1) * MB + ml) * 8;
        Fr = q[0];
        Fi = q[1];
    }
#pragma unroll
    for (int i = 0; i < kSpikeR; ++i) {
        if (i < nr) {
            const double xr = yr[i] + al[i] * Lr + be[i] * Fr;
            const double xi = yi[i] + al[i] * Li + be[i] * Fi;
            d[(long)(k0 + i) * M + m] = make_double2(xr, xi);
        }
    }
}

// ---------------------------------------------------------------------------
// projection u -= dt grad p from the plane-major (unnormalised) inverse FFT
// ---------------------------------------------------------------------------
// Also writes the interior of the ghost-shaped pressure p = P / (nx ny).
// t0: (kT+1) x (kT+2), t1: kT x (kT+1) doubles of LDS.  Each point
// also writes the ghost entries that take their values from it, in place of
// a ghost fill afterwards.

__device__ inline void project_planes_body(const Grid& g, double* __restrict__ u,
                                           double* __restrict__ v, double* __restrict__ w,
                                           const double* __restrict__ P, double inv_n, double dt,
                                           const double* __restrict__ dz_c,
                                           double* __restrict__ p, int i, int j0, int k0,
                                           double (*t0)[kT + 2], double (*t1)[kT + 1]) {
    const int nx = g.nx, ny = g.ny, nz = g.nz;
    const int i1 = (i + 1 == nx) ? 0 : i + 1;
    const int t = threadIdx.x;
    // load (j fastest: plane rows are contiguous in j)
    for (int e = t; e < (kT + 1) * (kT + 1); e += 256) {
        int jj = e % (kT + 1), kk = e / (kT + 1);
        int j = j0 + jj, k = k0 + kk;
        if (k < nz && j <= ny && jj <= kT) {
            int jw = (j == ny) ? 0 : j;
            t0[jj][kk] = P[((long)k * nx + i) * ny + jw];
        }
    }
    for (int e = t; e < kT * kT; e += 256) {
        int jj = e % kT, kk = e / kT;
        int j = j0 + jj, k = k0 + kk;
        if (k < nz && j < ny) t1[jj][kk] = P[((long)k * nx + i1) * ny + j];
    }
    __syncthreads();
    // update (k fastest: fields are z-contiguous)
    const int I = i + 1;
    const int kk = t % kT;
    for (int jj = t / kT; jj < kT; jj += 256 / kT) {
        int j = j0 + jj, k = k0 + kk;
        if (j >= ny || k >= nz) continue;
        const int J = j + 1, K = k + 1;
        double pc = t0[jj][kk] * inv_n;
        double pxp = t1[jj][kk] * inv_n;
        double pyp = t0[jj + 1][kk] * inv_n;
        double un = 0.0, vn = 0.0, wn = 0.0;
        if (u) {
            long ui = ((long)I * (ny + 2) + J) * (nz + 2) + K;
            un = u[ui] - dt * ((pxp - pc) / g.dx);
            u[ui] = un;
            long vi = ((long)I * (ny + 1) + J) * (nz + 2) + K;
            vn = v[vi] - dt * ((pyp - pc) / g.dy);
            v[vi] = vn;
        }
        if (u && k < nz - 1) {
            double pzp = t0[jj][kk + 1] * inv_n;
            long wi = ((long)I * (ny + 2) + J) * (nz + 1) + K;
            wn = w[wi] - dt * ((pzp - pc) / dz_c[K]);
            w[wi] = wn;
        }
        if (p) p[((long)I * (ny + 2) + J) * (nz + 2) + K] = pc;
        if (u) {
            put_ghosts(g, u, 0, I, J, K, un);
            put_ghosts(g, v, 1, I, J, K, vn);
            put_ghosts(g, w, 2, I, J, K, wn);
        }
        if (p) put_ghosts(g, p, 3, I, J, K, pc);
    }
}

// ---------------------------------------------------------------------------
// bulk velocity and the exact flux shift
// ---------------------------------------------------------------------------
// sum_{ijk} u_ijk * (dx dy dz_f[k]) / V, reduced over a fixed partition and a
// fixed tree (deterministic).  scal: [0] correction, [1] forcing, [2] u_bulk
// after the shift, [3] u_bulk before it.

constexpr int kRedBlock = 256;

__host__ __device__ inline int bulk_blocks(int nx, int ny, int nz) {
    long N = (long)nx * ny * nz;
    long nb = (N + kRedBlock * 8 - 1) / (kRedBlock * 8);
    return (int)(nb < 2048 ? nb : 2048);
}

// red: kRedBlock doubles of LDS; every thread gets the block sum
__device__ inline double block_sum(double v, double* red) {
    __syncthreads();
    red[threadIdx.x] = v;
    __syncthreads();
    for (int s = kRedBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    return red[0];
}

// Partial sum number blk of nb over u*cv, on every thread; SHIFT: u += corr
// first, and the ghost entries of the shifted values are written.
template <bool SHIFT>
__device__ inline double bulk_partial_body(const Grid& g, double* __restrict__ u,
                                           const double* __restrict__ cv, double corr, long blk,
                                           long nb, double* red) {
    const long N = (long)g.nx * g.ny * g.nz;
    const long chunk = (N + nb - 1) / nb;
    const long beg = blk * chunk;
    const long end = beg + chunk < N ? beg + chunk : N;
    double acc = 0.0;
    long n = beg + threadIdx.x;
    if (n < end) {
        // (i, j, k) of the first element, then steps of kRedBlock elements in
        // the mixed radix (ny, nz): dk < nz and dj < ny, so one carry per
        // digit suffices.  Same elements in the same order as a division per
        // element.
        const unsigned un = (unsigned)n;
        int k = (int)(un % (unsigned)g.nz);
        const unsigned r = un / (unsigned)g.nz;
        int j = (int)(r % (unsigned)g.ny), i = (int)(r / (unsigned)g.ny);
        const int dk = kRedBlock % g.nz, t = kRedBlock / g.nz;
        const int dj = t % g.ny, di = t / g.ny;
        // kB elements at a time, so that their loads are in flight together
        // (the shift's stores would hold back each next load)
        constexpr int kB = 4;
        while (n < end) {
            double val[kB];
            long ui[kB];
            int ii[kB], jj[kB], kk[kB];
#pragma unroll
            for (int b = 0; b < kB; ++b) {
                ii[b] = i;
                jj[b] = j;
                kk[b] = k;
                ui[b] = ((long)(i + 1) * (g.ny + 2) + (j + 1)) * (g.nz + 2) + (k + 1);
                val[b] = n + b * kRedBlock < end ? u[ui[b]] : 0.0;
                k += dk;
                if (k >= g.nz) {
                    k -= g.nz;
                    ++j;
                }
                j += dj;
                if (j >= g.ny) {
                    j -= g.ny;
                    ++i;
                }
                i += di;
            }
#pragma unroll
            for (int b = 0; b < kB; ++b) {
                if (n + b * kRedBlock >= end) break;
                if (SHIFT) {
                    val[b] = val[b] + corr;
                    u[ui[b]] = val[b];
                    put_ghosts(g, u, 0, ii[b] + 1, jj[b] + 1, kk[b] + 1, val[b]);
                }
                acc += val[b] * cv[kk[b]];
            }
            n += kB * kRedBlock;
        }
    }
    return block_sum(acc, red);
}

// The count of the blocks that have finished the shift, behind both sums.
__device__ inline unsigned* bulk_ticket(double* partials, int np) {
    return reinterpret_cast<unsigned*>(partials + 2 * np);
}

// First pass, block blk of np.
__device__ inline void bulk_before_body(const Grid& g, const double* u,
                                        const double* __restrict__ cv, double* partials, int blk,
                                        int np, double* red) {
    const double s = bulk_partial_body<false>(g, const_cast<double*>(u), cv, 0.0, blk, np, red);
    if (threadIdx.x != 0) return;
    partials[blk] = s;
    if (blk == 0) *bulk_ticket(partials, np) = 0u;
}

// The np partial sums over the volume, on every thread (a fixed tree).  AGENT:
// the partials were written by other blocks of this launch.
template <bool AGENT = false>
__device__ inline double bulk_mean(const double* partials, int np, double total_volume,
                                   double* red) {
    double acc = 0.0;
    for (int b = threadIdx.x; b < np; b += kRedBlock)
        acc += AGENT ? __hip_atomic_load(partials + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                     : partials[b];
    return block_sum(acc, red) / total_volume;
}

// Second pass, block blk of np: every block forms the mean from the partial
// sums (a few thousand cached loads in place of a launch of its own), shifts
// its chunk and the ghost entries that follow it, and sums the shifted
// values.  The last block to finish forms the mean after the shift, fills
// scal -- [0] correction, [1] forcing, [2] mean after the shift, [3] before
// it -- and returns true (on every thread).  The sums cross blocks as
// agent-scope accesses, each ahead of its block's ticket.  The order rests on
// gfx950, not on the language's memory model: there an agent-scope store has
// reached the device's point of coherence once vmcnt has counted it, so the
// wait before the ticket publishes the sum.  A release at agent scope would
// also write back the shifted values of the whole L2 with every block.
// Two launches in place of five (sums, mean, shift and sums, mean, ghosts):
// 24 -> 14 us at 64^3, 120 -> 117 us at 256^3 (bound by memory there).
__device__ inline bool bulk_shift_body(const Grid& g, double* __restrict__ u,
                                       const double* __restrict__ cv, double* partials, int blk,
                                       int np, double total_volume, double U_bulk, double dt,
                                       double* __restrict__ scal, double* red, bool* last) {
    const double ub = bulk_mean(partials, np, total_volume, red);
    const double corr = U_bulk - ub;
    double* after = partials + np;
    const double s = bulk_partial_body<true>(g, u, cv, corr, blk, np, red);
    if (threadIdx.x == 0) {
        __hip_atomic_store(after + blk, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        *last = __hip_atomic_fetch_add(bulk_ticket(partials, np), 1u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT) == (unsigned)np - 1u;
    }
    __syncthreads();
    if (!*last) return false;
    const double ua = bulk_mean<true>(after, np, total_volume, red);
    if (threadIdx.x == 0) {
        scal[0] = corr;
        scal[1] = corr / dt;
        scal[2] = ua;
        scal[3] = ub;
    }
    return true;
}

}  // namespace slc
