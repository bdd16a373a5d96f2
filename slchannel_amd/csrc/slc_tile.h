// slc_tile.h -- the LDS-tiled "trace, then gather" tile of the semi-Lagrangian
// step, shared by the single-run kernels (slc_step.hip) and the batched
// ensemble kernels (slc_ens_kernels.hip).
//
// One kernel template covers the four uses of "trace, then gather":
//   MODE_ADVECT  foot at dt of the given trajectory velocity, gather F
//                (SLAdvector.advect, semilag.py:584-671)
//   MODE_BDF1    as ADVECT with U* = V^n, plus dt * nu L_xy V^n
//                (solver.py:737-765)
//   MODE_FAR     BOTH feet of the frozen U* (depths dt and 2dt, each an
//                independent iterated midpoint from the arrival point; their
//                first sample, at the arrival point itself, is shared), the
//                near foot stored for MODE_NEAR, V^{n-1} gathered at the far
//                foot into out                          (solver.py:870-882)
//   MODE_NEAR    V^n gathered at the stored near foot, then
//                out = 4/3 near - 1/3 out + (2dt/3)(2 R^n - R^{n-1})
//                                                       (solver.py:885-903)
//   MODE_BDF2    MODE_FAR and MODE_NEAR in one pass: the near foot's stencil
//                waits in LDS while the far box is staged and contracted,
//                then the near box is staged into the same buffer; the far
//                value stays in a register.  The same operations as the two
//                passes, so the same doubles, without the near foot and the
//                far value going through HBM.
// A workgroup owns a TI x TJ x TK tile of arrival points (z fastest).  Phase 1
// traces the tile's feet and keeps each foot's stencil (base indices,
// fractional offsets, clamped z) in registers; the tile's stencil bounding
// box (its trajectory-CFL halo, measured) is reduced and staged in LDS; phase 2
// contracts every P^3 stencil from LDS (z, then y, then x, with FMAs -- the
// same order as the direct gather).
//
// What bounds it (fused BDF2 pass of u, 256^3, order 6; counters per
// wavefront): 2272 VALU instructions (74% of the launch; half of them FP64),
// 216 stencil values per foot from LDS (62%), the trajectory corners and z
// tables through the vector cache (78%): no unit is full, four waves per SIMD
// (128 VGPRs) do not hide the rest.  Measured with the index arithmetic in 32
// bits and scalar registers, the row stride on the LDS banks and the boxes in
// direct-to-LDS pieces: 1.61 -> 1.40 ms (w, whose odd rows went through
// registers, 1.70 -> 1.48), order 4 with FP32 storage at 256x192x160
// 0.63 -> 0.55 ms, advection of a component at 768x768x180, order 4,
// 4.36 -> 3.74 ms.
#pragma once

#include <climits>

#include "slc_device.h"
#include "slc_internal.h"

namespace slc {

// threads per workgroup (compile-time overridable for tile sweeps)
#ifndef SLC_TILE_NT
#define SLC_TILE_NT 256
#endif
constexpr int kSB = SLC_TILE_NT;

// threadIdx.x, opaque to the optimiser: what a phase derives from it is
// formed there, not formed once at entry and spilled in between.
__device__ inline int phase_tid() {
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

enum { MODE_ADVECT = 0, MODE_BDF1 = 1, MODE_FAR = 2, MODE_NEAR = 3, MODE_GATHER = 4,
       MODE_BDF2 = 5 };

// Foot coordinates of one component (flat arrival order): written by
// MODE_FAR (near feet), read by MODE_NEAR and MODE_GATHER.
struct Feet {
    double* x;
    double* y;
    double* z;
};

struct SBox {
    int xmin, xmax, ymin, ymax, kmin, kmax;
};

// Wavefront min / max with DPP lane moves (registers only): swaps within
// quads, half-row and row mirrors give every lane its 16-lane row's value;
// row broadcasts of lanes 15 and 31 fold the rows into lane 63, read back as
// a uniform value.  A lane with no DPP source receives the operation's
// identity (INT_MAX for min, INT_MIN for max), which lets the compiler fold
// each lane move into the min / max itself (one DPP-modified instruction).
template <bool MIN>
__device__ inline int s_wave_reduce(int v) {
    constexpr int id = MIN ? INT_MAX : INT_MIN;
    auto op = [](int a, int b) { return MIN ? min(a, b) : max(a, b); };
    v = op(v, __builtin_amdgcn_update_dpp(id, v, 0xB1, 0xF, 0xF, false));   // quad_perm 1,0,3,2
    v = op(v, __builtin_amdgcn_update_dpp(id, v, 0x4E, 0xF, 0xF, false));   // quad_perm 2,3,0,1
    v = op(v, __builtin_amdgcn_update_dpp(id, v, 0x141, 0xF, 0xF, false));  // row_half_mirror
    v = op(v, __builtin_amdgcn_update_dpp(id, v, 0x140, 0xF, 0xF, false));  // row_mirror
    v = op(v, __builtin_amdgcn_update_dpp(id, v, 0x142, 0xA, 0xF, false));  // row_bcast:15
    v = op(v, __builtin_amdgcn_update_dpp(id, v, 0x143, 0xC, 0xF, false));  // row_bcast:31
    return __builtin_amdgcn_readlane(v, 63);
}

__device__ inline int s_wave_min(int v) { return s_wave_reduce<true>(v); }

__device__ inline int s_wave_max(int v) { return s_wave_reduce<false>(v); }

constexpr int kTileWaves = kSB / 64;

// The workgroup unions of the lanes' boxes, without atomics: every wavefront
// reduces its lanes' boxes in registers and leaves them in red; after one
// barrier (the caller's) box_union reads them back as wave-uniform values.
struct BoxRed {
    int v[2][kTileWaves][8];
};

__device__ inline void box_reduce(const SBox& l, int (&dst)[kTileWaves][8]) {
    const int v0 = s_wave_min(l.xmin), v1 = s_wave_max(l.xmax), v2 = s_wave_min(l.ymin),
              v3 = s_wave_max(l.ymax), v4 = s_wave_min(l.kmin), v5 = s_wave_max(l.kmax);
    if ((threadIdx.x & 63) == 0) {
        int* d = dst[threadIdx.x >> 6];
        *reinterpret_cast<int4*>(d) = make_int4(v0, v1, v2, v3);
        *reinterpret_cast<int2*>(d + 4) = make_int2(v4, v5);
    }
}

__device__ inline SBox box_union(const int (&src)[kTileWaves][8]) {
    int r[6];
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) {
        const int4 a = *reinterpret_cast<const int4*>(src[w]);
        const int2 c = *reinterpret_cast<const int2*>(src[w] + 4);
        r[0] = w ? min(r[0], a.x) : a.x;
        r[1] = w ? max(r[1], a.y) : a.y;
        r[2] = w ? min(r[2], a.z) : a.z;
        r[3] = w ? max(r[3], a.w) : a.w;
        r[4] = w ? min(r[4], c.x) : c.x;
        r[5] = w ? max(r[5], c.y) : c.y;
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) r[q] = __builtin_amdgcn_readfirstlane(r[q]);
    return SBox{r[0], r[1], r[2], r[3], r[4], r[5]};
}

// Element i of p, addressed by a byte offset in 32 bits (one scalar base and
// one lane offset per load, no 64-bit lane arithmetic) when every field of the
// grid is below 4 GiB; BIG: in 64 bits.
template <bool BIG, typename T>
__device__ inline T* elem(T* p, unsigned i) {
    if (BIG) return p + (size_t)i;
    return reinterpret_cast<T*>(
        const_cast<char*>(reinterpret_cast<const char*>(p)) + (size_t)(i * (unsigned)sizeof(T)));
}

// Two consecutive doubles as one 16-byte load (8-byte aligned).
struct __attribute__((packed, aligned(8))) Pair {
    double a, b;
};

template <bool BIG>
__device__ inline Pair pair_at(const double* p, unsigned i) {
    return *reinterpret_cast<const Pair*>(elem<BIG>(p, i));
}

// The two trilinear columns of one axis: wrapped node indices i0, i1 of the
// cell and the fraction t in it.
struct Cell {
    int i0, i1;
    double t;
};

// Wrap by unsigned minima: for f in [-n, 2n) the first one adds a period to
// a negative f, the second takes one from an f >= n (the other candidate is
// then beyond 2^31).  *far collects lanes where f lies farther out.
__device__ inline Cell cell_of(double s, int n) {
    const double fl = floor(s);
    const unsigned un = (unsigned)n, f = (unsigned)floor_int(fl);
    unsigned r = min(f, f + un);
    r = min(r, r - un);
    const unsigned r1 = min(r + 1u, r + 1u - un);
    return Cell{(int)r, (int)r1, s - fl};
}

__device__ inline void cell_far(double s, int n, Cell& c) {
    const int f = floor_int(floor(s));
    c.i0 = wrap_far(f, n);
    c.i1 = c.i0 + 1 == n ? 0 : c.i0 + 1;
}

// x and y cells of a point for nodes on faces (shift 0) and centres (shift
// -1/2): u sits at (x face, y centre), v at (x centre, y face), w at (x
// centre, y centre), so four cells serve the three components.
struct XYCells {
    Cell xf, xc, yf, yc;
};

__device__ inline XYCells xy_cells(const Grid& g, double xdx, double ydy) {
    XYCells q;
    const double xh = xdx + -0.5, yh = ydy + -0.5;
    q.xf = cell_of(xdx, g.nx);
    q.xc = cell_of(xh, g.nx);
    q.yf = cell_of(ydy, g.ny);
    q.yc = cell_of(yh, g.ny);
    const bool far = max((unsigned)q.xf.i0, (unsigned)q.xc.i0) >= (unsigned)g.nx ||
                     max((unsigned)q.yf.i0, (unsigned)q.yc.i0) >= (unsigned)g.ny;
    if (__builtin_expect(far, 0)) {
        // a point more than one period outside the domain, or not finite
        cell_far(xdx, g.nx, q.xf);
        cell_far(xh, g.nx, q.xc);
        cell_far(ydy, g.ny, q.yf);
        cell_far(yh, g.ny, q.yc);
    }
    return q;
}

// The eight corner values of component C's trilinear cell: (i, j) columns,
// levels k0, k0 + 1.  Without BIG the indices and strides are below 2^24
// (big_index), so the products are full-rate 24-bit ones (a 32-bit product
// takes four times as long).  PACKED: a (nx, ny, levels) node buffer.
template <int C, bool BIG, bool PACKED>
__device__ inline void cell_cols(const Grid& g, const double* F, const Cell& x, const Cell& y,
                                 int k0, Pair (&v)[2][2]) {
    const unsigned SZ = (unsigned)Comp<C>::SZ(g);
    const unsigned PS = (unsigned)(PACKED ? g.ny : Comp<C>::SY(g)) * SZ;
    const double* base =
        PACKED ? F : F + ((size_t)Comp<C>::ox * PS + (size_t)Comp<C>::oy * SZ);
    auto mul = [](int a, unsigned b) { return BIG ? (unsigned)a * b : __umul24((unsigned)a, b); };
    const unsigned x0 = mul(x.i0, PS), x1 = mul(x.i1, PS);
    const unsigned y0 = mul(y.i0, SZ) + (unsigned)k0, y1 = mul(y.i1, SZ) + (unsigned)k0;
    v[0][0] = pair_at<BIG>(base, x0 + y0);
    v[0][1] = pair_at<BIG>(base, x0 + y1);
    v[1][0] = pair_at<BIG>(base, x1 + y0);
    v[1][1] = pair_at<BIG>(base, x1 + y1);
}

// The sequential (i, j, k) sum of the trilinear sample (semilag.py:44-59) with
// the order-2 weights (1 - t, t) of the cells: the terms and the order of
// trilinear<C> (slc_device.h), so the same doubles.
__device__ inline double cell_sum(const Cell& x, const Cell& y, const double (&wz)[2],
                                  const Pair (&v)[2][2]) {
    const double wx[2] = {1.0 - x.t, x.t}, wy[2] = {1.0 - y.t, y.t};
    double out = 0.0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const double wij = wx[i] * wy[j];
            const double t0 = (wij * wz[0]) * v[i][j].a, t1 = (wij * wz[1]) * v[i][j].b;
            out = (i == 0 && j == 0) ? t0 : out + t0;
            out = out + t1;
        }
    return out;
}

// Trajectory samples of the three U* components at (xdx, ydy) = (x/dx, y/dy)
// and the clamped z, whose face interval c and centre node interval m are
// known (semilag.py:512-528 recomputes them per component with identical
// results).  TV: TrajA or TrajNodes.
template <bool BIG, typename TV>
__device__ inline void sample3_at(const Grid& g, const TV& V, double xdx, double ydy,
                                  double zc, int c, int m, double& us, double& vs, double& ws) {
    const XYCells q = xy_cells(g, xdx, ydy);
    const Pair nf = pair_at<false>(g.z_f, (unsigned)c), nc = pair_at<false>(g.z_c, (unsigned)m);
    const Pair pc = pair_at<false>(g.dinv_c2, 2u * (unsigned)m);
    const Pair pf = pair_at<false>(g.dinv_f2, 2u * (unsigned)c);
    Pair uv[2][2], vv[2][2], wv[2][2];
    cell_cols<0, BIG, TV::packed>(g, V.a[0], q.xf, q.yc, m, uv);
    cell_cols<1, BIG, TV::packed>(g, V.a[1], q.xc, q.yf, m, vv);
    cell_cols<2, BIG, TV::packed>(g, V.a[2], q.xc, q.yc, c, wv);
    const double wzc[2] = {(zc - nc.b) * pc.a, (zc - nc.a) * pc.b};
    const double wzf[2] = {(zc - nf.b) * pf.a, (zc - nf.a) * pf.b};
    us = cell_sum(q.xf, q.yc, wzc, uv);
    vs = cell_sum(q.xc, q.yf, wzc, vv);
    ws = cell_sum(q.xc, q.yc, wzf, wv);
}

// sample3_at for a point whose z interval is not known, in one round of
// loads, for a point traced from the arrival
// (za, K) of component C.  The face interval c and the centred components'
// node interval m = c + s (s: z >= z_c[c+1]) are predicted without loads, and
// the faces, centre nodes, inverse denominators and the three components'
// columns of that prediction are read at once (every index inside its table
// or field for c in [0, nz-1], s in {0, 1}).  Near the arrival the
// prediction is exact: for C = u, v, za = z_c[K] is the split of face
// interval K-1; for C = w, za = z_f[K] is the face between intervals K-1 and
// K.  Elsewhere c is the float estimate of face_cell_fast and s comes from
// split_predict.  The loaded faces and centre then decide: where they confirm
// the prediction and z is outside the faces' 1e-10 band, c is the interval
// face_cell_fast returns (the one interval bracketing z) and m the node
// interval of locate_split.  Otherwise (a few lanes in 1e5 on stretched
// production grids) c and m are located as face_cell_fast does and the values
// read again.  Either way the sums are the same operations on the same
// values as with a located interval.
template <int C, bool BIG, typename TV>
__device__ inline void sample3(const Grid& g, const TV& V, double x, double y, double z,
                               double za, int K, double& us, double& vs, double& ws) {
    const double zc = clampd(z, g.z_lo, g.z_hi);
    const XYCells q = xy_cells(g, over_dx(g, x), over_dy(g, y));
    float kfe, a;
    int c = face_estimate(g, zc, kfe, a);
    if (!Comp<C>::centers && (c == K - 1 || c == K)) c = zc >= za ? K : K - 1;
    bool s = split_predict(g, c, kfe, a);
    if (Comp<C>::centers && c == K - 1) s = zc >= za;
    int m = c + (s ? 1 : 0);
    for (bool located = false;; located = true) {
        const Pair nf = pair_at<false>(g.z_f, (unsigned)c);
        const Pair nc = pair_at<false>(g.z_c, (unsigned)m);
        const Pair pc = pair_at<false>(g.dinv_c2, 2u * (unsigned)m);
        const Pair pf = pair_at<false>(g.dinv_f2, 2u * (unsigned)c);
        Pair uv[2][2], vv[2][2], wv[2][2];
        cell_cols<0, BIG, TV::packed>(g, V.a[0], q.xf, q.yc, m, uv);
        cell_cols<1, BIG, TV::packed>(g, V.a[1], q.xc, q.yf, m, vv);
        cell_cols<2, BIG, TV::packed>(g, V.a[2], q.xc, q.yc, c, wv);
        const double split = m > c ? nc.a : nc.b;  // z_c[c + 1]
        if (located || (face_estimate_holds(g, c, zc, nf.a, nf.b) && (zc >= split) == (m > c))) {
            const double wzc[2] = {(zc - nc.b) * pc.a, (zc - nc.a) * pc.b};
            const double wzf[2] = {(zc - nf.b) * pf.a, (zc - nf.a) * pf.b};
            us = cell_sum(q.xf, q.yc, wzc, uv);
            vs = cell_sum(q.xc, q.yf, wzc, vv);
            ws = cell_sum(q.xc, q.yc, wzf, wv);
            return;
        }
        double sp;
        c = face_cell_fast(g, zc, sp);
        m = locate_split<0>(c, sp, zc);
    }
}

// Per-foot stencil data kept between the phases.
struct FootSt {
    int bx, by, bk;      // unwrapped x/y base, clamped z base
    double tx, ty, z;    // fractional offsets, clamped z
};

template <int C, int P>
__device__ inline void make_st(const Grid& g, double x, double y, double z, FootSt& f,
                               int& ncl) {
    ncl += (z < g.z_lo || z > g.z_hi) ? 1 : 0;
    f.z = clampd(z, g.z_lo, g.z_hi);
    stencil_base<C, P>(g, x, y, f.z, f.bx, f.by, f.bk, f.tx, f.ty);
}

// How a tile's stencil box reaches the contraction (uniform over the block):
//   whole   the box in LDS with row stride kLZ: the usual case (the stencils of
//           a 16-level tile span 20-23 levels at the usual CFL)
//   slabs   the box goes through LDS in runs of x planes, each staged with
//           the box's own z extent; a lane adds its stencil planes as they
//           come by.  Boxes over the LDS budget (high CFL, rough fields)
//   direct  loads from memory, when not even one plane fits (feet far apart
//           or not finite)
// Every way adds the same products in the same order, so the doubles agree.
//
// kLZ = 32 doubles: a multiple of the 64 LDS banks, so the bank of a value
// depends on its level alone and the 16 consecutive levels that 16 lanes read
// do not collide when some of their columns lie in another row (a stride of
// 24 took 1.57 ms per fused pass of u at 256^3, order 6, this one 1.45 ms; the
// unpadded box extent 1.54 ms).
constexpr int kLZ = 32;

enum { BOX_NONE = 0, BOX_WHOLE, BOX_SLABS, BOX_DIRECT };

constexpr int kFar = 1 << 30;  // bases beyond: x0 + x could leave 32 bits

struct BoxPlan {
    int how;
    int x0, y0, k0;   // first node of the box (x, y before the periodic wrap)
    int BX, BY, BZ;   // extents
    int LD;           // row stride in LDS: kLZ (whole), else the slabs' own
    int ns;           // planes per slab
    int pairs;        // staged in 16-byte pieces (double fields)
    int ax, ay, c;    // level k of row (x, y) sits at k - k0 + ((ax x + ay y + c) & 1)
};

// Double fields are staged in aligned 16-byte pieces, two levels each.  Row
// (x, y) starts at element (rowidx SZ + k0) of the field, whose parity (and
// that of the field's base address) decides whether its pieces start at level
// k0 or k0 - 1; the row is shifted in LDS accordingly.  Rows of even length
// (u, v at even nz) all shift alike, rows of odd length (w there) by turns in
// y, and in x too when a plane holds an odd number of rows; a wrapped box
// keeps the turns where the period is even.  A piece may reach one or two
// elements out of its row, into a neighbouring row of the field (the first
// and last rows of a field are ghost rows, never staged).  A row's pieces are
// one load of a wavefront: rows of more than kPairRow doubles go in 4-byte
// pieces, unshifted.
constexpr int kPairRow = 128;

template <typename T, int C, int P>
__device__ inline BoxPlan plan_box(const Grid& g, const T* S, const SBox& b, int cap_bytes) {
    BoxPlan r{BOX_NONE, b.xmin, b.ymin, b.kmin, 0, 1, 1, 1, 0, 0, 0, 0, 0};
    if (b.xmin > b.xmax) return r;  // no live point
    r.how = BOX_DIRECT;
    // extents in 64 bits, each bounded before a product: feet far outside
    // the domain (or non-finite ones, whose floors saturate) would overflow
    // int extents and take the direct loads
    const long ex = (long)b.xmax - b.xmin + P, ey = (long)b.ymax - b.ymin + P;
    const int ez = b.kmax - b.kmin + P;  // bases are clamped to the column
    const long cap = cap_bytes / (int)sizeof(T);
    if (ex > 65536 || ey > cap || b.xmin < -kFar || b.xmax > kFar || b.ymin < -kFar ||
        b.ymax > kFar)
        return r;
    r.BX = (int)ex;
    r.BY = (int)ey;
    r.BZ = ez;
    int ld = ez;
    if (sizeof(T) == 8) {
        const int SZ = (int)Comp<C>::SZ(g), SY = (int)Comp<C>::SY(g);
        const int ay = SZ & 1, ax = SZ & SY & 1;
        const bool oky = !ay || g.ny % 2 == 0 || (b.ymin >= 0 && b.ymin + r.BY <= g.ny);
        const bool okx = !ax || g.nx % 2 == 0 || (b.xmin >= 0 && b.xmin + r.BX <= g.nx);
        if (okx && oky) {
            r.pairs = 1;
            r.ax = ax;
            r.ay = ay;
            const int row0 = (wrap_idx(b.xmin, g.nx) + Comp<C>::ox) * SY +
                             wrap_idx(b.ymin, g.ny) + Comp<C>::oy;
            r.c = (int)((reinterpret_cast<uintptr_t>(S) >> 3) + (unsigned)(row0 * SZ + b.kmin)) & 1;
            ld = (ez + (ay | r.c) + 1) & ~1;
        }
    }
    if (ld <= kLZ && ex * ey * kLZ <= cap) {
        r.how = BOX_WHOLE;
        r.LD = kLZ;
        r.ns = r.BX;
        return r;
    }
    if (ld > kPairRow) {  // no pieces, so no row shifted
        r.pairs = r.ax = r.ay = r.c = 0;
        ld = ez;
    }
    // past eight slabs the box holds about as many values as the stencils do
    if (ey * ld > cap || ex * ey * ld > 8 * cap) return r;
    r.how = BOX_SLABS;
    r.LD = ld;
    // planes per slab: floor by a float reciprocal, corrected by one (both
    // below 2^24, so the error is below one)
    const int pl = r.BY * ld;
    int ns = (int)((float)cap / (float)pl);
    if ((long)ns * pl > cap) --ns;
    r.ns = min(max(ns, 1), r.BX);
    return r;
}

// Boxes of doubles are staged by gfx950's direct global-to-LDS loads (no
// register round trip, no vector arithmetic per load): lane l of a wavefront's
// load lands 16 l (4 l) bytes behind the wave-uniform LDS address.  staged()
// waits for them.
__device__ inline void load16_to_lds(const void* src, void* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

__device__ inline void load4_to_lds(const void* src, void* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)lds, 4, 0, 0);
}

__device__ inline void staged() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// Planes [s0, s0 + n) of the box in 16-byte pieces.  A wavefront takes every
// kTileWaves-th plane, RPI rows of LD / 2 pieces per load (lane = rr LD / 2 +
// zp; the pieces that hold levels of the box are loaded), so a plane's address
// is scalar and a row's offset is formed once for all planes (twice where the
// shift turns in x).
template <int C, bool BIG>
__device__ inline void stage_pairs(const Grid& g, const double* __restrict__ S, const BoxPlan& b,
                                   int s0, int n, int LD, int RPI, int tid, int rr, int zp,
                                   double* __restrict__ lds) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned SZ = (unsigned)Comp<C>::SZ(g), SY = (unsigned)Comp<C>::SY(g);
    for (int y0 = 0; y0 < b.BY; y0 += RPI) {
        const int y = y0 + rr;
        const int sh = (b.ay * y + b.c + b.ax * (s0 + wave)) & 1;  // kTileWaves is even
        if (rr >= RPI || y >= b.BY || 2 * zp >= b.BZ + sh) continue;
        const int yg = wrap_idx(b.y0 + y, g.ny);
        const unsigned off = (BIG ? (unsigned)yg * SZ : __umul24((unsigned)yg, SZ)) +
                             (unsigned)(2 * zp - sh);
        for (int x = wave; x < n; x += kTileWaves) {
            const int xg = wrap_idx(b.x0 + s0 + x, g.nx);
            const double* plane = S + (((unsigned)(xg + Comp<C>::ox) * SY + Comp<C>::oy) * SZ +
                                       (unsigned)b.k0);
            load16_to_lds(plane + (long)(int)off, lds + (x * b.BY + y0) * LD);
        }
    }
}

// Planes [s0, s0 + n) of the box into rows of LD elements, in 4-byte pieces: a
// row of up to 64 of them per load (any alignment and extent), rows dealt
// round robin to the wavefronts, addresses scalar but for the lane's place in
// the row.
template <typename T, int C>
__device__ inline void stage_rows(const Grid& g, const T* __restrict__ S, const BoxPlan& b,
                                  int s0, int n, int LD, T* __restrict__ lds) {
    const int tid = phase_tid();
    const unsigned lane = (unsigned)tid & 63u;
    const unsigned nd = (unsigned)b.BZ * (unsigned)(sizeof(T) / 4);
    const unsigned SZ = (unsigned)Comp<C>::SZ(g), SY = (unsigned)Comp<C>::SY(g);
    for (unsigned d = 0; d < nd; d += 64) {  // one turn but for boxes over 32 levels
        if (d + lane >= nd) break;
        // row (x, y): y advances by kTileWaves <= P <= BY, one carry
        int x = 0, y = __builtin_amdgcn_readfirstlane(tid >> 6);
        while (x < n) {
            const int xg = wrap_idx(b.x0 + s0 + x, g.nx), yg = wrap_idx(b.y0 + y, g.ny);
            const T* row = S + (((unsigned)(xg + Comp<C>::ox) * SY +
                                 (unsigned)(yg + Comp<C>::oy)) * SZ + (unsigned)b.k0);
            load4_to_lds(reinterpret_cast<const unsigned*>(row) + (d + lane),
                         reinterpret_cast<unsigned*>(lds + (x * b.BY + y) * LD) + d);
            y += kTileWaves;
            if (y >= b.BY) {
                y -= b.BY;
                ++x;
            }
        }
    }
}

// A whole box of floats, four levels per lane and load (the last may reach out
// of its row, as the pieces above), through registers
// (unaligned 16-byte loads; in 4-byte direct loads the fused pass of u took
// 590 us at 256x192x160, order 4, against 548).
template <int C, bool BIG>
__device__ inline void stage_quads(const Grid& g, const float* __restrict__ S, const BoxPlan& b,
                                   float* __restrict__ lds) {
    constexpr int NP = kLZ / 4, RPI = 64 / NP;
    const int tid = phase_tid(), lane = tid & 63, rr = lane / NP, zp = lane % NP;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned SZ = (unsigned)Comp<C>::SZ(g), SY = (unsigned)Comp<C>::SY(g);
    struct __attribute__((packed, aligned(4))) Quad {
        float a, b, c, d;
    };
    for (int y0 = 0; y0 < b.BY; y0 += RPI) {
        const int y = y0 + rr;
        if (y >= b.BY || 4 * zp >= b.BZ) continue;
        const int yg = wrap_idx(b.y0 + y, g.ny);
        const unsigned off =
            (BIG ? (unsigned)yg * SZ : __umul24((unsigned)yg, SZ)) + (unsigned)(4 * zp);
        // three loads in flight per lane
#pragma unroll 3
        for (int x = wave; x < b.BX; x += kTileWaves) {
            const int xg = wrap_idx(b.x0 + x, g.nx);
            const float* plane = S + (((unsigned)(xg + Comp<C>::ox) * SY + Comp<C>::oy) * SZ +
                                      (unsigned)b.k0);
            const Quad q = *reinterpret_cast<const Quad*>(elem<BIG>(plane, off));
            *reinterpret_cast<float4*>(lds + (x * b.BY + y) * kLZ + 4 * zp) =
                make_float4(q.a, q.b, q.c, q.d);
        }
    }
}

template <typename T, int C, bool BIG>
__device__ inline void stage_whole(const Grid& g, const T* __restrict__ S, const BoxPlan& b,
                                   T* __restrict__ lds) {
    if constexpr (sizeof(T) == 4) {
        stage_quads<C, BIG>(g, S, b, lds);
    } else if (b.pairs) {
        constexpr int NP = kLZ / 2;
        const int tid = phase_tid(), lane = tid & 63;
        stage_pairs<C, BIG>(g, S, b, 0, b.BX, kLZ, 64 / NP, tid, lane / NP, lane % NP, lds);
    } else {
        stage_rows<T, C>(g, S, b, 0, b.BX, kLZ, lds);
    }
}

template <typename T, int C, bool BIG>
__device__ inline void stage_slab(const Grid& g, const T* __restrict__ S, const BoxPlan& b,
                                  int s0, int n, T* __restrict__ lds) {
    if constexpr (sizeof(T) == 8) {
        if (b.pairs) {
            // lane / NP and 64 / NP by a float reciprocal: the operands are small
            // integers, and half a unit keeps the quotient off the integers
            const int tid = phase_tid(), lane = tid & 63, NP = b.LD >> 1;
            const float rz = 1.0f / (float)NP;
            const int RPI = __builtin_amdgcn_readfirstlane((int)(64.5f * rz));
            const int rr = (int)(((float)lane + 0.5f) * rz);
            stage_pairs<C, BIG>(g, S, b, s0, n, b.LD, RPI, tid, rr, lane - rr * NP, lds);
            return;
        }
    }
    stage_rows<T, C>(g, S, b, s0, n, b.LD, lds);
}

// Weights of one foot's order-P stencil (z against the node tables,
// semilag.py:441-454).
// The x weights are formed after the planes' sums, which take their place in
// the registers.
template <int P>
struct Weights {
    double y[P], z[P];
};

template <int C, int P>
__device__ inline void weights(const Grid& g, const FootSt& f, Weights<P>& w) {
    const double* zn = znodes<C>(g);
    const double* dinv = Comp<C>::centers ? g.dinv_cP : g.dinv_fP;
    z_weights<P>(zn, dinv, f.z, f.bk, w.z);
    uniform_weights<P>(f.ty, w.y);
}

// The x sum over the stencil planes' values a.
template <int P>
__device__ inline double x_sum(const FootSt& f, const double (&a)[P]) {
    double wx[P], acc = 0.0;
    uniform_weights<P>(f.tx, wx);
#pragma unroll
    for (int i = 0; i < P; ++i) acc = fma(wx[i], a[i], acc);
    return acc;
}

// One stencil plane, z then y, from LDS with row stride LD: even rows from c0,
// odd rows from c1 (their levels may sit one place apart, BoxPlan).
template <typename T, int P>
__device__ inline double plane_sum(const Weights<P>& w, const T* __restrict__ c0,
                                   const T* __restrict__ c1, int LD) {
    double ai = 0.0;
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const T* col = (j & 1 ? c1 : c0) + j * LD;
        double sj = 0.0;
#pragma unroll
        for (int k = 0; k < P; ++k) sj = fma(w.z[k], (double)col[k], sj);
        ai = fma(w.y[j], sj, ai);
    }
    return ai;
}

// First values of the even and odd rows of the stencil's planes in a staged
// box whose plane s0 comes first: c[0], c[1] in its even planes, c[2], c[3] in
// its odd ones (plane 0 of the stencil may lie before the box).
template <typename T>
__device__ inline void stencil_rows(const FootSt& f, const BoxPlan& b, int ox, int LD,
                                    const T* __restrict__ lds, const T* (&c)[4]) {
    const int oy = f.by - b.y0;
    const T* col = lds + ((ox * b.BY + oy) * LD + (f.bk - b.k0));
    const int sh = (b.ax * (f.bx - b.x0) + b.ay * oy + b.c) & 1;
    c[0] = col + sh;
    c[1] = col + (sh ^ b.ay);
    c[2] = col + (sh ^ b.ax);
    c[3] = col + (sh ^ b.ay ^ b.ax);
}

// The staged z -> y -> x contraction with FMAs from a whole box.  The row
// stride is a compile-time constant: a plane's rows are read at immediate
// offsets from two lane addresses.
template <typename T, int P>
__device__ inline double contract_whole(const FootSt& f, const Weights<P>& w, const BoxPlan& b,
                                        const T* __restrict__ lds) {
    const T* c[4];
    stencil_rows<T>(f, b, f.bx - b.x0, kLZ, lds, c);
    const int step = b.BY * kLZ;
    double a[P];
#pragma unroll
    for (int i = 0; i < P; ++i)
        a[i] = plane_sum<T, P>(w, c[2 * (i & 1)] + i * step, c[2 * (i & 1) + 1] + i * step, kLZ);
    return x_sum<P>(f, a);
}

// The planes of the slab [s0, s0 + n) that belong to the lane's stencil, into
// their places of a.
template <typename T, int P>
__device__ inline void contract_slab(const FootSt& f, const Weights<P>& w, const BoxPlan& b,
                                     int s0, int n, const T* __restrict__ lds, double (&a)[P]) {
    const int ox = f.bx - b.x0 - s0;
    const T* c[4];
    stencil_rows<T>(f, b, ox, b.LD, lds, c);
    const int step = b.BY * b.LD;
#pragma unroll
    for (int i = 0; i < P; ++i)
        if ((unsigned)(ox + i) < (unsigned)n)
            a[i] = plane_sum<T, P>(w, c[2 * (i & 1)] + i * step, c[2 * (i & 1) + 1] + i * step,
                                   b.LD);
}

// The same sum by loads from the field S; rolled over the planes.
template <typename T, int C, int P>
__device__ inline double contract_direct(const Grid& g, const FootSt& f, const Weights<P>& w,
                                         const T* __restrict__ S) {
    // the base wrapped, then a step at a time, as build_stencil does (a
    // saturated base must not leave 32 bits)
    double acc = 0.0;
    int gx = wrap_idx(f.bx, g.nx);
    const int gy0 = wrap_idx(f.by, g.ny);
#pragma unroll 1
    for (int i = 0; i < P; ++i) {
        double ai = 0.0;
        int gy = gy0;
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const T* col = S + node_addr<C>(g, gx, gy, f.bk);
            double sj = 0.0;
#pragma unroll
            for (int k = 0; k < P; ++k) sj = fma(w.z[k], (double)col[k], sj);
            ai = fma(w.y[j], sj, ai);
            gy = gy + 1 == g.ny ? 0 : gy + 1;
        }
        acc = fma(uniform_weight_m<P>(f.tx, i), ai, acc);
        gx = gx + 1 == g.nx ? 0 : gx + 1;
    }
    return acc;
}

// Arrival point of interior index (i, j, k) (arrival<C> without the linear
// index).
template <int C>
__device__ inline void arrival_at(const Grid& g, int i, int j, int k, double& xa, double& ya,
                                  double& za) {
    const double ar = (double)(i + 1), aj = (double)(j + 1);
    xa = (C == 0 ? ar : ar - 0.5) * g.dx;
    ya = (C == 1 ? aj : aj - 0.5) * g.dy;
    za = *elem<false>(znodes<C>(g), (unsigned)(k + 1));
}

// Element (i+1, j+1, k+1) of component C's ghost-shaped array.
template <int C>
__device__ inline unsigned field_elem(const Grid& g, int i, int j, int k) {
    const unsigned SZ = (unsigned)Comp<C>::SZ(g), SY = (unsigned)Comp<C>::SY(g);
    return ((unsigned)(i + 1) * SY + (unsigned)(j + 1)) * SZ + (unsigned)(k + 1);
}

// Elements of the five-point xy stencil around interior point (i, j, .) at
// element o (operators.py:293-367; periodic extension for u in x, v in y).
struct XYStar {
    unsigned o, xp, xm, yp, ym;
};

template <int C>
__device__ inline XYStar xy_star(const Grid& g, int i, int j, unsigned o) {
    const unsigned SZ = (unsigned)Comp<C>::SZ(g), PS = (unsigned)Comp<C>::SY(g) * SZ;
    XYStar q{o, o + PS, o - PS, o + SZ, o - SZ};
    if (C == 0 && i == g.nx - 1) q.xp = o - (unsigned)(g.nx - 1) * PS;
    if (C == 1 && j == g.ny - 1) q.yp = o - (unsigned)(g.ny - 1) * SZ;
    return q;
}

// rhs_xy (slc_device.h) over those elements.
template <bool BIG>
__device__ inline double rhs_star(const Grid& g, const double* __restrict__ F, const XYStar& q,
                                  double rdx2, double rdy2) {
    const double c = *elem<BIG>(F, q.o);
    const double d2x = ((*elem<BIG>(F, q.xp) - 2.0 * c) + *elem<BIG>(F, q.xm)) * rdx2;
    const double d2y = ((*elem<BIG>(F, q.yp) - 2.0 * c) + *elem<BIG>(F, q.ym)) * rdy2;
    return g.nu * (d2x + d2y);
}

__device__ inline void box_add(SBox& l, const FootSt& f) {
    l.xmin = min(l.xmin, f.bx); l.xmax = max(l.xmax, f.bx);
    l.ymin = min(l.ymin, f.by); l.ymax = max(l.ymax, f.by);
    l.kmin = min(l.kmin, f.bk); l.kmax = max(l.kmax, f.bk);
}

// Iterated midpoint (semilag.py:534-552) from the arrival point with its
// shared first sample (u0, v0, w0); returns the unclamped foot.
template <int C, bool BIG, typename TV>
__device__ inline void trace_foot(const Grid& g, const TV& V, double xa, double ya,
                                  double za, int K, double u0, double v0, double w0, double h,
                                  double& x, double& y, double& z) {
    double xm = xa - h * u0, ym = ya - h * v0;
    double zm = clampd(za - h * w0, g.z_lo, g.z_hi);
    for (int it = 1; it < g.n_iters; ++it) {
        double us, vs, ws;
        sample3<C, BIG, TV>(g, V, xm, ym, zm, za, K, us, vs, ws);
        xm = xa - h * us;
        ym = ya - h * vs;
        zm = clampd(za - h * ws, g.z_lo, g.z_hi);
    }
    if (g.n_iters == 0) { xm = xa; ym = ya; zm = za; }
    x = 2.0 * xm - xa;
    y = 2.0 * ym - ya;
    z = 2.0 * zm - za;
}

// T: storage type of the gathered field (double, or float for the FP32-storage
// variant: values are staged and read as float, weights and accumulation stay
// FP64).  F / Fm are always the FP64 fields (explicit xy-diffusion);
// Sn / Sm are the gathered copies (== F / Fm when T is double).
// One tile of the step kernel (tile = linear tile index, k fastest).  The
// caller provides the block's LDS (TileLds).
// defer (MODE_GATHER): when non-null, one flag per tile: 1 for a tile whose
// box does not fit the LDS budget (it is not gathered here but left for a
// pass with a larger budget), 0 for the others.
// redo (MODE_GATHER): when redo.flags is non-null, only the points whose tile
// of an earlier pass (redo.ti x redo.tj x redo.tk tiles, same numbering) has
// its defer flag set are gathered; the others were done by that pass.
struct Redo {
    const unsigned* flags = nullptr;
    int ti = 1, tj = 1, tk = 1;
};

__device__ inline bool redo_point(const Redo& r, const Grid& g, int nzi, int i, int j, int k) {
    if (!r.flags) return true;
    const int rtk = (nzi + r.tk - 1) / r.tk, rtj = (g.ny + r.tj - 1) / r.tj;
    return r.flags[((long)(i / r.ti) * rtj + j / r.tj) * rtk + k / r.tk] != 0u;
}

// LDS of a tile workgroup.
template <typename T, int MODE, int NPT, int LDS_BYTES>
struct TileLds {
    static constexpr int NN = MODE == MODE_BDF2 ? NPT : 1;
    __align__(16) T box[LDS_BYTES / sizeof(T)];
    __align__(16) BoxRed red;
    // near stencils (MODE_BDF2), waiting for the far gather
    double ntx[NN], nty[NN], nz[NN];
    int nbx[NN], nby[NN], nbk[NN];
};

template <typename T, int C, int P, int MODE, int TI, int TJ, int TK, int LDS_BYTES, bool BIG>
__device__ __forceinline__ void sl_tile_body(
    const Grid& g, const ArrivalTabs& A, const TrajVel& V, const double* __restrict__ F,
    const double* __restrict__ Fm, const T* __restrict__ Sn, const T* __restrict__ Sm,
    double dt, double* __restrict__ out, const Feet& ft, unsigned long long* nclamp, unsigned tile,
    TileLds<T, MODE, TI * TJ * TK, LDS_BYTES>& L, unsigned* defer = nullptr,
    Redo redo = Redo{}) {
    constexpr int NPT = TI * TJ * TK;
    static_assert(NPT % kSB == 0, "tile must be a multiple of the block");
    constexpr int PT = NPT / kSB;
    constexpr bool BOTH = MODE == MODE_FAR || MODE == MODE_BDF2;  // both feet traced
    constexpr bool RHS = MODE == MODE_BDF1 || MODE == MODE_NEAR || MODE == MODE_BDF2;
    const int nzi = Comp<C>::NZI(g);
    const unsigned ntk = (unsigned)(nzi + TK - 1) / TK, ntj = (unsigned)(g.ny + TJ - 1) / TJ;
    // the step kernels' trajectory velocity is always a stored field
    const TrajA VA{{V.a[0], V.a[1], V.a[2]}};
    const unsigned r0 = tile / ntk, tk = tile - r0 * ntk;
    const unsigned ti = r0 / ntj, tj = r0 - ti * ntj;
    const int i0 = (int)ti * TI, j0 = (int)tj * TJ, k0t = (int)tk * TK;

    // ---- phase 1: feet and stencils --------------------------------------
    // lane's point p: (i, j, k), z fastest
    auto point = [&](int tid, int p, int& i, int& j, int& k) {
        const int q = tid + kSB * p;
        i = i0 + q / (TK * TJ);
        j = j0 + (q / TK) % TJ;
        k = k0t + q % TK;
    };
    bool live[PT];
    FootSt st[PT];
    SBox l{INT_MAX, INT_MIN, INT_MAX, INT_MIN, INT_MAX, INT_MIN};
    SBox ln{INT_MAX, INT_MIN, INT_MAX, INT_MIN, INT_MAX, INT_MIN};  // MODE_BDF2 near box
    int ncl = 0;
#pragma unroll
    for (int p = 0; p < PT; ++p) {
        int i, j, k;
        point((int)threadIdx.x, p, i, j, k);
        live[p] = i < g.nx && j < g.ny && k < nzi &&
                  (MODE != MODE_GATHER || redo_point(redo, g, nzi, i, j, k));
        if (live[p]) {
            const unsigned n = ((unsigned)i * g.ny + j) * nzi + k;
            double x, y, z;
            if (MODE == MODE_NEAR || MODE == MODE_GATHER) {
                x = *elem<BIG>(ft.x, n);
                y = *elem<BIG>(ft.y, n);
                z = *elem<BIG>(ft.z, n);
            } else {
                const int K = k + 1;
                double xa, ya, za;
                arrival_at<C>(g, i, j, k, xa, ya, za);
                // the first sample is at the arrival point for every foot depth
                double u0, v0, w0;
                const int csel = A.csel[k], c = csel >> 1;
                sample3_at<BIG>(g, VA, over_dx(g, xa), over_dy(g, ya),
                                clampd(za, g.z_lo, g.z_hi), c, c + (csel & 1), u0, v0, w0);
                if (BOTH) {
                    // the near foot first: it leaves the registers (to LDS or
                    // to the feet arrays) before the far foot is traced
                    double xn, yn, zn;
                    trace_foot<C, BIG>(g, VA, xa, ya, za, K, u0, v0, w0, 0.5 * dt, xn, yn, zn);
                    if (MODE == MODE_FAR) {
                        *elem<BIG>(ft.x, n) = xn;
                        *elem<BIG>(ft.y, n) = yn;
                        *elem<BIG>(ft.z, n) = zn;
                    } else {
                        FootSt sn;
                        make_st<C, P>(g, xn, yn, zn, sn, ncl);
                        box_add(ln, sn);
                        const int q = threadIdx.x + kSB * p;
                        L.ntx[q] = sn.tx;
                        L.nty[q] = sn.ty;
                        L.nz[q] = sn.z;
                        L.nbx[q] = sn.bx;
                        L.nby[q] = sn.by;
                        L.nbk[q] = sn.bk;
                    }
                }
                trace_foot<C, BIG>(g, VA, xa, ya, za, K, u0, v0, w0,
                                   BOTH ? 0.5 * (2.0 * dt) : 0.5 * dt, x, y, z);
            }
            make_st<C, P>(g, x, y, z, st[p], ncl);
            box_add(l, st[p]);
        }
    }
    box_reduce(l, L.red.v[0]);
    if (MODE == MODE_BDF2) box_reduce(ln, L.red.v[1]);
    __syncthreads();

    // ---- phase 2: stage a foot's box, contract; far foot, then near ---------
    constexpr int NF = MODE == MODE_BDF2 ? 2 : 1;
    double val[PT], farv[PT];
#pragma unroll 1
    for (int f = 0; f < NF; ++f) {
        const T* __restrict__ S = (MODE == MODE_FAR || (MODE == MODE_BDF2 && f == 0)) ? Sm : Sn;
        const BoxPlan b = plan_box<T, C, P>(g, S, box_union(L.red.v[f]), LDS_BYTES);
        if (MODE == MODE_GATHER && defer) {
            const bool later = b.how == BOX_DIRECT || (b.how == BOX_SLABS && b.BX > b.ns);
            if (threadIdx.x == 0) defer[tile] = later ? 1u : 0u;
            if (later) return;
        }
        if (b.how == BOX_WHOLE) stage_whole<T, C, BIG>(g, S, b, L.box);
        // in flight with the box: the near stencils and the z tables
        if (MODE == MODE_BDF2 && f == 1) {
            const int tid = phase_tid();
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                const int q = tid + kSB * p;
                if (live[p])
                    st[p] = FootSt{L.nbx[q], L.nby[q], L.nbk[q], L.ntx[q], L.nty[q], L.nz[q]};
            }
        }
        Weights<P> w[PT];
#pragma unroll
        for (int p = 0; p < PT; ++p)
            if (live[p]) weights<C, P>(g, st[p], w[p]);
        if (b.how == BOX_WHOLE) {
            staged();
#pragma unroll
            for (int p = 0; p < PT; ++p)
                if (live[p]) val[p] = contract_whole<T, P>(st[p], w[p], b, L.box);
        } else if (b.how == BOX_SLABS) {
            double a[PT][P] = {};
            for (int s0 = 0; s0 < b.BX; s0 += b.ns) {
                const int n = min(b.ns, b.BX - s0);
                if (s0) __syncthreads();  // every lane is done with the last slab
                stage_slab<T, C, BIG>(g, S, b, s0, n, L.box);
                staged();
#pragma unroll
                for (int p = 0; p < PT; ++p)
                    if (live[p]) contract_slab<T, P>(st[p], w[p], b, s0, n, L.box, a[p]);
            }
#pragma unroll
            for (int p = 0; p < PT; ++p) val[p] = x_sum<P>(st[p], a[p]);
        } else {
#pragma unroll
            for (int p = 0; p < PT; ++p)
                if (live[p]) val[p] = contract_direct<T, C, P>(g, st[p], w[p], S);
        }
        if (f + 1 < NF) {
#pragma unroll
            for (int p = 0; p < PT; ++p) farv[p] = val[p];
            __syncthreads();  // every lane is done with the far box
        }
    }
    const int tid = phase_tid();
#pragma unroll
    for (int p = 0; p < PT; ++p) {
        if (!live[p]) continue;
        int i, j, k;
        point(tid, p, i, j, k);
        const unsigned o = field_elem<C>(g, i, j, k);
        double rh = 0.0;
        if (RHS) {
            const double rdx2 = 1.0 / (g.dx * g.dx), rdy2 = 1.0 / (g.dy * g.dy);
            const XYStar q = xy_star<C>(g, i, j, o);
            rh = rhs_star<BIG>(g, F, q, rdx2, rdy2);
            // Rh: 2R^n - R^{n-1} ('extrap') or R^n ('lagged'), solver.py:848-854
            if (MODE != MODE_BDF1 && !g.xy_lagged)
                rh = 2.0 * rh - rhs_star<BIG>(g, Fm, q, rdx2, rdy2);
        }
        if (MODE == MODE_GATHER) {
            *elem<BIG>(out, ((unsigned)i * g.ny + j) * nzi + k) = val[p];
        } else if (MODE == MODE_ADVECT || MODE == MODE_FAR) {
            *elem<BIG>(out, o) = val[p];
        } else if (MODE == MODE_BDF1) {
            *elem<BIG>(out, o) = val[p] + dt * rh;
        } else {
            const double far = (MODE == MODE_BDF2) ? farv[p] : *elem<BIG>(out, o);
            const double dt_eff = (2.0 / 3.0) * dt;
            const double pred = fma(far, -1.0 / 3.0, val[p] * (4.0 / 3.0));
            *elem<BIG>(out, o) = pred + dt_eff * rh;
        }
    }
    if (nclamp) {
        // one or two clamped feet per lane, counted over the wavefront
        int tot = 0;
#pragma unroll
        for (int c = 0; c < PT * (BOTH ? 2 : 1); ++c) tot += __popcll(__ballot(ncl > c));
        if (tot && (threadIdx.x & 63) == 0) atomicAdd(nclamp, (unsigned long long)tot);
    }
}

}  // namespace slc
