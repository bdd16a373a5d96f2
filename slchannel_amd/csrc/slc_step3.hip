// slc_step3.hip -- the step kernels of slc_step.hip for the three components in
// one launch.
#include "slc_step.h"

namespace slc {

// The three components' tiles of a step kernel in one launch: a small grid's
// tiles fill the GPU together (32x24x32 has 96 tiles per component for 256
// CUs), and two drained tails and launches go.  For grids up to kMergeTiles
// tiles; on a larger one the launches saved are a few percent of the passes, at
// 256^3 nothing (kMergeTiles).  A grid of so few tiles never needs 64-bit
// addressing.
struct Tile3 {
    Grid g;
    TrajVel V;
    ArrivalTabs A[3];
    const double* F[3];
    const double* Fm[3];
    const void* Sn[3];  // gathered copies (double or float)
    const void* Sm[3];
    double* out[3];
    double dt;
    unsigned long long* ncl;
    unsigned n[3];  // tiles
};

// The kernel's argument (its only one) behind an opaque pointer: each of the
// three bodies reads it for itself.  Read at entry for all of them, the
// scalars overflowed into vector lanes (2200 v_readlane in the code; fused
// pass of u at 256^3, order 6, 1.40 -> 1.62 ms).
__device__ inline const Tile3& tile3_arg() {
    auto p = (const __attribute__((address_space(4))) Tile3*)(
        __builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(p));
    return *(const Tile3*)p;
}

template <typename T, int P, int MODE, int LDS_BYTES, int WAVES>
__global__ __launch_bounds__(kSB) __attribute__((amdgpu_waves_per_eu(WAVES))) void sl_tile3_kernel(
    Tile3 arg) {
    __shared__ TileLds<T, MODE, kTI * kTJ * kTK, LDS_BYTES> L;
    const Comp3 w = comp3_unit(blockIdx.x, arg.n);
#define SLC_TILE3(C)                                                                             \
    do {                                                                                         \
        const Tile3& a = tile3_arg();                                                            \
        sl_tile_body<T, C, P, MODE, kTI, kTJ, kTK, LDS_BYTES, false>(                              \
            a.g, a.A[C], a.V, a.F[C], a.Fm[C], (const T*)a.Sn[C], (const T*)a.Sm[C], a.dt,       \
            a.out[C], Feet{nullptr, nullptr, nullptr}, a.ncl, w.u, L);                           \
    } while (0)
    if (w.c == 0) SLC_TILE3(0);
    else if (w.c == 1) SLC_TILE3(1);
    else if (w.c == 2) SLC_TILE3(2);
#undef SLC_TILE3
}

template <typename T, int MODE>
static void launch_tile3(const Tile3& a, hipStream_t s) {
    constexpr int LDS = MODE == MODE_BDF2 ? kTileLdsBdf2 : kTileLds, W = kTileWavesPerSimd;
    const dim3 grid(pad8(a.n[0]) + pad8(a.n[1]) + pad8(a.n[2])), blk(kSB);
    if (grid.x == 0) return;
    if (a.g.order == 4)
        hipLaunchKernelGGL((sl_tile3_kernel<T, 4, MODE, LDS, W>), grid, blk, 0, s, a);
    else
        hipLaunchKernelGGL((sl_tile3_kernel<T, 6, MODE, LDS, W>), grid, blk, 0, s, a);
}

hipError_t run_tile_step3(const Grid& g, int mode, const ArrivalTabs A[3], const TrajVel& V,
                          const double* const F[3], const double* const Fm[3],
                          const float* const Fn32[3], const float* const Fm32[3], double dt,
                          double* const out[3], unsigned long long* ncl, hipStream_t s) {
    Tile3 a{};
    a.g = g;
    a.V = V;
    a.dt = dt;
    a.ncl = ncl;
    for (int c = 0; c < 3; ++c) {
        a.A[c] = A[c];
        a.F[c] = F[c];
        a.Fm[c] = Fm ? Fm[c] : nullptr;
        a.Sn[c] = Fn32 ? (const void*)Fn32[c] : F[c];
        a.Sm[c] = Fm32 ? (const void*)Fm32[c] : a.Fm[c];
        a.out[c] = out[c];
        a.n[c] = (unsigned)step_tiles(g, c);
    }
    const bool f32 = Fn32 != nullptr;
    switch (mode) {
        case MODE_ADVECT:
            if (f32) launch_tile3<float, MODE_ADVECT>(a, s);
            else launch_tile3<double, MODE_ADVECT>(a, s);
            break;
        case MODE_BDF1:
            if (f32) launch_tile3<float, MODE_BDF1>(a, s);
            else launch_tile3<double, MODE_BDF1>(a, s);
            break;
        default:
            if (f32) launch_tile3<float, MODE_BDF2>(a, s);
            else launch_tile3<double, MODE_BDF2>(a, s);
    }
    return hipGetLastError();
}

}  // namespace slc
