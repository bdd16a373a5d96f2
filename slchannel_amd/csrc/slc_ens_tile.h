// slc_ens_tile.h -- the batched SL tile kernel of the ensemble step:
// PASS 0 far pass (BDF2 members), PASS 1 near / bootstrap pass (BDF2 / BDF1
// members), PASS 2 fused pass (MODE_BDF2 / BDF1), each unit one sl_tile_body
// tile of its member.  Included once per
// (storage type, order) by slc_ens_tile_{d4,d6,f4,f6}.hip.
#pragma once

#include "slc_ens_dev.h"
#include "slc_tile.h"

namespace slc {

// One workgroup per tile, the three components (or one, n[c] = 0 for the
// others) in one launch: its member from the per-unit member map (the
// persistent chunk walk of the other batched kernels keeps ~25 more registers
// live here and halves the occupancy).
template <typename T, int C, int P, int PASS, int TI, int TJ, int TK, int kEnsLds, bool BIG,
          typename LdsT>
__device__ __forceinline__ void ens_tile_unit(const EnsMember* __restrict__ mem,
                                              const unsigned* __restrict__ start,
                                              const int* __restrict__ umap, unsigned uu, LdsT& L) {
    // one of the two tile bodies runs: the bootstrap's LDS is the fused pass's
    TileLds<T, MODE_BDF1, TI * TJ * TK, kEnsLds>& L1 =
        reinterpret_cast<TileLds<T, MODE_BDF1, TI * TJ * TK, kEnsLds>&>(L);
    // member and state are the same for the whole workgroup: broadcast them
    // so the member table is read with scalar loads and its pointers stay in
    // scalar registers
    const int m = __builtin_amdgcn_readfirstlane(umap[uu]);
    const unsigned u = uu - start[m];
    const EnsMember& M = mem[m];
    const int st = __builtin_amdgcn_readfirstlane(*M.state);
    const int a = ens_a(st), b = ens_b(st), c = ens_c(st);
    const long NA = (long)M.g.nx * M.g.ny * M.g.nz;
    const Feet ft{M.nfoot, M.nfoot + NA, M.nfoot + 2 * NA};
    const double* Fa = M.fld[a][C];
    const double* Fb = M.fld[b][C];
    const T* Sa;
    const T* Sb;
    if constexpr (sizeof(T) == 4) {
        Sa = reinterpret_cast<const T*>(M.f32n[C]);
        Sb = reinterpret_cast<const T*>(M.f32m[C]);
    } else {
        Sa = reinterpret_cast<const T*>(Fa);
        Sb = reinterpret_cast<const T*>(Fb);
    }
    if (ens_bdf2(st)) {
        const TrajVel V{{M.us[0], M.us[1], M.us[2]}, {nullptr, nullptr, nullptr}};
        if constexpr (PASS == 0)
            sl_tile_body<T, C, P, MODE_FAR, TI, TJ, TK, kEnsLds, BIG>(
                M.g, M.at[C], V, Fa, Fb, Sa, Sb, M.dt, M.fld[c][C], ft, M.ncl, u, L);
        else if constexpr (PASS == 2)
            sl_tile_body<T, C, P, MODE_BDF2, TI, TJ, TK, kEnsLds, BIG>(
                M.g, M.at[C], V, Fa, Fb, Sa, Sb, M.dt, M.fld[c][C], ft, M.ncl, u, L);
        else
            sl_tile_body<T, C, P, MODE_NEAR, TI, TJ, TK, kEnsLds, BIG>(
                M.g, M.at[C], V, Fa, Fb, Sa, Sb, M.dt, M.fld[c][C], ft, M.ncl, u, L);
    } else if constexpr (PASS >= 1) {
        const TrajVel V{{M.fld[a][0], M.fld[a][1], M.fld[a][2]}, {nullptr, nullptr, nullptr}};
        sl_tile_body<T, C, P, MODE_BDF1, TI, TJ, TK, kEnsLds, BIG>(
            M.g, M.at[C], V, Fa, nullptr, Sa, nullptr, M.dt, M.fld[c][C], ft, M.ncl, u, L1);
    }
}

template <typename T, int P, int PASS, int TI, int TJ, int TK, int kEnsLds, int WAVES, bool BIG>
__global__ __launch_bounds__(kSB) __attribute__((amdgpu_waves_per_eu(WAVES))) void
ens_tile_kernel(const EnsMember* __restrict__ mem, EnsTiles t) {
    constexpr int M0 = PASS == 0 ? MODE_FAR : PASS == 1 ? MODE_NEAR : MODE_BDF2;
    __shared__ TileLds<T, M0, TI * TJ * TK, kEnsLds> L;
    const Comp3 w = comp3_unit(blockIdx.x, t.n);
    if (w.c == 0)
        ens_tile_unit<T, 0, P, PASS, TI, TJ, TK, kEnsLds, BIG>(mem, t.start[0], t.umap[0], w.u, L);
    else if (w.c == 1)
        ens_tile_unit<T, 1, P, PASS, TI, TJ, TK, kEnsLds, BIG>(mem, t.start[1], t.umap[1], w.u, L);
    else if (w.c == 2)
        ens_tile_unit<T, 2, P, PASS, TI, TJ, TK, kEnsLds, BIG>(mem, t.start[2], t.umap[2], w.u, L);
}

template <typename T, int P, int PASS>
inline void launch_tile_shape(const EnsMember* mem, const EnsTiles& t, int shape, hipStream_t s) {
    const dim3 grid(pad8(t.n[0]) + pad8(t.n[1]) + pad8(t.n[2])), blk(kSB);
    if (t.big) {  // a member past the 32-bit offsets: one shape
        hipLaunchKernelGGL((ens_tile_kernel<T, P, PASS, 4, 4, 16, 31104, 4, true>), grid, blk, 0, s,
                           mem, t);
        return;
    }
    switch (shape) {
        case 1:
            hipLaunchKernelGGL((ens_tile_kernel<T, P, PASS, 4, 4, 32, 40960, 1, false>), grid, blk,
                               0, s, mem, t);
            break;
        case 2:
            hipLaunchKernelGGL((ens_tile_kernel<T, P, PASS, 2, 8, 16, 31104, 4, false>), grid, blk,
                               0, s, mem, t);
            break;
        default:
            hipLaunchKernelGGL((ens_tile_kernel<T, P, PASS, 4, 4, 16, 31104, 4, false>), grid, blk,
                               0, s, mem, t);
    }
}

template <typename T, int P>
inline void launch_tile_pass(const EnsMember* mem, const EnsTiles& t, int pass, int shape,
                             hipStream_t s) {
    if (pass == 0) launch_tile_shape<T, P, 0>(mem, t, shape, s);
    else if (pass == 1) launch_tile_shape<T, P, 1>(mem, t, shape, s);
    else launch_tile_shape<T, P, 2>(mem, t, shape, s);
}

}  // namespace slc
