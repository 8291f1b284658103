// Fused Yee step for rows of any width: fused_tile with XS = 0, one wave per
// row segment of 64 cells, TY rows (plus the halo row) per workgroup.
//
// The whole-row kernel (k_yee_fused) exists for padded rows of 128, 256 and
// 512 cells; every other width (a grid 64, 180 or 301 cells long) stepped H
// and E in two launches, which moves every field twice.  Segments of 64
// cells divide any padded row (the pitch is a multiple of 64), so no lane is
// idle beyond the padding, and a workgroup is TY + 1 waves whatever the row:
// FP64 takes 3 rows in 4 waves here, two workgroups on a compute unit, where
// whole rows of 256 cells fit 2 rows in 12 waves.  The price is the x halo of
// every segment (one lane-spread load per plane and the recomputed H of one
// cell).
#pragma once
#include "fused_kernel.h"

namespace pm {

// Waves per SIMD the register allocation aims at: 4 in FP32 (128 VGPRs),
// 2 in FP64.
template <typename T>
constexpr int kSegWaves = sizeof(T) == 4 ? 4 : 2;

template <typename T, int CK, int TY, bool ADE>
__global__ __launch_bounds__(64 * (TY + 1), kSegWaves<T>) void k_yee_seg(
    const KGrid g, const KFz z, int nseg, int kchunk, int ntile_y, int nchunk, int n_out,
    int n_in, int seg, int order, TileBox bx) {
  __shared__ FusedLds<T, 1, 1, TY, 0> lds;
  __shared__ KAde ade_tab[ADE ? kMaxAde : 1];
  __shared__ T ade_cf[ADE ? kMaxAde : 1][12];
  if constexpr (ADE) stage_ade<T>(g, ade_tab, ade_cf);
  const int b = blockIdx.x;
  if (b < seg)
    fused_tile<T, CK, 1, 1, TY, 0, true, ADE>(g, z, kchunk, ntile_y, nchunk, n_out, order, bx, b,
                                              lds, ade_tab, ade_cf, nseg);
  else
    fused_tile<T, CK, 1, 1, TY, 0, false, ADE>(g, z, kchunk, ntile_y, nchunk, n_in, order, bx,
                                               b - seg, lds, ade_tab, ade_cf, nseg);
}

template <typename T, int CK, int TY>
int launch_seg_one(const KGrid& g, const KFz& z, int kchunk, int order, hipStream_t s) {
  const int nseg = (int)(g.sy / 64);
  const int ntile_y = (g.ny + TY - 1) / TY;
  const int nchunk = (g.nz + kchunk - 1) / kchunk;
  const TileBox bx = interior_tiles(g, TY, kchunk);
  const int n_in = (bx.ty1 - bx.ty0) * (bx.kc1 - bx.kc0) * nseg;
  const int n_out = ntile_y * nchunk * nseg - n_in;
  const int seg = ((n_out + 7) / 8) * 8;
  const dim3 grid(seg + ((n_in + 7) / 8) * 8), block(64 * (TY + 1));
  if (g.n_ade)
    hipLaunchKernelGGL((k_yee_seg<T, CK, TY, true>), grid, block, 0, s, g, z, nseg, kchunk,
                       ntile_y, nchunk, n_out, n_in, seg, order, bx);
  else
    hipLaunchKernelGGL((k_yee_seg<T, CK, TY, false>), grid, block, 0, s, g, z, nseg, kchunk,
                       ntile_y, nchunk, n_out, n_in, seg, order, bx);
  return 0;
}

// Tile heights built: 3 and 7 rows (4 and 8 waves).
template <typename T, int CK>
int launch_seg_ck(const KGrid& g, const KFz& z, int ty, int kchunk, int order, hipStream_t s) {
  if (ty == 3) return launch_seg_one<T, CK, 3>(g, z, kchunk, order, s);
  if (ty == 7) return launch_seg_one<T, CK, 7>(g, z, kchunk, order, s);
  return -1;
}

}  // namespace pm
