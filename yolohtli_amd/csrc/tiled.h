// tiled.h -- the temporally blocked kernel of the plain stepper and its
// dispatch for one ionic model.  Its instantiations (tile shapes, masks,
// outputs) are compiled in one file per model, tiled_2v.hip and tiled_fk.hip.
#pragma once

#include "tile.h"
#include "yh_internal.h"

namespace yh {

template <int MODEL, bool MASKED, int R, int NW, int CW, bool APD, bool PREV, int ISO = -1,
          bool WT = false>
__global__ __launch_bounds__(64 * NW) void k_tiled(const KParams k, CFields in, Fields out,
                                                   const uint8_t* __restrict__ codes, int K,
                                                   int tiles_x, int ntiles, const ApdState apd,
                                                   float* __restrict__ prev) {
  __shared__ TileLds<MODEL, NW, CW> lds;
  const int tile = xcd_tile(blockIdx.x, ntiles);
  const int ty = tile / tiles_x;
  tile_advance<MODEL, MASKED, R, NW, CW, APD, PREV, ISO, WT>(k, in, out, codes, K,
                                                             tile - ty * tiles_x, ty, lds, apd,
                                                             prev);
}

template <int MODEL, bool MASKED, int R, int NW, int CW, bool APD, bool PREV = false,
          int ISO = -1, bool WT = false>
static hipError_t launch_tiled_t(int K, const KParams& k, CFields in, Fields out,
                                 const uint8_t* codes, hipStream_t s, const ApdState& apd,
                                 float* prev = nullptr, int* occ = nullptr) {
  if (occ)  // the workgroups of this instantiation one CU holds at once; no launch
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(
        occ, k_tiled<MODEL, MASKED, R, NW, CW, APD, PREV, ISO, WT>, 64 * NW, 0);
  const int wout = 64 * CW - 2 * K, hout = NW * R - 2 * K;
  if (K < 1 || wout <= 0 || hout <= 0) return hipErrorInvalidValue;
  const int tiles_x = (k.nx + wout - 1) / wout;
  const int tiles_y = (k.ny + hout - 1) / hout;
  const int ntiles = tiles_x * tiles_y;
  hipLaunchKernelGGL((k_tiled<MODEL, MASKED, R, NW, CW, APD, PREV, ISO, WT>), dim3(ntiles),
                     dim3(64 * NW), 0, s, k, in, out, codes, K, tiles_x, ntiles, apd, prev);
  return hipGetLastError();
}

template <int MODEL, bool MASKED>
hipError_t launch_tiled_m(int rows, int waves, int cols, int K, const KParams& k,
                                 CFields in, Fields out, const uint8_t* codes, hipStream_t s,
                                 const ApdState* apd, float* prev, int* occ) {
  const ApdState a = apd ? *apd : ApdState();
  if (apd) {
    if (prev) return hipErrorInvalidValue;
#define YH_TILE_APD_I(RR, WW, I) \
  launch_tiled_t<MODEL, MASKED, RR, WW, 1, true, false, I>(K, k, in, out, codes, s, a, nullptr, occ)
#define YH_TILE_APD(RR, WW)                    \
  if (rows == RR && waves == WW && cols == 1) \
    return k.iso ? YH_TILE_APD_I(RR, WW, 1) : YH_TILE_APD_I(RR, WW, 0);
    YH_TILE_APD(4, 8)
    YH_TILE_APD(8, 8)
    YH_TILE_APD(4, 16)
    YH_TILE_APD(8, 16)
#undef YH_TILE_APD
#undef YH_TILE_APD_I
    return hipErrorInvalidValue;
  }
  // the shapes the automatic choice takes come with isotropic or anisotropic
  // diffusion fixed at compile time (the run-time test of both in the row loop
  // costs registers, and with them the second workgroup of a CU), with and
  // without the previous-u output, and with write-through stores (k.wt) for
  // launches of two workgroups per CU
#define YH_TILE_PW(RR, WW, I, W)                                              \
  return prev ? launch_tiled_t<MODEL, MASKED, RR, WW, 1, false, true, I, W>(   \
                    K, k, in, out, codes, s, a, prev, occ)                    \
              : launch_tiled_t<MODEL, MASKED, RR, WW, 1, false, false, I, W>(  \
                    K, k, in, out, codes, s, a, nullptr, occ);
#define YH_TILE_MAIN(RR, WW)                       \
  if (rows == RR && waves == WW && cols == 1) {    \
    if (k.iso) {                                   \
      if (k.wt) YH_TILE_PW(RR, WW, 1, true)        \
      YH_TILE_PW(RR, WW, 1, false)                 \
    }                                              \
    if (k.wt) YH_TILE_PW(RR, WW, 0, true)          \
    YH_TILE_PW(RR, WW, 0, false)                   \
  }
  YH_TILE_MAIN(4, 8)
  YH_TILE_MAIN(8, 8)
  YH_TILE_MAIN(4, 16)
  YH_TILE_MAIN(5, 16)
  YH_TILE_MAIN(7, 16)
  YH_TILE_MAIN(8, 16)
#undef YH_TILE_MAIN
#undef YH_TILE_PW
  if (prev) return hipErrorInvalidValue;
#define YH_TILE_CASE(RR, WW, CC)                 \
  if (rows == RR && waves == WW && cols == CC) \
    return launch_tiled_t<MODEL, MASKED, RR, WW, CC, false>(K, k, in, out, codes, s, a, nullptr, \
                                                            occ);
  YH_TILE_CASE(4, 4, 1)
  YH_TILE_CASE(8, 4, 1)
  YH_TILE_CASE(16, 4, 1)
  YH_TILE_CASE(16, 8, 1)
  YH_TILE_CASE(4, 4, 2)
  YH_TILE_CASE(8, 4, 2)
  YH_TILE_CASE(4, 8, 2)
  YH_TILE_CASE(8, 8, 2)
  YH_TILE_CASE(4, 16, 2)
#undef YH_TILE_CASE
  return hipErrorInvalidValue;
}

}  // namespace yh
