// gr_star7_k5.hip -- dispatch of kernel 5's temporally blocked passes (gr_star7.hpp).
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include "../../include/girih_gpu.h"
#include "gr_internal.hpp"
#include "gr_star7_launch.hpp"

namespace gr {

// Tiles per precision and depth; `tile` 0 is the default, the autotuner tries them all.
// What bounds a pass is the memory fabric: it moves the coefficients and the field of
// the computed region (tile + margins, less what neighbouring tiles find in the L2) once
// per TL steps.  So the tile is as large as the registers allow at one workgroup per
// CU: TL x 7 coefficient words, 3 x TL queue words and the next plane's 8 per cell.
// Lanes own 4 cells in x (FP32, bf16) or 2 (FP64): fewer instructions per cell, and a
// 256-VGPR budget at 7-8 waves per CU.  512^3, one box, 4 passes, GLUP/s, against the
// pass with one barrier per level and coefficients loaded where level 1 uses them:
//   FP32 depth 4: 64 x 16, 448 lanes x 4 cells 459 (2.75 GB/pass HBM write+fetch 5.9 GB,
//     5.1 TB/s), 832 lanes x 2 cells 360 (spills); before 284
//   bf16 depth 4: 128 x 16, 768 lanes x 4 cells 714; 64 x 32, 704 lanes x 4 668; 64 x 16,
//     832 lanes x 2 636; before 388.  Depth 6, 64 x 16, 1024 lanes x 2: 703; before 322
//   FP64 depth 4: 64 x 8, 512 lanes x 2 cells 245 (6.6 TB/s); 1024 lanes x 1 187
//     (spills), 32 x 18 210; before 128
//   The tiles that 64 does not divide fill their lanes (56 + 8 margin cells are 16 slots
//   of 4) and compute fewer margin cells per cell of output, and grids that 64-wide tiles
//   overhang have another width to choose.  One call of 24 steps, GLUP/s, 64-wide tile /
//   the other, FP32 64 x 16 / 56 x 22 / 48 x 26: 389 x 270 x 331 337 / 357 / 339, 448 x 330 x
//   260 327 / 393 / 325, 130 x 410 x 90 248 / 310 / 312, 300 x 310 x 250 320 / 331 / 366, 512^3
//   416 / 394 / 390; bf16 depth 6 64 x 16 / 52 x 22: 674 / 727, 600 x 130 x 333 463 / 624; FP64
//   64 x 8 / 56 x 10: 448 x 330 x 260 182 / 199, 130 x 410 x 90 147 / 204, 512^3 212 / 176.
//   Never the fastest: FP32 64 x 18, 32 x 38; bf16 56 x 38, 48 x 42, 40 x 28; FP64 40 x 14, 32 x 18.
//   depth 2: FP32 64 x 32 245, 128 x 16 262 (before 217); bf16 64 x 32 382 (258);
//     FP64 64 x 16 138 (104)
template <typename T, typename C>
static hipError_t k5_dispatch(int tl, int tile, const S7Args<T, C> &a, hipStream_t st) {
  constexpr bool B16 = std::is_same<C, __hip_bfloat16>::value;
  if constexpr (B16) {
    if (tl == 2) return launch_s7<T, C, 5, 2, 64, 32, 640, 4, 1, false>(a, st);
    if (tl == 4) {
      if (tile == 1) return launch_s7<T, C, 5, 4, 128, 16, 768, 4, 1, false>(a, st);
      if (tile == 2) return launch_s7<T, C, 5, 4, 64, 16, 832, 2, 1, false>(a, st);
      return launch_s7<T, C, 5, 4, 64, 32, 704, 4, 1, false>(a, st);
    }
    if (tl == 6) {
      if (tile == 1) return launch_s7<T, C, 5, 6, 52, 22, 1024, 2, 1, false>(a, st);
      return launch_s7<T, C, 5, 6, 64, 16, 1024, 2, 1, false>(a, st);
    }
  } else if constexpr (sizeof(T) == 4) {
    if (tl == 2) {
      if (tile == 1) return launch_s7<T, C, 5, 2, 128, 16, 704, 4, 1, false>(a, st);
      return launch_s7<T, C, 5, 2, 64, 32, 640, 2, 1, false>(a, st);
    }
    if (tl == 4) {
      if (tile == 1) return launch_s7<T, C, 5, 4, 56, 22, 448, 4, 1, false>(a, st);
      if (tile == 2) return launch_s7<T, C, 5, 4, 48, 26, 448, 4, 1, false>(a, st);
      return launch_s7<T, C, 5, 4, 64, 16, 448, 4, 1, false>(a, st);
    }
  } else {
    if (tl == 2) return launch_s7<T, C, 5, 2, 64, 16, 704, 2, 1, false>(a, st);
    if (tl == 4) {
      if (tile == 1) return launch_s7<T, C, 5, 4, 56, 10, 512, 2, 1, false>(a, st);
      return launch_s7<T, C, 5, 4, 64, 8, 512, 2, 1, false>(a, st);
    }
  }
  return hipErrorInvalidValue;
}

int k5_tiles(const Problem &P, int tl) {
  if (P.flags & GR_COEF_BF16) return tl == 4 ? 3 : tl == 6 ? 2 : 1;
  if (P.dtype == GR_F64) return tl == 4 ? 2 : 1;
  return tl == 2 ? 2 : tl == 4 ? 3 : 1;
}

template <typename T, typename C>
static hipError_t k5_pass_t(const Problem &P, int tl, const void *Y, void *Z1, void *Z, const void *src, long long src_idx,
                            const LaunchCfg &lc, hipStream_t st) {
  S7Args<T, C> a = s7_args<T, C>(P, Y, Z1, Z, src, src_idx, lc);
  a.coef = (const C *)P.coef - P.xoff;  // addressed with the fields' element index
  a.cstride = P.field_elems;
  return k5_dispatch<T, C>(tl, lc.ftile, a, st);
}

// One pass of tl kernel-5 steps: Y -> Z (level tl-1 -> Z1 unless null).
hipError_t k5_pass(const Problem &P, int tl, const void *Y, void *Z1, void *Z, const void *src, long long src_idx,
                   const LaunchCfg &lc, hipStream_t st) {
  if (P.dtype == GR_F64) return k5_pass_t<double, double>(P, tl, Y, Z1, Z, src, src_idx, lc, st);
  if (P.flags & GR_COEF_BF16) return k5_pass_t<float, __hip_bfloat16>(P, tl, Y, Z1, Z, src, src_idx, lc, st);
  return k5_pass_t<float, float>(P, tl, Y, Z1, Z, src, src_idx, lc, st);
}

}  // namespace gr
