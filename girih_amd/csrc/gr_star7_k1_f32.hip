// gr_star7_k1_f32.hip -- dispatch of kernel 1's temporally blocked passes (gr_star7.hpp), FP32.
#include <hip/hip_runtime.h>

#include "gr_internal.hpp"
#include "gr_star7_launch.hpp"

namespace gr {

// A pass is bound by the vector ALU (12.3 instructions per computed cell, 10 of them the
// stencil; 77% busy on 64 x 50 at depth 4) and by the LDS reads behind each barrier, not by
// memory (1.80 GB a pass at 512^3), so a tile trades the margins it computes twice (1.33x the tile at 128 x 24, depth 4)
// against two workgroups per CU, which cover each other's barriers.  512^3, one box,
// GLUP/s, against one-cell lanes (1029-1179 at depth 4); in parentheses with the input
// loaded one plane ahead instead of two:
//   depth 2: 128 x 32 1280 (1020), 128 x 16 1231 (1066);
//   depth 3: 128 x 16 1624 (1478);
//   depth 4: 128 x 24 1714 three planes ahead, 1694 two (1472), 128 x 16 1690 (1279);
//   depth 5: 128 x 16 1663 (1597; 1394 with 2 cells per lane);  depth 6: 64 x 20 1150 (1099).
// The narrower tiles are for grids that 128-wide tiles would overhang: one call of 24 steps
// at depth 4, 128 x 24 / 64 x 50 (1.26x the tile computed) / 48 x 26: 512^3 1539 / 1543 / 1365,
// 448 x 330 x 260 1357 / 1625 / 1203, 389 x 270 x 331 1198 / 1366 / 1216, 130 x 410 x 90 577 /
// 674 / 764, 192 x 180 x 230 873 / 1041 / 1059.  600 x 130 x 333 1320 / 1319 / 1268 and 1459
// on 56 x 26.  Depth 3, 128 x 16 / 64 x 24: 512^3 1449 / 1404, 251 x 420 x 140 1135 / 1368, 192 x
// 180 x 230 754 / 1101.  Never the fastest: 64 x 16 at depths 3 and 4, 64 x 22 and 96 x 32 at 4,
// 120 x 12 at 3, 56 x 44 at 5.
template <bool STRM>
static hipError_t k1_dispatch(int tl, int tile, const S7Args<float, float> &a, hipStream_t st) {
  switch (tl) {
    case 2:
      if (tile == 1) return launch_s7<float, float, 1, 2, 128, 16, 704, 2, 2, STRM>(a, st);
      return launch_s7<float, float, 1, 2, 128, 32, 832, 2, 2, STRM>(a, st);
    case 3:
      if (tile == 1) return launch_s7<float, float, 1, 3, 64, 24, 512, 4, 2, STRM>(a, st);
      return launch_s7<float, float, 1, 3, 128, 16, 704, 2, 2, STRM>(a, st);
    case 4:
      if (tile == 1) return launch_s7<float, float, 1, 4, 128, 24, 1024, 4, 3, STRM>(a, st);
      if (tile == 2) return launch_s7<float, float, 1, 4, 64, 50, 1024, 4, 3, STRM>(a, st);
      if (tile == 3) return launch_s7<float, float, 1, 4, 48, 26, 448, 4, 2, STRM>(a, st);
      if (tile == 4) return launch_s7<float, float, 1, 4, 56, 26, 512, 4, 2, STRM>(a, st);
      return launch_s7<float, float, 1, 4, 128, 16, 768, 2, 2, STRM>(a, st);
    case 5: return launch_s7<float, float, 1, 5, 128, 16, 896, 4, 2, STRM>(a, st);
    case 6: return launch_s7<float, float, 1, 6, 64, 20, 640, 4, 2, STRM>(a, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t k1_pass_f32(const Problem &P, int tl, const void *Y, void *Z1, void *Z, const void *src, long long src_idx,
                       const LaunchCfg &lc, hipStream_t st) {
  const S7Args<float, float> a = s7_args<float, float>(P, Y, Z1, Z, src, src_idx, lc);
  return streaming_sweep(P) ? k1_dispatch<true>(tl, lc.ftile, a, st) : k1_dispatch<false>(tl, lc.ftile, a, st);
}

}  // namespace gr
