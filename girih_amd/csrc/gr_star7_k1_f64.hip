// gr_star7_k1_f64.hip -- dispatch of kernel 1's temporally blocked passes (gr_star7.hpp), FP64.
#include <hip/hip_runtime.h>

#include "gr_internal.hpp"
#include "gr_star7_launch.hpp"

namespace gr {

// Two cells per lane (16-byte accesses).  512^3, one box, GLUP/s, against one-cell lanes
// (557-640 at depth 3); in parentheses with the input loaded one plane ahead instead of
// two: depth 2: 64 x 16 652 (559; three workgroups per CU), 128 x 16 699 (568); depth 3:
// 64 x 16 899 (798; two per CU, 4.7 TB/s), 64 x 24 666, 128 x 8 472; depth 4: 64 x 22 944
// (812), 64 x 16 839 (703); depth 5: 64 x 14 685 (693); depth 6: 64 x 8 556 (569).  128^3
// in the caches, 8-plane chunks: depth 3 at 64 x 16 432 (412; before 294), 4 at 64 x 16 413.
// 48 x 30 at depth 4 is for grids that 64-wide tiles overhang; one call of 24 steps, 64 x 22 /
// 48 x 30: 389 x 270 x 331 673 / 817, 130 x 410 x 90 455 / 589, 192 x 180 x 230 691 / 741, 512^3 830 /
// 798; 32 x 42 gained nothing over the better of the two.
template <bool STRM>
static hipError_t k1_dispatch(int tl, int tile, const S7Args<double, double> &a, hipStream_t st) {
  switch (tl) {
    case 2:
      if (tile == 1) return launch_s7<double, double, 1, 2, 128, 16, 640, 2, 2, STRM>(a, st);
      return launch_s7<double, double, 1, 2, 64, 16, 640, 2, 2, STRM>(a, st);
    case 3: return launch_s7<double, double, 1, 3, 64, 16, 768, 2, 2, STRM>(a, st);
    case 4:
      if (tile == 1) return launch_s7<double, double, 1, 4, 64, 22, 1024, 2, 2, STRM>(a, st);
      if (tile == 2) return launch_s7<double, double, 1, 4, 48, 30, 1024, 2, 2, STRM>(a, st);
      return launch_s7<double, double, 1, 4, 64, 16, 832, 2, 2, STRM>(a, st);
    case 5: return launch_s7<double, double, 1, 5, 64, 14, 1024, 2, 1, STRM>(a, st);
    case 6: return launch_s7<double, double, 1, 6, 64, 8, 768, 2, 1, STRM>(a, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t k1_pass_f64(const Problem &P, int tl, const void *Y, void *Z1, void *Z, const void *src, long long src_idx,
                       const LaunchCfg &lc, hipStream_t st) {
  const S7Args<double, double> a = s7_args<double, double>(P, Y, Z1, Z, src, src_idx, lc);
  return streaming_sweep(P) ? k1_dispatch<true>(tl, lc.ftile, a, st) : k1_dispatch<false>(tl, lc.ftile, a, st);
}

}  // namespace gr
