// gr_star7_launch.hpp -- host-side launch of star7_tb_kernel (gr_star7.hpp).
#pragma once
#include "gr_star7.hpp"

namespace gr {

template <typename T, typename C, int KID, int TL, int TX, int TY, int NT, int P, int PD, bool STRM>
static hipError_t launch_s7(S7Args<T, C> a, hipStream_t st) {
  if (g_fused_tile_probe) {
    g_fused_tile_probe[0] = TX;
    g_fused_tile_probe[1] = TY;
    return hipSuccess;
  }
  a.tiles_x = (a.nx + TX - 1) / TX;
  a.tiles_y = (a.ny + TY - 1) / TY;
  a.zchunk = (a.zchunk <= 0 || a.zchunk > a.nz) ? a.nz : a.zchunk;
  a.nzc = (a.nz + a.zchunk - 1) / a.zchunk;
  a.nwork = a.tiles_x * a.tiles_y * a.nzc;
  const dim3 grid(a.nwork + (a.H ? (unsigned)((halo_waves(a.ny, a.nz, 1) + NT / 64 - 1) / (NT / 64)) : 0u));
  const bool gen = a.src_k >= 0 || a.Z1;
  if constexpr (KID == 5) {
    if (a.down) {  // plane k of the arguments is plane nz + 1 - k of the fields
      const long long top = (a.nz + 1) * a.sz;
      a.Y += top;
      a.Z += top;
      if (a.Z1) a.Z1 += top;
      a.coef += top;
      if (a.src_k >= 0) a.src_k = a.nz + 1 - a.src_k;
      a.sz = -a.sz;
      if (gen)
        hipLaunchKernelGGL((star7_tb_kernel<T, C, KID, TL, TX, TY, NT, P, PD, STRM, true, true>), grid, dim3(NT), 0, st,
                           a);
      else
        hipLaunchKernelGGL((star7_tb_kernel<T, C, KID, TL, TX, TY, NT, P, PD, STRM, false, true>), grid, dim3(NT), 0, st,
                           a);
      return hipGetLastError();
    }
  }
  if (gen)
    hipLaunchKernelGGL((star7_tb_kernel<T, C, KID, TL, TX, TY, NT, P, PD, STRM, true, false>), grid, dim3(NT), 0, st, a);
  else
    hipLaunchKernelGGL((star7_tb_kernel<T, C, KID, TL, TX, TY, NT, P, PD, STRM, false, false>), grid, dim3(NT), 0, st, a);
  return hipGetLastError();
}

// Arguments of a pass Y -> Z over problem P (fields given with the x offset applied); Z1,
// when given, receives level tl-1.
template <typename T, typename C>
static S7Args<T, C> s7_args(const Problem &P, const void *Y, void *Z1, void *Z, const void *src, long long src_idx,
                            const LaunchCfg &lc) {
  S7Args<T, C> a{};
  a.Y = (const T *)Y - P.xoff;
  a.Z = (T *)Z - P.xoff;
  a.Z1 = Z1 ? (T *)Z1 - P.xoff : nullptr;
  a.c0 = (T)P.c[0];
  a.c1 = (T)P.c[1];
  a.sz = (long long)P.pitch * P.rows;
  a.sy = P.pitch;
  a.xoff = P.xoff;
  a.nx = P.nx;
  a.ny = P.ny;
  a.nz = P.nz;
  a.xcd_order = lc.xcd_order;
  a.zchunk = lc.zchunk;
  a.down = lc.down;
  a.HS = (const T *)Y;
  a.H = (T *)lc.halo;
  a.src = (const T *)src;
  a.src_k = src_idx < 0 ? -1 : (int)(src_idx / a.sz);
  a.src_off = src_idx < 0 ? 0 : (int)(src_idx % a.sz) + P.xoff;
  return a;
}

}  // namespace gr
