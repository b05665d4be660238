// gr_star7.hpp -- TL steps of a 7-point stencil (girih's kernels 1 and 5) per HBM pass.
//
// The GPU analogue of a diamond of height TL with the z wavefront of
// stencils_1wf.ic:19-82: a pass reads the field and the coefficients once and
// writes the field once for TL updates.
//
// Scheme (z streaming, one barrier per plane step):
//   * a workgroup owns an output tile of TX x TY cells and a chunk of z planes;
//     every level is computed over the tile plus a margin (the ghost zone of the
//     last level that makes the tile independent of its neighbours);
//   * a lane owns slots of P cells adjacent in x (P = 2 where the registers allow:
//     half the load, store, LDS and address instructions per cell, and one x
//     neighbour of each cell in the lane itself), in row-major order;
//   * in plane step k, level t computes plane k-t: its z neighbours are level
//     t-1's planes k-t-1 .. k-t+1 (the same lane's queue, the newest computed in
//     this step), its xy neighbours come from level t-1's plane k-t in LDS,
//     written one step earlier (levels >= 1) or at the start of this step (the
//     input).  Every level writes its plane into a double-buffered LDS slot, so
//     one barrier per step orders all levels;
//   * kernel 5's coefficients of a plane are loaded one step before level 1 needs
//     them and then stay in the lane's registers while the plane passes through the
//     levels (one per step), so they are read from memory once;
//   * the input is loaded PD planes ahead: kernel 1's plane step (0.3-0.8 us) is shorter
//     than the latency of a load from HBM (512^3 with PD 2 against 1: FP32 depth 4 1694
//     against 1472 GLUP/s, FP64 944 against 812); kernel 5, whose steps stream eight
//     arrays, gains nothing;
//   * the x margin is a whole number of slots and covers the input's ring, so only
//     the ring rows above and below the region are loaded apart;
//   * the plane loop is unrolled by UN steps, so queue (mod 3), LDS (mod 2) and
//     coefficient (mod TL) slots are compile-time constants.
//
// The arithmetic is the single sweep's (girih's operand order, no contraction),
// so a pass is bit-identical to TL sweeps.  Boundary cells (girih's halo) keep
// their input value at every level; the host runs this path only when U1 and U2
// hold the same halo.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <type_traits>

#include "gr_internal.hpp"
#include "gr_plane.hpp"
#include "gr_sweep.hpp"

namespace gr {

// Fields are addressed from the start of their rows (the x offset NOT applied):
// element (i, j, k) at base[k*sz + j*sy + xoff + i].  xoff + R and sy are even, so a
// slot of two cells that starts an even distance from the first interior cell never
// straddles a row end.  The coefficient base is moved so that the fields' element
// index addresses it.
template <typename T, typename C>
struct S7Args {
  const T *Y;     // input level
  T *Z;           // level TL
  const C *coef;  // kernel 5: array m at coef + m*cstride
  long long cstride, sz;
  T c0, c1;       // kernel 1
  int sy, xoff;
  int nx, ny, nz;  // interior; boxes are [1, n+1)
  int tiles_x, tiles_y, nzc, zchunk, xcd_order;
  // read by the GEN instantiations only
  T *Z1;         // level TL-1 (null: not written)
  const T *src;  // level t adds src[t-1] at plane src_k, in-plane element src_off from the
                 // row start (src_k < 0: no source)
  int src_k, src_off;
  bool down;  // read by the host only: the DN instantiation, its planes numbered from the top
  // Workgroups from nwork on copy the halo of HS to H (x offset applied; null: there are none)
  // while the others compute.  Cost per call, a launch of its own / here: 128^3 FP64 5.4 / 0.5
  // us, 389 x 270 x 331 FP32 18 / 2, 512^3 FP32 30 / 21.
  const T *HS;
  T *H;
  int nwork;
};

// P adjacent elements at byte offset `off` of a uniform base.
template <typename X, int P>
struct Slot {
  typedef X type __attribute__((ext_vector_type(P)));
};
template <typename X>
struct Slot<X, 1> {
  typedef X type;
};
template <typename X, int P>
__device__ __forceinline__ void ld_slot(const X *base, unsigned off, X (&v)[P]) {
  const auto r = *reinterpret_cast<const typename Slot<X, P>::type *>(reinterpret_cast<const char *>(base) + off);
  if constexpr (P == 1)
    v[0] = r;
  else
#pragma unroll
    for (int e = 0; e < P; ++e) v[e] = r[e];
}
template <typename X, int P>
__device__ __forceinline__ void st_slot(X *p, const X (&v)[P]) {
  typename Slot<X, P>::type r;
  if constexpr (P == 1)
    r = v[0];
  else
#pragma unroll
    for (int e = 0; e < P; ++e) r[e] = v[e];
  *reinterpret_cast<typename Slot<X, P>::type *>(p) = r;
}

template <typename X, int P, bool NT>
__device__ __forceinline__ void st_slot_strm(X *base, unsigned off, const X (&v)[P]) {
  typename Slot<X, P>::type r;
  if constexpr (P == 1)
    r = v[0];
  else
#pragma unroll
    for (int e = 0; e < P; ++e) r[e] = v[e];
  stb_stream<typename Slot<X, P>::type, NT>(base, off, r);
}

template <typename T, typename C, int KID, int TL, int TX, int TY, int NT, int P>
struct Star7 {
  static constexpr int PAD = P == 4 ? 4 : 2;
  static constexpr int MX = (TL + P - 1) / P * P, MY = TL - 1;  // margins of the computed region
  static constexpr int W = TX + 2 * MX, H = TY + 2 * MY;        // computed region
  static constexpr int WS = W / P;                              // slots per row
  static constexpr int NS = (WS * H + NT - 1) / NT;             // slots per lane
  static constexpr int NR = (2 * WS + NT - 1) / NT;             // ring slots per lane
  static constexpr int PL = (H + 2) * W + 2 * PAD;  // one LDS plane: ring rows, slack at both ends
  static constexpr int NC = kncoef(KID);
  // bf16 coefficients stay packed as loaded, P to a 32-bit register
  static constexpr bool PK = std::is_same<C, __hip_bfloat16>::value;
  static constexpr int UN = (TL == 4 && NC > 0) ? 12 : 6;       // multiple of 2, 3 and (kernel 5) TL
  static_assert(TX % P == 0 && UN % 6 == 0 && (NC == 0 || UN % TL == 0), "tile and unroll");
};

template <typename T, typename C, int KID, int TL, int TX, int TY, int NT, int P, int PD, bool STRM,
          bool GEN, bool DN>
__global__ __launch_bounds__(NT) void star7_tb_kernel(const S7Args<T, C> a) {
  using G = Star7<T, C, KID, TL, TX, TY, NT, P>;
  constexpr int W = G::W, H = G::H, WS = G::WS, NS = G::NS, NR = G::NR, NC = G::NC, UN = G::UN;
  constexpr bool PK = G::PK;
  constexpr int PAD = G::PAD;
  __shared__ __align__(16) T lds[TL][2][G::PL];  // level t's latest planes (t = 0: the input)

  if (a.H && (int)blockIdx.x >= a.nwork) {
    const long long w = (long long)((int)blockIdx.x - a.nwork) * (NT / 64) + threadIdx.x / 64;
    for_halo_cells(w, threadIdx.x % 64, a.nx, a.ny, a.nz, 1, a.sy, [&](long long o) { a.H[o] = a.HS[o]; });
    return;
  }
  const int ntile = a.tiles_x * a.tiles_y;
  const int lb = tile_order(blockIdx.x, ntile * a.nzc, ntile, a.xcd_order);
  const int tile = lb % ntile;
  const int tx0 = 1 + (tile % a.tiles_x) * TX;  // first output cell (girih indices)
  const int ty0 = 1 + (tile / a.tiles_x) * TY;
  const int zs = 1 + (lb / ntile) * a.zchunk;
  const int ze = min(zs + a.zchunk, a.nz + 1);
  const int nny = a.ny + 2, nnz = a.nz + 2;
  const int tid = threadIdx.x;

  // byte offset of the slot at (gx, gy) from the row start of its plane, clamped into the plane
  auto boff = [&](int gx, int gy) {
    gy = min(max(gy, 0), nny - 1);
    return (unsigned)(gy * a.sy + min(gx + a.xoff, a.sy - P)) * (unsigned)sizeof(T);
  };
  unsigned off[NS];
  int lo[NS];  // LDS index of the cell's (-PAD, -1) neighbour: every read has a non-negative immediate offset
  int nout[NS];  // leading cells of the slot that are output cells
  bool inner[NS][P];
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    // spare lanes repeat the last slot: they compute and stage its values again
    const int s = min(tid + j * NT, WS * H - 1);
    const int cx = (s % WS) * P, cy = s / WS;
    const int gx = tx0 - G::MX + cx, gy = ty0 - G::MY + cy;
    off[j] = boff(gx, gy);
    lo[j] = cy * W + cx;
#pragma unroll
    for (int e = 0; e < P; ++e)
      inner[j][e] = gx + e >= 1 && gx + e < a.nx + 1 && gy >= 1 && gy < a.ny + 1;
    const bool o = tid + j * NT < WS * H && cx >= G::MX && cx < G::MX + TX && cy >= G::MY && cy < G::MY + TY &&
                   gy < a.ny + 1;
    nout[j] = o ? min(a.nx + 1 - gx, P) : 0;
  }
  // ring rows -1 and H of the region (input only)
  unsigned roff[NR];
  int rl[NR];
  bool rw[NR];  // lanes that own a ring slot
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    const int c = min(tid + s * NT, 2 * WS - 1);
    rw[s] = tid + s * NT < 2 * WS;
    const int ry = c < WS ? -1 : H, cx = (c < WS ? c : c - WS) * P;
    roff[s] = boff(tx0 - G::MX + cx, ty0 - G::MY + ry);
    rl[s] = (ry + 1) * W + cx + PAD;
  }
  auto yplane = [&](int k) { return a.Y + (long long)min(max(k, 0), nnz - 1) * a.sz; };
  const T c0 = a.c0, c1 = a.c1;

  // queues: level t's plane p in the slot of the step that computed it, mod 3
  T q[TL][NS][3][P];
#pragma unroll
  for (int t = 0; t < TL; ++t)
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int e = 0; e < P; ++e) q[t][j][i][e] = T(0);
  // coefficients: plane p's set in slot p mod TL, and the next plane's in nc
  using W1 = typename std::conditional<PK, unsigned, T>::type;
  constexpr int CP = PK ? (P + 1) / 2 : P;  // words per slot and array
  W1 cs[TL][NS][NC > 0 ? NC : 1][CP], nc[NS][NC > 0 ? NC : 1][CP];
  auto ld_coefs = [&](int p, int j, W1 (&c)[NC > 0 ? NC : 1][CP]) {  // plane p's coefficients of slot j
    const C *cp = a.coef + (long long)min(max(p, 0), nnz - 1) * a.sz;
#pragma unroll
    for (int m = 0; m < NC; ++m) {
      const C *pm = cp + m * a.cstride;
      if constexpr (PK && P == 1)
        c[m][0] = ldb<unsigned short>(pm, off[j] / 2u);
      else if constexpr (PK)
        ld_slot<unsigned, CP>(reinterpret_cast<const unsigned *>(pm), off[j] / 2u, c[m]);
      else
        ld_slot<T, P>(reinterpret_cast<const T *>(pm), off[j], c[m]);
    }
  };

  const int kfirst = zs - TL, kend = ze + TL;  // step k: the input's plane k enters; level t computes k - t
  // input planes in flight: plane k's slots and the ring rows of plane k - 1 in k mod PD
  T nv[PD][NS][P], hv[PD][NR][P];
  auto fetch = [&](int k, int slot) {  // input plane k and the ring rows of plane k - 1
    const T *vp = yplane(k), *hp = yplane(k - 1);
#pragma unroll
    for (int j = 0; j < NS; ++j) ld_slot<T, P>(vp, off[j], nv[slot][j]);
#pragma unroll
    for (int s = 0; s < NR; ++s)
      if (rw[s]) ld_slot<T, P>(hp, roff[s], hv[slot][s]);
  };
#pragma unroll
  for (int i = 0; i < PD; ++i) fetch(kfirst + i, i);
  if constexpr (NC > 0) {
#pragma unroll
    for (int j = 0; j < NS; ++j) ld_coefs(kfirst - 1, j, nc[j]);
  }

  auto put = [&](T *z, int p, int j, const T (&val)[P]) {  // the slot's output cells of plane p
    T *zp = z + (long long)p * a.sz;
    if (nout[j] == P) {
      st_slot_strm<T, P, STRM>(zp, off[j], val);
    } else {  // the grid ends inside the slot
#pragma unroll
      for (int e = 0; e < P - 1; ++e)
        if (e < nout[j]) stb_stream<T, STRM>(zp, off[j] + e * (unsigned)sizeof(T), val[e]);
    }
  };

  auto step = [&](int kb, auto PHC) __attribute__((always_inline)) -> bool {
    constexpr int ph = decltype(PHC)::value;
    constexpr int qs = ph % 3, qm1 = (ph + 2) % 3, qm2 = (ph + 1) % 3;  // slots of steps k, k-1, k-2
    constexpr int bs = ph % 2, bm1 = (ph + 1) % 2;                      // LDS slots of steps k, k-1
    const int k = kb + ph;
    if (k >= kend) return false;
    // the input's plane k enters its queue; its plane k-1 (level 1's centre plane) goes to
    // LDS; plane k-1's coefficients take the slot of plane k-1-TL, which level TL has done
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
      for (int e = 0; e < P; ++e) q[0][j][qs][e] = nv[ph % PD][j][e];
    {
      T *L0 = lds[0][bs];
#pragma unroll
      for (int j = 0; j < NS; ++j)
        st_slot<T, P>(L0 + lo[j] + W + PAD, q[0][j][qm1]);
#pragma unroll
      for (int s = 0; s < NR; ++s)
        if (rw[s]) st_slot<T, P>(L0 + rl[s], hv[ph % PD][s]);
    }
    if constexpr (NC > 0) {
#pragma unroll
      for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int m = 0; m < NC; ++m)
#pragma unroll
          for (int e = 0; e < CP; ++e) cs[(ph + TL - 1) % TL][j][m][e] = nc[j][m][e];
    }
    // packed words are widened by every level that uses them: keep the compiler from
    // widening them once and holding the (twice as many) FP32 registers instead
    if constexpr (PK && NC > 0) {
#pragma unroll
      for (int t = 0; t < TL; ++t)
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
          for (int m = 0; m < NC; ++m)
#pragma unroll
            for (int e = 0; e < CP; ++e) asm("" : "+v"(cs[t][j][m][e]));
    }
    fetch(k + PD, ph % PD);
    if constexpr (NC > 0) {
#pragma unroll
      for (int j = 0; j < NS; ++j) ld_coefs(k, j, nc[j]);  // level 1's next centre plane
    }
    __syncthreads();

#pragma unroll
    for (int t = 1; t <= TL; ++t) {
      const int p = k - t;
      const bool zin = p >= 1 && p < a.nz + 1;
      // (p runs below plane 0 for the first chunk: src_k = -1 means "no source" and must not match it)
      const bool srcp = GEN && a.src_k >= 0 && p == a.src_k;
      const T *Lp = lds[t - 1][t == 1 ? bs : bm1];  // level t-1's plane p
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const T *Lc = Lp + lo[j];
        const T xl = Lc[W + PAD - 1], xr = Lc[W + PAD + P];
        T ym[P], yp[P], val[P];
        ld_slot<T, P>(Lc + PAD, 0, ym);
        ld_slot<T, P>(Lc + 2 * W + PAD, 0, yp);
#pragma unroll
        for (int e = 0; e < P; ++e) {
          const T v0 = q[t - 1][j][qm1][e];                           // plane p
          const T zm = q[t - 1][j][qm2][e], zp = q[t - 1][j][qs][e];  // planes p-1, p+1
          const T xm = e == 0 ? xl : q[t - 1][j][qm1][e > 0 ? e - 1 : 0];
          const T xp = e == P - 1 ? xr : q[t - 1][j][qm1][e < P - 1 ? e + 1 : e];
          T out;
          if constexpr (KID == 1) {  // stencils.c:73-78, operand order kept
            out = c0 * v0 + c1 * (xp + xm) + c1 * (yp[e] + ym[e]) + c1 * (zp + zm);
          } else {  // KID == 5, stencils.c:193-201
            T c[7];
#pragma unroll
            for (int m = 0; m < 7; ++m) {
              const W1 w = cs[(ph + 2 * TL - t) % TL][j][m][PK ? e / 2 : e];
              if constexpr (PK)  // a bf16 value is the top half of its FP32 value
                c[m] = __uint_as_float(e & 1 ? (w & 0xffff0000u) : (w << 16));
              else
                c[m] = w;
            }
            out = c[0] * v0 + c[1] * xm + c[2] * xp + c[3] * ym[e] + c[4] * yp[e] + c[5] * (DN ? zp : zm) +
                  c[6] * (DN ? zm : zp);
          }
          if (GEN && srcp && off[j] + e * (unsigned)sizeof(T) == (unsigned)a.src_off * (unsigned)sizeof(T))
            out = out + a.src[t - 1];
          val[e] = (inner[j][e] && zin) ? out : v0;  // girih's halo keeps its value
        }
        if (GEN && t == TL - 1 && a.Z1 && p >= zs && p < ze) put(a.Z1, p, j, val);
        if (t < TL) {
#pragma unroll
          for (int e = 0; e < P; ++e) q[t < TL ? t : 0][j][qs][e] = val[e];
          st_slot<T, P>(lds[t < TL ? t : 0][bs] + lo[j] + W + PAD, val);
        } else if (p >= zs && p < ze) {
          put(a.Z, p, j, val);
        }
      }
    }
    return true;
  };
  for (int kb = kfirst; kb < kend; kb += UN) static_for<UN>([&](auto PHC) __attribute__((always_inline)) {
    return step(kb, PHC);
  });
}

}  // namespace gr
