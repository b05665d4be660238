// gr_runtime.hip -- host side of the C ABI declared in include/girih_gpu.h.
//
// Owns the device fields of one problem, converts between girih's padded host
// layout (src/utils.c:367-374) and the device layout, and drives the sweep
// kernels with girih's step pairing (src/kernels/nb_naive_ts.c:187-203).
//
// Device layout of one field: element (i, j, k) (halo-inclusive girih indices)
// at  base + x_offset + (k*rows_y + j)*pitch_x + i, rows_y = ny+2R,
// planes = nz+2R.  x_offset puts the first interior cell (i = R) on a 128-byte
// boundary and pitch_x is a multiple of 128 bytes, so every wavefront row
// access of the interior is cache-line aligned.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "../../include/girih_gpu.h"
#include "gr_internal.hpp"
#include "gr_launch.hpp"
#include "gr_plane.hpp"

namespace {

thread_local char g_err[512] = "";
constexpr int kSrcPad = 64;  // zero source values past the end (fused passes read up to 64 ahead)

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

#define HIP_TRY(expr)                                                                     \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess)                                                                 \
      return fail(GR_EHIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, \
                  __LINE__);                                                              \
  } while (0)

}  // namespace

namespace gr {

int set_error(int code, const char *msg) { return fail(code, "%s", msg); }
int set_errorf(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

size_t elem_size(int dtype) { return dtype == GR_F64 ? 8 : 4; }

// Bytes per cell that a sweep of P streams: both fields and the coefficient arrays.
static double cell_bytes(const Problem &P) {
  const double cbytes = (P.flags & GR_COEF_BF16) ? 2.0 : (double)elem_size(P.dtype);
  return 2.0 * elem_size(P.dtype) + cbytes * (P.ncoef + (P.roc2 ? 1 : 0));
}
static double sweep_bytes(const Problem &P) { return (double)P.field_elems * cell_bytes(P); }

// Whether sweeps and kernel-1 passes mark what they touch once as non-temporal: where the 256
// MB Infinity Cache no longer holds it from one sweep to the next.  The fields with their rows'
// padding must exceed it (kernel 1 FP64 384 x 384 x 100, 250 MB: 51 us a sweep without the hints,
// 55 with), and their cells a line that differs by kernel, as sweeps of more arrays lose more
// below it (kernel 5 FP32 128 x 300 x 128 has 175 MB of cells in 259 MB: 67 us without, 85 with).
// us per sweep without / with, cubes and 128-wide boxes (MB of cells):
//   kernel 0 FP64 225 67 / 72, 262 98 / 99, 301 121 / 119; FP32 201 60 / 64, 222 80 / 80, 294 95 / 90
//   kernel 1 FP64 240 56 / 55, 278 71 / 66; FP32 184 47.5 / 44.9, 239 57 / 56, 274 69 / 64
//   kernel 2 FP64 206 42 / 43, 240 51 / 50; FP32 186 43.9 / 42.6, 206 48.5 / 45.5
//   kernel 3 FP64 309 61 / 63, 346 71 / 69; FP32 186 39.3 / 38.9, 206 44 / 42, 240 52 / 48
//   kernel 4 FP64 332 61 / 66, 356 77 / 77, 393 74 / 73; FP32 312 64 / 65, 345 69 / 67
//   kernel 5 FP64 289 64 / 70, 308 65 / 65, 346 72 / 70; FP32 288 53 / 56, 309 67 / 67, 342 71 / 67;
//     bf16 206 43.3 / 43.1, 241 52 / 51, 309 65 / 63
// Passes of kernel 1 gain 1..5% from 250 MB on, those of kernel 5 do not care.
int streaming_sweep(const Problem &P) {
  if (P.strm_mode >= 0) return P.strm_mode;
  static const int line_mb[6][3] = {{256, 225, 210}, {235, 180, 180}, {230, 180, 180},  // FP64, FP32, bf16 arrays
                                    {330, 180, 180}, {340, 330, 300}, {310, 310, 235}};
  constexpr double mb = 1024.0 * 1024.0;
  const double cells = (double)(P.nx + 2 * P.R) * (P.ny + 2 * P.R) * (P.nz + 2 * P.R);
  const int type = P.dtype == GR_F64 ? 0 : (P.flags & GR_COEF_BF16) ? 2 : 1;
  return sweep_bytes(P) > 256 * mb && cells * cell_bytes(P) > line_mb[P.kernel][type] * mb ? 1 : 0;
}

// ------------------------------------------------------------------ tile variants
// Tile variants selectable at run time for the kernels on the hot path (the
// other kernels use their default tile).  Lanes are 64*BX x BY, RY rows per lane:
//   0: default (64 x 16)                 1: 64x32 (8 x 4)   2: 64x16 (8 x 2)
//   3: 64x32 (8 x 4), >= 4 (FP32) / 3 (FP64) waves per SIMD
//   4: 64x16 (4 x 4), >= 4 (FP32) / 3 (FP64) waves per SIMD
//   5: as 3 with the LDS plane ring (halo fetched with the plane interior)
//   6: 64x16 (8 x 2) with the LDS plane ring
//   7: as 4 with the LDS plane ring
//   8: 128x16 (2 waves wide, 4 x 4)      9: 128x32 (8 x 4, 1024 lanes)
//  10: as 8 with the LDS plane ring     11: as 8 with >= 4 / 3 waves per SIMD
//  12: 128x8 (2 x 4) ring, 256 lanes    13: 128x16 (8 x 2) ring, 1024 lanes
//  14: as 10 with >= 4 / 3 waves per SIMD
//  15: 256x8 (4 waves wide, 2 x 4) ring (double-buffered tile where the ring does not fit in LDS)
//  16: kernel 0 only: as 13, with u^(n-1) (and roc2) of plane k+1 loaded while plane k is computed
int num_tile_variants(int kid, int dtype) {
  (void)dtype;
  return kid == 0 ? 17 : (kid == 1 || kid == 5) ? 16 : 1;
}
void tile_of_variant(int kid, int dtype, int variant, int *tx, int *ty) {
  static const int rows[17] = {16, 32, 16, 32, 16, 32, 16, 16, 16, 32, 16, 16, 8, 16, 16, 8, 16};
  static const int cols[17] = {64, 64, 64, 64, 64, 64, 64, 64, 128, 128, 128, 128, 128, 128, 128, 256, 128};
  const bool ok = variant > 0 && variant < num_tile_variants(kid, dtype);
  *tx = ok ? cols[variant] : 64;
  *ty = ok ? rows[variant] : 16;
}

// The settings of a sweep that nobody tuned (gr_sweep_dev, and steppers until gr_set_config,
// gr_set_xcd_order or gr_autotune), by kernel and box.  Measured on the sweep entry
// point over 32^3 .. 600 x 600 x 300 in FP32 and FP64 (times per call, with its synchronisation):
//  * chunks: whole-z items leave most CUs idle (403 x 300 x 219 FP32: kernel 0 317 us against
//    119, kernel 5 540 against 262).  Enough chunks for two 512-lane workgroups per CU
//    (64^3 kernel 1 FP64: 54 us whole, 20 at 8 planes, 18 at 4), but not longer than the
//    kernel gains from: 32 planes for kernel 0, whose chunks re-read 8 planes (512^3 FP32
//    32 planes 486 us, 16 500; on 64-wide tiles, more of which fit a CU, 16: 403 x 300 x
//    219 FP32 119 us, 32 planes 135), 16 for kernel 1 (512^3 FP32 247 us, 32 planes 248, 128
//    251), 4 where coefficient arrays are streamed (600 x 600 x 300 kernel 5 FP64 4 planes
//    1490 us, 8 1534, 16 1558; 403 x 300 x 219 kernel 4 384, 405, 419), but 16 for kernel 4 in FP64,
//    whose chunks re-read 8 planes, from 200000 cells a plane on (us per four sweeps at 4 / 16
//    planes: 512 x 512 x 256 6097 / 5839, 700 x 500 x 200 6601 / 6495, 448 x 330 x 260 3516 / 3578);
//  * tile: 128 x 16 of 1024 lanes (for kernel 0 with the operand prefetch) where it overhangs
//    the box no further than 64 x 16 does (256^3 kernel 0 FP32 60 us against 62, 512^3
//    486 against 520; but 320^3 138 against 133) and there is work for 256 of them, or with
//    chunks of the caller's for 256 (kernel 0) or 150 (us per four sweeps, wide / 64 x 16: 152
//    workgroups, 128 x 300 x 128 at 16 planes, kernel 0 FP32 102 / 97, kernel 1 FP64 73 / 79; 144, kernel 0
//    FP64 384 x 384 x 100 at 64 planes 638 / 468; 64, kernel 5 FP64 250 x 120 x 200 936 / 583);
//    else 64 x 16 of 512 lanes (64^3 kernel 0 19 us against 22);
//  * order: XCD bands of tile rows (403 x 300 x 219 kernel 3 157 us, plain runs 164).
LaunchCfg sweep_cfg(int kid, int dtype, const LaunchCfg &lc, int nx, int ny, int nz) {
  LaunchCfg c = lc;
  const bool hot = kid == 0 || kid == 1 || kid == 5;  // kernels with tile variants
  if (lc.auto_variant) {
    const long long chunks = lc.zchunk > 0 && lc.zchunk < nz ? (nz + lc.zchunk - 1) / lc.zchunk : 1;  // the caller's
    const bool enough = lc.auto_zchunk ? (long long)nx * ny * nz >= (1 << 21)
                                       : (nx + 127) / 128 * ((ny + 15) / 16) * chunks >= (kid == 0 ? 256 : 150);
    const bool wide = (nx + 127) / 128 * 2 == (nx + 63) / 64 && enough;
    c.variant = !hot ? 0 : !wide ? 2 : kid == 0 ? 16 : 13;
  }
  if (lc.auto_zchunk) {
    int tx = 64, ty = 16;
    tile_of_variant(kid, 0, c.variant, &tx, &ty);
    const long long tiles = (long long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
    const bool wide4 = kid == 4 && dtype == GR_F64 && (long long)nx * ny >= 200000;
    const int most = kid == 0 ? (tx > 64 ? 32 : 16) : kid == 1 || wide4 ? 16 : 4;
    c.zchunk = (int)std::min<long long>(most, std::max<long long>(4, tiles * nz / (tx > 64 ? 256 : 512)));
  }
  if (lc.auto_order) c.xcd_order = 2;
  c.auto_variant = c.auto_zchunk = c.auto_order = false;
  return c;
}

// Whether successive sweeps or passes over P run up and down z in turn (LaunchCfg::down), so
// that each starts with the planes that the one before touched last, while the 256 MB
// Infinity Cache still holds them.  Kernel-0 sweeps, GLUP/s one way / in turn: FP32 with
// roc2 at 288^2 x 316 (300 MB) 251 / 269 and at 400^3 (1 GB) 315 / 320, FP64 at 500 x 330 x
// 270 (1.4 GB) 162 / 168 and at 768^2 x 512 (9 GB) 166 / 167; the same at 12 GB and within
// the cache.  Kernel-5 passes: FP64 at 192^2 x 200 (500 MB) 190 / 205 and at 320^3 (2.2 GB)
// 205 / 209, FP32 at 192^2 x 200 306 / 327, but FP64 at 512^3 (9 GB) 241 / 235.  Kernel-1
// passes, bound by their arithmetic, gained nothing.
static bool z_turns(const Problem &P) {
  const double mb = sweep_bytes(P) / (1024 * 1024);
  return P.kernel == 5 ? mb < 4096 : streaming_sweep(P) && mb < 10240;
}

// The same sweep with its planes numbered from the top: plane k of the arguments is plane
// zb + ze - 1 - k of the fields.  Kernels 0 to 4 add the planes below and above in pairs, and
// so give the same bits either way; kernel 5 does not (its passes have an instantiation
// for it, its sweeps run up only).
template <typename T, typename C>
static void turn(SweepArgs<T, C> &a) {
  const long long top = (a.g.zb + a.g.ze - 1) * a.g.sz;
  a.u += top;
  a.v += top;
  if (a.uold) a.uold += top;
  if (a.roc2) a.roc2 += top;
  if (a.coef) a.coef += top;
  if (a.src_k >= 0) a.src_k = a.g.zb + a.g.ze - 1 - a.src_k;
  a.g.sz = -a.g.sz;
}

// One sweep u <- f(v) with the handle's configuration.
hipError_t sweep_fields(const Problem &P, void *u, const void *v, const void *src, long long src_idx,
                        const LaunchCfg &cfg, hipStream_t st, const void *uold) {
  const LaunchCfg lc = sweep_cfg(P.kernel, P.dtype, cfg, P.nx, P.ny, P.nz);
  const bool down = lc.down && P.kernel != 5 && z_turns(P);
  const bool fast = (P.flags & GR_FAST) != 0;
  const bool rocs = (P.flags & GR_ROC2_SCALAR) != 0;
  const bool bf16 = (P.flags & GR_COEF_BF16) != 0;
  Geom g;
  g.sy = P.pitch;
  g.sz = (long long)P.pitch * P.rows;
  g.xb = P.R;
  g.yb = P.R;
  g.zb = P.R;
  g.xe = P.nx + P.R;
  g.ye = P.ny + P.R;
  g.ze = P.nz + P.R;
  if (P.dtype == GR_F64) {
    SweepArgs<double, double> a{};
    a.u = (double *)u;
    a.v = (const double *)v;
    a.uold = (const double *)uold;
    a.roc2 = (const double *)P.roc2;
    a.coef = (const double *)P.coef;
    a.cstride = P.field_elems;
    for (int r = 0; r < 5; ++r) a.c[r] = P.c[r];
    a.roc2s = P.roc2s;
    a.g = g;
    a.src = (const double *)src;
    a.src_k = src_idx < 0 ? -1 : (int)(src_idx / g.sz);
    a.src_off = src_idx < 0 ? 0 : (int)(src_idx % g.sz);
    if (down) turn(a);
    return launch_sweep_f64(P.kernel, false, rocs, a, lc, st, streaming_sweep(P));
  }
  if (bf16) {
    SweepArgs<float, __hip_bfloat16> a{};
    a.u = (float *)u;
    a.v = (const float *)v;
    a.uold = (const float *)uold;
    a.roc2 = (const __hip_bfloat16 *)P.roc2;
    a.coef = (const __hip_bfloat16 *)P.coef;
    a.cstride = P.field_elems;
    for (int r = 0; r < 5; ++r) a.c[r] = (float)P.c[r];
    a.csum = fast_csum(P.c);
    a.roc2s = (float)P.roc2s;
    a.g = g;
    a.src = (const float *)src;
    a.src_k = src_idx < 0 ? -1 : (int)(src_idx / g.sz);
    a.src_off = src_idx < 0 ? 0 : (int)(src_idx % g.sz);
    if (down) turn(a);
    return launch_sweep_bf16(P.kernel, fast, rocs, a, lc, st, streaming_sweep(P));
  }
  SweepArgs<float, float> a{};
  a.u = (float *)u;
  a.v = (const float *)v;
  a.uold = (const float *)uold;
  a.roc2 = (const float *)P.roc2;
  a.coef = (const float *)P.coef;
  a.cstride = P.field_elems;
  for (int r = 0; r < 5; ++r) a.c[r] = (float)P.c[r];
  a.csum = fast_csum(P.c);
  a.roc2s = (float)P.roc2s;
  a.g = g;
  a.src = (const float *)src;
  a.src_k = src_idx < 0 ? -1 : (int)(src_idx / g.sz);
  a.src_off = src_idx < 0 ? 0 : (int)(src_idx % g.sz);
  if (down) turn(a);
  return launch_sweep_f32(P.kernel, fast, rocs, a, lc, st, streaming_sweep(P));
}

}  // namespace gr

using namespace gr;

// What a captured step sequence depends on besides the (fixed) field allocations.
struct GraphKey {
  int napply, parity, lu0, lu1, variant, zchunk, t_block, xcd_order, ftile, autos, fuse, exposed;
  long long napplied;  // -1 unless a source is active (its pointers are baked into the graph)
  bool operator==(const GraphKey &o) const {
    return napply == o.napply && parity == o.parity && lu0 == o.lu0 && lu1 == o.lu1 && variant == o.variant &&
           zchunk == o.zchunk && t_block == o.t_block && xcd_order == o.xcd_order && ftile == o.ftile && autos == o.autos && fuse == o.fuse &&
           exposed == o.exposed && napplied == o.napplied;
  }
};

struct gr_handle {
  Problem P;
  LaunchCfg lc;
  // Physical field buffers: 0 and 1 always exist; 2 and 3 are spares for fused
  // kernel-0 passes and for the autotuner.  lu[] maps logical U1 / U2 onto them.
  void *fbuf[4] = {nullptr, nullptr, nullptr, nullptr};
  int lu[2] = {0, 1};
  bool spares_synced = false;  // spares hold the same halo as U1/U2
  bool no_spare = false;       // no memory for a third buffer: not asked for again until the fields are set
  int halo_equal = -1;         // U1 and U2 hold the same halo (-1: not yet checked)
  bool exposed = false;        // gr_field_ptr gave a field's pointer away: the caller may write halos between calls
  void *alloc_roc2 = nullptr, *alloc_coef = nullptr;
  void *flag = nullptr;  // one device int for checks
  void *src = nullptr;  // device source values (padded with zeros)
  int nsrc = 0;
  long long src_idx = -1;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  int parity = 0;      // 0: next application writes U1
  long long napplied = 0;
  gr_stats stats{};
  int device = 0;
  int ncu = 1;         // compute units of the device
  // pinned slots of the host-field copies (copy_rows), one event each
  void *stage = nullptr;
  size_t stage_bytes = 0;
  hipEvent_t stage_ev[8] = {};
  // graph mode (gr_set_graph): the last captured step sequence and the state it leaves
  bool use_graph = false;
  hipGraphExec_t gexec = nullptr;
  GraphKey gkey{};
  int gparity = 0, glu[2] = {0, 1}, glaunches = 0;
  int captures = 0;  // sequences captured so far
};

static void drop_graph(gr_handle *h);
static void free_stage(gr_handle *h);

static void *field_base(const gr_handle *h, void *alloc) {
  return alloc ? (char *)alloc + (size_t)h->P.xoff * elem_size(h->P.dtype) : nullptr;
}
// base of logical field l (0 = U1, 1 = U2)
static void *ubase(const gr_handle *h, int l) { return field_base(h, h->fbuf[h->lu[l]]); }
static void spare_ids(const gr_handle *h, int out[2]) {
  int n = 0;
  for (int i = 0; i < 4 && n < 2; ++i)
    if (i != h->lu[0] && i != h->lu[1]) out[n++] = i;
}
// the fields were (re)written from outside: parity restarts, spares and halo facts are stale
static void state_reset(gr_handle *h) {
  h->parity = 0;
  h->napplied = 0;
  h->spares_synced = false;
  h->no_spare = false;
  h->halo_equal = -1;
}

extern "C" const char *gr_last_error(void) { return g_err; }

extern "C" int gr_mwd_round_nt(int nt, int t_dim) {
  const int w = (t_dim + 1) * 2;
  const int rem = (nt - 2) % w;
  return rem != 0 ? nt + w - rem : nt;
}

extern "C" int gr_create(const gr_desc *d, gr_handle **out) {
  if (!d || !out) return fail(GR_EINVAL, "gr_create: null argument");
  *out = nullptr;
  if (d->kernel < 0 || d->kernel > 5)
    return fail(GR_EINVAL, "gr_create: kernel %d not supported (regular star kernels 0-5)", d->kernel);
  if (d->dtype != GR_F64 && d->dtype != GR_F32) return fail(GR_EINVAL, "gr_create: bad dtype %d", d->dtype);
  if (d->nx < 1 || d->ny < 1 || d->nz < 1) return fail(GR_EINVAL, "gr_create: empty grid");
  if ((d->flags & GR_FAST) && d->dtype != GR_F32)
    return fail(GR_EINVAL, "gr_create: GR_FAST applies to GR_F32 only");
  if ((d->flags & GR_FAST) && d->kernel != 0)
    return fail(GR_EUNSUPPORTED, "gr_create: GR_FAST is implemented for kernel 0");
  if ((d->flags & GR_COEF_BF16) && d->dtype != GR_F32)
    return fail(GR_EINVAL, "gr_create: GR_COEF_BF16 applies to GR_F32 fields");
  if ((d->flags & GR_ROC2_SCALAR) && d->kernel != 0)
    return fail(GR_EINVAL, "gr_create: GR_ROC2_SCALAR applies to kernel 0");
  gr_handle *h = new gr_handle();
  Problem &P = h->P;
  P.kernel = d->kernel;
  P.dtype = d->dtype;
  P.flags = d->flags;
  P.nx = d->nx;
  P.ny = d->ny;
  P.nz = d->nz;
  P.R = kradius(d->kernel);
  P.ncoef = kncoef(d->kernel);
  for (int r = 0; r < 5; ++r) P.c[r] = d->coef[r];
  P.roc2s = d->roc2;
  const int es = (int)elem_size(P.dtype);
  const int line = 128 / es;                      // elements per 128-byte line
  P.xoff = (line - P.R % line) % line;            // (xoff + R) % line == 0
  // bf16 roc2 / coefficient storage: rows of a whole number of 128-byte lines (pitch a
  // multiple of 64 elements) and its own x offset, so that its first interior cell
  // (i = R) starts a line too; its element index equals the fields'
  const bool bf16_store = (P.flags & GR_COEF_BF16) != 0;
  const int pline = bf16_store ? 64 : line;
  P.pitch = ((P.xoff + P.nx + 2 * P.R + pline - 1) / pline) * pline;
  P.cxoff = bf16_store ? (64 - P.R % 64) % 64 : P.xoff;
  P.rows = P.ny + 2 * P.R;
  P.planes = P.nz + 2 * P.R;
  P.field_elems = (long long)P.pitch * P.rows * P.planes;
  h->lc.zchunk = 0;
  h->lc.auto_variant = h->lc.auto_zchunk = true;
  {  // GIRIH_XCD_ORDER=0, 1 or 2 starts from that workgroup order (the autotuner tries all three)
    const char *e = getenv("GIRIH_XCD_ORDER");
    h->lc.auto_order = !(e && e[0] >= '0' && e[0] <= '2');
    h->lc.xcd_order = h->lc.auto_order ? 0 : e[0] - '0';
  }
  h->lc.t_block = d->t_block <= 0 ? 1 : d->t_block;  // 0: single sweeps until gr_autotune picks a depth
  if (h->lc.t_block > 1) {
    int depths[8];
    const int nd = tb_depths(P.kernel, P.dtype, depths, 8);
    bool have = false;
    for (int i = 0; i < nd; ++i) have |= depths[i] == h->lc.t_block;
    if (!have) {
      delete h;
      return fail(GR_EUNSUPPORTED, "gr_create: fused depth %d not available for kernel %d", d->t_block, d->kernel);
    }
  }
  const size_t fbytes = (size_t)P.field_elems * es;
  hipError_t e;
  int rc = GR_OK;
  if ((e = hipGetDevice(&h->device)) != hipSuccess ||
      (e = hipDeviceGetAttribute(&h->ncu, hipDeviceAttributeMultiprocessorCount, h->device)) != hipSuccess)
    rc = fail(GR_EHIP, "hipGetDevice: %s", hipGetErrorString(e));
  // Zero fills go on the handle's own (non-blocking) stream, which does not order with
  // the null stream: a null-stream hipMemset could still be running when the first
  // kernel on the handle's stream writes the same memory.
  if (rc == GR_OK && (e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking)) != hipSuccess)
    rc = fail(GR_EHIP, "hipStreamCreate: %s", hipGetErrorString(e));
  if (rc == GR_OK && ((e = hipEventCreate(&h->ev0)) != hipSuccess || (e = hipEventCreate(&h->ev1)) != hipSuccess))
    rc = fail(GR_EHIP, "hipEventCreate: %s", hipGetErrorString(e));
  auto alloc = [&](void **p, size_t n) {
    if (rc != GR_OK) return;
    if ((e = hipMalloc(p, n)) != hipSuccess) {
      rc = fail(GR_ENOMEM, "hipMalloc(%zu) failed: %s", n, hipGetErrorString(e));
      return;
    }
    if ((e = hipMemsetAsync(*p, 0, n, h->stream)) != hipSuccess)
      rc = fail(GR_EHIP, "hipMemsetAsync: %s", hipGetErrorString(e));
  };
  alloc(&h->fbuf[0], fbytes);
  alloc(&h->fbuf[1], fbytes);
  // bf16 storage: 64 elements of slack for its x offset (up to 63 past the fields')
  const size_t cbytes = bf16_store ? (size_t)P.field_elems * 2 : fbytes;
  const size_t cslack = bf16_store ? 128 : 0;
  if (P.kernel == 0 && !(P.flags & GR_ROC2_SCALAR)) alloc(&h->alloc_roc2, cbytes + cslack);
  if (P.ncoef > 0) alloc(&h->alloc_coef, cbytes * P.ncoef + cslack);
  // the fields are zero before any other stream (a batch, torch) can touch them
  if (rc == GR_OK && (e = hipStreamSynchronize(h->stream)) != hipSuccess)
    rc = fail(GR_EHIP, "hipStreamSynchronize: %s", hipGetErrorString(e));
  if (rc != GR_OK) {
    gr_destroy(h);
    return rc;
  }
  const size_t ces = (P.flags & GR_COEF_BF16) ? 2 : es;
  P.roc2 = h->alloc_roc2 ? (char *)h->alloc_roc2 + (size_t)P.cxoff * ces : nullptr;
  P.coef = h->alloc_coef ? (char *)h->alloc_coef + (size_t)P.cxoff * ces : nullptr;
  h->stats.device_bytes = (int64_t)(2 * fbytes + (h->alloc_roc2 ? cbytes + cslack : 0) +
                                    (h->alloc_coef ? (size_t)P.ncoef * cbytes + cslack : 0));
  *out = h;
  return GR_OK;
}

extern "C" int gr_destroy(gr_handle *h) {
  if (!h) return GR_OK;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  if (h->gexec) (void)hipGraphExecDestroy(h->gexec);
  for (void *p : {h->fbuf[0], h->fbuf[1], h->fbuf[2], h->fbuf[3], h->alloc_roc2, h->alloc_coef, h->src, h->flag})
    if (p) (void)hipFree(p);
  free_stage(h);
  if (h->ev0) (void)hipEventDestroy(h->ev0);
  if (h->ev1) (void)hipEventDestroy(h->ev1);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return GR_OK;
}

__global__ void to_bf16_kernel(const float *src, __hip_bfloat16 *dst, long long n) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) dst[t] = __float2bfloat16(src[t]);  // round to nearest even
}

// ------------------------------------------------------------------ host fields
// host girih layout <-> device layout: both store rows (k*nny + j) at a constant pitch.
// hipMemcpy2DAsync moves pageable pitched rows one by one (256 x 256 x 128 FP32, two
// fields down: 495 ms, 0.15 GB/s).  Here a few host threads each take chunks of rows
// through a pinned slot of their own: a kernel packs the rows into the slot (or unpacks
// them from it) over the bus while the other threads copy theirs between slot and
// array, which also spreads the page faults of fresh arrays.
constexpr int kStageThreads = 8;                  // host threads and slots
constexpr size_t kStageBytes = (size_t)2 << 20;   // one slot (a copy that is smaller takes what it needs)

// rows of `width` words at `pitch` <-> rows at `width` (one wavefront per row)
template <typename W, bool PACK>
__global__ __launch_bounds__(256) void stage_rows_kernel(W *pitched, long long pitch, W *packed, int width, int nrows) {
  const int row = blockIdx.x * 4 + threadIdx.x / 64;
  if (row >= nrows) return;
  W *a = pitched + row * pitch, *b = packed + (long long)row * width;
  for (int i = threadIdx.x % 64; i < width; i += 64)
    if (PACK)
      b[i] = a[i];
    else
      a[i] = b[i];
}

template <typename W>
static hipError_t stage_rows(bool pack, void *dev, long long pitch, void *slot, int width, int nrows, hipStream_t st) {
  const dim3 grid((nrows + 3) / 4);
  if (pack)
    hipLaunchKernelGGL((stage_rows_kernel<W, true>), grid, dim3(256), 0, st, (W *)dev, pitch, (W *)slot, width, nrows);
  else
    hipLaunchKernelGGL((stage_rows_kernel<W, false>), grid, dim3(256), 0, st, (W *)dev, pitch, (W *)slot, width, nrows);
  return hipGetLastError();
}

static void free_stage(gr_handle *h) {
  for (hipEvent_t &e : h->stage_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (h->stage) (void)hipHostFree(h->stage);
  h->stage = nullptr;
  h->stage_bytes = 0;
}

// At least `bytes` of pinned slots, kept until the handle is destroyed or a copy needs more
// (false: not available).  A handle holds what its largest copy uses, at most 16 MB: one of 30^3
// 128 KB.
static bool ensure_stage(gr_handle *h, size_t bytes) {
  if (h->stage_bytes >= bytes) return true;
  free_stage(h);
  bool ok = hipHostMalloc(&h->stage, bytes, hipHostMallocDefault) == hipSuccess;
  if (!ok) h->stage = nullptr;
  for (int i = 0; i < kStageThreads && ok; ++i)
    ok = hipEventCreateWithFlags(&h->stage_ev[i], hipEventDisableTiming) == hipSuccess;
  if (ok) {
    h->stage_bytes = bytes;
  } else {
    (void)hipGetLastError();
    free_stage(h);
  }
  return ok;
}

// Makes a device current for a scope; the caller's own is current again after it.
class CurrentDevice {
 public:
  explicit CurrentDevice(int device) {
    int now = 0;
    status = hipGetDevice(&now);
    if (status == hipSuccess && now != device && (status = hipSetDevice(device)) == hipSuccess) back_ = now;
  }
  ~CurrentDevice() {
    if (back_ >= 0) (void)hipSetDevice(back_);
  }
  CurrentDevice(const CurrentDevice &) = delete;
  CurrentDevice &operator=(const CurrentDevice &) = delete;
  hipError_t status;

 private:
  int back_ = -1;
};

// Host threads this process may use.
static int host_threads() {
  cpu_set_t set;
  CPU_ZERO(&set);
  return sched_getaffinity(0, sizeof(set), &set) == 0 ? std::max(1, CPU_COUNT(&set)) : 1;
}

// Copies nrows rows through the slots; *done false where there is no memory for them.
static int copy_rows(gr_handle *h, char *dev, size_t dev_pitch, char *host, size_t host_pitch, size_t width, int nrows,
                     size_t es, bool to_dev, bool *done) {
  const int per = (int)std::max<size_t>(1, std::min<size_t>(nrows, kStageBytes / width));  // rows per chunk
  const int nchunk = (nrows + per - 1) / per;
  const int nt = std::min({kStageThreads, nchunk, host_threads()});
  const size_t slot_bytes = (per * width + 63) / 64 * 64;
  *done = ensure_stage(h, nt * slot_bytes);
  if (!*done) return GR_OK;
  std::atomic<int> next{0}, err{(int)hipSuccess};
  auto work = [&](int t) {
    char *slot = (char *)h->stage + (size_t)t * slot_bytes;
    hipError_t e = t > 0 ? hipSetDevice(h->device) : hipSuccess;  // current on the caller's thread already
    bool busy = false;  // the slot is still being read by the unpacking kernel
    for (int c; e == hipSuccess && err.load() == (int)hipSuccess && (c = next.fetch_add(1)) < nchunk;) {
      const int r0 = c * per, n = std::min(per, nrows - r0);
      char *d = dev + (size_t)r0 * dev_pitch, *u = host + (size_t)r0 * host_pitch;
      if (busy) e = hipEventSynchronize(h->stage_ev[t]);
      busy = false;
      if (to_dev)
        for (int r = 0; r < n; ++r) memcpy(slot + r * width, u + r * host_pitch, width);
      if (e == hipSuccess)
        e = es == 8 ? stage_rows<double>(!to_dev, d, (long long)(dev_pitch / 8), slot, (int)(width / 8), n, h->stream)
                    : stage_rows<float>(!to_dev, d, (long long)(dev_pitch / 4), slot, (int)(width / 4), n, h->stream);
      if (e == hipSuccess) e = hipEventRecord(h->stage_ev[t], h->stream);
      if (e != hipSuccess) break;
      busy = to_dev;
      if (!to_dev && (e = hipEventSynchronize(h->stage_ev[t])) == hipSuccess)
        for (int r = 0; r < n; ++r) memcpy(u + r * host_pitch, slot + r * width, width);
    }
    if (busy) (void)hipEventSynchronize(h->stage_ev[t]);
    if (e != hipSuccess) err.store((int)e);
  };
  std::vector<std::thread> pool;
  try {
    for (int t = 1; t < nt; ++t) pool.emplace_back(work, t);
  } catch (const std::exception &) {
    // no more threads: those that run, and this one, take all chunks
  }
  work(0);
  for (std::thread &t : pool) t.join();
  const hipError_t e = (hipError_t)err.load();
  return e == hipSuccess ? GR_OK : fail(GR_EHIP, "field copy: %s", hipGetErrorString(e));
}

static int copy_field(gr_handle *h, const int ld[3], void *dev_base, size_t dev_es, const void *host,
                      size_t host_es, bool to_dev) {
  const Problem &P = h->P;
  const size_t width = (size_t)(P.nx + 2 * P.R) * host_es;
  const size_t dpitch = (size_t)P.pitch * dev_es, hpitch = (size_t)ld[0] * host_es;
  const size_t nrows = (size_t)P.rows * P.planes;
  if (dev_es != host_es) return fail(GR_EINVAL, "copy_field: element size mismatch");
  // slots, events and kernels belong to the handle's GPU, whichever is current
  const CurrentDevice current(h->device);
  if (current.status != hipSuccess) return fail(GR_EHIP, "copy_field: %s", hipGetErrorString(current.status));
  // memory that host threads cannot touch (a device pointer), pinned arrays, which the runtime
  // moves at the bus's rate (two 256 x 256 x 128 FP32 fields up 1.3 ms, through the slots 2.0),
  // and rows longer than a slot go to the runtime's copy
  hipPointerAttribute_t at{};
  const bool direct = hipPointerGetAttributes(&at, host) == hipSuccess &&
                      (at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeHost);
  (void)hipGetLastError();
  if (!direct && width <= kStageBytes && nrows <= (size_t)INT_MAX) {
    bool done = false;
    const int rc = copy_rows(h, (char *)dev_base, dpitch, (char *)const_cast<void *>(host), hpitch, width, (int)nrows,
                             dev_es, to_dev, &done);
    if (done) return rc;
  }
  if (to_dev)
    HIP_TRY(hipMemcpy2DAsync(dev_base, dpitch, host, hpitch, width, nrows, hipMemcpyHostToDevice, h->stream));
  else
    HIP_TRY(hipMemcpy2DAsync((void *)host, hpitch, dev_base, dpitch, width, nrows, hipMemcpyDeviceToHost, h->stream));
  return GR_OK;
}

static int check_ld(const gr_handle *h, const int ld[3]) {
  const Problem &P = h->P;
  if (!ld) return fail(GR_EINVAL, "ldomain_shape is NULL");
  if (ld[0] < P.nx + 2 * P.R || ld[1] != P.ny + 2 * P.R || ld[2] != P.nz + 2 * P.R)
    return fail(GR_EINVAL, "ldomain_shape {%d,%d,%d} does not fit grid %dx%dx%d with radius %d", ld[0], ld[1],
                ld[2], P.nx, P.ny, P.nz, P.R);
  return GR_OK;
}

extern "C" int gr_upload(gr_handle *h, const int ld[3], const void *U1, const void *U2, const void *U3,
                         const void *coef) {
  if (!h) return fail(GR_EINVAL, "gr_upload: null handle");
  int rc = check_ld(h, ld);
  if (rc) return rc;
  const Problem &P = h->P;
  const size_t es = elem_size(P.dtype);
  if (U1 && U2) {  // both fields are overwritten: back to the first buffer pair
    drop_graph(h);
    h->lu[0] = 0;
    h->lu[1] = 1;
  }
  if (U1 && (rc = copy_field(h, ld, ubase(h, 0), es, U1, es, true))) return rc;
  if (U2 && (rc = copy_field(h, ld, ubase(h, 1), es, U2, es, true))) return rc;
  const size_t hstride = (size_t)ld[0] * ld[1] * ld[2] * es;
  if (P.flags & GR_COEF_BF16) {
    // bf16 roc2 / coefficient fields: FP32 host arrays staged through one FP32
    // field on the device and rounded to nearest even
    const bool want_r = U3 && P.roc2, want_c = coef && P.coef;
    if (want_r || want_c) {
      void *tmp = nullptr;
      HIP_TRY(hipMalloc(&tmp, (size_t)P.field_elems * sizeof(float)));
      float *tbase = (float *)tmp + P.xoff;
      auto one = [&](const void *host, __hip_bfloat16 *dst) -> int {
        int r = copy_field(h, ld, tbase, sizeof(float), host, es, true);
        if (r) return r;
        const unsigned nb = (unsigned)((P.field_elems + 255) / 256);
        hipLaunchKernelGGL(to_bf16_kernel, dim3(nb), dim3(256), 0, h->stream, (const float *)tmp,
                           dst - P.xoff, P.field_elems);
        const hipError_t e = hipGetLastError();
        return e == hipSuccess ? GR_OK : fail(GR_EHIP, "bf16 conversion: %s", hipGetErrorString(e));
      };
      if (want_r) rc = one(U3, (__hip_bfloat16 *)P.roc2);
      for (int m = 0; rc == GR_OK && want_c && m < P.ncoef; ++m)
        rc = one((const char *)coef + m * hstride, (__hip_bfloat16 *)P.coef + (size_t)m * P.field_elems);
      const hipError_t e = hipStreamSynchronize(h->stream);
      (void)hipFree(tmp);
      if (rc) return rc;
      if (e != hipSuccess) return fail(GR_EHIP, "gr_upload: %s", hipGetErrorString(e));
    }
  } else {
    if (U3 && P.roc2 && (rc = copy_field(h, ld, P.roc2, es, U3, es, true))) return rc;
    if (coef && P.coef) {
      const size_t dstride = (size_t)P.field_elems * es;
      for (int m = 0; m < P.ncoef; ++m)
        if ((rc = copy_field(h, ld, (char *)P.coef + m * dstride, es, (const char *)coef + m * hstride, es, true)))
          return rc;
    }
  }
  HIP_TRY(hipStreamSynchronize(h->stream));
  state_reset(h);
  return GR_OK;
}

extern "C" int gr_download(gr_handle *h, const int ld[3], void *U1, void *U2) {
  if (!h) return fail(GR_EINVAL, "gr_download: null handle");
  int rc = check_ld(h, ld);
  if (rc) return rc;
  const size_t es = elem_size(h->P.dtype);
  if (U1 && (rc = copy_field(h, ld, ubase(h, 0), es, U1, es, false))) return rc;
  if (U2 && (rc = copy_field(h, ld, ubase(h, 1), es, U2, es, false))) return rc;
  HIP_TRY(hipStreamSynchronize(h->stream));
  return GR_OK;
}

extern "C" int gr_set_source(gr_handle *h, int i, int j, int k, const double *values, int n) {
  if (!h) return fail(GR_EINVAL, "gr_set_source: null handle");
  const Problem &P = h->P;
  drop_graph(h);  // a captured step sequence holds the old source pointers
  if (h->src) {
    HIP_TRY(hipFree(h->src));
    h->src = nullptr;
  }
  h->nsrc = 0;
  h->src_idx = -1;
  if (n <= 0) return GR_OK;
  if (!values) return fail(GR_EINVAL, "gr_set_source: values is NULL");
  if (i < P.R || i >= P.nx + P.R || j < P.R || j >= P.ny + P.R || k < P.R || k >= P.nz + P.R)
    return fail(GR_EINVAL, "gr_set_source: point (%d,%d,%d) is not an interior cell", i, j, k);
  const size_t es = elem_size(P.dtype);
  std::vector<char> buf((size_t)(n + kSrcPad) * es, 0);  // zeros past n: fused passes read ahead
  for (int s = 0; s < n; ++s) {
    if (P.dtype == GR_F64)
      ((double *)buf.data())[s] = values[s];
    else
      ((float *)buf.data())[s] = (float)values[s];
  }
  HIP_TRY(hipMalloc(&h->src, buf.size()));
  HIP_TRY(hipMemcpy(h->src, buf.data(), buf.size(), hipMemcpyHostToDevice));
  h->nsrc = n;
  h->src_idx = ((long long)k * P.rows + j) * P.pitch + i;
  return GR_OK;
}

static int check_halo_equal(gr_handle *h);
static int ensure_spares(gr_handle *h, int n = 2);
static int sync_spares(gr_handle *h);
static int enqueue_apps(gr_handle *h, int napply, bool fuse, int *nlaunch);
static int finish_step(gr_handle *h, int napply, int launches);
static bool trades_buffers(const gr_handle *h, int napply);
static int rest_depth(const gr_handle *h, int rest);
static void drop_graph(gr_handle *h) {
  if (h->gexec) {
    (void)hipStreamSynchronize(h->stream);  // a replay may still be running
    (void)hipGraphExecDestroy(h->gexec);
  }
  h->gexec = nullptr;
}

// One application U(w) <- f(U(r)) with the handle's sweep configuration.
static hipError_t single_app(gr_handle *h, long long app) {
  const size_t es = elem_size(h->P.dtype);
  const bool has_src = h->src && app < h->nsrc;
  const void *srcp = has_src ? (const char *)h->src + (size_t)app * es : nullptr;
  const long long sidx = has_src ? h->src_idx : -1;
  const int w = h->parity, r = 1 - w;
  LaunchCfg lc = h->lc;
  lc.down = w == 1;
  hipError_t e = sweep_fields(h->P, ubase(h, w), ubase(h, r), srcp, sidx, lc, h->stream);
  h->parity ^= 1;
  return e;
}

// Whether fused passes of depth tl may run for this handle.
static int fused_depth_ok(gr_handle *h, int tl, bool *ok) {
  *ok = false;
  if (tl < 2) return GR_OK;
  int depths[8];
  const int nd = tb_depths(h->P.kernel, h->P.dtype, depths, 8);
  bool have = false;
  for (int i = 0; i < nd; ++i) have |= depths[i] == tl;
  if (!have) return GR_OK;
  // bf16-stored fields fuse for kernel 5 (coefficient arrays) and kernel 0 (roc2)
  if ((h->P.flags & GR_COEF_BF16) != 0 && h->P.kernel != 5 && h->P.kernel != 0) return GR_OK;
  int rc = check_halo_equal(h);
  if (rc) return rc;
  *ok = h->halo_equal == 1;
  return GR_OK;
}

extern "C" int gr_step(gr_handle *h, int napply) {
  if (!h) return fail(GR_EINVAL, "gr_step: null handle");
  if (napply < 0) return fail(GR_EINVAL, "gr_step: negative step count");
  const int tl = h->lc.t_block;
  bool fuse = false;
  int rc = fused_depth_ok(h, tl, &fuse);
  if (rc) return rc;
  const bool wave = h->P.kernel == 0;
  if (fuse && wave) {
    if ((rc = ensure_spares(h)) || (rc = sync_spares(h))) return rc;
  } else if (fuse && !h->no_spare) {
    // a third buffer lets the last pass write both levels that a call leaves; without the
    // memory for it a call ends with a single sweep
    if (ensure_spares(h, 1) == GR_OK) {
      const bool in_pass = h->exposed && star7_pass(h->P, rest_depth(h, napply));  // enqueue_first_order
      if (napply > 1 && !in_pass && (rc = sync_spares(h))) return rc;
    } else {
      (void)hipGetLastError();
      h->no_spare = true;
    }
  }
  // graph mode: replay the launch sequence of an identical earlier call
  GraphKey key{napply, h->parity, h->lu[0], h->lu[1], h->lc.variant, h->lc.zchunk, h->lc.t_block, h->lc.xcd_order,
               h->lc.ftile, h->lc.auto_variant + 2 * h->lc.auto_zchunk + 4 * h->lc.auto_order, fuse ? 1 : 0,
               h->exposed ? 1 : 0, -1};
  if (h->src && h->napplied < h->nsrc) key.napplied = h->napplied;  // source pointers are baked in
  if (h->use_graph && napply > 0 && !(fuse && trades_buffers(h, napply))) {
    if (!(h->gexec && h->gkey == key)) {
      drop_graph(h);
      const int parity0 = h->parity, lu0 = h->lu[0], lu1 = h->lu[1];
      hipGraph_t g = nullptr;
      HIP_TRY(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
      int launches = 0;
      const int erc = enqueue_apps(h, napply, fuse, &launches);
      hipError_t e = hipStreamEndCapture(h->stream, &g);
      if (erc == GR_OK && e == hipSuccess) e = hipGraphInstantiate(&h->gexec, g, nullptr, nullptr, 0);
      if (g) (void)hipGraphDestroy(g);
      h->gparity = h->parity;
      h->glu[0] = h->lu[0];
      h->glu[1] = h->lu[1];
      h->glaunches = launches;
      h->parity = parity0;  // the state advances when the graph runs, below
      h->lu[0] = lu0;
      h->lu[1] = lu1;
      if (erc != GR_OK) {
        drop_graph(h);
        return erc;
      }
      if (e != hipSuccess) {
        drop_graph(h);
        return fail(GR_EHIP, "step graph capture: %s", hipGetErrorString(e));
      }
      h->gkey = key;
      ++h->captures;
    }
    HIP_TRY(hipEventRecord(h->ev0, h->stream));
    HIP_TRY(hipGraphLaunch(h->gexec, h->stream));
    h->parity = h->gparity;
    h->lu[0] = h->glu[0];
    h->lu[1] = h->glu[1];
    return finish_step(h, napply, h->glaunches);
  }
  HIP_TRY(hipEventRecord(h->ev0, h->stream));
  int launches = 0;
  if ((rc = enqueue_apps(h, napply, fuse, &launches))) return rc;
  return finish_step(h, napply, launches);
}

// The z chunk with which a pass of depth tl has at most `rounds` workgroups per CU, as
// near to that as whole chunks allow, but no chunk shorter than 2*tl planes: those would
// mostly compute each other's ghost planes (0: the whole z).
static int round_chunk(const gr_handle *h, int tl, const LaunchCfg &lc, int rounds) {
  const Problem &P = h->P;
  int tx = 0, ty = 0;
  if (!fused_tile(P, tl, lc, &tx, &ty)) return 0;
  const int ntile = ((P.nx + tx - 1) / tx) * ((P.ny + ty - 1) / ty);
  const int nzc = rounds * h->ncu / ntile;
  if (nzc < 1) return 0;
  const int zc = std::max(2 * tl, (P.nz + nzc - 1) / nzc);
  return zc < P.nz ? zc : 0;
}

// The z chunk of an untuned pass: one round of the CUs where the tiles leave room for chunks,
// else the number of chunks with the shortest rounds in all, as one that is nearly empty costs
// as much as a full one (FP64 Jacobi, 512 x 512 x 256 at depth 5: 296 tiles, 21 steps on whole z
// 3218 us, on the chunks 2362; before, with another kernel, 2508).  A chunk computes 2*R*tl planes more than it writes.
static int untuned_chunk(const gr_handle *h, int tl, const LaunchCfg &lc) {
  const Problem &P = h->P;
  int tx = 0, ty = 0;
  if (!fused_tile(P, tl, lc, &tx, &ty)) return 0;
  const long long ntile = (long long)((P.nx + tx - 1) / tx) * ((P.ny + ty - 1) / ty);
  if (ntile <= h->ncu) return round_chunk(h, tl, lc, 1);
  const int margin = 2 * P.R * tl;
  int best = 0;
  long long cost = LLONG_MAX;
  for (int nzc = 1; nzc <= 16; ++nzc) {
    const int zc = (P.nz + nzc - 1) / nzc;
    if (nzc > 1 && zc < margin) break;
    const long long c = (ntile * nzc + h->ncu - 1) / h->ncu * (zc + margin);
    if (c < cost) {
      cost = c;
      best = zc;
    }
  }
  return best < P.nz ? best : 0;
}

// h's settings for fused passes of depth tl: chunks for whole rounds of the CUs and, in FP32,
// the XCD bands (512^3 kernel 5 FP32 1163 us a pass against 1261 in plain order, FP64 2457
// against 2178) where the caller has set neither.
static LaunchCfg fused_cfg(const gr_handle *h, int tl) {
  LaunchCfg lc = h->lc;
  if (tl != lc.t_block) lc.ftile = 0;  // a rest shallower than the configured depth
  if (lc.auto_order) lc.xcd_order = h->P.dtype == GR_F32 && h->P.kernel != 0 ? 2 : 0;
  if (lc.auto_zchunk || tl != lc.t_block) lc.zchunk = untuned_chunk(h, tl, lc);
  return lc;
}

// Depth of the next launch of a first-order call with `rest` applications to go (1: a single
// sweep).  tb_kernel's pass (kernel 5, depth 6, without bf16 coefficients) ends no call: the
// two shallower passes in its place take 2.2 ms against 10.0 at 512 x 512 x 256 in FP64 (six
// sweeps 5.0), and 1.2 against 3.3 (2.8) in FP32.
static int rest_depth(const gr_handle *h, int rest) {
  const bool tb6 = h->P.kernel == 5 && !(h->P.flags & GR_COEF_BF16);
  int depths[8], d = 1;
  const int nd = tb_depths(h->P.kernel, h->P.dtype, depths, 8);
  for (int i = 0; i < nd; ++i)
    if (depths[i] <= std::min(rest, h->lc.t_block) && !(tb6 && depths[i] == 6 && rest == 6)) d = std::max(d, depths[i]);
  return d;
}

// Whether a fused first-order call ends on other buffers than it began with
// (enqueue_first_order): one pass, or one pass and an odd step's sweep.  Its one or two
// launches are not captured: the sequence would differ at every call (128^3 FP64, 4 steps at
// depth 4: 48 us, captured anew each time 61).
static bool trades_buffers(const gr_handle *h, int napply) {
  int sp[2];
  spare_ids(h, sp);
  if (h->P.kernel == 0 || napply < 2 || !h->fbuf[sp[0]]) return false;
  const int d = rest_depth(h, napply);
  return d == napply || (d == napply - 1 && (napply & 1));
}

// Launch napply applications of a first-order kernel as fused passes, the last of which
// writes the field's last two levels (the U1/U2 pair a call leaves) into different
// buffers, so that no single sweep is needed to make both exact: at 512^3, 20 kernel-5
// FP64 steps at depth 4 were 4 passes and 4 sweeps, and the sweeps took 40% of the time.
// A rest shorter than the depth runs as one shallower pass, and as a sweep where one
// application is left.  Three buffers take part: U1, U2 and a spare.  A pass may write
// any buffer but the one it reads, so the sequence is led such that the call ends on
// the buffers it began with (a captured graph then stays valid); only a call of one
// pass has to trade the read field for the spare (trades_buffers).
static int enqueue_first_order(gr_handle *h, int napply, int *nlaunch) {
  const Problem &P = h->P;
  const size_t es = elem_size(P.dtype);
  std::vector<int> ops;  // depth of each launch (1: a single sweep)
  for (int rest = napply; rest > 0; rest -= ops.back()) ops.push_back(rest_depth(h, rest));
  int sp[2];
  spare_ids(h, sp);
  const int m = (int)ops.size(), w = h->parity, r = 1 - w;
  const int newest = (napply & 1) ? w : r;            // the logical field that ends newest
  int end[2] = {h->lu[0], h->lu[1]};                   // buffers of U1 and U2 after the call
  const bool both = m > 0 && ops[m - 1] > 1;           // the last launch writes both levels
  int x = h->lu[r];                                    // buffer read next
  if (m == 1 && both) end[r] = sp[0];                  // one pass reads end[r]'s buffer
  if (m == 2 && !both && newest == w) end[r] = sp[0];  // one pass and one sweep: the same
  // the buffer the last launch reads: for a pass the one that stays free, for a sweep the older level's
  const int last_in = both ? (m == 1 ? x : sp[0]) : end[1 - newest];
  long long app = h->napplied;
  for (int i = 0; i < m; ++i) {
    const bool has_src = h->src && app < h->nsrc;
    const void *srcp = has_src ? (const char *)h->src + (size_t)app * es : nullptr;
    const long long sidx = has_src ? h->src_idx : -1;
    LaunchCfg lc = ops[i] > 1 ? fused_cfg(h, ops[i]) : h->lc;
    // the first pass brings the spare the halo, which the caller may have rewritten
    if (i == 0 && h->exposed && star7_pass(P, ops[0])) lc.halo = field_base(h, h->fbuf[sp[0]]);
    lc.down = (i & 1) && P.kernel == 5 && z_turns(P);
    const void *in = field_base(h, h->fbuf[x]);
    hipError_t e;
    if (i == m - 1) {
      void *out = field_base(h, h->fbuf[end[newest]]);
      e = both ? tblock_pass(P, ops[i], nullptr, in, field_base(h, h->fbuf[end[1 - newest]]), out, srcp, sidx, lc,
                             h->stream)
               : sweep_fields(P, out, in, srcp, sidx, lc, h->stream);
    } else {
      // the next buffer: any other one, such that the last launch finds its input in last_in
      int y = last_in;
      if (i < m - 2 || y == x)
        for (int c : {h->lu[w], h->lu[r], sp[0]})
          if (c != x && (i < m - 3 || c != last_in)) {
            y = c;
            break;
          }
      e = tblock_pass(P, ops[i], nullptr, in, nullptr, field_base(h, h->fbuf[y]), srcp, sidx, lc, h->stream);
      x = y;
    }
    if (e != hipSuccess) return fail(GR_EHIP, "fused pass launch failed: %s", hipGetErrorString(e));
    app += ops[i];
  }
  h->parity ^= napply & 1;
  h->lu[0] = end[0];
  h->lu[1] = end[1];
  *nlaunch = m;
  return GR_OK;
}

// Launch napply applications on the handle's stream (fused passes where enabled,
// then single sweeps), advancing the host-side parity and buffer mapping.  Only
// kernel launches: the sequence may be captured into a HIP graph.
static int enqueue_apps(gr_handle *h, int napply, bool fuse, int *nlaunch) {
  const Problem &P = h->P;
  const size_t es = elem_size(P.dtype);
  const int tl = h->lc.t_block;
  const bool wave = P.kernel == 0;
  int s = 0, launches = 0;
  if (fuse && !wave && napply > 1) {
    int sp[2];
    spare_ids(h, sp);
    if (h->fbuf[sp[0]]) return enqueue_first_order(h, napply, nlaunch);
  }
  if (fuse) {
    // kernel 0 keeps (u^(n-1), u^n) exact after every pass; first-order kernels
    // keep the last application as a single sweep so U1 and U2 end exact.
    const int reserve = wave ? 0 : 1;
    const LaunchCfg flc = fused_cfg(h, tl);
    while (napply - reserve - s >= tl) {
      const long long app = h->napplied + s;
      const bool has_src = h->src && app < h->nsrc;
      const void *srcp = has_src ? (const char *)h->src + (size_t)app * es : nullptr;
      const long long sidx = has_src ? h->src_idx : -1;
      const int w = h->parity, r = 1 - w;
      hipError_t e;
      if (wave) {
        int sp[2];
        spare_ids(h, sp);
        e = tblock_pass(P, tl, ubase(h, w), ubase(h, r), field_base(h, h->fbuf[sp[0]]), field_base(h, h->fbuf[sp[1]]),
                        srcp, sidx, flc, h->stream);
        h->parity ^= (tl & 1);
        h->lu[h->parity] = sp[0];      // written next: holds level tl-1
        h->lu[1 - h->parity] = sp[1];  // read next: level tl
      } else {
        const int pw = h->lu[w], pr = h->lu[r];
        e = tblock_pass(P, tl, nullptr, ubase(h, r), nullptr, ubase(h, w), srcp, sidx, flc, h->stream);
        h->parity ^= (tl & 1);
        h->lu[1 - h->parity] = pw;  // newest (level tl) is read next
        h->lu[h->parity] = pr;
      }
      if (e != hipSuccess) return fail(GR_EHIP, "fused pass launch failed: %s", hipGetErrorString(e));
      s += tl;
      ++launches;
    }
  }
  for (; s < napply; ++s, ++launches) {
    hipError_t e = single_app(h, h->napplied + s);
    if (e != hipSuccess) return fail(GR_EHIP, "sweep launch failed: %s", hipGetErrorString(e));
  }
  *nlaunch = launches;
  return GR_OK;
}

static int finish_step(gr_handle *h, int napply, int launches) {
  const Problem &P = h->P;
  HIP_TRY(hipEventRecord(h->ev1, h->stream));
  HIP_TRY(hipEventSynchronize(h->ev1));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, h->ev0, h->ev1));
  h->napplied += napply;
  h->stats.last_ms = ms;
  h->stats.last_updates = (int64_t)napply * P.nx * P.ny * P.nz;
  h->stats.last_launches = launches;
  return GR_OK;
}

extern "C" int gr_set_graph(gr_handle *h, int on) {
  if (!h) return fail(GR_EINVAL, "gr_set_graph: null handle");
  h->use_graph = on != 0;
  if (!h->use_graph) drop_graph(h);
  return GR_OK;
}

extern "C" int gr_run_ts(gr_handle *h, int ts, int nt, int t_dim, int *nt_applied) {
  if (!h) return fail(GR_EINVAL, "gr_run_ts: null handle");
  if (nt < 0) return fail(GR_EINVAL, "gr_run_ts: negative nt");
  const Problem &P = h->P;
  if (ts == 0 || ts == 1) {
    if (nt_applied) *nt_applied = nt;
    return gr_step(h, 2 * ((nt + 1) / 2));
  }
  if (ts != 2) return fail(GR_EINVAL, "gr_run_ts: unknown time stepper %d", ts);
  // validity rules of the diamond stepper (diamond_utils.c:1023-1098), single rank
  if (t_dim < 1) return fail(GR_EINVAL, "Diamond method does not support unrolling in time less than 1");
  if (t_dim % 2 == 0) return fail(GR_EINVAL, "diamond method does not supports even time unrolling");
  const int dw = P.R * (t_dim + 1) * 2;
  if (P.ny < dw || P.ny % dw != 0)
    return fail(GR_EINVAL, "Intra-diamond method requires the sub-domain size to be multiples of the diamond width: %d elements",
                dw);
  if (P.nz < t_dim * 2 * P.R + 1)
    return fail(GR_EINVAL, "The single core wavefront requires a minimum size of %d at the Z direction",
                t_dim * 2 * P.R + 1);
  const int ntr = gr_mwd_round_nt(nt, t_dim);
  if (nt_applied) *nt_applied = ntr;
  return gr_step(h, ntr - 1);
}

// gr_set_config's and gr_stats' tile variant v + kTileBase * (t + 1) is the sweeps' variant v
// with the passes' output tile t; below kTileBase the pass's tile goes by v, where the depth
// has that many.
constexpr int kTileBase = 64;
static int default_ftile(const Problem &P, int depth, int variant) {
  return variant < fused_tiles(P, depth) ? variant : 0;
}

extern "C" int gr_get_stats(gr_handle *h, gr_stats *out) {
  if (!h || !out) return fail(GR_EINVAL, "gr_get_stats: null argument");
  gr_stats s = h->stats;
  s.t_block = h->lc.t_block;
  LaunchCfg lc = sweep_cfg(h->P.kernel, h->P.dtype, h->lc, h->P.nx, h->P.ny, h->P.nz);  // the settings in use
  if (lc.t_block > 1) {
    const LaunchCfg f = fused_cfg(h, lc.t_block);
    lc.zchunk = f.zchunk;
    lc.xcd_order = f.xcd_order;
  }
  // the fused pass's tile when the configuration fuses steps, else the sweep's
  if (lc.t_block < 2 || !fused_tile(h->P, lc.t_block, lc, &s.tile_x, &s.tile_y))
    tile_of_variant(h->P.kernel, h->P.dtype, lc.variant, &s.tile_x, &s.tile_y);
  s.zchunk = lc.zchunk;
  s.parity = h->parity;
  s.pitch_x = h->P.pitch;
  s.rows_y = h->P.rows;
  s.planes_z = h->P.planes;
  s.x_offset = h->P.xoff;
  s.tile_variant = lc.variant;  // one number that gr_set_config reads back to the same tiles
  if (lc.t_block > 1 && lc.ftile != default_ftile(h->P, lc.t_block, lc.variant))
    s.tile_variant += kTileBase * (lc.ftile + 1);
  s.xcd_order = lc.xcd_order;
  *out = s;
  return GR_OK;
}

extern "C" int gr_set_config(gr_handle *h, int variant, int zchunk, int t_block) {
  if (!h) return fail(GR_EINVAL, "gr_set_config: null handle");
  const int depth = t_block >= 1 ? t_block : h->lc.t_block;
  const int ftile = variant / kTileBase - 1;  // the pass's tile; -1: by the sweep's variant
  if (variant >= kTileBase && (depth < 2 || ftile >= fused_tiles(h->P, depth)))
    return fail(GR_EINVAL, "gr_set_config: pass tile %d not available for kernel %d at depth %d", ftile, h->P.kernel,
                depth);
  if (variant >= 0) {
    if (variant % kTileBase >= num_tile_variants(h->P.kernel, h->P.dtype))
      return fail(GR_EINVAL, "gr_set_config: tile variant %d not available for kernel %d", variant % kTileBase,
                  h->P.kernel);
    h->lc.variant = variant % kTileBase;
    h->lc.auto_variant = false;
  }
  if (zchunk >= 0) {
    h->lc.zchunk = zchunk;
    h->lc.auto_zchunk = false;
  }
  const bool new_depth = t_block >= 1 && t_block != h->lc.t_block;
  if (t_block >= 1) {
    if (t_block > 1) {
      int depths[8];
      const int nd = tb_depths(h->P.kernel, h->P.dtype, depths, 8);
      bool have = false;
      for (int i = 0; i < nd; ++i) have |= depths[i] == t_block;
      if (!have) return fail(GR_EUNSUPPORTED, "gr_set_config: fused depth %d not available for kernel %d", t_block,
                             h->P.kernel);
    }
    h->lc.t_block = t_block;
  }
  if (variant >= kTileBase)
    h->lc.ftile = ftile;
  else if (variant >= 0 || new_depth)
    h->lc.ftile = default_ftile(h->P, h->lc.t_block, h->lc.variant);
  return GR_OK;
}

extern "C" int gr_set_streaming(gr_handle *h, int mode) {
  if (!h) return fail(GR_EINVAL, "gr_set_streaming: null handle");
  if (mode < -1 || mode > 1) return fail(GR_EINVAL, "gr_set_streaming: mode must be -1, 0 or 1");
  if (mode != h->P.strm_mode) drop_graph(h);  // a captured sequence holds the other instantiations
  h->P.strm_mode = mode;
  return GR_OK;
}

extern "C" int gr_set_xcd_order(gr_handle *h, int xcd_order) {
  if (!h) return fail(GR_EINVAL, "gr_set_xcd_order: null handle");
  if (xcd_order < 0 || xcd_order > 2) return fail(GR_EINVAL, "gr_set_xcd_order: 0, 1 or 2");
  h->lc.xcd_order = xcd_order;
  h->lc.auto_order = false;
  return GR_OK;
}

// The first n spare buffers.
static int ensure_spares(gr_handle *h, int n) {
  const size_t fbytes = (size_t)h->P.field_elems * elem_size(h->P.dtype);
  for (int i = 2; i < 2 + n; ++i)
    if (!h->fbuf[i]) {
      void *p = nullptr;
      HIP_TRY(hipMalloc(&p, fbytes));
      drop_graph(h);  // a captured sequence runs without it
      h->fbuf[i] = p;
      h->no_spare = false;
      HIP_TRY(hipMemsetAsync(h->fbuf[i], 0, fbytes, h->stream));  // ordered before the spares' first use
      h->spares_synced = false;
      h->stats.device_bytes += (int64_t)fbytes;
    }
  return GR_OK;
}

extern "C" int gr_autotune(gr_handle *h, int steps, gr_stats *best) {
  if (!h) return fail(GR_EINVAL, "gr_autotune: null handle");
  if (steps < 1) steps = 4;
  int rc = ensure_spares(h);
  if (rc) return rc;
  const Problem &P = h->P;
  const size_t fbytes = (size_t)P.field_elems * elem_size(P.dtype);
  int sp[2];
  spare_ids(h, sp);
  HIP_TRY(hipMemcpyAsync(h->fbuf[sp[0]], h->fbuf[h->lu[0]], fbytes, hipMemcpyDeviceToDevice, h->stream));
  HIP_TRY(hipMemcpyAsync(h->fbuf[sp[1]], h->fbuf[h->lu[1]], fbytes, hipMemcpyDeviceToDevice, h->stream));
  h->spares_synced = true;  // copies of the fields: same halo
  void *a = field_base(h, h->fbuf[sp[0]]), *b = field_base(h, h->fbuf[sp[1]]);
  const int nz = P.nz;
  std::vector<int> zchunks = {0};
  for (int zc : {512, 256, 128, 64, 32})
    if (zc < nz) zchunks.push_back(zc);
  if (nz <= 256)  // small grids need short chunks to fill 256 CUs
    for (int zc : {16, 8})
      if (zc < nz) zchunks.push_back(zc);
  LaunchCfg best_lc = h->lc;
  best_lc.auto_variant = best_lc.auto_zchunk = best_lc.auto_order = false;
  const LaunchCfg lc0 = best_lc;
  float best_ms = 1e30f;
  std::vector<std::pair<float, LaunchCfg>> tried;  // sweep trials: time of `steps` sweeps
  // one untimed sweep, then n timed sweeps
  auto time_sweeps = [&](LaunchCfg lc, int n, float *ms) -> int {
    hipError_t e = sweep_fields(P, a, b, nullptr, -1, lc, h->stream);
    if (e != hipSuccess) return fail(GR_EHIP, "autotune launch: %s", hipGetErrorString(e));
    HIP_TRY(hipEventRecord(h->ev0, h->stream));
    for (int s = 0; s < n; ++s) {
      lc.down = !(s & 1);  // as steps do
      e = (s & 1) ? sweep_fields(P, a, b, nullptr, -1, lc, h->stream) : sweep_fields(P, b, a, nullptr, -1, lc, h->stream);
      if (e != hipSuccess) return fail(GR_EHIP, "autotune launch: %s", hipGetErrorString(e));
    }
    HIP_TRY(hipEventRecord(h->ev1, h->stream));
    HIP_TRY(hipEventSynchronize(h->ev1));
    HIP_TRY(hipEventElapsedTime(ms, h->ev0, h->ev1));
    return GR_OK;
  };
  auto trial = [&](const LaunchCfg &lc) -> int {
    float ms = 0.f;
    if (int r = time_sweeps(lc, steps, &ms)) return r;
    tried.emplace_back(ms, lc);
    if (ms < best_ms) {
      best_ms = ms;
      best_lc = lc;
    }
    return GR_OK;
  };
  // stage 1: tile variant x workgroup order at each z-chunk size of a coarse set;
  // stage 2: all z-chunk sizes and orders for the best variant
  // (a variant whose plain order is far from the best so far skips the other orders)
  for (int var = 0; var < num_tile_variants(P.kernel, P.dtype); ++var) {
    float var_ms = 1e30f;
    for (int order = 0; order < 3 && !(order > 0 && var_ms > 1.4f * best_ms); ++order)
      for (int zc : {0, std::min(128, nz)}) {
        LaunchCfg lc = lc0;
        lc.variant = var;
        lc.xcd_order = order;
        lc.zchunk = zc;
        lc.t_block = 1;
        if ((rc = trial(lc))) return rc;
        var_ms = std::min(var_ms, tried.back().first);
      }
  }
  {
    const LaunchCfg base = best_lc;
    for (int order = 0; order < 3; ++order)
      for (int zc : zchunks) {
        LaunchCfg lc = base;
        lc.xcd_order = order;
        lc.zchunk = zc;
        if ((rc = trial(lc))) return rc;
      }
  }
  // stage 2b: the four fastest distinct sweep configurations again, 4x as many steps,
  // twice each in alternation; short trials alone do not separate candidates a few
  // percent apart
  {
    std::stable_sort(tried.begin(), tried.end(),
                     [](const std::pair<float, LaunchCfg> &x, const std::pair<float, LaunchCfg> &y) {
                       return x.first < y.first;
                     });
    std::vector<LaunchCfg> top;
    for (const auto &t : tried) {
      bool seen = false;
      for (const LaunchCfg &c : top)
        seen = seen || (c.variant == t.second.variant && c.zchunk == t.second.zchunk &&
                        c.xcd_order == t.second.xcd_order);
      if (!seen) top.push_back(t.second);
      if (top.size() == 4) break;
    }
    std::vector<float> tmin(top.size(), 1e30f);
    for (int round = 0; round < 2; ++round)
      for (size_t i = 0; i < top.size(); ++i) {
        float ms = 0.f;
        if ((rc = time_sweeps(top[i], 4 * steps, &ms))) return rc;
        tmin[i] = std::min(tmin[i], ms / 4);
      }
    for (size_t i = 0; i < top.size(); ++i)
      if (i == 0 || tmin[i] < best_ms) {
        best_ms = tmin[i];
        best_lc = top[i];
      }
  }
  const float sweep_ms = best_ms;
  // stage 3: fused passes (time per application) on the scratch copies; kernel 0
  // reads the fields themselves (never written here) and writes the scratch pair
  {
    int depths[8];
    const int nd = tb_depths(P.kernel, P.dtype, depths, 8);
    std::vector<std::pair<float, LaunchCfg>> fused;
    // one untimed pass, then npass timed passes: ms per `steps` applications, comparable with the sweep trials
    auto time_passes = [&](LaunchCfg lc, int npass, float *per_step) -> int {
      const int tl = lc.t_block;
      auto pass = [&](int q) {
        lc.down = (q & 1) && P.kernel == 5 && z_turns(P);
        if (P.kernel == 0) return tblock_pass(P, tl, ubase(h, 0), ubase(h, 1), a, b, nullptr, -1, lc, h->stream);
        return tblock_pass(P, tl, nullptr, q & 1 ? b : a, nullptr, q & 1 ? a : b, nullptr, -1, lc, h->stream);
      };
      hipError_t e = pass(0);
      if (e != hipSuccess) return fail(GR_EHIP, "autotune fused launch: %s", hipGetErrorString(e));
      HIP_TRY(hipEventRecord(h->ev0, h->stream));
      for (int q = 1; q <= npass; ++q)
        if ((e = pass(q)) != hipSuccess) return fail(GR_EHIP, "autotune fused launch: %s", hipGetErrorString(e));
      HIP_TRY(hipEventRecord(h->ev1, h->stream));
      HIP_TRY(hipEventSynchronize(h->ev1));
      float ms = 0.f;
      HIP_TRY(hipEventElapsedTime(&ms, h->ev0, h->ev1));
      *per_step = ms * steps / (float)(npass * tl);
      return GR_OK;
    };
    for (int i = 0; i < nd; ++i) {
      bool ok = false;
      if ((rc = fused_depth_ok(h, depths[i], &ok))) return rc;
      if (!ok) continue;
      const int tl = depths[i];
      const int npass = (steps + tl - 1) / tl;
      for (int ft = 0; ft < fused_tiles(P, tl); ++ft) {
        LaunchCfg lc = best_lc;
        lc.t_block = tl;
        lc.ftile = ft;
        // chunk lengths: first those that make the workgroups one to four full rounds of
        // the GPU's CUs (at 512^3 they are up to 15% faster than the powers of two)
        std::vector<int> zcs;
        auto add = [&](int zc) {
          if (std::find(zcs.begin(), zcs.end(), zc) == zcs.end()) zcs.push_back(zc);
        };
        for (int r = 1; r <= 4; ++r) {
          const int zc = round_chunk(h, tl, lc, r);
          if (zc > 0) add(zc);
        }
        for (int zc : zchunks) add(zc);
        // two lengths in every order (XCD-contiguous orders keep the margins' re-reads in
        // one L2), then the others in the tile's best order, unless the tile is far from
        // the best configuration so far
        float tile_ms = 1e30f;
        int tile_order = 0;
        for (size_t iz = 0; iz < zcs.size() && !(iz >= 2 && tile_ms > 1.4f * best_ms); ++iz)
          for (int order = 0; order < 3; ++order) {
            if (iz >= 2 && order != tile_order) continue;
            lc.zchunk = zcs[iz];
            lc.xcd_order = order;
            float ms = 0.f;
            if ((rc = time_passes(lc, npass, &ms))) return rc;
            fused.emplace_back(ms, lc);
            if (ms < tile_ms) {
              tile_ms = ms;
              tile_order = order;
            }
            best_ms = std::min(best_ms, ms);
          }
      }
    }
    // the four fastest again, over four times as many applications, as in stage 2b
    std::stable_sort(fused.begin(), fused.end(),
                     [](const std::pair<float, LaunchCfg> &x, const std::pair<float, LaunchCfg> &y) {
                       return x.first < y.first;
                     });
    const size_t ntop = std::min<size_t>(4, fused.size());
    float tmin[4] = {1e30f, 1e30f, 1e30f, 1e30f};
    for (int round = 0; round < 2; ++round)
      for (size_t i = 0; i < ntop; ++i) {
        if (fused[i].first > 1.1f * best_ms) continue;
        float ms = 0.f;
        if ((rc = time_passes(fused[i].second, std::max(3, 4 * steps / fused[i].second.t_block), &ms))) return rc;
        tmin[i] = std::min(tmin[i], ms);
      }
    best_ms = sweep_ms;
    for (size_t i = 0; i < ntop; ++i)
      if (tmin[i] < best_ms) {
        best_ms = tmin[i];
        best_lc = fused[i].second;
      }
  }
  h->spares_synced = true;  // the scratch pair holds tuning garbage in the interior; halos still match
  h->lc = best_lc;
  if (best) {
    rc = gr_get_stats(h, best);
    if (rc) return rc;
    best->last_ms = best_ms / steps;
  }
  return GR_OK;
}

static size_t coef_elem_size(const Problem &P) { return (P.flags & GR_COEF_BF16) ? 2 : elem_size(P.dtype); }

extern "C" int gr_field_ptr(gr_handle *h, int which, void **p) {
  if (!h || !p) return fail(GR_EINVAL, "gr_field_ptr: null argument");
  if (which != 2 && which != 3) h->exposed = true;
  switch (which) {
    case 0: *p = h->fbuf[h->lu[0]]; break;
    case 1: *p = h->fbuf[h->lu[1]]; break;
    // roc2 / coefficients: the pointer for which base + x_offset + index holds element index
    // (bf16 storage sits at its own offset inside its allocation)
    case 2: *p = h->P.roc2 ? (char *)h->P.roc2 - (size_t)h->P.xoff * coef_elem_size(h->P) : nullptr; break;
    case 3: *p = h->P.coef ? (char *)h->P.coef - (size_t)h->P.xoff * coef_elem_size(h->P) : nullptr; break;
    case 4:
    case 5: {
      int sp[2];
      spare_ids(h, sp);
      *p = h->fbuf[sp[which - 4]];
      break;
    }
    default: return fail(GR_EINVAL, "gr_field_ptr: bad field %d", which);
  }
  return GR_OK;
}

extern "C" int gr_sweep_dev(int kernel, int dtype, const int shape[3], int xb, int yb, int zb, int xe, int ye,
                            int ze, const void *coef, void *u, const void *v, const void *roc2) {
  if (kernel < 0 || kernel > 5) return fail(GR_EINVAL, "gr_sweep_dev: bad kernel %d", kernel);
  if (dtype != GR_F64 && dtype != GR_F32) return fail(GR_EINVAL, "gr_sweep_dev: bad dtype");
  if (!shape || !u || !v || !coef) return fail(GR_EINVAL, "gr_sweep_dev: null argument");
  const int R = kradius(kernel);
  if (xb < R || yb < R || zb < R || xe > shape[0] - R || ye > shape[1] - R || ze > shape[2] - R || xb >= xe ||
      yb >= ye || zb >= ze)
    return fail(GR_EINVAL, "gr_sweep_dev: box must be non-empty and keep %d cells from every face", R);
  if (kernel == 0 && !roc2) return fail(GR_EINVAL, "gr_sweep_dev: kernel 0 needs roc2");
  Problem P{};
  P.kernel = kernel;
  P.dtype = dtype;
  P.R = R;
  P.ncoef = kncoef(kernel);
  P.pitch = shape[0];
  P.rows = shape[1];
  P.field_elems = (long long)shape[0] * shape[1] * shape[2];
  if (P.ncoef == 0) {
    for (int r = 0; r <= R; ++r) P.c[r] = dtype == GR_F64 ? ((const double *)coef)[r] : ((const float *)coef)[r];
  } else {
    P.coef = (void *)coef;
  }
  P.roc2 = (void *)roc2;
  // Rows of the caller's layout start anywhere in a cache line, and a non-temporal store
  // then writes parts of lines: for a 64-cell tile 2 of 3 lines in FP32, 2 of 5 in FP64.
  // us per sweep without / with the hints: kernel 0 FP32 at 291^2 x 288 (300 MB) 113 / 130
  // and at 515^2 x 494 486 / 593, kernel 5 FP32 at 291^2 x 309 207 / 238 and FP64 at 291^2 x
  // 257 325 / 337; kernel 0 FP64 at 355^2 x 312 (1 GB) 314 / 300, kernel 1 FP64 at 355^2 x 312
  // 168 / 159.
  P.strm_mode = dtype == GR_F64 && P.ncoef == 0 && sweep_bytes(P) > 512.0 * 1024 * 1024;
  // express the box through the generic geometry
  Geom g;
  g.sy = shape[0];
  g.sz = (long long)shape[0] * shape[1];
  g.xb = xb; g.yb = yb; g.zb = zb; g.xe = xe; g.ye = ye; g.ze = ze;
  LaunchCfg lc;
  lc.auto_variant = lc.auto_zchunk = lc.auto_order = true;
  hipError_t e = sweep_box(P, g, u, v, sweep_cfg(kernel, dtype, lc, xe - xb, ye - yb, ze - zb), nullptr);
  if (e != hipSuccess) return fail(GR_EHIP, "gr_sweep_dev: %s", hipGetErrorString(e));
  HIP_TRY(hipStreamSynchronize(nullptr));
  return GR_OK;
}

namespace gr {
hipError_t sweep_box(const Problem &P, const Geom &g, void *u, const void *v, const LaunchCfg &lc, hipStream_t st) {
  if (P.dtype == GR_F64) {
    SweepArgs<double, double> a{};
    a.u = (double *)u;
    a.v = (const double *)v;
    a.roc2 = (const double *)P.roc2;
    a.coef = (const double *)P.coef;
    a.cstride = P.field_elems;
    for (int r = 0; r < 5; ++r) a.c[r] = P.c[r];
    a.g = g;
    a.src_k = -1;
    return launch_sweep_f64(P.kernel, false, false, a, lc, st, streaming_sweep(P));
  }
  SweepArgs<float, float> a{};
  a.u = (float *)u;
  a.v = (const float *)v;
  a.roc2 = (const float *)P.roc2;
  a.coef = (const float *)P.coef;
  a.cstride = P.field_elems;
  for (int r = 0; r < 5; ++r) a.c[r] = (float)P.c[r];
  a.g = g;
  a.src_k = -1;
  return launch_sweep_f32(P.kernel, false, false, a, lc, st, streaming_sweep(P));
}
}  // namespace gr

// ------------------------------------------------------------------ device initial states
namespace {

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__device__ __forceinline__ double u01(uint64_t seed, uint64_t stream, uint64_t i) {
  return (double)(splitmix64(seed ^ splitmix64(stream * 0x632BE59BD9B4E019ull + i)) >> 11) * 0x1.0p-53;
}

// girih's closed-form state (utils.c:605-697, one rank) / uniform / zero
template <typename T>
__global__ void init_fields_kernel(T *u1, T *u2, T *r2, int mode, uint64_t seed, int nx, int ny, int nz, int R,
                                   long long pitch, long long rows, long long total) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int nnx = nx + 2 * R;
  const long long row = t / nnx;
  const int i = (int)(t - row * nnx);
  const int j = (int)(row % rows);
  const int k = (int)(row / rows);
  const long long o = row * pitch + i;
  const bool inner = i >= R && i < nx + R && j >= R && j < ny + R && k >= R && k < nz + R;
  T val = T(0);
  if (mode == 0) {
    if (inner) {
      const T r = (T)(1.0 / 3 * (1.0 * i / nx + 1.0 * j / ny + 1.0 * k / nz));
      val = (T)(r * 1.845703);
    }
    if (r2) r2[o] = val;
    if (i == 0 || i == nnx - 1) val = (T)(val + 100.1);
  } else if (mode == 1) {
    if (inner) val = (T)u01(seed, 0, (uint64_t)((k - R) * (long long)ny + (j - R)) * nx + (i - R));
  }
  u1[o] = val;
  u2[o] = val;
}

// Workgroups of 256 lanes of a kernel over P's halo cells.
static unsigned halo_blocks(const Problem &P) { return (unsigned)((halo_waves(P.ny, P.nz, P.R) + 3) / 4); }
__device__ __forceinline__ long long block_wave() {
  return (long long)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
}

// flag = 1 if U1 and U2 differ (bitwise) anywhere outside the interior box
template <typename U>
__global__ void halo_diff_kernel(const U *a, const U *b, int nx, int ny, int nz, int R, long long pitch, int *flag) {
  for_halo_cells(block_wave(), threadIdx.x % 64, nx, ny, nz, R, pitch, [&](long long o) {
    if (a[o] != b[o]) *flag = 1;
  });
}

// the halo of src into d0 (and d1 unless null)
template <typename U>
__global__ void halo_copy_kernel(const U *src, U *d0, U *d1, int nx, int ny, int nz, int R, long long pitch) {
  for_halo_cells(block_wave(), threadIdx.x % 64, nx, ny, nz, R, pitch, [&](long long o) {
    const U v = src[o];
    d0[o] = v;
    if (d1) d1[o] = v;
  });
}

// Coefficient m of halo-inclusive cell (i, j, k) is drawn from its logical index
// (k*(ny+2R) + j)*(nx+2R) + i, so the values do not depend on the device layout
// (precision, pitch) and FP32 / FP64 / bf16 problems get the same coefficients.
template <typename C>
__global__ void init_coef_kernel(C *coef, int ncoef, uint64_t seed, double lo0, double hi0, double lo1, double hi1,
                                 int nx, int R, long long pitch, long long total, long long field_elems) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const int nnx = nx + 2 * R;
  const long long row = t / nnx;
  const int i = (int)(t - row * nnx);
  const long long o = row * pitch + i;
  for (int m = 0; m < ncoef; ++m) {
    const double x = u01(seed, 1 + m, (uint64_t)t);
    const double val = m == 0 ? lo0 + (hi0 - lo0) * x : lo1 + (hi1 - lo1) * x;
    coef[(long long)m * field_elems + o] = (C)val;
  }
}

}  // namespace

static int check_halo_equal(gr_handle *h) {
  if (h->halo_equal >= 0) return GR_OK;
  const Problem &P = h->P;
  if (!h->flag) HIP_TRY(hipMalloc(&h->flag, sizeof(int)));
  HIP_TRY(hipMemsetAsync(h->flag, 0, sizeof(int), h->stream));
  const int bs = 256;
  const unsigned nb = halo_blocks(P);
  if (P.dtype == GR_F64)
    hipLaunchKernelGGL(halo_diff_kernel<unsigned long long>, dim3(nb), dim3(bs), 0, h->stream,
                       (const unsigned long long *)ubase(h, 0), (const unsigned long long *)ubase(h, 1), P.nx, P.ny,
                       P.nz, P.R, (long long)P.pitch, (int *)h->flag);
  else
    hipLaunchKernelGGL(halo_diff_kernel<unsigned>, dim3(nb), dim3(bs), 0, h->stream, (const unsigned *)ubase(h, 0),
                       (const unsigned *)ubase(h, 1), P.nx, P.ny, P.nz, P.R, (long long)P.pitch, (int *)h->flag);
  HIP_TRY(hipGetLastError());
  int hflag = 1;
  HIP_TRY(hipMemcpyAsync(&hflag, h->flag, sizeof(int), hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(hipStreamSynchronize(h->stream));
  h->halo_equal = hflag == 0 ? 1 : 0;
  return GR_OK;
}

// The spares get the fields' halo, which passes read but never write.  Once per upload or
// initial state, and at every call of a handle whose field pointers the caller holds (where
// the call's first pass cannot bring it along: 4 us at 128^3 FP64, 30 at 512^3 FP32).
static int sync_spares(gr_handle *h) {
  if (h->exposed) h->spares_synced = false;
  if (h->spares_synced) return GR_OK;
  const Problem &P = h->P;
  int sp[2];
  spare_ids(h, sp);
  const unsigned nb = halo_blocks(P);
  void *d0 = field_base(h, h->fbuf[sp[0]]), *d1 = field_base(h, h->fbuf[sp[1]]);
  if (h->exposed && P.kernel != 0) d1 = nullptr;  // a first-order call uses the first spare only
  if (P.dtype == GR_F64)
    hipLaunchKernelGGL(halo_copy_kernel<double>, dim3(nb), dim3(256), 0, h->stream, (const double *)ubase(h, 1),
                       (double *)d0, (double *)d1, P.nx, P.ny, P.nz, P.R, (long long)P.pitch);
  else
    hipLaunchKernelGGL(halo_copy_kernel<float>, dim3(nb), dim3(256), 0, h->stream, (const float *)ubase(h, 1),
                       (float *)d0, (float *)d1, P.nx, P.ny, P.nz, P.R, (long long)P.pitch);
  HIP_TRY(hipGetLastError());
  h->spares_synced = true;
  return GR_OK;
}

extern "C" int gr_init_fields(gr_handle *h, int mode, uint64_t seed) {
  if (!h) return fail(GR_EINVAL, "gr_init_fields: null handle");
  if (mode < 0 || mode > 2) return fail(GR_EINVAL, "gr_init_fields: bad mode %d", mode);
  const Problem &P = h->P;
  const long long total = (long long)(P.nx + 2 * P.R) * P.rows * P.planes;
  const int bs = 256;
  const unsigned nb = (unsigned)((total + bs - 1) / bs);
  if (h->lu[0] != 0 || h->lu[1] != 1) {  // both fields are rewritten: back to the first buffer pair
    drop_graph(h);
    h->lu[0] = 0;
    h->lu[1] = 1;
  }
  void *b1 = ubase(h, 0), *b2 = ubase(h, 1);
  if (P.dtype == GR_F64) {
    hipLaunchKernelGGL(init_fields_kernel<double>, dim3(nb), dim3(bs), 0, h->stream, (double *)b1, (double *)b2,
                       (P.roc2 && mode == 0) ? (double *)P.roc2 : nullptr, mode, seed, P.nx, P.ny, P.nz, P.R,
                       (long long)P.pitch, (long long)P.rows, total);
  } else {
    if ((P.flags & GR_COEF_BF16) && P.roc2 && mode == 0)
      return fail(GR_EUNSUPPORTED, "gr_init_fields: closed-form roc2 is not stored as bf16");
    hipLaunchKernelGGL(init_fields_kernel<float>, dim3(nb), dim3(bs), 0, h->stream, (float *)b1, (float *)b2,
                       (P.roc2 && mode == 0) ? (float *)P.roc2 : nullptr, mode, seed, P.nx, P.ny, P.nz, P.R,
                       (long long)P.pitch, (long long)P.rows, total);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(h->stream));
  state_reset(h);
  return GR_OK;
}

extern "C" int gr_init_coef_uniform(gr_handle *h, uint64_t seed, double lo0, double hi0, double lo1, double hi1) {
  if (!h) return fail(GR_EINVAL, "gr_init_coef_uniform: null handle");
  const Problem &P = h->P;
  if (P.ncoef == 0 || !h->alloc_coef) return fail(GR_EINVAL, "gr_init_coef_uniform: kernel has no coefficient arrays");
  const int bs = 256;
  const long long total = (long long)(P.nx + 2 * P.R) * P.rows * P.planes;
  const unsigned nb = (unsigned)((total + bs - 1) / bs);
  const long long pitch = P.pitch;
  if (P.flags & GR_COEF_BF16)
    hipLaunchKernelGGL(init_coef_kernel<__hip_bfloat16>, dim3(nb), dim3(bs), 0, h->stream,
                       (__hip_bfloat16 *)P.coef, P.ncoef, seed, lo0, hi0, lo1, hi1, P.nx, P.R, pitch, total,
                       P.field_elems);
  else if (P.dtype == GR_F64)
    hipLaunchKernelGGL(init_coef_kernel<double>, dim3(nb), dim3(bs), 0, h->stream, (double *)P.coef, P.ncoef, seed,
                       lo0, hi0, lo1, hi1, P.nx, P.R, pitch, total, P.field_elems);
  else
    hipLaunchKernelGGL(init_coef_kernel<float>, dim3(nb), dim3(bs), 0, h->stream, (float *)P.coef, P.ncoef, seed,
                       lo0, hi0, lo1, hi1, P.nx, P.R, pitch, total, P.field_elems);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(h->stream));
  return GR_OK;
}

// ------------------------------------------------------------------ FP64 reductions
namespace {

template <typename TA, typename TB>
__global__ __launch_bounds__(256) void compare_kernel(const TA *a, long long asy, long long asz, const TB *b,
                                                      long long bsy, long long bsz, int nx, int ny, int nz, int R,
                                                      double *part) {
  // one workgroup per (j, k) row block; grid-stride over rows
  double sd = 0.0, sr = 0.0, md = 0.0, mr = 0.0;
  const long long nrows = (long long)ny * nz;
  for (long long row = blockIdx.x; row < nrows; row += gridDim.x) {
    const int j = (int)(row % ny) + R, k = (int)(row / ny) + R;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) {
      const double x = (double)a[k * asz + j * asy + i + R];
      const double y = (double)b[k * bsz + j * bsy + i + R];
      const double d = x - y;
      sd += d * d;
      sr += y * y;
      md = fmax(md, fabs(d));
      mr = fmax(mr, fabs(y));
    }
  }
  __shared__ double s[4][256];
  s[0][threadIdx.x] = sd;
  s[1][threadIdx.x] = sr;
  s[2][threadIdx.x] = md;
  s[3][threadIdx.x] = mr;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s[0][threadIdx.x] += s[0][threadIdx.x + w];
      s[1][threadIdx.x] += s[1][threadIdx.x + w];
      s[2][threadIdx.x] = fmax(s[2][threadIdx.x], s[2][threadIdx.x + w]);
      s[3][threadIdx.x] = fmax(s[3][threadIdx.x], s[3][threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int q = 0; q < 4; ++q) part[blockIdx.x * 4 + q] = s[q][0];
}

template <typename TA, typename TB>
hipError_t launch_compare(const gr::Problem &A, const void *a, const gr::Problem &B, const void *b, double *part,
                          int nblk, hipStream_t st) {
  hipLaunchKernelGGL((compare_kernel<TA, TB>), dim3(nblk), dim3(256), 0, st, (const TA *)a, (long long)A.pitch,
                     (long long)A.pitch * A.rows, (const TB *)b, (long long)B.pitch, (long long)B.pitch * B.rows,
                     A.nx, A.ny, A.nz, A.R, part);
  return hipGetLastError();
}

}  // namespace

// Partial sums per workgroup of the comparison (compare_kernel's grid).
constexpr int kComparePartials = 2048;

static int compare_args(gr_handle *a, int fa, gr_handle *b, int fb, const char *who) {
  if (!a || !b) return fail(GR_EINVAL, "%s: null argument", who);
  if (fa < 0 || fa > 1 || fb < 0 || fb > 1) return fail(GR_EINVAL, "%s: field must be 0 (U1) or 1 (U2)", who);
  const Problem &A = a->P, &B = b->P;
  if (A.nx != B.nx || A.ny != B.ny || A.nz != B.nz || A.R != B.R) return fail(GR_EINVAL, "%s: grids differ", who);
  return GR_OK;
}

static hipError_t launch_compare_any(gr_handle *a, int fa, gr_handle *b, int fb, double *part, int nblk) {
  const Problem &A = a->P, &B = b->P;
  const void *pa = ubase(a, fa);
  const void *pb = ubase(b, fb);
  if (A.dtype == GR_F64 && B.dtype == GR_F64) return launch_compare<double, double>(A, pa, B, pb, part, nblk, a->stream);
  if (A.dtype == GR_F32 && B.dtype == GR_F64) return launch_compare<float, double>(A, pa, B, pb, part, nblk, a->stream);
  if (A.dtype == GR_F64 && B.dtype == GR_F32) return launch_compare<double, float>(A, pa, B, pb, part, nblk, a->stream);
  return launch_compare<float, float>(A, pa, B, pb, part, nblk, a->stream);
}

extern "C" int gr_compare_fields(gr_handle *a, int fa, gr_handle *b, int fb, double out[4]) {
  int rc = compare_args(a, fa, b, fb, "gr_compare_fields");
  if (rc) return rc;
  if (!out) return fail(GR_EINVAL, "gr_compare_fields: null argument");
  const int nblk = kComparePartials;
  double *part = nullptr;
  HIP_TRY(hipMalloc(&part, sizeof(double) * 4 * nblk));
  HIP_TRY(hipStreamSynchronize(b->stream));
  hipError_t e = launch_compare_any(a, fa, b, fb, part, nblk);
  if (e != hipSuccess) {
    (void)hipFree(part);
    return fail(GR_EHIP, "compare launch: %s", hipGetErrorString(e));
  }
  std::vector<double> h(4 * nblk);
  e = hipMemcpyAsync(h.data(), part, sizeof(double) * 4 * nblk, hipMemcpyDeviceToHost, a->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(a->stream);
  (void)hipFree(part);
  if (e != hipSuccess) return fail(GR_EHIP, "compare copy: %s", hipGetErrorString(e));
  out[0] = out[1] = out[2] = out[3] = 0.0;
  for (int i = 0; i < nblk; ++i) {
    out[0] += h[4 * i];
    out[1] += h[4 * i + 1];
    out[2] = std::max(out[2], h[4 * i + 2]);
    out[3] = std::max(out[3], h[4 * i + 3]);
  }
  return GR_OK;
}

// ------------------------------------------------------------------ comparison without allocation
// gr_compare_fields_static keeps the partial sums in `scratch`, one copy per GPU
// (a file-scope device array: the library holds it on every GPU it runs on until
// the process ends), and reduces them on the device in gr_compare_fields's order.
// Host code never names `scratch` as device memory: it uses the address that
// hipGetSymbolAddress returned for the current device.  Every call writes all
// partials before reading them, so nothing needs clearing between calls; calls
// that overlap on one GPU share the array and race.
namespace {

constexpr int kScratchDoubles = 4 * kComparePartials + 4;  // partials, then the 4 results
static __device__ __align__(256) double scratch[kScratchDoubles];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

// The reduction of the host loop of gr_compare_fields, in the same order.
__global__ void compare_finish_kernel(const double *part, int nblk, double *res) {
  if (threadIdx.x != 0) return;
  double o0 = 0.0, o1 = 0.0, o2 = 0.0, o3 = 0.0;
  for (int i = 0; i < nblk; ++i) {
    o0 += part[4 * i];
    o1 += part[4 * i + 1];
    o2 = (o2 < part[4 * i + 2]) ? part[4 * i + 2] : o2;
    o3 = (o3 < part[4 * i + 3]) ? part[4 * i + 3] : o3;
  }
  res[0] = o0;
  res[1] = o1;
  res[2] = o2;
  res[3] = o3;
}

// This device's copy of `scratch` (looked up once per device, with it current).
int scratch_ptr(int dev, double **out) {
  if (dev < 0 || dev >= kMaxDevices) return fail(GR_EUNSUPPORTED, "gr_compare_fields_static: device %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(GR_EHIP, "gr_compare_fields_static: hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = (double *)p;
  }
  *out = g_scratch_ptr[dev];
  return GR_OK;
}

}  // namespace

extern "C" int gr_compare_fields_static(gr_handle *a, int fa, gr_handle *b, int fb, double out[4]) {
  int rc = compare_args(a, fa, b, fb, "gr_compare_fields_static");
  if (rc) return rc;
  if (!out) return fail(GR_EINVAL, "gr_compare_fields_static: null argument");
  const int nblk = kComparePartials;
  if (4 * nblk + 4 > kScratchDoubles)
    return fail(GR_EUNSUPPORTED, "gr_compare_fields_static: %d partials exceed the %d-double scratch array", nblk,
                kScratchDoubles);
  int cur = 0;
  HIP_TRY(hipGetDevice(&cur));
  if (cur != a->device) HIP_TRY(hipSetDevice(a->device));  // the handle's GPU is current for the call
  double *base = nullptr;
  rc = scratch_ptr(a->device, &base);
  hipError_t e = hipSuccess;
  if (rc == GR_OK) e = hipStreamSynchronize(b->stream);
  if (rc == GR_OK && e == hipSuccess) e = launch_compare_any(a, fa, b, fb, base, nblk);
  if (rc == GR_OK && e == hipSuccess) {
    hipLaunchKernelGGL(compare_finish_kernel, dim3(1), dim3(64), 0, a->stream, (const double *)base, nblk,
                       base + 4 * nblk);
    e = hipGetLastError();
  }
  if (rc == GR_OK && e == hipSuccess)
    e = hipMemcpyAsync(out, base + 4 * nblk, 4 * sizeof(double), hipMemcpyDeviceToHost, a->stream);
  if (rc == GR_OK && e == hipSuccess) e = hipStreamSynchronize(a->stream);
  if (cur != a->device) (void)hipSetDevice(cur);
  if (rc) return rc;
  if (e != hipSuccess) return fail(GR_EHIP, "gr_compare_fields_static: %s", hipGetErrorString(e));
  return GR_OK;
}

// ------------------------------------------------------------------ internals for gr_batch.hip
const gr::Problem &gr_internal_problem(const gr_handle *h) { return h->P; }
void *gr_internal_field(const gr_handle *h, int logical) { return ubase(h, logical); }
void *gr_internal_spare(gr_handle *h, int which) {
  if (ensure_spares(h) != GR_OK) return nullptr;
  int sp[2];
  spare_ids(h, sp);
  return field_base(h, h->fbuf[sp[which & 1]]);
}
int gr_internal_parity(const gr_handle *h) { return h->parity; }
long long gr_internal_napplied(const gr_handle *h) { return h->napplied; }
const void *gr_internal_source(const gr_handle *h, int *n, long long *idx) {
  *n = h->nsrc;
  *idx = h->src_idx;
  return h->src;
}
hipStream_t gr_internal_stream(const gr_handle *h) { return h->stream; }
const gr::LaunchCfg &gr_internal_launch_cfg(const gr_handle *h) { return h->lc; }
extern "C" int gr_internal_graph_captures(const gr_handle *h) { return h->captures; }
extern "C" int gr_internal_streaming(const gr_handle *h) { return streaming_sweep(h->P); }
extern "C" long long gr_internal_pinned_bytes(const gr_handle *h) { return (long long)h->stage_bytes; }
int gr_internal_fused_prepare(gr_handle *h, bool *ok) {
  *ok = false;
  bool depth_ok = false;
  int rc = fused_depth_ok(h, 2, &depth_ok);
  if (rc || !depth_ok || h->P.kernel != 0) return rc;
  if ((rc = ensure_spares(h))) return rc;
  if (!h->spares_synced || h->exposed) {
    if ((rc = sync_spares(h))) return rc;
    HIP_TRY(hipStreamSynchronize(h->stream));
  }
  *ok = true;
  return GR_OK;
}
void gr_internal_fused_buffers(const gr_handle *h, int npasses, void *buf[4]) {
  // the mapping (written-next, read-next) after npasses two-step passes, and its spares;
  // a pass writes (u^(n+1), u^(n+2)) into the spares, which then become the fields
  int lu[2] = {h->lu[0], h->lu[1]};
  const int w = h->parity, r = 1 - w;
  for (int p = 0; p <= npasses; ++p) {
    int sp[2], n = 0;
    for (int i = 0; i < 4 && n < 2; ++i)
      if (i != lu[0] && i != lu[1]) sp[n++] = i;
    if (p == npasses) {
      buf[0] = field_base(h, h->fbuf[lu[w]]);
      buf[1] = field_base(h, h->fbuf[lu[r]]);
      buf[2] = field_base(h, h->fbuf[sp[0]]);
      buf[3] = field_base(h, h->fbuf[sp[1]]);
      return;
    }
    lu[w] = sp[0];
    lu[r] = sp[1];
  }
}
void gr_internal_fused_advance(gr_handle *h, int npasses, int napply, double ms) {
  for (int p = 0; p < npasses; ++p) {  // the rotation of gr_step's kernel-0 fused path
    int sp[2];
    spare_ids(h, sp);
    h->lu[h->parity] = sp[0];
    h->lu[1 - h->parity] = sp[1];
  }
  h->parity ^= (napply - 2 * npasses) & 1;
  h->napplied += napply;
  h->stats.last_ms = ms;
  h->stats.last_updates = (int64_t)napply * h->P.nx * h->P.ny * h->P.nz;
  h->stats.last_launches = npasses + (napply - 2 * npasses);
}
int gr_internal_copy_field(gr_handle *h, const int ld[3], void *dev_base, void *host, bool to_dev) {
  const size_t es = elem_size(h->P.dtype);
  return copy_field(h, ld, dev_base, es, host, es, to_dev);
}
void gr_internal_advance(gr_handle *h, int napply, double ms) {
  h->parity ^= napply & 1;
  h->napplied += napply;
  h->stats.last_ms = ms;
  h->stats.last_updates = (int64_t)napply * h->P.nx * h->P.ny * h->P.nz;
  h->stats.last_launches = napply;
}
