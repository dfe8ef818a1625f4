/*
 * ax_step_tiled.hip - Abelian-Higgs and Moore steps of one lattice, one
 * 64-lane wave per (chunk of 64 sites of the (y, z) plane, x segment) marching
 * along x (the updates themselves are ah_march in ax_march.h and moore_march
 * in ax_march_moore.h).  FP64 and FP32, every boundary (boundary planes and
 * rows are left to the boundary kernels).
 *
 * Work items are numbered in the XCD-aware order of make_tile_grid
 * (ax_internal.h): each XCD takes bands of consecutive rows with all their
 * chunks, so y-neighbour rows and chunk-edge lines are read from its own L2.
 */
#include <algorithm>
#include <cstdlib>
#include <limits>

#include "ax_internal.h"
#include "ax_march.h"
#include "ax_march_moore.h"

namespace ax {

/* The chunk and the planes [x0, x1) a work item steps; with non-periodic x/y
 * (ex) the boundary planes are left alone (their neighbours would wrap),
 * evolution.cpp:161-186.  Returns false for an empty item. */
__device__ __forceinline__ bool tile_range(const TileGrid &g, int nx, int ex, int w, int &chunk, int &x0, int &x1) {
  int seg;
  if (!tile_item(g, w, chunk, seg)) return false;
  x0 = seg * g.xseg;
  x1 = min(nx, x0 + g.xseg);
  if (ex) {
    x0 = max(x0, 1);
    x1 = min(x1, nx - 1);
  }
  return x0 < x1;
}

template <typename R, bool POW2, bool PLAIN, bool BIG, bool PF, bool FLAT>
__global__ void __launch_bounds__(64, sizeof(R) == 8 ? 3 : 1) ah_tiled_kernel(MarchConsts<R> k, Levels<R> L, int nx, int ny, int nz,
                                                      TileGrid g, int ex, int ez) {
  int chunk, x0, x1;
  if (!tile_range(g, nx, ex, (int)blockIdx.x, chunk, x0, x1)) return;
  const uint32_t p0 = (uint32_t)chunk * 64;
  if (!FLAT && ex && (p0 < (uint32_t)nz || p0 >= (uint32_t)nz * (ny - 1))) return;   /* a boundary row */
  ah_march<R, POW2, PLAIN ? 1 : 0, BIG, PF, 0, false, FLAT>(k, L, nx, ny, nz, p0, x0, x1, ex != 0, ez != 0);
}

/* FD: FP64 with divisors in the FixedDivisor range on a periodic lattice.
 * band[3] are the per-level band flags (ax_march_moore.h), indexed by
 * TimeStep mod 3: this step (TimeStep t) divides through FixedDivisor when
 * use_band is set and band[t % 3] is clear, ORs its output's check into
 * band[(t + 1) % 3] and clears band[(t + 2) % 3] for the next step. */
template <typename R, bool POW2, bool BUF, bool FD, bool FLAT>
__global__ void __launch_bounds__(64, 3) moore_tiled_kernel(MooreConsts<R> k, Levels<R> L, int nx, int ny, int nz,
                                                         TileGrid g, int ex, int ez, int *band, int t,
                                                         int use_band) {
  if (FD && blockIdx.x == 0 && threadIdx.x == 0) band[(t + 2) % 3] = 0;
  int chunk, x0, x1;
  if (!tile_range(g, nx, ex, (int)blockIdx.x, chunk, x0, x1)) return;
  const uint32_t p0 = (uint32_t)chunk * 64;
  if (!FLAT && ex && (p0 < (uint32_t)nz || p0 >= (uint32_t)nz * (ny - 1))) return;   /* a boundary row */
  if constexpr (FD) {
    int *out = band + (t + 1) % 3;
    if (use_band && band[t % 3] == 0)
      moore_march<R, POW2, BUF, FLAT, true, true>(k, L, nx, ny, nz, p0, x0, x1, false, false, out);
    else
      moore_march<R, POW2, BUF, FLAT, false, true>(k, L, nx, ny, nz, p0, x0, x1, false, false, out);
  } else {
    moore_march<R, POW2, BUF, FLAT>(k, L, nx, ny, nz, p0, x0, x1, ex != 0, ez != 0);
  }
}

template <typename R>
hipError_t launch_step_tiled_moore(const StepConsts &k, const Levels<R> &L, int xseg, hipStream_t st, int *band,
                                   int t, bool use_band, bool *fd_used) {
  const TileGrid g = make_tile_grid(k.nx, k.ny, k.nz, xseg);
  MooreConsts<R> m;
  moore_consts_from<R>(k, m);
  const bool pow2 = is_pow2(k.dx2) && is_pow2(k.dy2) && is_pow2(k.dz2);
  /* buffer path when both levels of a field lie within 4 GiB of its lower plane */
  const size_t lev = (size_t)std::llabs((const char *)L.cur[0] - (const char *)L.prv[0]);
  const bool buf = lev + (size_t)k.nx * k.ny * k.nz * sizeof(R) < ((size_t)1 << 32) &&
                   getenv("AX_BIG_PLANES") == nullptr;   /* forces the global path, for tests */
  /* FP64 divisions by dx^2, dy^2, dz^2 through FixedDivisor, guarded by the
   * band flags (every site written by this kernel: periodic lattices only);
   * with the buffer path only: on the global path (planes of 4 GiB or
   * more) it spills 67 VGPRs at 3 waves per SIMD and is no faster than the
   * site kernel, the plain divisions spill none */
  const bool fd = sizeof(R) == 8 && buf && !pow2 && band != nullptr && !k.ex && !k.ez && fixed_divisor_range(k.dx2) &&
                  fixed_divisor_range(k.dy2) && fixed_divisor_range(k.dz2) && moore_band_charge((int)k.q1) &&
                  moore_band_charge((int)k.q2) && getenv("AX_MOORE_PLAIN_DIV") == nullptr;
  *fd_used = fd;
  dim3 grid(g.work), block(64);
  const bool flat = k.nz % 64 != 0;   /* as launch_step_tiled_ah */
#define AX_MRK(P2, B, FD, FL)                                                                                      \
  hipLaunchKernelGGL((moore_tiled_kernel<R, P2, B, FD, FL>), grid, block, 0, st, m, L, k.nx, k.ny, k.nz, g, k.ex, k.ez, \
                     band, t, use_band ? 1 : 0)
#define AX_MRL(P2, B, FD)                  \
  do {                                     \
    if (flat) AX_MRK(P2, B, FD, true);     \
    else AX_MRK(P2, B, FD, false);         \
  } while (0)
  if (pow2 && buf) AX_MRL(true, true, false);
  else if (pow2) AX_MRL(true, false, false);
  else if (buf && fd) AX_MRL(false, true, true);
  else if (buf) AX_MRL(false, true, false);
  else AX_MRL(false, false, false);
#undef AX_MRK
#undef AX_MRL
  return hipGetLastError();
}

template hipError_t launch_step_tiled_moore<double>(const StepConsts &, const Levels<double> &, int, hipStream_t,
                                                    int *, int, bool, bool *);
template hipError_t launch_step_tiled_moore<float>(const StepConsts &, const Levels<float> &, int, hipStream_t, int *,
                                                   int, bool, bool *);

/* Every Abelian-Higgs and Moore lattice marches, whatever its plane (chunks
 * cross rows, and the last of a plane may run with lanes idle) and whatever
 * its size (planes of 4 GiB or more take the 64-bit plane addressing of
 * ah_march and moore_march). */
bool use_tiled_ah(const ax_params &p) {
  return (p.model == AX_MODEL_AH || p.model == AX_MODEL_MOORE) && p.nx >= 3 && p.ny >= 3 &&
         getenv("AX_FORCE_SITE_KERNEL") == nullptr;
}

/* x planes per wave: tile_xseg's rule, up to the length that is best on
 * large lattices (measured at 512^3 AH, 256^3 Moore, on one box each):
 * Abelian-Higgs FP64 32 (3.607 ms; 8: 3.746, 16: 3.644, 24: 3.631, 48: 3.603;
 * 256^3 32: 0.459, 16: 0.468), FP32 16 (1.737 ms; 8: 1.762, 12: 1.758, 32:
 * 1.756); Moore FP32 8 (0.422 ms; 32: 0.444).  Moore's prologue is cheap
 * against a plane, so it takes half the rule's length (rule / half, us: FP64
 * 201x201x51 fixed 141.6 / 133.8, 100^3 fixed 70.1 / 65.4, 150^3 fixed 203 /
 * 197, periodic 181 / 179, 200^3 fixed 464 / 452, 128^3 110.5 / 108.1; FP32
 * 128^3 65 / 60, 160^3 135 / 118), in FP64 from 3 planes on (64^3 2: 19.2, 1:
 * 21.0).  On whole chunks in FP64 longer segments catch up from about 10
 * planes on, so it is the rule's length less 4 there, up to 12 (periodic, half
 * / this / 16 planes: 192^3 356 / 354 / 364, 128x300x192 366 / 365 / 388, 256^3
 * 814 / 804 / 804); across rows half is best or within 1 % (250^3 814, 11
 * planes 826, 16 823; 260^3 889, 882, 881; 300^3 1344, 1354, 1351; fixed 250^3
 * 889, 896, 897; 300^3 1464, 1459, 1469). */
int default_xseg(const ax_params &p) {
  const char *xe = getenv("AX_TILED_XSEG");
  if (xe) return atoi(xe);
  const bool f32 = p.precision == 32;
  if (p.model != AX_MODEL_MOORE) return tile_xseg(p.nx, p.ny, p.nz, f32 ? 16 : 32);
  const int xs = tile_xseg(p.nx, p.ny, p.nz, 16), half = (xs + 1) / 2;
  if (f32) return half;
  return xs <= 2 ? xs : p.nz % 64 == 0 ? std::max(half, xs - 4) : half;
}

/* The LDS prefetch of the FP64 march applies: whole 64-site chunks (across
 * rows it costs registers that spill: 200^3 251 us against 245 without),
 * three field planes within 32-bit offsets, and the [comp][level] plane order
 * its pairs of rows rely on (AX_NO_PREFETCH turns it off). */
template <typename R>
static bool prefetch_ok(const StepConsts &k, const Levels<R> &L) {
  const ptrdiff_t cs = L.cur[1] - L.cur[0];   /* [comp][level]: two planes */
  const bool order = cs > 0 && L.cur[3] - L.cur[2] == cs && L.cur[4] - L.cur[3] == cs && L.prv[1] - L.prv[0] == cs &&
                     L.prv[3] - L.prv[2] == cs;
  return k.nz % 64 == 0 && order &&
         (size_t)k.nx * k.ny * k.nz * sizeof(double) * 3 + ((size_t)1 << 20) < ((size_t)1 << 32) &&
         getenv("AX_NO_PREFETCH") == nullptr;
}

template <typename R>
hipError_t launch_step_tiled_ah(const StepConsts &k, const Levels<R> &L, int xseg, hipStream_t st) {
  const TileGrid g = make_tile_grid(k.nx, k.ny, k.nz, xseg);
  MarchConsts<R> m;
  march_consts_from<R>(k, rate_limit<R>((R)k.dt), m);
  const bool pow2 = is_pow2(k.dx2) && is_pow2(k.dy2) && is_pow2(k.dz2);
  /* a field plane of 4 GiB or more: 64-bit plane addressing (AX_BIG_PLANES
   * forces it on smaller lattices, for tests) */
  const bool big = (size_t)k.nx * k.ny * k.nz * sizeof(R) >= ((size_t)1 << 32) || getenv("AX_BIG_PLANES") != nullptr;
  dim3 grid(g.work), block(64);
  /* FP64, whole chunks and three planes within 32-bit offsets: a plane's
   * rows are prefetched into LDS (ah_march).  Every variant keeps 3 waves per
   * SIMD with it, with the stores issued one plane late. */
  const bool pf = sizeof(R) == 8 && !big && prefetch_ok(k, L);
  /* rows of whole chunks, whose row offsets stay scalars, else chunks across
   * rows.  us per step with partial chunks at the row ends / across rows:
   * FP64 101^3 50 / 43, 200^3 290 / 245, 300^3 949 / 781, 201x201x51 90 / 76;
   * FP32 101^3 33 / 24, 200^3 162 / 121, 300^3 582 / 417 (those lattices'
   * rows now keep to one XCD too).  Whole chunks taken across rows lose: with
   * 64-bit planes, FP64, whole / across 512^3 3.93 / 4.09 ms, 520x512x1024 7.76 /
   * 8.08 (8 VGPRs spilled) */
  const bool flat = k.nz % 64 != 0;
#define AX_AHK(P2, PL, BG, PF, FL)                                                                             \
  hipLaunchKernelGGL((ah_tiled_kernel<R, P2, PL, BG, PF, FL>), grid, block, 0, st, m, L, k.nx, k.ny, k.nz, g, k.ex, \
                     k.ez)
#define AX_AHL(BG, PF, FL)                          \
  do {                                              \
    if (pow2 && m.plain) AX_AHK(true, true, BG, PF, FL);  \
    else if (pow2) AX_AHK(true, false, BG, PF, FL);       \
    else if (m.plain) AX_AHK(false, true, BG, PF, FL);    \
    else AX_AHK(false, false, BG, PF, FL);                \
  } while (0)
  if (pf) {
    if constexpr (sizeof(R) == 8) AX_AHL(false, true, false);
  } else if (big) {
    if (flat) AX_AHL(true, false, true);
    else AX_AHL(true, false, false);
  } else {
    if (flat) AX_AHL(false, false, true);
    else AX_AHL(false, false, false);
  }
#undef AX_AHL
#undef AX_AHK
  return hipGetLastError();
}

/* The FP64 periodic Abelian-Higgs step with its current level's divergence
 * stored (MODE 1) or its current level's diagnostics taken (MODE 2), see
 * ah_march.  One partial-sum triple per work item (MODE 2).  PF: the LDS
 * prefetch of the plain step (MODE 1 keeps 3 waves per SIMD with it, 168
 * VGPRs; MODE 2 runs at 2 either way). */
template <bool POW2, bool P2D, int MODE, bool PF, bool FLAT>
__global__ void __launch_bounds__(64, MODE == 1 ? 3 : 2) ah_fused_kernel(MarchConsts<double> k, Levels<double> L, int nx, int ny, int nz,
                                                      TileGrid g, FusedDiag fd) {
  const int w = (int)blockIdx.x;
  int chunk, x0, x1;
  if (!tile_range(g, nx, 0, w, chunk, x0, x1)) {
    if (MODE == 2 && threadIdx.x < 3) fd.part[3 * (size_t)w + threadIdx.x] = 0;
    return;
  }
  ah_march<double, POW2, 2, false, PF, MODE, P2D, FLAT>(k, L, nx, ny, nz, (uint32_t)chunk * 64, x0, x1, false, false, fd,
                                                        w);
}

int fused_work_items(int nx, int ny, int nz, int xseg) { return make_tile_grid(nx, ny, nz, xseg).work; }

hipError_t launch_step_fused(const StepConsts &k, const Levels<double> &L, int xseg, hipStream_t st, int mode,
                             bool p2d, const FusedDiag &fd) {
  const TileGrid g = make_tile_grid(k.nx, k.ny, k.nz, xseg);
  MarchConsts<double> m;
  march_consts_from<double>(k, rate_limit<double>(k.dt), m);
  const bool pow2 = is_pow2(k.dx2) && is_pow2(k.dy2) && is_pow2(k.dz2);
  /* the plain step's prefetch conditions (launch_step_tiled_ah) */
  const bool pf = prefetch_ok(k, L);
  dim3 grid(g.work), block(64);
  const bool flat = k.nz % 64 != 0;
#define AX_FK(P2, PD, MD, PF, FL)                                                                               \
  hipLaunchKernelGGL((ah_fused_kernel<P2, PD, MD, PF, FL>), grid, block, 0, st, m, L, k.nx, k.ny, k.nz, g, fd)
#define AX_FL(P2, PD, MD)                          \
  do {                                             \
    if (pf) AX_FK(P2, PD, MD, true, false);        \
    else if (flat) AX_FK(P2, PD, MD, false, true); \
    else AX_FK(P2, PD, MD, false, false);          \
  } while (0)
  if (mode == 1) {
    if (pow2) AX_FL(true, false, 1);
    else AX_FL(false, false, 1);
  } else {
    if (pow2 && p2d) AX_FL(true, true, 2);
    else if (pow2) AX_FL(true, false, 2);
    else AX_FL(false, false, 2);
  }
#undef AX_FL
#undef AX_FK
  return hipGetLastError();
}

template hipError_t launch_step_tiled_ah<double>(const StepConsts &, const Levels<double> &, int, hipStream_t);
template hipError_t launch_step_tiled_ah<float>(const StepConsts &, const Levels<float> &, int, hipStream_t);

}  // namespace ax
