/*
 * ax_internal.h - declarations shared by the library's translation units.
 */
#ifndef AXIONS_AX_INTERNAL_H
#define AXIONS_AX_INTERNAL_H

#include <cmath>
#include <cstdarg>
#include <cstdlib>

#include "ax_device.h"

struct ax_lattice;

namespace ax {

/* Work items of a marching kernel: one 64-lane wave per (chunk of 64
 * consecutive sites of the (y, z) plane, x segment of xseg planes).  A chunk
 * lies in one row where nz is a multiple of 64 and crosses rows otherwise.
 *
 * Workgroups are handed to the eight XCDs round-robin (workgroup w to XCD w
 * mod 8), each XCD with its own L2.  With chunk = w mod nc, neighbouring
 * chunks, which share the cache lines at their z edges and the rows at their
 * y edges, would sit on different XCDs.  So XCD x gets the x-th eighth of each
 * segment's chunks, a band of consecutive rows (512^3 FP64 reads 15.4 -> 12.9
 * GB per step, FP32 9.0 -> 6.1 GB); where the chunks are no multiple of 8 a
 * few of the workgroups find nothing to do.  Planes of fewer than 14 chunks
 * take the natural order once the fullest XCD would get more than 128 waves,
 * one for each of its SIMDs, while others idle (us per step, eighths / natural:
 * 4000x3x3, one chunk, AH FP64 53.7 / 12.2, Moore 88 / 18.6; 1000x10x10, two,
 * 22.5 / 9.5 and 32.6 / 12.9; 600x24x24, nine, 23.0 / 16.2 and 73 / 50;
 * 150x4x4, one, 6.9 / 5.9 and 11.4 / 9.1).  With fewer waves one XCD's L2 counts
 * for more (100x4x4 5.8 / 6.1 and 7.5 / 8.0; 43x28x29, 13 chunks, 7.0 / 7.6),
 * and so it does on wider planes (43x43x22, 15, 6.9 / 7.5 and 8.3 / 9.7; 50^3,
 * 40, 9.4 / 9.6 and 11.9 / 13.5; 101^3, 160, 41 / 48 and 69 / 74). */
struct TileGrid {
  int nc;      /* chunks of a plane */
  int xseg;    /* x planes marched by one wave */
  int work;    /* workgroups, with the empty ones */
  int per;     /* chunks per XCD per x segment, 0 = natural order */
};

inline int tile_chunks(int ny, int nz) { return (int)(((long long)ny * nz + 63) / 64); }

inline TileGrid make_tile_grid(int nx, int ny, int nz, int xseg) {
  TileGrid g;
  g.xseg = (xseg <= 0 || xseg > nx) ? nx : xseg;
  g.nc = tile_chunks(ny, nz);
  const char *o = getenv("AX_TILE_ORDER");        /* "natural" for measurements */
  const int nseg = (nx + g.xseg - 1) / g.xseg, per = (g.nc + 7) / 8;
  const bool natural = (o && o[0] == 'n') || (g.nc < 14 && (long long)per * nseg > 128);
  g.per = natural ? 0 : per;
  g.work = (natural ? g.nc : 8 * per) * nseg;
  return g;
}

/* Workgroups of a march in whichever order takes more: what a buffer of one
 * entry per workgroup holds, so that it serves launches of either order
 * (AX_TILE_ORDER is read at each launch). */
inline size_t tile_items_max(int nx, int ny, int nz, int xseg) {
  const int xs = (xseg <= 0 || xseg > nx) ? nx : xseg;
  return (size_t)8 * ((tile_chunks(ny, nz) + 7) / 8) * ((nx + xs - 1) / xs);
}

/* chunk and x segment of workgroup w; false for an empty one */
__device__ __forceinline__ bool tile_item(const TileGrid &g, int w, int &chunk, int &seg) {
  if (g.per) {
    const int i = w >> 3;
    seg = i / g.per;
    chunk = (w & 7) * g.per + (i - seg * g.per);
    return chunk < g.nc;
  }
  seg = w / g.nc;
  chunk = w - seg * g.nc;
  return true;
}

/* This lane's site of the chunk that begins at site p0 of the (y, z) plane.
 * FLAT: chunks cross rows, so rows that are no multiple of 64 long leave no
 * lanes idle (101^3: 160 waves a plane instead of 202); lanes past the
 * plane's last site hold that site (act false).  Otherwise nz is a multiple
 * of 64, a chunk lies in one row, and the byte offset of a neighbour in its
 * plane splits into a scalar row part and a lane part (two to four VGPRs
 * fewer). */
template <bool FLAT>
struct LaneSite {
  uint32_t p;
  int y, z, ym, yp, zm, zp, nz;
  bool act;
  __device__ __forceinline__ LaneSite(int ny, int nz_, uint32_t p0) : nz(nz_) {
    const uint32_t n = (uint32_t)ny * nz_, q = p0 + (threadIdx.x & 63);
    act = !FLAT || q < n;
    p = act ? q : n - 1;
    y = (int)((FLAT ? p : p0) / (uint32_t)nz_);
    if (!FLAT) {
      /* opaque from here on: seen as the quotient it is, the row makes the
       * compiler give every row address registers of its own (Moore with
       * 64-bit planes: 30 VGPRs spilled, 192^3 FP64 656 us a step; 415 with
       * this) */
      y = __builtin_amdgcn_readfirstlane(y);
      asm("" : "+s"(y));
    }
    z = (int)(p - (uint32_t)y * nz_);
    ym = y == 0 ? ny - 1 : y - 1;
    yp = y == ny - 1 ? 0 : y + 1;
    zm = z == 0 ? nz_ - 1 : z - 1;
    zp = z == nz_ - 1 ? 0 : z + 1;
  }
  /* row and lane byte offsets of the site (y + r, z + c), elements of E bytes */
  __device__ __forceinline__ uint32_t row(int r, uint32_t E) const {
    return FLAT ? 0u : (uint32_t)(r < 0 ? ym : r > 0 ? yp : y) * nz * E;
  }
  __device__ __forceinline__ uint32_t col(int r, int c, uint32_t E) const {
    const uint32_t zz = (uint32_t)(c < 0 ? zm : c > 0 ? zp : z);
    return (FLAT ? (uint32_t)(r < 0 ? ym : r > 0 ? yp : y) * nz + zz : zz) * E;
  }
};

/* n / d for n < 2^31 and d >= 2 by a multiplication: m = floor(2^(31+s)/d) + 1
 * with 2^(s-1) < d <= 2^s exceeds 2^(31+s)/d by less than 2^s/d <= 2, so the
 * quotient's error stays below 1/d */
struct FastDiv {
  uint32_t d, m, s;
};
inline FastDiv fast_div(uint32_t d) {
  uint32_t s = 1;
  while (((uint64_t)1 << s) < d) ++s;
  return {d, (uint32_t)(((uint64_t)1 << (31 + s)) / d + 1), s - 1};
}
__device__ __forceinline__ uint32_t quotient(uint32_t n, const FastDiv &f) { return __umulhi(n, f.m) >> f.s; }

/* x planes per wave of a march over the whole lattice, at most cap.  A wave
 * pays a prologue worth about one plane, so long segments do the least work;
 * but a lattice of few chunks then fills few of the chip's 1024 SIMDs, and
 * the launch ends with a tail that lasts as long as one segment.  With W
 * (chunks) x (planes) per SIMD, work W (1 + c / xseg) plus a tail of
 * xseg planes is least near xseg = sqrt(W), which is what the sweeps show
 * (AH FP64 step, us per step with 32 planes / with this rule / best of 1 ...
 * 32: 32^3 68 / 6.6 / 6.6, 64^3 64 / 12.6 / 12.6, 128^3 74 / 66 / 63, 192^3
 * 223 / 202 / 201, 256^3 475 / 477 / 475).  The length is then evened out over the segments. */
inline int tile_xseg(int nx, int ny, int nz, int cap) {
  const double w = (double)tile_chunks(ny, nz) * nx / 1024.0;
  const double x = std::sqrt(w) + 0.5;
  const int xs = x >= cap ? cap : x < 1 ? 1 : (int)x;
  const int nseg = (nx + xs - 1) / xs;
  return (nx + nseg - 1) / nseg;
}

struct DiagConsts {
  int nx, ny, nz, ex, ez, model, energy_form, ncomp;
  double dx, dy, dz, dt, g, lambda, eta;
  double lambda1, lambda2, lambda12, eta1, eta2, q1, q2;
  double inner; /* (nx-2)(ny-2)(nz-2) as a double */
};

int fail(int code, const char *fmt, ...);
int hip_fail(hipError_t e, const char *what);
int check_params(const ax_params *p);
StepConsts step_consts(const ax_params *p, int n);
DiagConsts diag_consts(const ax_params *p);

template <typename T>
Levels<T> levels_of(ax_lattice *L, int n);
hipStream_t lattice_stream(ax_lattice *L);
const ax_params &lattice_params(const ax_lattice *L);
void *lattice_state(ax_lattice *L);
size_t lattice_sites(const ax_lattice *L);
size_t lattice_pitch(const ax_lattice *L);
int lattice_device(const ax_lattice *L);
int lattice_timestep(const ax_lattice *L);
void lattice_reset_timestep(ax_lattice *L);

/* Partial sums of a diagnostic pass: triples at p (room for
 * diag_part_blocks), n of them once the pass is launched; launch_sums adds
 * them up. */
struct Partials {
  double *p;
  int n;
};

int launch_step(ax_lattice *L, int n);
int ensure_winding_buffer(ax_lattice *L);
int ensure_phase_buffer(ax_lattice *L);
hipError_t launch_march_diag(ax_lattice *L, bool phases, Partials &part);
hipError_t launch_phase_winding(ax_lattice *L, int8_t *out, Partials &part);
int prepare_faces(ax_lattice *L);
/* the Neumann faces prepared (prepare_faces); out may be null.  With faces
 * the counts are NaN where FP32 edge values did not hold the links, and
 * launch_site_winding evaluates the windings then (the counts and out). */
int launch_site_winding(ax_lattice *L, int field, int8_t *out, Partials &part);
int launch_winding_field(ax_lattice *L, int field, int8_t *out, Partials &part);

template <typename R>
hipError_t launch_step_site(const StepConsts &k, const Levels<R> &L, int model, hipStream_t st);
bool use_tiled_ah(const ax_params &p);
int default_xseg(const ax_params &p);
template <typename R>
hipError_t launch_step_tiled_ah(const StepConsts &k, const Levels<R> &L, int xseg, hipStream_t st);
/* band: the lattice's three per-level band flags (nullptr: none); t the
 * TimeStep; use_band: band[t % 3] was written by the previous step; *fd_used
 * tells whether the kernel kept the flags (FP64 FixedDivisor path) */
template <typename R>
hipError_t launch_step_tiled_moore(const StepConsts &k, const Levels<R> &L, int xseg, hipStream_t st, int *band, int t,
                                   bool use_band, bool *fd_used);

template <typename R>
hipError_t launch_global_step(const ax_params &p, void *state, size_t pitch, int n, hipStream_t st);
size_t global_energy_blocks(const ax_params &p);   /* partial-sum blocks of launch_global_energy, whatever the pitch */
template <typename R>
hipError_t launch_global_energy(const ax_params &p, const void *state, size_t pitch, int n, Partials &part,
                                hipStream_t st);

template <typename T>
hipError_t launch_diag(const DiagConsts &k, const Levels<T> &L, Partials &part, hipStream_t st);
/* Abelian-Higgs: energy/Gauss march, with phase != NULL also the FP32 edge
 * values [3][V] (forward edge phase + link angle, ax_wind.h);
 * launch_wind_phase turns them into windings (the field into out when out !=
 * NULL, the counts into part; ex, ez: x and y, z not periodic, and the counts
 * are NaN where an edge value exceeds kEdgeExact) */
/* x planes per wave of the diagnostics and winding marches (us per
 * ax_diagnostics call without / with windings; this rule against the best of
 * 1 ... 32 planes: 64^3 27.5 / 41.8 against 27.4 / 41.7, 160^3 125 / 244
 * against 125 / 244; with 32 planes the energy march alone took 84 at 101^3,
 * with this rule 35) */
inline int diag_xseg(int nx, int ny, int nz) { return tile_xseg(nx, ny, nz, 32); }
bool use_diag_march(const ax_params &p);
size_t diag_part_blocks(const ax_params &p);
template <typename T>
hipError_t launch_diag_march(const DiagConsts &k, const Levels<T> &L, float *phase, Partials &part, hipStream_t st);
hipError_t launch_wind_phase(int nx, int ny, int nz, int ex, int ez, const float *E, int8_t *out, Partials &part,
                             hipStream_t st);
/* the FP32 edge values of field (fr, fi) of charge q into E, then the
 * windings from them, as launch_wind_phase */
template <typename T>
hipError_t launch_edge_winding(int nx, int ny, int nz, int ex, int ez, const T *fr, const T *fi, const T *tx,
                               const T *ty, const T *tz, double q, float *E, int8_t *out, Partials &part,
                               hipStream_t st);
template <typename T>
hipError_t launch_winding(int nx, int ny, int nz, const T *fr, const T *fi, const T *tx, const T *ty, const T *tz,
                          double q, int ex, int ez, int8_t *out, Partials &part, hipStream_t st);
/* Crossings: sites of one wave's group (a multiple of 64), and the groups of
 * a lattice, which is how many counts (bcount) and offsets (boff)
 * launch_crossings uses.  512 sites a group, fewer where that would leave
 * the chip short of waves (8192 resident); at most max(2^14, V / 512 + 1)
 * groups. */
inline uint32_t cross_sites(size_t V) {
  const size_t s = V / 8192 / 64 * 64;
  return (uint32_t)(s < 64 ? 64 : s > 512 ? 512 : s);
}
inline size_t cross_groups(size_t V) { return (V + cross_sites(V) - 1) / cross_sites(V); }
template <typename T>
hipError_t launch_crossings(int nx, int ny, int nz, double dx, double dy, double dz, const T *fr, const T *fi,
                            int ex, int ez, int *bcount, long long *boff, long long *total, double *xyz,
                            long long cap, uint64_t *masks, hipStream_t st, bool write);
/* the face masks (masks, may be null) of a lattice of V sites */
inline size_t cross_mask_bytes(size_t V) { return (V + 63) / 64 * 3 * sizeof(uint64_t); }

/* Fused diagnostics (ax_march.h MODE 1/2, FP64 periodic Abelian-Higgs) */
struct FusedDiag;
struct EnergyConsts;
int fused_work_items(int nx, int ny, int nz, int xseg);   /* of the launch, at most tile_items_max */
hipError_t launch_step_fused(const StepConsts &k, const Levels<double> &L, int xseg, hipStream_t st, int mode,
                             bool p2d, const FusedDiag &fd);
/* the sums of a into out3 and, where b holds any, of b into outb3 (which
 * may be pinned host memory) in one launch */
hipError_t launch_sums(const Partials &a, double *out3, const Partials &b, double *outb3, hipStream_t st);
hipError_t launch_level_div(int nx, int ny, int nz, const double *tx, const double *ty, const double *tz,
                            const EnergyConsts &ek, bool pow2, double *div, hipStream_t st);
bool diag_pow2(double dx, double dy, double dz, double gg);

/* Boundary work of one TimeStep on a lattice that is not periodic
 * (ax_bound.hip).  launch_neumann_faces sets the faces of level tN from
 * their inner neighbours; launch_absorbing steps the x/y faces and corners
 * and must run before the bulk update, which overwrites the level-tP values
 * they read. */
template <typename R>
hipError_t launch_neumann_faces(const ax_params &p, void *state, size_t pitch, int tN, hipStream_t st);
template <typename R>
hipError_t launch_absorbing(const StepConsts &k, const ax_params &p, void *state, size_t pitch, int tN, int tP,
                            hipStream_t st);

}  // namespace ax

#endif
