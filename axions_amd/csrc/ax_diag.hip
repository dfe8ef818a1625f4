/*
 * ax_diag.hip - read-only diagnostic passes over one lattice state.
 *
 *  diag_kernel      energy density and Gauss-law deviation per site
 *                   (evolution.cpp:298-427, Moore mooreEvol.cpp:259-389) in
 *                   FP64 whatever the storage type, plus a finiteness flag
 *                   over every stored value; per-block FP64 partial sums are
 *                   reduced by one block in a fixed order, so the result is
 *                   deterministic for a given lattice shape.
 *  winding_kernel   per-plaquette winding numbers (no reference
 *                   counterpart) and their absolute sum.
 *  crossing kernels the bilinear face-crossing test of
 *                   mpi_evolution.cpp:536-789, in FP32 with an error bound
 *                   first, in FP64 where it is needed (ax_cross.h),
 *                   compacted in site order.
 *
 * The diagnostics must read the current level of every neighbour and the
 * previous level (the Gauss law needs the neighbours' previous level,
 * evolution.cpp:390-391), so they run as a separate pass before the in-place
 * update of the same TimeStep.
 */
#include <algorithm>

#include "ax_cross.h"
#include "ax_energy.h"
#include "ax_internal.h"
#include "ax_march.h"
#include "ax_wind.h"

namespace ax {

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

/* Block-wide sum of 256 values in a fixed pairing order; valid in thread 0. */
__device__ __forceinline__ double block_sum256(double v, double *sh) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0;
  if (threadIdx.x == 0) r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  return r;
}

template <typename T>
__device__ __forceinline__ void site_energy_ah(const DiagConsts &k, const Levels<T> &L, int i, int j, int kk,
                                               double &rho, double &absG) {
  const int nx = k.nx, ny = k.ny, nz = k.nz;
  auto id = [&](int a, int b, int c) { return (a * ny + b) * nz + c; };
  const int s = id(i, j, kk);
  const int sxp = id(wrapp(i, nx), j, kk), sxm = id(wrapm(i, nx), j, kk);
  const int syp = id(i, wrapp(j, ny), kk), sym = id(i, wrapm(j, ny), kk);
  const int szp = id(i, j, wrapp(kk, nz)), szm = id(i, j, wrapm(kk, nz));
  const double dx = k.dx, dy = k.dy, dz = k.dz, dt = k.dt, g = k.g;
  const double pr = ld(L.cur[0], s), pi = ld(L.cur[1], s);
  const double mag2 = pr * pr + pi * pi;
  double vel[2], gx[2], gy[2], gz[2];
  double sxm_, cxm_, sym_, cym_, szm_, czm_;
  ax_sincos(ld(L.cur[2], sxm), &sxm_, &cxm_);
  ax_sincos(ld(L.cur[3], sym), &sym_, &cym_);
  ax_sincos(ld(L.cur[4], szm), &szm_, &czm_);
  {
    vel[0] = (pr - ld(L.prv[0], s)) / dt;
    gx[0] = (pr - cxm_ * ld(L.cur[0], sxm) + sxm_ * ld(L.cur[1], sxm)) / dx;
    gy[0] = (pr - cym_ * ld(L.cur[0], sym) + sym_ * ld(L.cur[1], sym)) / dy;
    gz[0] = (pr - czm_ * ld(L.cur[0], szm) + szm_ * ld(L.cur[1], szm)) / dz;
    vel[1] = (pi - ld(L.prv[1], s)) / dt;
    gx[1] = (pi - cxm_ * ld(L.cur[1], sxm) + (-sxm_) * ld(L.cur[0], sxm)) / dx;
    gy[1] = (pi - cym_ * ld(L.cur[1], sym) + (-sym_) * ld(L.cur[0], sym)) / dy;
    gz[1] = (pi - czm_ * ld(L.cur[1], szm) + (-szm_) * ld(L.cur[0], szm)) / dz;
  }
  const double X = ld(L.cur[2], s), Y = ld(L.cur[3], s), Z = ld(L.cur[4], s);
  const double pxy = X + ld(L.cur[3], sxp) - ld(L.cur[2], syp) - Y;
  const double pxz = X + ld(L.cur[4], sxp) - ld(L.cur[2], szp) - Z;
  const double pyz = Y + ld(L.cur[4], syp) - ld(L.cur[3], szp) - Z;
  const double oX = ld(L.prv[2], s), oY = ld(L.prv[3], s), oZ = ld(L.prv[4], s);
  double tdc, fcont, G = 0;
  const double vv = mag2 - k.eta * k.eta;
  if (k.energy_form == 0) {
    if (g == 0) {
      tdc = 0;
      fcont = 0;
    } else {
      double divN = (X - ld(L.cur[2], sxm)) / (dx * dx) + (Y - ld(L.cur[3], sym)) / (dy * dy) +
                    (Z - ld(L.cur[4], szm)) / (dz * dz);
      double divP = (oX - ld(L.prv[2], sxm)) / (dx * dx) + (oY - ld(L.prv[3], sym)) / (dy * dy) +
                    (oZ - ld(L.prv[4], szm)) / (dz * dz);
      double divT = (divN - divP) / dt;
      G = divT / g - 2 * g * (pi * vel[0] - pr * vel[1]);
      double ex = (X - oX) / (g * dt * dx), ey = (Y - oY) / (g * dt * dy), ez = (Z - oZ) / (g * dt * dz);
      tdc = 0.5 * (ex * ex + ey * ey + ez * ez);
      double bxy = (1 - ax_cos(pxy)) / ((g * dx * dy) * (g * dx * dy));
      double bxz = (1 - ax_cos(pxz)) / ((g * dx * dz) * (g * dx * dz));
      double byz = (1 - ax_cos(pyz)) / ((g * dy * dz) * (g * dy * dz));
      fcont = bxy + bxz + byz;
    }
    double r = vel[0] * vel[0] + vel[1] * vel[1] + gx[0] * gx[0] + gx[1] * gx[1] + gy[0] * gy[0] +
               gy[1] * gy[1] + gz[0] * gz[0] + gz[1] * gz[1] + tdc + fcont + 0.25 * k.lambda * (vv * vv);
    rho = dx * dy * dz * r;
  } else {
    double ex = (X - oX) / dt, ey = (Y - oY) / dt, ez = (Z - oZ) / dt;
    tdc = 0.5 * (ex * ex + ey * ey + ez * ez);
    double bxy = (1 - ax_cos(pxy)) / ((g * dx * dy) * (g * dx * dy));
    double bxz = (1 - ax_cos(pxz)) / ((g * dx * dz) * (g * dx * dz));
    double byz = (1 - ax_cos(pyz)) / ((g * dy * dz) * (g * dy * dz));
    fcont = bxy + bxz + byz;
    rho = (vel[0] * vel[0] + vel[1] * vel[1] + gx[0] * gx[0] + gx[1] * gx[1] + gy[0] * gy[0] +
           gy[1] * gy[1] + gz[0] * gz[0] + gz[1] * gz[1] + tdc + fcont + 0.25 * k.lambda * (vv * vv)) *
          dx * dy * dz;
  }
  absG = fabs(G);
}

template <typename T>
__device__ __forceinline__ void site_energy_moore(const DiagConsts &k, const Levels<T> &L, int i, int j, int kk,
                                                  double &rho, double &absG) {
  const int nx = k.nx, ny = k.ny, nz = k.nz;
  auto id = [&](int a, int b, int c) { return (a * ny + b) * nz + c; };
  const int s = id(i, j, kk);
  const int sxp = id(wrapp(i, nx), j, kk), sxm = id(wrapm(i, nx), j, kk);
  const int syp = id(i, wrapp(j, ny), kk), sym = id(i, wrapm(j, ny), kk);
  const int szp = id(i, j, wrapp(kk, nz)), szm = id(i, j, wrapm(kk, nz));
  const double dx = k.dx, dy = k.dy, dz = k.dz, dt = k.dt, g = k.g;
  const double q[2] = {k.q1, k.q2};
  double v[2][2], gx[2][2], gy[2][2], gz[2][2], m[2];
  for (int f = 0; f < 2; ++f) {
    const T *re = L.cur[2 * f], *im = L.cur[2 * f + 1];
    const double ar = ld(re, s), ai = ld(im, s);
    m[f] = ar * ar + ai * ai;
    double sxm_, cxm_, sym_, cym_, szm_, czm_;
    ax_sincos(q[f] * ld(L.cur[4], sxm), &sxm_, &cxm_);
    ax_sincos(q[f] * ld(L.cur[5], sym), &sym_, &cym_);
    ax_sincos(q[f] * ld(L.cur[6], szm), &szm_, &czm_);
    gx[f][0] = (ar - cxm_ * ld(re, sxm) + sxm_ * ld(im, sxm)) / dx;
    gy[f][0] = (ar - cym_ * ld(re, sym) + sym_ * ld(im, sym)) / dy;
    gz[f][0] = (ar - czm_ * ld(re, szm) + szm_ * ld(im, szm)) / dz;
    gx[f][1] = (ai - cxm_ * ld(im, sxm) + (-sxm_) * ld(re, sxm)) / dx;
    gy[f][1] = (ai - cym_ * ld(im, sym) + (-sym_) * ld(re, sym)) / dy;
    gz[f][1] = (ai - czm_ * ld(im, szm) + (-szm_) * ld(re, szm)) / dz;
    v[f][0] = (ar - ld(L.prv[2 * f], s)) / dt;
    v[f][1] = (ai - ld(L.prv[2 * f + 1], s)) / dt;
  }
  const double X = ld(L.cur[4], s), Y = ld(L.cur[5], s), Z = ld(L.cur[6], s);
  const double oX = ld(L.prv[4], s), oY = ld(L.prv[5], s), oZ = ld(L.prv[6], s);
  double tdc = 0, fcont = 0, G = 0;
  if (g != 0) {
    double divN = (X - ld(L.cur[4], sxm)) / (dx * dx) + (Y - ld(L.cur[5], sym)) / (dy * dy) +
                  (Z - ld(L.cur[6], szm)) / (dz * dz);
    double divP = (oX - ld(L.prv[4], sxm)) / (dx * dx) + (oY - ld(L.prv[5], sym)) / (dy * dy) +
                  (oZ - ld(L.prv[6], szm)) / (dz * dz);
    double divT = (divN - divP) / dt;
    G = divT / g - 2 * g * (q[0] * (ld(L.cur[1], s) * v[0][0] - ld(L.cur[0], s) * v[0][1]) +
                            q[1] * (ld(L.cur[3], s) * v[1][0] - ld(L.cur[2], s) * v[1][1]));
    double ex = (X - oX) / (g * dt * dx), ey = (Y - oY) / (g * dt * dy), ez = (Z - oZ) / (g * dt * dz);
    tdc = 0.5 * (ex * ex + ey * ey + ez * ez);
    double bxy = (1 - ax_cos(X + ld(L.cur[5], sxp) - ld(L.cur[4], syp) - Y)) / ((g * dx * dy) * (g * dx * dy));
    double bxz = (1 - ax_cos(X + ld(L.cur[6], sxp) - ld(L.cur[4], szp) - Z)) / ((g * dx * dz) * (g * dx * dz));
    double byz = (1 - ax_cos(Y + ld(L.cur[6], syp) - ld(L.cur[5], szp) - Z)) / ((g * dy * dz) * (g * dy * dz));
    fcont = bxy + bxz + byz;
  }
  const double w1 = m[0] - k.eta1 * k.eta1, w2 = m[1] - k.eta2 * k.eta2;
  double r = v[0][0] * v[0][0] + v[0][1] * v[0][1] + gx[0][0] * gx[0][0] + gx[0][1] * gx[0][1] +
             gy[0][0] * gy[0][0] + gy[0][1] * gy[0][1] + gz[0][0] * gz[0][0] + gz[0][1] * gz[0][1] +
             v[1][0] * v[1][0] + v[1][1] * v[1][1] + gx[1][0] * gx[1][0] + gx[1][1] * gx[1][1] +
             gy[1][0] * gy[1][0] + gy[1][1] * gy[1][1] + gz[1][0] * gz[1][0] + gz[1][1] * gz[1][1] + tdc +
             fcont + 0.25 * k.lambda1 * (w1 * w1) + 0.25 * k.lambda2 * (w2 * w2) + 0.5 * k.lambda12 * w1 * w2;
  rho = dx * dy * dz * r;
  absG = k.ex ? fabs(G) / k.inner : fabs(G);
}

/* Sites per thread of the winding pass (each thread takes sites 256 apart,
 * so loads stay coalesced); the energy pass takes one site per thread. */
constexpr int kSitesPerThread = 2;
constexpr int kSitesPerBlock = 256 * kSitesPerThread;
constexpr int kDiagSitesPerThread = 1;
constexpr int kDiagSitesPerBlock = 256 * kDiagSitesPerThread;

/* out: per block [energy, sum|G|, nonfinite count] */
template <typename T, int MODEL>
__global__ void __launch_bounds__(256) diag_kernel(DiagConsts k, Levels<T> L, int V, double *part) {
  __shared__ double sh[4];
  double rho = 0, aG = 0, bad = 0;
  for (int q = 0; q < kDiagSitesPerThread; ++q) {
    const int s = blockIdx.x * kDiagSitesPerBlock + q * 256 + threadIdx.x;
    if (s >= V) break;
    const int kk = s % k.nz, r = s / k.nz, j = r % k.ny, i = r / k.ny;
    const bool inner = !((k.ex && (i == 0 || i == k.nx - 1 || j == 0 || j == k.ny - 1)) ||
                         (k.ez && (kk == 0 || kk == k.nz - 1)));
    if (inner) {
      double r1 = 0, g1 = 0;
      if (MODEL == AX_MODEL_AH)
        site_energy_ah<T>(k, L, i, j, kk, r1, g1);
      else
        site_energy_moore<T>(k, L, i, j, kk, r1, g1);
      rho += r1;
      aG += g1;
    }
    for (int c = 0; c < k.ncomp; ++c) {
      if (!isfinite(ld(L.cur[c], s))) bad += 1;
      if (!isfinite(ld(L.prv[c], s))) bad += 1;
    }
  }
  double e = block_sum256(rho, sh);
  double g = block_sum256(aG, sh);
  double b = block_sum256(bad, sh);
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x] = e;
    part[3 * blockIdx.x + 1] = g;
    part[3 * blockIdx.x + 2] = b;
  }
}

/* One block sums the na triples of a, and a second block the nb of b where
 * there are any: thread t adds triples t, t+1024, ... in order, then a fixed
 * tree; deterministic for a given number.  The results may go straight to
 * pinned host memory. */
__global__ void __launch_bounds__(1024) sum3_kernel(const double *a, int na, double *outa, const double *b, int nb,
                                                    double *outb) {
  __shared__ double sh[3][16];
  const double *part = blockIdx.x ? b : a;
  double *out = blockIdx.x ? outb : outa;
  const int n = blockIdx.x ? nb : na;
  double v[3] = {0, 0, 0};
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += 1024)
    for (int c = 0; c < 3; ++c) v[c] += part[3 * (size_t)i + c];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  for (int c = 0; c < 3; ++c) {
    double x = wave_sum(v[c]);
    if (l == 0) sh[c][w] = x;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double acc = 0;
    for (int q = 0; q < 16; ++q) acc += sh[threadIdx.x][q];
    out[threadIdx.x] = acc;
  }
}

/* ------------------------------- winding -------------------------------- */
template <typename T>
__global__ void __launch_bounds__(256) winding_kernel(int nx, int ny, int nz, const T *fr, const T *fi,
                                                      const T *tx, const T *ty, const T *tz, double q,
                                                      int ex, int ez, int8_t *out, double *part) {
  __shared__ double sh[4];
  const int V = nx * ny * nz;
  double tot[3] = {0, 0, 0};
  for (int qq = 0; qq < kSitesPerThread; ++qq) {
    const int s = blockIdx.x * kSitesPerBlock + qq * 256 + threadIdx.x;
    if (s >= V) break;
    const int kk = s % nz, r = s / nz, j = r % ny, i = r / ny;
    int w[3];
    site_winding<T>(nx, ny, nz, fr, fi, tx, ty, tz, q, i, j, kk, w);
    /* plaquettes that would wrap across a non-periodic axis do not exist */
    const bool xe = ex && i == nx - 1, ye = ex && j == ny - 1, ze = ez && kk == nz - 1;
    if (xe || ye) w[0] = 0;
    if (xe || ze) w[1] = 0;
    if (ye || ze) w[2] = 0;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      out[(size_t)pl * V + s] = (int8_t)w[pl];
      tot[pl] += (double)(w[pl] < 0 ? -w[pl] : w[pl]);
    }
  }
  double a = block_sum256(tot[0], sh);
  double b = block_sum256(tot[1], sh);
  double c = block_sum256(tot[2], sh);
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x] = a;
    part[3 * blockIdx.x + 1] = b;
    part[3 * blockIdx.x + 2] = c;
  }
}


/* ------------------------------ crossings -------------------------------
 * The face equations of mpi_evolution.cpp:552-623 cost some 280 instructions
 * with six divisions and a root in FP64, for three faces a site.  Most faces
 * are settled without them: face_class solves the face in FP32 in its own
 * coordinates, with a bound on how far that may lie from the FP64 solution,
 * and tells how many roots FP64 finds or that it cannot tell.  A wave takes
 * a group of consecutive sites; what needs FP64 (the count: the undecided
 * faces; the points: every face with a root) goes through a queue in LDS, in
 * site and face order, and is solved 64 at a time with every lane at work.
 * The points of a round are put in order with two ballots and stored through
 * LDS as one contiguous run.  Two launches (counts, then points at their
 * offsets) with a scan in between.  512^3 FP64, 1.2 points a site: counts
 * 2.67 -> 1.56 ms, scan 0.92 -> 0.15, points 6.96 -> 2.94 (3.9 GB written);
 * FP32 2.63 -> 1.45, 0.92 -> 0.15, 6.29 -> 2.72; with the faces handed on as
 * masks the whole call 4.65 -> 3.88, FP32 4.15 -> 3.27 (301^3 FP64 0.98 ->
 * 0.81, 101^3 78 -> 69 us).  Faces of zeros and NaNs, which the equations leave
 * at once, are not queued either (a field of zeros, 128^3 FP64: 114 us a call
 * when they were, 53 now, 57 for the equations alone); that check costs other
 * fields 1 to 2 %.  Bound by instructions. */

struct CrossGeom {
  int nx, ny, nz, ex, ez, x0, y0, z0;
  uint32_t V, sites, groups, per;   /* sites; sites of a group (a multiple of 64); groups; groups per XCD */
  FastDiv by_nz, by_ny;
  double dx, dy, dz;
  float k;                          /* face_class's relative error bound; >= 1: solve every face in FP64 */
};

/* WRITE: the points of each group from its offset on; else its count.
 * masks: three words per 64 sites, the lanes whose xy, xz, yz face is not
 * known to hold no point.  The count pass stores them and the point pass
 * (MASKED) takes its faces from them instead of reading and classifying
 * every face again; without the memory for them it classifies. */
template <typename T, bool WRITE, bool MASKED>
__global__ void __launch_bounds__(64) cross_kernel(CrossGeom g, const T *__restrict__ fr, const T *__restrict__ fi,
                                                   int *__restrict__ count, const long long *__restrict__ offset,
                                                   double *__restrict__ xyz, long long cap, uint64_t *masks) {
  /* consecutive groups on one XCD, so that rows y + 1 are read from its L2 */
  const uint32_t grp = (blockIdx.x & 7) * g.per + (blockIdx.x >> 3);
  if (grp >= g.groups) return;
  /* queue: site in the group, face; at most 63 left over + 192 of a chunk */
  __shared__ uint16_t queue[256];
  __shared__ double stage[WRITE ? 384 : 1];
  const int lane = (int)threadIdx.x;
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  const uint32_t base = grp * g.sites;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  auto id = [&](int i, int j, int k) { return (uint32_t)((i * ny + j) * nz + k); };
  uint32_t head = 0, tail = 0;   /* of the queue (mod 256) */
  long long out = WRITE ? offset[grp] : 0;
  int own = 0;                   /* roots counted by this lane */

  auto solve = [&](uint32_t n) {
    int m = 0;
    double r1 = 0, r2 = 0, q1 = 0, q2 = 0, third = 0;
    int face = 0;
    if ((uint32_t)lane < n) {
      const uint32_t e = queue[(head + lane) & 255];
      face = (int)(e & 3);
      const uint32_t s = base + (e >> 2);
      const uint32_t r = quotient(s, g.by_nz), i = quotient(r, g.by_ny);
      const int k = (int)(s - r * nz), j = (int)(r - i * ny);
      const int ip = wrapp((int)i, nx), jp = wrapp(j, ny), kp = wrapp(k, nz);
      /* the face spans axes a < b: xy, xz, yz */
      const int ia = face == 2 ? (int)i : ip, ja = face == 2 ? jp : j;
      const int jb = face == 0 ? jp : j, kb = face == 0 ? k : kp;
      const uint32_t sa = id(ia, ja, k), sb = id((int)i, jb, kb), sab = id(ia, face == 1 ? j : jp, kb);
      const double x = ((int)i - g.x0) * g.dx, y = (j - g.y0) * g.dy, z = (k - g.z0) * g.dz;
      const double v[2] = {ld(fr, s), ld(fi, s)}, va[2] = {ld(fr, sa), ld(fi, sa)};
      const double vb[2] = {ld(fr, sb), ld(fi, sb)}, vab[2] = {ld(fr, sab), ld(fi, sab)};
      third = face == 0 ? z : face == 1 ? y : x;
      m = face_roots(v, va, vb, vab, face == 2 ? y : x, face == 2 ? g.dy : g.dx, face == 0 ? y : z,
                     face == 0 ? g.dy : g.dz, r1, r2, q1, q2);
    }
    const uint64_t one = __builtin_amdgcn_ballot_w64(m >= 1), two = __builtin_amdgcn_ballot_w64(m == 2);
    const int tot = __popcll(one) + __popcll(two);
    if (WRITE && tot) {
      auto put = [&](int at, double s1, double s2) {
        stage[3 * at] = face == 2 ? third : s1;
        stage[3 * at + 1] = face == 0 ? s2 : face == 1 ? third : s1;
        stage[3 * at + 2] = face == 0 ? third : s2;
      };
      const int at = __popcll(one & below) + __popcll(two & below);
      if (m >= 1) put(at, r1, r2);
      if (m == 2) put(at + 1, q1, q2);
      __syncthreads();
      /* beyond the caller's capacity only the count goes on */
      const int fit = (int)min((long long)tot, max(cap - out, 0ll));
      for (int d = lane; d < 3 * fit; d += 64) xyz[3 * out + d] = stage[d];
      __syncthreads();
    }
    out += tot;
    head += n;
  };

  /* Re phi or Im phi zero on the corners of a face of site s.  (s opaque: its
   * addresses are formed again rather than held in registers for this.) */
  auto zero_face = [&](uint32_t s, int f) {
    asm("" : "+v"(s));
    const uint32_t r = quotient(s, g.by_nz), i = quotient(r, g.by_ny);
    const int k = (int)(s - r * nz), j = (int)(r - i * ny);
    const int ia = f == 2 ? (int)i : wrapp((int)i, nx), ja = f == 2 ? wrapp(j, ny) : j;
    const int jb = f == 0 ? wrapp(j, ny) : j, kb = f == 0 ? k : wrapp(k, nz);
    const uint32_t at[4] = {s, id(ia, ja, k), id((int)i, jb, kb), id(ia, f == 1 ? j : wrapp(j, ny), kb)};
    auto zero = [&](const T *p) { return p[at[0]] == 0 && p[at[1]] == 0 && p[at[2]] == 0 && p[at[3]] == 0; };
    return zero(fr) || zero(fi);
  };

  for (uint32_t c = 0; c < g.sites; c += 64) {
    if (base + c >= g.V) break;
    uint64_t mask[3];   /* lanes whose xy, xz, yz face goes to the queue */
    if constexpr (MASKED && WRITE) {
#pragma unroll
      for (int f = 0; f < 3; ++f) mask[f] = masks[3 * (size_t)((base + c) >> 6) + f];
    } else {
      const uint32_t s = min(base + c + lane, g.V - 1);
      const uint32_t r = quotient(s, g.by_nz), i = quotient(r, g.by_ny);
      const int k = (int)(s - r * nz), j = (int)(r - i * ny);
      /* only the sites the bulk update covers (evolution.cpp:731-743) */
      const bool bulk = base + c + lane < g.V &&
                        !((g.ex && ((int)i == 0 || (int)i == nx - 1 || j == 0 || j == ny - 1)) ||
                          (g.ez && (k == 0 || k == nz - 1)));
      const int ip = wrapp((int)i, nx), jp = wrapp(j, ny), kp = wrapp(k, nz);
      const uint32_t at7[7] = {s, id(ip, j, k), id((int)i, jp, k), id((int)i, j, kp), id(ip, jp, k), id(ip, j, kp),
                               id((int)i, jp, kp)};
      float re[7], im[7];
#pragma unroll
      for (int q = 0; q < 7; ++q) re[q] = (float)fr[at7[q]];
#pragma unroll
      for (int q = 0; q < 7; ++q) im[q] = (float)fi[at7[q]];
      uint64_t some[3];
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        const int a = f == 2 ? 2 : 1, b = f == 0 ? 2 : 3, ab = 4 + f;
        int n = 0;
        const bool open = bulk && !one_sign(re[0], re[a], re[b], re[ab], g.k);
        if (__builtin_amdgcn_ballot_w64(open) && open)
          n = face_class(re[0], re[a], re[b], re[ab], im[0], im[a], im[b], im[ab], g.k);
        if (n == 4) n = zero_face(base + c + lane, f) ? 0 : 3;   /* zero in FP32: exactly zero? */
        if (!WRITE) own += n == 3 ? 0 : n;
        some[f] = __builtin_amdgcn_ballot_w64(n != 0);
        mask[f] = WRITE ? some[f] : __builtin_amdgcn_ballot_w64(n == 3);
      }
      if (MASKED && lane < 3)
        masks[3 * (size_t)((base + c) >> 6) + lane] = lane == 0 ? some[0] : lane == 1 ? some[1] : some[2];
    }
    uint32_t at = tail;
#pragma unroll
    for (int f = 0; f < 3; ++f) at += __popcll(mask[f] & below);
#pragma unroll
    for (int f = 0; f < 3; ++f)
      if ((mask[f] >> lane) & 1) queue[at++ & 255] = (uint16_t)((c + lane) << 2 | f);
#pragma unroll
    for (int f = 0; f < 3; ++f) tail += __popcll(mask[f]);
    __syncthreads();
    while (tail - head >= 64) solve(64);
  }
  if (tail != head) solve(tail - head);
  if (!WRITE) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) own += __shfl_xor(own, off, 64);
    if (lane == 0) count[grp] = own + (int)out;
  }
}

/* Exclusive scan of n counts by one workgroup, 8192 a round, the next
 * round's counts loaded ahead (262 144 counts, 512^3: 0.15 ms; one count at a
 * time per thread it was 0.92 ms). */
__global__ void __launch_bounds__(1024) scan_kernel(const int *__restrict__ in, long long *__restrict__ out, int n,
                                                    long long *total) {
  __shared__ int sums[16];
  const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
  auto load = [&](int b, int v[8]) {
    const int i = b + 8 * t;
    if (i + 8 <= n) {
      const int4 lo = *(const int4 *)(in + i), hi = *(const int4 *)(in + i + 4);
      v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
      v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = i + q < n ? in[i + q] : 0;
    }
  };
  int v[8], next[8];
  load(0, v);
  long long carry = 0;
  for (int b = 0; b < n; b += 8192) {
    if (b + 8192 < n) load(b + 8192, next);
    int own = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) own += v[q];
    int inc = own;   /* a round's counts sum to below 2^25 */
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(inc, off, 64);
      if (lane >= off) inc += o;
    }
    if (lane == 63) sums[w] = inc;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      if (q < w) before += sums[q];
      all += sums[q];
    }
    long long run = carry + before + inc - own;
    const int i = b + 8 * t;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      if (i + q < n) out[i + q] = run;
      run += v[q];
    }
    carry += all;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = next[q];
  }
  if (t == 0) *total = carry;
}

/* ------------------- marching diagnostics (Abelian-Higgs) -----------------
 * One 64-lane wave per (chunk of 64 sites of a plane, x segment) marching along x,
 * as the step kernel.  Per site it evaluates the energy density and Gauss
 * residual with the expressions of site_energy_ah (the same per-site bits;
 * with x/y or z not periodic only the bulk region's terms are summed, as
 * diag_kernel does),
 * carrying the x-backward field, link and link trig from the previous
 * plane, and, with PH, the three forward edge phases
 *   delta_a(s) = arg( conj(phi(s)) exp(-i theta_a(s)) phi(s+a) )
 * from the same link sincos, stored as the FP32 edge values
 * e_a(s) = delta_a(s) + theta_a(s) that wind_march_kernel combines
 * (ax_wind.h).  The winding of a plaquette needs four edges of three
 * sites; computing each edge once here instead of nine per site in
 * winding_kernel is the saving. */

/* link_phase_sc (ax_energy.h): link_phase with the link's sin/cos already at hand */

/* P2: dx, dy, dz and g (when g != 0) are powers of two, so every division by
 * dx, dx*dx, g or (g*dx*dy)^2 is the multiplication by its exact reciprocal
 * (the same correctly rounded value).  Divisions by dt stay divisions.
 * FP64 is held to 3 waves per SIMD (the phase-storing variant needs 173
 * VGPRs otherwise, i.e. 2 waves; capped it spills 4 and runs 3.5 % faster
 * per 512^3 call); FP32 keeps the compiler's choice (already 3 waves; the
 * same cap there changed its schedule and cost 36 %). */
template <typename T, bool PH, bool P2>
__global__ void __launch_bounds__(64, sizeof(T) == 8 ? 3 : 1) diag_march_kernel(DiagConsts k, Levels<T> L, TileGrid g, float *phase,
                                                        double *part) {
  const int w = (int)blockIdx.x;
  const int lane = (int)(threadIdx.x & 63);
  int chunk, seg;
  if (!tile_item(g, w, chunk, seg)) {
    if (lane < 3) part[3 * (size_t)w + lane] = 0;
    return;
  }
  const int x0 = seg * g.xseg, x1 = min(k.nx, x0 + g.xseg);
  const int NX = k.nx, NY = k.ny, NZ = k.nz;
  const LaneSite<true> ls(NY, NZ, (uint32_t)chunk * 64);
  const bool act = ls.act;
  const bool in_yz = !(k.ex && (ls.y == 0 || ls.y == NY - 1)) && !(k.ez && (ls.z == 0 || ls.z == NZ - 1));
  const uint32_t E = (uint32_t)sizeof(T);
  /* byte offsets in a plane of the site and of y+-1, z+-1 (in the lane for
   * every nz: with scalar row offsets the march holds more registers) */
  const uint32_t o0 = ls.col(0, 0, E), oyp = ls.col(1, 0, E), oym = ls.col(-1, 0, E);
  const uint32_t ozp = ls.col(0, 1, E), ozm = ls.col(0, -1, E);
  const T *PR = L.cur[0], *PI = L.cur[1], *TX = L.cur[2], *TY = L.cur[3], *TZ = L.cur[4];
  const T *OPR = L.prv[0], *OPI = L.prv[1], *OTX = L.prv[2], *OTY = L.prv[3], *OTZ = L.prv[4];
  /* value of field b in x plane x at offsets in it: the plane's 64-bit
   * address is formed on the scalar unit, so planes of any size work */
  const size_t NYNZ = (size_t)NY * NZ;
  auto ld_ = [NYNZ](const T *b, int x, uint32_t o) { return (double)ldo(b + (size_t)x * NYNZ, 0u, o); };
  const double dx = k.dx, dy = k.dy, dz = k.dz, dt = k.dt, gg = k.g;
  const size_t V = (size_t)NX * NY * NZ;
  const double dxx = dx * dx, dyy = dy * dy, dzz = dz * dz;
  const double bxyd = (gg * dx * dy) * (gg * dx * dy), bxzd = (gg * dx * dz) * (gg * dx * dz),
               byzd = (gg * dy * dz) * (gg * dy * dz);
  const double idx = 1 / dx, idy = 1 / dy, idz = 1 / dz, idxx = 1 / dxx, idyy = 1 / dyy, idzz = 1 / dzz;
  const double igg = 1 / gg, ibxy = 1 / bxyd, ibxz = 1 / bxzd, ibyz = 1 / byzd;
  auto dv = [](double a, double d, double inv) { return P2 ? a * inv : a / d; };
  /* divisions by dt and g dt dx_a as multiplications by the reciprocal: the
   * per-site terms change by at most an ulp, far inside the 1e-12 the sums
   * are held to (the site kernels divide).  Not in the FP64 pass that also
   * stores the edge phases, where the extra live reciprocals cost more
   * spills than the divisions (512^3: 6.50 -> 6.79 ms with them; FP32
   * 5.30 -> 5.01 ms, FP64 without phases 2.67 -> 2.51 ms) */
  constexpr bool RECIP = !(PH && sizeof(T) == 8);
  const double idt = 1 / dt;
  const double iedx = 1 / (gg * dt * dx), iedy = 1 / (gg * dt * dy), iedz = 1 / (gg * dt * dz);
  auto by_dt = [&](double a) { return RECIP ? a * idt : a / dt; };
  auto by_e = [&](double a, double d, double inv) { return RECIP ? a * inv : a / (gg * dt * d); };

  /* carried from plane x-1: phi, theta_x (both levels), sin/cos theta_x */
  const int xm0 = x0 == 0 ? NX - 1 : x0 - 1;
  double PRm = ld_(PR, xm0, o0), PIm = ld_(PI, xm0, o0);
  double TXm = ld_(TX, xm0, o0), oXm = ld_(OTX, xm0, o0);
  double sxm, cxm;
  ax_sincos(TXm, &sxm, &cxm);
  double PRc = ld_(PR, x0, o0), PIc = ld_(PI, x0, o0);
  double X = ld_(TX, x0, o0), Y = ld_(TY, x0, o0), Z = ld_(TZ, x0, o0);
  double rho_sum = 0, g_sum = 0;
  int bad = 0;

  for (int x = x0; x < x1; ++x) {
    const int xp = x == NX - 1 ? 0 : x + 1;
    const double PRn = ld_(PR, xp, o0), PIn = ld_(PI, xp, o0);
    const double TXn = ld_(TX, xp, o0), TYn = ld_(TY, xp, o0), TZn = ld_(TZ, xp, o0);
    const double oPR = ld_(OPR, x, o0), oPI = ld_(OPI, x, o0);
    const double oX = ld_(OTX, x, o0), oY = ld_(OTY, x, o0), oZ = ld_(OTZ, x, o0);
    const double PRyp = ld_(PR, x, oyp), PIyp = ld_(PI, x, oyp);
    const double TXyp = ld_(TX, x, oyp), TZyp = ld_(TZ, x, oyp);
    const double PRzp = ld_(PR, x, ozp), PIzp = ld_(PI, x, ozp);
    const double TXzp = ld_(TX, x, ozp), TYzp = ld_(TY, x, ozp);
    const double PRym = ld_(PR, x, oym), PIym = ld_(PI, x, oym);
    const double TYym = ld_(TY, x, oym), oYym = ld_(OTY, x, oym);
    const double PRzm = ld_(PR, x, ozm), PIzm = ld_(PI, x, ozm);
    const double TZzm = ld_(TZ, x, ozm), oZzm = ld_(OTZ, x, ozm);

    /* site_energy_ah at s, operands by name */
    const double pr = PRc, pi = PIc;
    const double mag2 = pr * pr + pi * pi;
    double sym_, cym_, szm_, czm_;
    ax_sincos(TYym, &sym_, &cym_);
    ax_sincos(TZzm, &szm_, &czm_);
    double vel[2], gx[2], gy[2], gz[2];
    vel[0] = by_dt(pr - oPR);
    gx[0] = dv(pr - cxm * PRm + sxm * PIm, dx, idx);
    gy[0] = dv(pr - cym_ * PRym + sym_ * PIym, dy, idy);
    gz[0] = dv(pr - czm_ * PRzm + szm_ * PIzm, dz, idz);
    vel[1] = by_dt(pi - oPI);
    gx[1] = dv(pi - cxm * PIm + (-sxm) * PRm, dx, idx);
    gy[1] = dv(pi - cym_ * PIym + (-sym_) * PRym, dy, idy);
    gz[1] = dv(pi - czm_ * PIzm + (-szm_) * PRzm, dz, idz);
    const double pxy = X + TYn - TXyp - Y;
    const double pxz = X + TZn - TXzp - Z;
    const double pyz = Y + TZyp - TYzp - Z;
    /* cosines of the three plaquette angles; the short k = 0 form when every
     * lane's angles qualify (bit-identical to ax_cos there) */
    auto plaq_cos = [&](double &cxy, double &cxz, double &cyz) {
      if (__all(ax_sin_is_small(pxy) && ax_sin_is_small(pxz) && ax_sin_is_small(pyz))) {
        cxy = ax_cos_kernel(pxy, 0.0); cxz = ax_cos_kernel(pxz, 0.0); cyz = ax_cos_kernel(pyz, 0.0);
      } else {
        cxy = ax_cos(pxy); cxz = ax_cos(pxz); cyz = ax_cos(pyz);
      }
    };
    double tdc, fcont, G = 0, rho;
    const double vv = mag2 - k.eta * k.eta;
    if (k.energy_form == 0) {
      if (gg == 0) {
        tdc = 0;
        fcont = 0;
      } else {
        double divN = dv(X - TXm, dxx, idxx) + dv(Y - TYym, dyy, idyy) + dv(Z - TZzm, dzz, idzz);
        double divP = dv(oX - oXm, dxx, idxx) + dv(oY - oYym, dyy, idyy) + dv(oZ - oZzm, dzz, idzz);
        double divT = by_dt(divN - divP);
        G = dv(divT, gg, igg) - 2 * gg * (pi * vel[0] - pr * vel[1]);
        double ex = by_e(X - oX, dx, iedx), ey = by_e(Y - oY, dy, iedy), ez = by_e(Z - oZ, dz, iedz);
        tdc = 0.5 * (ex * ex + ey * ey + ez * ez);
        double cxy, cxz, cyz;
        plaq_cos(cxy, cxz, cyz);
        double bxy = dv(1 - cxy, bxyd, ibxy);
        double bxz = dv(1 - cxz, bxzd, ibxz);
        double byz = dv(1 - cyz, byzd, ibyz);
        fcont = bxy + bxz + byz;
      }
      double r_ = vel[0] * vel[0] + vel[1] * vel[1] + gx[0] * gx[0] + gx[1] * gx[1] + gy[0] * gy[0] +
                  gy[1] * gy[1] + gz[0] * gz[0] + gz[1] * gz[1] + tdc + fcont + 0.25 * k.lambda * (vv * vv);
      rho = dx * dy * dz * r_;
    } else {
      double ex = by_dt(X - oX), ey = by_dt(Y - oY), ez = by_dt(Z - oZ);
      tdc = 0.5 * (ex * ex + ey * ey + ez * ez);
      double cxy, cxz, cyz;
      plaq_cos(cxy, cxz, cyz);
      double bxy = dv(1 - cxy, bxyd, ibxy);
      double bxz = dv(1 - cxz, bxzd, ibxz);
      double byz = dv(1 - cyz, byzd, ibyz);
      fcont = bxy + bxz + byz;
      rho = (vel[0] * vel[0] + vel[1] * vel[1] + gx[0] * gx[0] + gx[1] * gx[1] + gy[0] * gy[0] +
             gy[1] * gy[1] + gz[0] * gz[0] + gz[1] * gz[1] + tdc + fcont + 0.25 * k.lambda * (vv * vv)) *
            dx * dy * dz;
    }
    double sx, cx;
    ax_sincos(X, &sx, &cx);
    if (PH) {
      double sy, cy, sz, cz;
      ax_sincos(Y, &sy, &cy);
      ax_sincos(Z, &sz, &cz);
      const double dX = link_phase_sc(pr, pi, PRn, PIn, sx, cx);
      const double dY = link_phase_sc(pr, pi, PRyp, PIyp, sy, cy);
      const double dZ = link_phase_sc(pr, pi, PRzp, PIzp, sz, cz);
      if (act) {
        /* edge values e_a(s) (ax_wind.h) */
        float *e = phase + (size_t)x * NYNZ;
        sto(e, 0u, ls.p * 4u, (float)(dX + X));
        sto(e + V, 0u, ls.p * 4u, (float)(dY + Y));
        sto(e + 2 * V, 0u, ls.p * 4u, (float)(dZ + Z));
      }
    }
    if (act) {
      /* energy and Gauss over the bulk region only when x/y or z are not
       * periodic (the boundary sites' terms, computed from wrapped
       * neighbours, are dropped), finiteness over every site -- as
       * diag_kernel */
      if (in_yz && !(k.ex && (x == 0 || x == NX - 1))) {
        rho_sum += rho;
        g_sum += fabs(G);
      }
    }
    const double vals[10] = {PRc, PIc, X, Y, Z, oPR, oPI, oX, oY, oZ};
    bad += nonfinite(vals, act);
    PRm = PRc; PIm = PIc; TXm = X; oXm = oX; sxm = sx; cxm = cx;
    PRc = PRn; PIc = PIn; X = TXn; Y = TYn; Z = TZn;
  }
  const double a = wave_sum(rho_sum), bsum = wave_sum(g_sum), c = (double)bad;
  if (lane == 0) {
    part[3 * w] = a;
    part[3 * w + 1] = bsum;
    part[3 * w + 2] = c;
  }
}

/* Windings of the current level from the edge values the marching
 * diagnostics stored (wind_march, ax_wind.h): one wave per work item of
 * the tile grid, carrying plane x+1's values.  out (the winding field
 * [3][V]) may be null when only the counts are wanted.  An edge value above
 * lim (kEdgeExact, or infinity) turns the counts into a NaN. */
__global__ void __launch_bounds__(64) wind_march_kernel(int nx, int ny, int nz, const float *E, TileGrid g, int ex,
                                                        int ez, double lim, int8_t *out, double *part) {
  const int item = (int)blockIdx.x;
  int chunk, seg;
  if (!tile_item(g, item, chunk, seg)) {
    if (threadIdx.x < 3) part[3 * (size_t)item + threadIdx.x] = 0;
    return;
  }
  const int x0 = seg * g.xseg, x1 = min(nx, x0 + g.xseg);
  const WindRow w(nx, ny, nz, chunk);
  double tot[3] = {0, 0, 0};
  /* plaquettes that would wrap across a non-periodic axis do not exist */
  const bool ye = ex && w.y == ny - 1, ze = ez && w.z == nz - 1;
  const double big = wind_march(w, E, x0, x1, [&](int x, size_t s, const int *wn) {
    const bool xe = ex && x == nx - 1;
    const bool none[3] = {xe || ye, xe || ze, ye || ze};
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      const int v = none[pl] ? 0 : wn[pl];
      if (out) out[(size_t)pl * w.V + s] = (int8_t)v;
      tot[pl] += (double)(v < 0 ? -v : v);
    }
  });
  if (big > lim) tot[0] = NAN;
  const double a = wave_sum(tot[0]), b = wave_sum(tot[1]), c = wave_sum(tot[2]);
  if ((threadIdx.x & 63) == 0) {
    part[3 * item] = a;
    part[3 * item + 1] = b;
    part[3 * item + 2] = c;
  }
}

/* ------------------ marching diagnostics (Moore model) -------------------
 * Energy density and Gauss residual of site_energy_moore (the same
 * expressions in the same order, so the same per-site terms) by one wave
 * per (chunk of 64 sites of a plane, x segment) marching along x: both scalars and
 * theta_x (both levels) of plane x-1 are carried from the previous plane,
 * and plane x+1's current level is loaded once, as the next plane's centre.
 * The site kernel reads the x-neighbour planes, which another pass over the
 * lattice had fetched, a second time.  Sums over the bulk region where x/y
 * or z are not periodic, finiteness over the fourteen stored values of
 * every site, as diag_kernel.  FP64 is held to 3 waves per SIMD (222 VGPRs
 * otherwise; 2 spilled with the cap): 256^3 0.83 -> 0.72 ms per call. */
template <typename T>
__global__ void __launch_bounds__(64, sizeof(T) == 8 ? 3 : 1) moore_diag_march_kernel(DiagConsts k, Levels<T> L,
                                                                                   TileGrid g, double *part) {
  const int w = (int)blockIdx.x;
  const int lane = (int)(threadIdx.x & 63);
  int chunk, seg;
  if (!tile_item(g, w, chunk, seg)) {
    if (lane < 3) part[3 * (size_t)w + lane] = 0;
    return;
  }
  const int x0 = seg * g.xseg, x1 = min(k.nx, x0 + g.xseg);
  const int NX = k.nx, NY = k.ny, NZ = k.nz;
  const LaneSite<true> ls(NY, NZ, (uint32_t)chunk * 64);
  const bool act = ls.act;
  const bool in_yz = !(k.ex && (ls.y == 0 || ls.y == NY - 1)) && !(k.ez && (ls.z == 0 || ls.z == NZ - 1));
  const uint32_t E = (uint32_t)sizeof(T);
  /* byte offsets in a plane of the site and of y+-1, z+-1 (in the lane for
   * every nz: with scalar row offsets the march spills more) */
  const uint32_t o0 = ls.col(0, 0, E), oyp = ls.col(1, 0, E), oym = ls.col(-1, 0, E);
  const uint32_t ozp = ls.col(0, 1, E), ozm = ls.col(0, -1, E);
  const size_t NYNZ = (size_t)NY * NZ;
  auto C = [&](int c, int x, uint32_t o) { return (double)ldo(L.cur[c] + (size_t)x * NYNZ, 0u, o); };
  auto P = [&](int c, int x, uint32_t o) { return (double)ldo(L.prv[c] + (size_t)x * NYNZ, 0u, o); };
  const double dx = k.dx, dy = k.dy, dz = k.dz, dt = k.dt, gg = k.g;
  const double q[2] = {k.q1, k.q2};
  /* plane x-1 (carried): both scalars, theta_x of both levels; plane x */
  const int xm0 = x0 == 0 ? NX - 1 : x0 - 1;
  double Fm[4], TXm = C(4, xm0, o0), oXm = P(4, xm0, o0), Fc[4], Tc[3];
  for (int c = 0; c < 4; ++c) {
    Fm[c] = C(c, xm0, o0);
    Fc[c] = C(c, x0, o0);
  }
  for (int a = 0; a < 3; ++a) Tc[a] = C(4 + a, x0, o0);
  double rho_sum = 0, g_sum = 0;
  int bad = 0;
  for (int x = x0; x < x1; ++x) {
    const int xp = x == NX - 1 ? 0 : x + 1;
    double Fn[4], Tn[3], Fo[4], Fy[4], Fz[4];
    for (int c = 0; c < 4; ++c) {
      Fn[c] = C(c, xp, o0);
      Fo[c] = P(c, x, o0);
      Fy[c] = C(c, x, oym);
      Fz[c] = C(c, x, ozm);
    }
    for (int a = 0; a < 3; ++a) Tn[a] = C(4 + a, xp, o0);
    const double oX = P(4, x, o0), oY = P(5, x, o0), oZ = P(6, x, o0);
    const double TYym = C(5, x, oym), oYym = P(5, x, oym);
    const double TZzm = C(6, x, ozm), oZzm = P(6, x, ozm);
    const double TXyp = C(4, x, oyp), TZyp = C(6, x, oyp);
    const double TXzp = C(4, x, ozp), TYzp = C(5, x, ozp);
    const double X = Tc[0], Y = Tc[1], Z = Tc[2];

    /* site_energy_moore at s, operands by name */
    double v[2][2], gx[2][2], gy[2][2], gz[2][2], m[2];
    for (int f = 0; f < 2; ++f) {
      const double ar = Fc[2 * f], ai = Fc[2 * f + 1];
      m[f] = ar * ar + ai * ai;
      double sxm_, cxm_, sym_, cym_, szm_, czm_;
      ax_sincos(q[f] * TXm, &sxm_, &cxm_);
      ax_sincos(q[f] * TYym, &sym_, &cym_);
      ax_sincos(q[f] * TZzm, &szm_, &czm_);
      const double rxm = Fm[2 * f], ixm = Fm[2 * f + 1], rym = Fy[2 * f], iym = Fy[2 * f + 1];
      const double rzm = Fz[2 * f], izm = Fz[2 * f + 1];
      gx[f][0] = (ar - cxm_ * rxm + sxm_ * ixm) / dx;
      gy[f][0] = (ar - cym_ * rym + sym_ * iym) / dy;
      gz[f][0] = (ar - czm_ * rzm + szm_ * izm) / dz;
      gx[f][1] = (ai - cxm_ * ixm + (-sxm_) * rxm) / dx;
      gy[f][1] = (ai - cym_ * iym + (-sym_) * rym) / dy;
      gz[f][1] = (ai - czm_ * izm + (-szm_) * rzm) / dz;
      v[f][0] = (ar - Fo[2 * f]) / dt;
      v[f][1] = (ai - Fo[2 * f + 1]) / dt;
    }
    double tdc = 0, fcont = 0, G = 0;
    if (gg != 0) {
      double divN = (X - TXm) / (dx * dx) + (Y - TYym) / (dy * dy) + (Z - TZzm) / (dz * dz);
      double divP = (oX - oXm) / (dx * dx) + (oY - oYym) / (dy * dy) + (oZ - oZzm) / (dz * dz);
      double divT = (divN - divP) / dt;
      G = divT / gg - 2 * gg * (q[0] * (Fc[1] * v[0][0] - Fc[0] * v[0][1]) +
                                q[1] * (Fc[3] * v[1][0] - Fc[2] * v[1][1]));
      double ex = (X - oX) / (gg * dt * dx), ey = (Y - oY) / (gg * dt * dy), ez = (Z - oZ) / (gg * dt * dz);
      tdc = 0.5 * (ex * ex + ey * ey + ez * ez);
      double bxy = (1 - ax_cos(X + Tn[1] - TXyp - Y)) / ((gg * dx * dy) * (gg * dx * dy));
      double bxz = (1 - ax_cos(X + Tn[2] - TXzp - Z)) / ((gg * dx * dz) * (gg * dx * dz));
      double byz = (1 - ax_cos(Y + TZyp - TYzp - Z)) / ((gg * dy * dz) * (gg * dy * dz));
      fcont = bxy + bxz + byz;
    }
    const double w1 = m[0] - k.eta1 * k.eta1, w2 = m[1] - k.eta2 * k.eta2;
    double r = v[0][0] * v[0][0] + v[0][1] * v[0][1] + gx[0][0] * gx[0][0] + gx[0][1] * gx[0][1] +
               gy[0][0] * gy[0][0] + gy[0][1] * gy[0][1] + gz[0][0] * gz[0][0] + gz[0][1] * gz[0][1] +
               v[1][0] * v[1][0] + v[1][1] * v[1][1] + gx[1][0] * gx[1][0] + gx[1][1] * gx[1][1] +
               gy[1][0] * gy[1][0] + gy[1][1] * gy[1][1] + gz[1][0] * gz[1][0] + gz[1][1] * gz[1][1] + tdc +
               fcont + 0.25 * k.lambda1 * (w1 * w1) + 0.25 * k.lambda2 * (w2 * w2) + 0.5 * k.lambda12 * w1 * w2;
    const double rho = dx * dy * dz * r;
    const double absG = k.ex ? fabs(G) / k.inner : fabs(G);
    if (act) {
      if (in_yz && !(k.ex && (x == 0 || x == NX - 1))) {
        rho_sum += rho;
        g_sum += absG;
      }
    }
    const double vals[14] = {Fc[0], Fc[1], Fc[2], Fc[3], X, Y, Z, Fo[0], Fo[1], Fo[2], Fo[3], oX, oY, oZ};
    bad += nonfinite(vals, act);
    for (int c = 0; c < 4; ++c) {
      Fm[c] = Fc[c];
      Fc[c] = Fn[c];
    }
    TXm = X;
    oXm = oX;
    for (int a = 0; a < 3; ++a) Tc[a] = Tn[a];
  }
  const double a = wave_sum(rho_sum), b = wave_sum(g_sum), c = (double)bad;
  if (lane == 0) {
    part[3 * w] = a;
    part[3 * w + 1] = b;
    part[3 * w + 2] = c;
  }
}

/* ------------------------------ launchers ------------------------------- */
template <typename T>
hipError_t launch_diag(const DiagConsts &k, const Levels<T> &L, Partials &part, hipStream_t st) {
  const int V = k.nx * k.ny * k.nz;
  int nb = (V + kDiagSitesPerBlock - 1) / kDiagSitesPerBlock;
  if (k.model == AX_MODEL_AH) {
    hipLaunchKernelGGL((diag_kernel<T, AX_MODEL_AH>), dim3(nb), dim3(256), 0, st, k, L, V, part.p);
  } else if (getenv("AX_DIAG_SITE_KERNEL") == nullptr) {
    /* part holds 3 doubles per work item (diag_part_blocks) */
    const TileGrid g = make_tile_grid(k.nx, k.ny, k.nz, diag_xseg(k.nx, k.ny, k.nz));
    hipLaunchKernelGGL((moore_diag_march_kernel<T>), dim3(g.work), dim3(64), 0, st, k, L, g, part.p);
    nb = g.work;
  } else {
    hipLaunchKernelGGL((diag_kernel<T, AX_MODEL_MOORE>), dim3(nb), dim3(256), 0, st, k, L, V, part.p);
  }
  part.n = nb;
  return hipGetLastError();
}

template <typename T>
hipError_t launch_winding(int nx, int ny, int nz, const T *fr, const T *fi, const T *tx, const T *ty,
                          const T *tz, double q, int ex, int ez, int8_t *out, Partials &part, hipStream_t st) {
  const int V = nx * ny * nz;
  const int nb = (V + kSitesPerBlock - 1) / kSitesPerBlock;
  hipLaunchKernelGGL((winding_kernel<T>), dim3(nb), dim3(256), 0, st, nx, ny, nz, fr, fi, tx, ty, tz, q, ex, ez,
                     out, part.p);
  part.n = nb;
  return hipGetLastError();
}

template <typename T>
hipError_t launch_crossings(int nx, int ny, int nz, double dx, double dy, double dz, const T *fr, const T *fi,
                            int ex, int ez, int *bcount, long long *boff, long long *total, double *xyz,
                            long long cap, uint64_t *masks, hipStream_t st, bool write) {
  CrossGeom g;
  g.nx = nx; g.ny = ny; g.nz = nz; g.ex = ex; g.ez = ez;
  g.x0 = int(0.5 * (nx - 1)); g.y0 = int(0.5 * (ny - 1)); g.z0 = int(0.5 * (nz - 1));
  g.V = (uint32_t)nx * ny * nz;
  g.sites = cross_sites(g.V);
  g.groups = (uint32_t)cross_groups(g.V);
  g.per = (g.groups + 7) / 8;
  g.by_nz = fast_div((uint32_t)nz);
  g.by_ny = fast_div((uint32_t)ny);
  g.dx = dx; g.dy = dy; g.dz = dz;
  g.k = cross_bound(nx, ny, nz, dx, dy, dz);
  const dim3 grid(8 * g.per), block(64);
#define AX_CROSS(W, M) \
  hipLaunchKernelGGL((cross_kernel<T, W, M>), grid, block, 0, st, g, fr, fi, bcount, boff, xyz, cap, masks)
  if (write && masks) AX_CROSS(false, true);
  else AX_CROSS(false, false);
  hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(1024), 0, st, bcount, boff, (int)g.groups, total);
  if (write && masks) AX_CROSS(true, true);
  else if (write) AX_CROSS(true, false);
#undef AX_CROSS
  return hipGetLastError();
}

/* The FP32 edge values of field (fr, fi) of charge q over the work items of
 * the tile grid (phase_march, ax_wind.h), where no energy pass stores them
 * along the way. */
template <typename T>
__global__ void __launch_bounds__(64) edge_march_kernel(int nx, int ny, int nz, const T *fr, const T *fi, const T *tx,
                                                        const T *ty, const T *tz, double q, TileGrid g, float *E) {
  int chunk, seg;
  if (!tile_item(g, (int)blockIdx.x, chunk, seg)) return;
  const int x0 = seg * g.xseg, x1 = min(nx, x0 + g.xseg);
  const WindRow w(nx, ny, nz, chunk);
  (void)phase_march<T>(w, fr, fi, tx, ty, tz, E, x0, x1, q);
}

template <typename T>
hipError_t launch_edge_winding(int nx, int ny, int nz, int ex, int ez, const T *fr, const T *fi, const T *tx,
                               const T *ty, const T *tz, double q, float *E, int8_t *out, Partials &part, hipStream_t st) {
  const TileGrid g = make_tile_grid(nx, ny, nz, diag_xseg(nx, ny, nz));
  hipLaunchKernelGGL((edge_march_kernel<T>), dim3(g.work), dim3(64), 0, st, nx, ny, nz, fr, fi, tx, ty, tz, q, g,
                     E);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? launch_wind_phase(nx, ny, nz, ex, ez, E, out, part, st) : e;
}

template <typename T>
hipError_t launch_diag_march(const DiagConsts &k, const Levels<T> &L, float *phase, Partials &part, hipStream_t st) {
  const TileGrid g = make_tile_grid(k.nx, k.ny, k.nz, diag_xseg(k.nx, k.ny, k.nz));
  /* without a gauge coupling the pass divides by dx, dy, dz alone
   * (energy_form 0 leaves out the gauge terms) */
  const bool p2 = diag_pow2(k.dx, k.dy, k.dz, k.g == 0 && k.energy_form == 0 ? 1.0 : k.g);
#define AX_DM(PH, P2) \
  hipLaunchKernelGGL((diag_march_kernel<T, PH, P2>), dim3(g.work), dim3(64), 0, st, k, L, g, phase, part.p)
  if (phase && p2) AX_DM(true, true);
  else if (phase) AX_DM(true, false);
  else if (p2) AX_DM(false, true);
  else AX_DM(false, false);
#undef AX_DM
  part.n = g.work;
  return hipGetLastError();
}

hipError_t launch_sums(const Partials &a, double *out3, const Partials &b, double *outb3, hipStream_t st) {
  hipLaunchKernelGGL(sum3_kernel, dim3(b.n ? 2 : 1), dim3(1024), 0, st, a.p, a.n, out3, b.p, b.n, outb3);
  return hipGetLastError();
}

/* div[s] = sum_a (theta_a(s) - theta_a(s-a))/dx_a^2 of one level (periodic),
 * the arithmetic of the fused step's stored divergence (ax_march.h). */
template <bool P2>
__global__ void __launch_bounds__(256) level_div_kernel(int nx, int ny, int nz, const double *tx, const double *ty,
                                                        const double *tz, EnergyConsts ek, double *div) {
  const size_t V = (size_t)nx * ny * nz;
  const size_t s = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (s >= V) return;
  const int kk = (int)(s % nz), r = (int)(s / nz), j = r % ny, i = r / ny;
  auto id = [&](int a, int b, int c) { return ((size_t)a * ny + b) * nz + c; };
  div[s] = link_div<P2>(ek, tx[s], tx[id(wrapm(i, nx), j, kk)], ty[s], ty[id(i, wrapm(j, ny), kk)], tz[s],
                        tz[id(i, j, wrapm(kk, nz))]);
}

hipError_t launch_level_div(int nx, int ny, int nz, const double *tx, const double *ty, const double *tz,
                            const EnergyConsts &ek, bool pow2, double *div, hipStream_t st) {
  const size_t V = (size_t)nx * ny * nz;
  const unsigned nb = (unsigned)((V + 255) / 256);
  if (pow2) hipLaunchKernelGGL((level_div_kernel<true>), dim3(nb), dim3(256), 0, st, nx, ny, nz, tx, ty, tz, ek, div);
  else hipLaunchKernelGGL((level_div_kernel<false>), dim3(nb), dim3(256), 0, st, nx, ny, nz, tx, ty, tz, ek, div);
  return hipGetLastError();
}

/* the P2 condition of the diagnostics march: dx, dy, dz, g and the derived
 * divisors are powers of two with finite reciprocals */
bool diag_pow2(double dx, double dy, double dz, double gg) {
  const double dvs[10] = {dx, dy, dz, dx * dx, dy * dy, dz * dz, gg, (gg * dx * dy) * (gg * dx * dy),
                          (gg * dx * dz) * (gg * dx * dz), (gg * dy * dz) * (gg * dy * dz)};
  bool p2 = gg != 0;
  for (double d : dvs) p2 = p2 && is_pow2(fabs(d)) && std::isfinite(1 / d);
  return p2;
}

hipError_t launch_wind_phase(int nx, int ny, int nz, int ex, int ez, const float *E, int8_t *out, Partials &part,
                             hipStream_t st) {
  /* part holds 3 doubles per work item (diag_part_blocks) */
  const TileGrid g = make_tile_grid(nx, ny, nz, diag_xseg(nx, ny, nz));
  const double lim = ex || ez ? kEdgeExact : INFINITY;
  hipLaunchKernelGGL(wind_march_kernel, dim3(g.work), dim3(64), 0, st, nx, ny, nz, E, g, ex, ez, lim, out, part.p);
  part.n = g.work;
  return hipGetLastError();
}

#define AX_INST(T)                                                                                             \
  template hipError_t launch_diag<T>(const DiagConsts &, const Levels<T> &, Partials &, hipStream_t);           \
  template hipError_t launch_winding<T>(int, int, int, const T *, const T *, const T *, const T *, const T *,   \
                                        double, int, int, int8_t *, Partials &, hipStream_t);                   \
  template hipError_t launch_crossings<T>(int, int, int, double, double, double, const T *, const T *, int,     \
                                          int, int *, long long *, long long *, double *, long long,            \
                                          uint64_t *, hipStream_t, bool);                                       \
  template hipError_t launch_diag_march<T>(const DiagConsts &, const Levels<T> &, float *, Partials &,          \
                                           hipStream_t);                                                        \
  template hipError_t launch_edge_winding<T>(int, int, int, int, int, const T *, const T *, const T *,          \
                                             const T *, const T *, double, float *, int8_t *, Partials &,       \
                                             hipStream_t);
AX_INST(double)
AX_INST(float)
#undef AX_INST

}  // namespace ax
