/*
 * ax_global.hip - global (ungauged) string: the momentum-form leapfrog of
 * leapfrog.cpp:166-347 on one lattice, FP64 or FP32.
 *
 * Device layout (planes of `pitch` elements): phi_re at level 0/1, phi_im at
 * level 0/1, pi_re, pi_im.  The field is double-buffered: TimeStep n reads
 * phi from level n%2 and writes level (n+1)%2, so the reference's two
 * passes (all phitt from the pre-step field, then the site-by-site update)
 * become one kernel.  The momentum is updated in place.
 *
 *  global_bc_kernel      Neumann copies of the x and y faces of the current
 *                        field (leapfrog.cpp:168-193): y faces for interior
 *                        x, then x faces over all y, folded into one pass by
 *                        reading the corner sources directly; written to both
 *                        field buffers.
 *  global_step_kernel    phitt = phixx + phiyy + phizz - (|phi|^2 - 1) phi,
 *                        pi += phitt dt, phi_new = phi + pi dt.
 *  global_energy_kernel  the energy the reference prints for that step
 *                        (leapfrog.cpp:301-321): recomputes phitt from the
 *                        pre-step field, takes the momentum rolled back by
 *                        dt/2 and central differences of the field as a
 *                        one-thread run holds it mid-loop -- neighbours
 *                        earlier in loop order already updated, later ones
 *                        not -- accumulated in FP64 per wave.
 *
 * The last two take one thread per site, or per two z neighbours where nz is
 * even, blocks of consecutive sites on one XCD.  With spacings that are
 * powers of two (POW2) the divisions by dx^2 and 2 dx are multiplications by
 * the exact reciprocals, the same bits.  200^3 FP64, Neumann faces: step 132
 * -> 103 us (64 bytes a site: 5.0 TB/s, a copy reaches 4.8), energy 192 ->
 * 121 us; before, every index was divided out for each neighbour, the twelve
 * quotients were divisions and every lane loaded 8 bytes at a time.  A march
 * along x with the planes in registers was slower (156 and 125 us).
 */
#include <algorithm>

#include "ax_internal.h"
#include "ax_march.h"

namespace ax {

/* What a kernel needs of the lattice, and no more: a small lattice's steps are
 * as fast as the host can launch them, and every argument byte goes over the
 * bus (Neumann faces, two launches a step, us: 16^3 FP32 7.4 with all of the
 * lattice's constants for each kernel, 6.5 with its own). */
struct GlobalGeom {
  int nx, ny, nz;
  int periodic;          /* 1: all sites updated, periodic wrap; 0: Neumann x/y faces */
  uint32_t V, per;       /* sites; blocks per XCD */
  uint32_t first;        /* first site stepped: Neumann x faces are left out, no XCD's share lies in them */
  FastDiv by_nz, by_ny;
};

/* dx^2, dy^2, dz^2 or, with POW2, their reciprocals */
template <typename R>
struct GlobalLap {
  R x, y, z;
};

template <typename R>
struct GlobalEnergy {
  R tx, ty, tz;          /* 2 dx ..., with POW2 their reciprocals */
  double dt, vol;        /* vol = dx dy dz */
  uint32_t runs;         /* of 256 threads' sites a block takes */
};

template <typename R, bool POW2>
__device__ __forceinline__ R gdiv(R a, R d) {
  return mdiv<R, POW2>(a, d, d);
}

template <typename R, bool POW2>
__device__ __forceinline__ R glap(const GlobalLap<R> &k, R f, R xp, R xm, R yp, R ym, R zp, R zm, R mag) {
  R xx = gdiv<R, POW2>(xp - 2 * f + xm, k.x);
  R yy = gdiv<R, POW2>(yp - 2 * f + ym, k.y);
  R zz = gdiv<R, POW2>(zp - 2 * f + zm, k.z);
  return xx + yy + zz - (mag - 1) * f;
}

template <typename R>
__global__ void __launch_bounds__(256) global_bc_kernel(int nx, int ny, int nz, R *pr, R *pi, R *qr,
                                                        R *qi) {
  /* boundary sites: the two x faces (all j), then the two y faces at interior x */
  const int nxf = 2 * ny * nz, nyf = 2 * (nx - 2) * nz;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= nxf + nyf) return;
  int i, j, k, si, sj;
  if (t < nxf) {
    const int f = t / (ny * nz), r = t % (ny * nz);
    j = r / nz;
    k = r % nz;
    i = f ? nx - 1 : 0;
    si = f ? nx - 2 : 1;
    sj = j == 0 ? 1 : (j == ny - 1 ? ny - 2 : j);   /* the y-face copy already applied at x = si */
  } else {
    const int u = t - nxf;
    const int f = u / ((nx - 2) * nz), r = u % ((nx - 2) * nz);
    i = 1 + r / nz;
    k = r % nz;
    j = f ? ny - 1 : 0;
    si = i;
    sj = f ? ny - 2 : 1;
  }
  const size_t d = ((size_t)i * ny + j) * nz + k, s = ((size_t)si * ny + sj) * nz + k;
  /* into the current field and into the buffer the step writes, whose
   * faces the step leaves alone: after the step the state holds the faces
   * the reference's array holds (copies of the pre-step interior) */
  const R vr = pr[s], vi = pi[s];
  pr[d] = vr;
  pi[d] = vi;
  qr[d] = vr;
  qi[d] = vi;
}

/* W sites of a thread: one, or two neighbours along z (nz and the planes'
 * pitch even, so that both lie in one row and their 16 (FP64) or 8 bytes are
 * aligned).  A request takes the addresser the same time whatever a lane's
 * width, and both kernels were bound by it (busy 78 % of the launch): with two
 * sites a lane issues 9 instead of 20 requests per site (step), 11 instead of
 * 26 (energy). */
template <typename R, int W>
struct Sites {
  typedef R vec __attribute__((ext_vector_type(W)));
  R v[W];
  __device__ static Sites load(const R *p, uint32_t s) {
    Sites o;
    const vec t = *(const vec *)(p + s);
#pragma unroll
    for (int q = 0; q < W; ++q) o.v[q] = t[q];
    return o;
  }
  __device__ void store(R *p, uint32_t s) const {
    vec t;
#pragma unroll
    for (int q = 0; q < W; ++q) t[q] = v[q];
    *(vec *)(p + s) = t;
  }
};
template <typename R>
struct Sites<R, 1> {
  R v[1];
  __device__ static Sites load(const R *p, uint32_t s) { return {{p[s]}}; }
  __device__ void store(R *p, uint32_t s) const { p[s] = v[0]; }
};

/* The first of this thread's W sites in run `run` of 256 threads, its
 * coordinates and its neighbours; on: the step updates them (they are within
 * the lattice and no Neumann face). */
template <int W>
struct GlobalSite {
  uint32_t s, xp, xm, yp, ym, zp, zm;   /* zp: after the last of the W sites */
  int i, j, k;
  bool on;
  __device__ GlobalSite(const GlobalGeom &g, uint32_t run) {
    const uint32_t at = g.first + (run * 256 + threadIdx.x) * W;
    s = min(at, g.V - W);               /* every lane holds loadable sites */
    const uint32_t r = quotient(s, g.by_nz);
    i = (int)quotient(r, g.by_ny);
    k = (int)(s - r * g.nz);
    j = (int)(r - i * g.ny);
    on = at < g.V && (g.periodic || (i > 0 && i < g.nx - 1 && j > 0 && j < g.ny - 1));
    const int nz = g.nz, nyz = g.ny * nz;
    xp = i == g.nx - 1 ? s - (g.nx - 1) * nyz : s + nyz;
    xm = i == 0 ? s + (g.nx - 1) * nyz : s - nyz;
    yp = j == g.ny - 1 ? s - (nyz - nz) : s + nz;
    ym = j == 0 ? s + (nyz - nz) : s - nz;
    zp = k + W == nz ? s - k : s + W;
    zm = k == 0 ? s + (nz - 1) : s - 1;
  }
  /* f at z - 1 and z + 1 of the W sites from f there: between lanes by a
   * shift, at the ends of the wave and of the row by a load */
  template <typename R>
  __device__ Sites<R, W> below(const GlobalGeom &g, const R *f, const Sites<R, W> &c) const {
    Sites<R, W> o;
    o.v[0] = lane_prev(c.v[W - 1], c.v[0]);
    if ((threadIdx.x & 63) == 0 || k == 0) o.v[0] = f[zm];
    if (W == 2) o.v[W - 1] = c.v[0];
    return o;
  }
  template <typename R>
  __device__ Sites<R, W> above(const GlobalGeom &g, const R *f, const Sites<R, W> &c) const {
    Sites<R, W> o;
    const R next = lane_next(c.v[0], c.v[0]);
    o.v[W - 1] = next;
    if ((threadIdx.x & 63) == 63 || k + W == g.nz) o.v[W - 1] = f[zp];
    if (W == 2) o.v[0] = c.v[W - 1];
    return o;
  }
};

template <typename R, bool POW2, int W>
__global__ void __launch_bounds__(256) global_step_kernel(GlobalGeom g, GlobalLap<R> c, R dt, const R *__restrict__ ar,
                                                          const R *__restrict__ ai, R *__restrict__ br,
                                                          R *__restrict__ bi, R *__restrict__ mr, R *__restrict__ mi) {
  typedef Sites<R, W> S;
  const GlobalSite<W> q(g, (blockIdx.x & 7) * g.per + (blockIdx.x >> 3));
  const R *f[2] = {ar, ai};
  R *n[2] = {br, bi}, *m[2] = {mr, mi};
  S here[2], xp[2], xm[2], yp[2], ym[2], mom[2];
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    here[v] = S::load(f[v], q.s);
    xp[v] = S::load(f[v], q.xp);
    xm[v] = S::load(f[v], q.xm);
    yp[v] = S::load(f[v], q.yp);
    ym[v] = S::load(f[v], q.ym);
    mom[v] = S::load(m[v], q.s);
  }
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    const S zm = q.below(g, f[v], here[v]), zp = q.above(g, f[v], here[v]);
    S p, o;
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const R mag = here[0].v[e] * here[0].v[e] + here[1].v[e] * here[1].v[e];
      const R t = glap<R, POW2>(c, here[v].v[e], xp[v].v[e], xm[v].v[e], yp[v].v[e], ym[v].v[e], zp.v[e], zm.v[e], mag);
      p.v[e] = mom[v].v[e] + t * dt;
      o.v[e] = here[v].v[e] + p.v[e] * dt;
    }
    if (q.on) {
      p.store(m[v], q.s);
      o.store(n[v], q.s);
    }
  }
}

/* o: the pre-step field, n: the step's result, m: its momentum.  A block
 * takes w.runs consecutive runs of 256 threads' sites: four, which leaves a
 * fourth of the partial sums, while the chip still gets four blocks a CU, and
 * fewer on small lattices, where one run after another is what the call waits
 * for (us per ax_diagnostics, FP64, periodic, dx 0.7, four runs / this rule:
 * 16^3 23.6 / 18.3, 33x47x80 24.6 / 19.2, 64^3 24.6 / 21.8, 128^3 and more
 * have four either way; one site a block's thread, without runs: 20.1, 21.6,
 * 24.2). */
constexpr uint32_t kEnergyRuns = 4;
template <typename R, bool POW2, int W>
__global__ void __launch_bounds__(256) global_energy_kernel(GlobalGeom g, GlobalLap<R> c, GlobalEnergy<R> w,
                                                            const R *__restrict__ ar, const R *__restrict__ ai,
                                                            const R *__restrict__ br, const R *__restrict__ bi,
                                                            const R *__restrict__ mr, const R *__restrict__ mi,
                                                            double *__restrict__ part) {
  typedef Sites<R, W> S;
  __shared__ double sh[2][4];
  double rho = 0, bad = 0;
  const uint32_t blk = (blockIdx.x & 7) * g.per + (blockIdx.x >> 3);
  const R *o[2] = {ar, ai}, *n[2] = {br, bi}, *m[2] = {mr, mi};
#pragma unroll 1
  for (uint32_t run = 0; run < w.runs; ++run) {
    const GlobalSite<W> q(g, blk * w.runs + run);
    /* a neighbour holds its new value when it is an updated site earlier in
     * loop order (x, then y, then z): x - 1 and y - 1 unless they wrap or are
     * faces, z - 1 unless it wraps; x + 1, y + 1, z + 1 only where they wrap */
    const int first = g.periodic ? 0 : 1;
    S here[2], now[2], mom[2];
    R t[2][W], gx[2][W], gy[2][W], gz[2][W];
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      here[v] = S::load(o[v], q.s);
      now[v] = S::load(n[v], q.s);
      mom[v] = S::load(m[v], q.s);
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      const S xp = S::load(o[v], q.xp), xm = S::load(o[v], q.xm), yp = S::load(o[v], q.yp), ym = S::load(o[v], q.ym);
      const S zp = q.above(g, o[v], here[v]), zm = q.below(g, o[v], here[v]);
      S xps = xp, yps = yp, zps = zp;
      S xms = S::load(n[v], q.xm), yms = S::load(n[v], q.ym), zms = q.below(g, n[v], now[v]);
      if (q.i <= first) xms = xm;
      if (q.j <= first) yms = ym;
      if (q.k == 0) zms.v[0] = zm.v[0];
      if (q.i == g.nx - 1) xps = S::load(n[v], q.xp);
      if (q.j == g.ny - 1) yps = S::load(n[v], q.yp);
      if (q.k + W == g.nz) zps.v[W - 1] = n[v][q.zp];
#pragma unroll
      for (int e = 0; e < W; ++e) {
        const R mag = here[0].v[e] * here[0].v[e] + here[1].v[e] * here[1].v[e];
        t[v][e] = glap<R, POW2>(c, here[v].v[e], xp.v[e], xm.v[e], yp.v[e], ym.v[e], zp.v[e], zm.v[e], mag);
        gx[v][e] = gdiv<R, POW2>(xps.v[e] - xms.v[e], w.tx);
        gy[v][e] = gdiv<R, POW2>(yps.v[e] - yms.v[e], w.ty);
        gz[v][e] = gdiv<R, POW2>(zps.v[e] - zms.v[e], w.tz);
      }
    }
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const R mag = here[0].v[e] * here[0].v[e] + here[1].v[e] * here[1].v[e];
      const double r0 = (double)mom[0].v[e] - 0.5 * (double)t[0][e] * w.dt;
      const double r1 = (double)mom[1].v[e] - 0.5 * (double)t[1][e] * w.dt;
      const double dm = (double)mag - 1;
      const double gx0 = gx[0][e], gx1 = gx[1][e], gy0 = gy[0][e], gy1 = gy[1][e], gz0 = gz[0][e], gz1 = gz[1][e];
      const double r = r0 * r0 + r1 * r1 + gx0 * gx0 + gx1 * gx1 + gy0 * gy0 + gy1 * gy1 + gz0 * gz0 + gz1 * gz1 +
                       0.5 * (dm * dm);
      if (q.on) {
        rho += w.vol * r;
        bad += (isfinite((double)now[0].v[e]) && isfinite((double)now[1].v[e]) && isfinite((double)mom[0].v[e]) &&
                isfinite((double)mom[1].v[e])) ? 0.0 : 1.0;
      }
    }
  }
  /* fixed-order block sums */
  rho = march_wave_sum(rho);
  bad = march_wave_sum(bad);
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) {
    sh[0][wv] = rho;
    sh[1][wv] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[3 * (size_t)blockIdx.x] = (sh[0][0] + sh[0][1]) + (sh[0][2] + sh[0][3]);
    part[3 * (size_t)blockIdx.x + 1] = 0;
    part[3 * (size_t)blockIdx.x + 2] = (sh[1][0] + sh[1][1]) + (sh[1][2] + sh[1][3]);
  }
}

/* How a lattice's kernels are launched. */
struct GlobalPlan {
  GlobalGeom g;
  bool wide;             /* two sites a thread */
  uint32_t eper, eruns;  /* blocks of the energy per XCD, runs of one */
};
/* pitch: of the planes, whose two-site loads need it even as well */
static GlobalPlan plan_of(const ax_params &p, size_t pitch) {
  GlobalPlan q;
  GlobalGeom &g = q.g;
  g.nx = p.nx; g.ny = p.ny; g.nz = p.nz;
  g.periodic = p.boundary == AX_BC_PERIODIC;
  g.V = (uint32_t)p.nx * p.ny * p.nz;
  q.wide = p.nz % 2 == 0 && pitch % 2 == 0;
  g.first = g.periodic ? 0 : (uint32_t)p.ny * p.nz;
  const uint32_t sites = g.V - 2 * g.first;
  const uint32_t runs = (sites + 255) / 256 / (q.wide ? 2 : 1) + 1;   /* of 256 threads */
  g.per = (runs + 7) / 8;
  q.eruns = std::min(kEnergyRuns, (runs + 1023) / 1024);
  q.eper = ((runs + q.eruns - 1) / q.eruns + 7) / 8;
  g.by_nz = fast_div((uint32_t)p.nz);
  g.by_ny = fast_div((uint32_t)p.ny);
  return q;
}

size_t global_energy_blocks(const ax_params &p) { return (size_t)8 * std::max(plan_of(p, 0).eper, plan_of(p, 1).eper); }

/* dx^2 ... and 2 dx ...; true when every one is a power of two with a normal
 * reciprocal, and then the reciprocals */
template <typename R>
static bool consts_of(const ax_params &p, GlobalLap<R> &l, R t[3]) {
  R d[6] = {(R)(p.dx * p.dx), (R)(p.dy * p.dy), (R)(p.dz * p.dz), 2 * (R)p.dx, 2 * (R)p.dy, 2 * (R)p.dz};
  bool p2 = true;
  for (R v : d) p2 = p2 && is_pow2(v) && std::isnormal(v) && std::isnormal(1 / v);
  if (p2)
    for (R &v : d) v = 1 / v;
  l = {d[0], d[1], d[2]};
  for (int a = 0; a < 3; ++a) t[a] = d[3 + a];
  return p2;
}

template <typename R>
hipError_t launch_global_step(const ax_params &p, void *state, size_t pitch, int n, hipStream_t st) {
  R *b = (R *)state;
  const int cur = n % 2, nw = 1 - cur;
  R *ar = b + (size_t)(0 + cur) * pitch, *ai = b + (size_t)(2 + cur) * pitch;
  R *br = b + (size_t)(0 + nw) * pitch, *bi = b + (size_t)(2 + nw) * pitch;
  R *mr = b + 4 * pitch, *mi = b + 5 * pitch;
  const GlobalPlan q = plan_of(p, pitch);
  if (!q.g.periodic) {
    const int nbs = 2 * p.ny * p.nz + 2 * (p.nx - 2) * p.nz;
    hipLaunchKernelGGL((global_bc_kernel<R>), dim3((nbs + 255) / 256), dim3(256), 0, st, p.nx, p.ny, p.nz, ar, ai, br, bi);
  }
  GlobalLap<R> l;
  R t[3];
  const bool p2 = consts_of<R>(p, l, t);
  const dim3 grid(8 * q.g.per), block(256);
#define AX_GS(P2, W) \
  hipLaunchKernelGGL((global_step_kernel<R, P2, W>), grid, block, 0, st, q.g, l, (R)p.dt, ar, ai, br, bi, mr, mi)
  if (p2 && q.wide) AX_GS(true, 2);
  else if (p2) AX_GS(true, 1);
  else if (q.wide) AX_GS(false, 2);
  else AX_GS(false, 1);
#undef AX_GS
  return hipGetLastError();
}

template <typename R>
hipError_t launch_global_energy(const ax_params &p, const void *state, size_t pitch, int n, Partials &part,
                                hipStream_t st) {
  const R *b = (const R *)state;
  const int cur = n % 2, nw = 1 - cur;   /* the pre-step field of TimeStep n and its result */
  GlobalPlan q = plan_of(p, pitch);
  q.g.per = q.eper;
  GlobalLap<R> l;
  R t[3];
  const bool p2 = consts_of<R>(p, l, t);
  const GlobalEnergy<R> w = {t[0], t[1], t[2], p.dt, p.dx * p.dy * p.dz, q.eruns};
  const dim3 grid(8 * q.eper), block(256);   /* part holds 3 doubles each (diag_part_blocks) */
#define AX_GE(P2, W)                                                                                               \
  hipLaunchKernelGGL((global_energy_kernel<R, P2, W>), grid, block, 0, st, q.g, l, w, b + (size_t)cur * pitch,      \
                     b + (size_t)(2 + cur) * pitch, b + (size_t)nw * pitch, b + (size_t)(2 + nw) * pitch, b + 4 * pitch, \
                     b + 5 * pitch, part.p)
  if (p2 && q.wide) AX_GE(true, 2);
  else if (p2) AX_GE(true, 1);
  else if (q.wide) AX_GE(false, 2);
  else AX_GE(false, 1);
#undef AX_GE
  part.n = (int)(8 * q.eper);
  return hipGetLastError();
}

template hipError_t launch_global_step<double>(const ax_params &, void *, size_t, int, hipStream_t);
template hipError_t launch_global_step<float>(const ax_params &, void *, size_t, int, hipStream_t);
template hipError_t launch_global_energy<double>(const ax_params &, const void *, size_t, int, Partials &,
                                                 hipStream_t);
template hipError_t launch_global_energy<float>(const ax_params &, const void *, size_t, int, Partials &, hipStream_t);

}  // namespace ax
