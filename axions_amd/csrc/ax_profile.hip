/*
 * ax_profile.hip - the straight-string initial-condition pipeline:
 *
 *  1. the radial profile f(r), A(r) of one straight string by successive
 *     over-relaxation (singleSemiAnalytic.cpp:54-134), and
 *  2. the lattice built from it by quadratic interpolation
 *     (straight_ic.cpp:59-146), written straight into a lattice's state.
 *
 * SOR.  The reference relaxes the 1-D grid r_j = j h in place, j = 1 ..
 * nx-2 in increasing order (one thread; its OpenMP loop over the same
 * in-place array races at chunk edges, so only the one-thread order is a
 * defined result): each point uses the new values at j-1 and the previous
 * sweep's values at j and j+1.  Sweep k at point j therefore depends only
 * on sweep k at j-1 and sweep k-1 at j, j+1.  Here lane L of a wave
 * runs sweep k0 + L, two points behind lane L-1: at time s lane L updates
 * j = s - 2L, and the two values of sweep k-1 it needs are what lane L-1
 * produced at times s-1 (point j+1) and s-2 (point j), moved by a DPP
 * row-crossing shift.  The last lane's sweep goes through device memory to
 * the next wave, a workgroup on another CU some 150 time steps behind, so a
 * launch keeps up to 512 waves x 64 sweeps in flight.  Every sweep sees
 * exactly the operands it sees in the reference loop, so the profile, the
 * sweep count and the stopping residual are the reference's bits.
 *
 * The loop stops after the first sweep whose largest |F| is not above tol
 * (or at max_iter).  A wave holding such a sweep ends the waves behind it;
 * the host finds the sweep in the residuals and runs that wave again up to
 * it.  A time step is a chain of some 250 dependent instructions, 16 waves
 * on one CU shared its issue slots: 5001 points x 6000 sweeps 51 -> 8.8 ms,
 * 30001 points x 23278 sweeps 1.04 s -> 51 ms.
 */
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "ax_internal.h"

namespace ax {

constexpr int SOR_MAX_WAVES = 512;           /* one per SIMD on half the chip */
constexpr size_t SOR_ROWS_BYTES = (size_t)1 << 30;   /* device memory the rows between waves may take */
constexpr int SOR_CHUNK = 32;                /* points a wave takes from the row before it at a time */
constexpr unsigned SOR_SPINS = 1u << 24;     /* polls (some 20 s) before a wave gives the launch up (AX_SOR_SPINS) */

struct SorConsts {
  int nx;
  double h, w, n, lambda, eta, g;
  double hh;          /* h*h */
  double two_hh;      /* 2/(h*h) */
  double half_lam;    /* 0.5*lambda */
  double eta2;        /* pow(eta, 2) */
};

/* One point of one sweep, singleSemiAnalytic.cpp:110-123, operands as the
 * reference reads them (pm, am: new j-1; p, a: old j; pp, ap: old j+1).
 * pow(x, 2) is x*x (GCC folds it so at -O1 and above). */
struct SorPoint {
  double phi, A, rphi, rA;
};

__host__ __device__ inline SorPoint sor_point(const SorConsts &k, int j, double pm, double p, double pp, double am,
                                              double a, double ap) {
  const double jh = j * k.h;
  const double den1 = (double)(2 * j) * k.h * k.h;
  const double q = (k.n - k.g * a) / jh;
  const double q2 = q * q;
  const double f0 = (q2 + k.half_lam * (p * p - k.eta2)) * p - (pp - pm) / den1 - (pp - 2 * p + pm) / k.hh;
  const double f1 = q2 + k.half_lam * (3 * (p * p) - k.eta2) + k.two_hh;
  const double gp = k.g * p;
  const double a0 = -2 * k.g * (k.n - k.g * a) * (p * p) + (ap - am) / den1 - (ap - 2 * a + am) / k.hh;
  const double a1 = 2 * (gp * gp) + k.two_hh;
  SorPoint r;
  r.phi = p + -k.w * f0 / f1;
  r.A = a + -k.w * a0 / a1;
  r.rphi = fabs(f0);
  r.rA = fabs(a0);
  return r;
}

/* value of lane-1 (DPP wave_shr:1); lane 0 gets `first` */
__device__ inline double from_prev_lane(double v, double first) {
  const long long bits = __double_as_longlong(v), fb = __double_as_longlong(first);
  const int lo = __builtin_amdgcn_update_dpp((int)fb, (int)bits, 0x138, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(fb >> 32), (int)(bits >> 32), 0x138, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

/* What the waves of a launch share besides the rows. */
struct SorControl {
  int ticket;     /* waves started */
  int stop;       /* lowest wave holding a sweep that meets the tolerance */
  int failed;     /* a wave waited longer than its polls */
};

/* "Not written yet" in a row: a signalling NaN, which no arithmetic returns. */
constexpr unsigned long long kSorUnset = 0x7ff40a5eab5e17edull;

__global__ void __launch_bounds__(256) sor_clear_kernel(unsigned long long *rows, size_t n, SorControl *ctl) {
  const size_t step = (size_t)gridDim.x * 256;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) rows[i] = kSorUnset;
  if (blockIdx.x == 0 && threadIdx.x == 0) *ctl = {0, 1 << 30, 0};
}

__device__ __forceinline__ unsigned long long sor_peek(const double *p) {
  return __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int sor_flag(const int *p) {
  return __builtin_amdgcn_readfirstlane(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void sor_post(double *p, double v) {
  __hip_atomic_store((unsigned long long *)p, (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

/* nb sweeps from (ip, ia) -> (op, oa); res[L] = the largest |F| of sweep L
 * (not of the sweeps in waves after one that stops).  Wave w = sweeps 64 w
 * ... 64 w + 63, in a workgroup of its own; rows[w] takes the last of them,
 * phi then A, and is what wave w + 1 starts from.  A value is handed over by
 * itself: the row holds kSorUnset until the producer's relaxed store, and the
 * consumer polls for it, so no order between two stores matters.  A wave
 * waits only for the one numbered before it, and numbers are handed out in
 * the order the waves start, so the lowest waiting wave always has a running
 * predecessor; the wait is bounded all the same, by `spins` polls, and after a
 * launch given up the host goes on with one wave a launch, which waits for
 * nobody. */
__global__ void __launch_bounds__(64) sor_kernel(SorConsts k, double tol, const double *__restrict__ ip,
                                                 const double *__restrict__ ia, double *rows, double *__restrict__ op,
                                                 double *__restrict__ oa, double *__restrict__ res, int nb,
                                                 SorControl *ctl, unsigned spins) {
  __shared__ double2 in[SOR_CHUNK];          /* in[t]: the previous sweep at point s0 + 2 + t */
  const int lane = (int)threadIdx.x;
  int ticket = 0;
  if (lane == 0) ticket = atomicAdd(&ctl->ticket, 1);
  const int w = __builtin_amdgcn_readfirstlane(ticket);
  const int nx = k.nx, L = 64 * w + lane;
  const int last = min(63, nb - 1 - 64 * w);             /* this wave's last sweep */
  const bool final = 64 * w + last == nb - 1;
  const double *bp = w ? rows + (size_t)2 * (w - 1) * nx : ip, *ba = w ? bp + nx : ia;
  double *rp = rows + (size_t)2 * w * nx, *ra = rp + nx;
  if (final && lane == last) {
    op[0] = 0;
    oa[0] = 0;
  }
  const bool live = lane <= last;
  const int s_end = nx - 2 + 2 * last;                   /* last time any sweep works */
  double o1p = 0, o1a = 0;                               /* own outputs at s-1 */
  double u1p = 0, u1a = 0;                               /* the previous sweep at point j + 1, j */
  double r = 0;
  /* point j of the row before, as raw bits; what is not needed reads as 0 */
  auto need = [&](int j) { return lane < SOR_CHUNK && j <= nx - 2; };
  unsigned long long np = 0, na = 0;
  auto fetch = [&](int j) {
    np = na = 0;
    if (need(j)) {
      np = sor_peek(bp + j);
      na = sor_peek(ba + j);
    }
  };
  /* true when every needed value has arrived */
  auto settle = [&](int j) {
    for (unsigned n = 0;; ++n) {
      const bool wait = need(j) && w && (np == kSorUnset || na == kSorUnset);
      if (__builtin_amdgcn_ballot_w64(wait) == 0) return true;
      if ((n & 63) == 63) {
        const bool over = n > spins;
        if (over && lane == 0) __hip_atomic_store(&ctl->failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (over || sor_flag(&ctl->failed) || sor_flag(&ctl->stop) < w) return false;
      }
      __builtin_amdgcn_s_sleep(2);
      fetch(j);
    }
  };
  /* point 1: u1 at time 0 */
  fetch(1 + lane);
  if (!settle(1 + lane)) return;
  u1p = __longlong_as_double((long long)__shfl((long long)np, 0, 64));
  u1a = __longlong_as_double((long long)__shfl((long long)na, 0, 64));
  if (lane) u1p = u1a = 0;
  fetch(2 + lane);
  for (int s0 = 0; s0 < s_end; s0 += SOR_CHUNK) {
    if (!settle(s0 + 2 + lane)) return;
    if (lane < SOR_CHUNK)
      in[lane] = make_double2(__longlong_as_double((long long)np), __longlong_as_double((long long)na));
    __syncthreads();
    /* the next chunk's values, and whether a wave before this one stops */
    fetch(s0 + SOR_CHUNK + 2 + lane);
    const bool stopped = sor_flag(&ctl->stop) < w;
    for (int t = 0; t < SOR_CHUNK; ++t) {
      const int s = s0 + 1 + t, j = s - 2 * lane;
      const double2 f = in[t];
      /* at point j + 1 the previous lane's output of the last time step; at
       * point j the one before, which is the last time's u1 */
      const double u2p = u1p, u2a = u1a;
      u1p = from_prev_lane(o1p, f.x);
      u1a = from_prev_lane(o1a, f.y);
      if (live && j >= 1 && j <= nx - 2) {
        const bool edge = j == nx - 2;              /* phi(nx-1) = phi(nx-2) of the previous sweep */
        const SorPoint q = sor_point(k, j, j == 1 ? 0.0 : o1p, u2p, edge ? u2p : u1p, j == 1 ? 0.0 : o1a, u2a,
                                     edge ? u2a : u1a);
        o1p = q.phi;
        o1a = q.A;
        if (q.rphi > r) r = q.rphi;
        if (q.rA > r) r = q.rA;
        if (lane == last) {
          if (final) {
            op[j] = o1p;
            oa[j] = o1a;
            if (edge) {
              op[nx - 1] = u2p;
              oa[nx - 1] = u2a;
            }
          } else {
            sor_post(rp + j, o1p);
            sor_post(ra + j, o1a);
          }
        }
      }
    }
    if (stopped) return;
    __syncthreads();
  }
  if (live) res[L] = r;
  if (__builtin_amdgcn_ballot_w64(live && !(r > tol)) && lane == 0) atomicMin(&ctl->stop, w);
}

/* straight_ic.cpp:63-134 at one (x, y): phi and the gauge field A */
struct StraightSite {
  double f0, f1, a0, a1;
  int offgrid;
};

__host__ __device__ inline StraightSite straight_site(const double *prof, int nprof, double dr, double nw, double g,
                                                      double x, double y) {
  StraightSite o;
  const double d = sqrt(x * x + y * y);
  const long long pc = llround(d / dr);
  double fm, am;
  o.offgrid = 0;
  if (pc == 0) {
    fm = (prof[2] * d - prof[0] * (d - dr)) / dr;
    am = (prof[3] * d - prof[1] * (d - dr)) / dr;
  } else if (pc + 1 < nprof) {
    const int p = (int)pc;
    const double e0 = d - p * dr, em = d - (p - 1) * dr, ep = d - (p + 1) * dr;
    const double den = 2 * dr * dr;
    fm = (prof[2 * (p - 1)] * e0 * ep - 2 * prof[2 * p] * em * ep + prof[2 * (p + 1)] * em * e0) / den;
    am = (prof[2 * (p - 1) + 1] * e0 * ep - 2 * prof[2 * p + 1] * em * ep + prof[2 * (p + 1) + 1] * em * e0) / den;
  } else {
    fm = 1;
    am = g == 0 ? 0 : nw / g;
    o.offgrid = 1;
  }
  const double d2 = d * d;
  if (x == 0) {
    o.f0 = 0;
    o.a1 = 0;
  } else {
    o.f0 = fm * x / d;
    o.a1 = am * x / d2;
  }
  if (y == 0) {
    o.f1 = 0;
    o.a0 = 0;
  } else {
    o.f1 = fm * y / d;
    o.a0 = -am * y / d2;
  }
  return o;
}

struct StraightArgs {
  int nx, ny, nz, nprof, global;
  double dx, dy, dz, dr, nw, g;
  size_t pitch;
};

/* one thread per site; the z column shares one (x, y) value */
template <typename T>
__global__ void __launch_bounds__(256) straight_kernel(StraightArgs a, const double *__restrict__ prof, T *state,
                                                       unsigned long long *offgrid) {
  const size_t V = (size_t)a.nx * a.ny * a.nz;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V) return;
  const int z = (int)(i % a.nz);
  const size_t xy = i / a.nz;
  const int y = (int)(xy % a.ny), x = (int)(xy / a.ny);
  const int x0 = (a.nx - 1) / 2, y0 = (a.ny - 1) / 2;
  const StraightSite s = straight_site(prof, a.nprof, a.dr, a.nw, a.g, (x - x0) * a.dx, (y - y0) * a.dy);
  if (s.offgrid && z == 0) atomicAdd(offgrid, 1ull);
  if (a.global) {
    /* (Re phi, Im phi) in both parity buffers, momentum 0 */
    for (int b = 0; b < 2; ++b) {
      state[(size_t)(2 * 0 + b) * a.pitch + i] = (T)s.f0;
      state[(size_t)(2 * 1 + b) * a.pitch + i] = (T)s.f1;
    }
    state[(size_t)4 * a.pitch + i] = 0;
    state[(size_t)5 * a.pitch + i] = 0;
    return;
  }
  /* link variables dx*g*A (straight_ic.cpp:146); both levels */
  const T v[5] = {(T)s.f0, (T)s.f1, (T)(a.dx * a.g * s.a0), (T)(a.dy * a.g * s.a1), (T)(a.dz * a.g * 0.0)};
  for (int c = 0; c < 5; ++c)
    for (int t = 0; t < 2; ++t) state[(size_t)(2 * c + t) * a.pitch + i] = v[c];
}

}  // namespace ax

using namespace ax;

namespace {

int sor_check(const ax_sor_params *p) {
  if (!p) return fail(AX_EINVAL, "NULL parameters");
  if (p->nx < 3) return fail(AX_EINVAL, "profile needs nx >= 3 (got %d)", p->nx);
  if (p->nx > (1 << 28)) return fail(AX_EINVAL, "profile nx %d too large", p->nx);
  if (!(p->h > 0)) return fail(AX_EINVAL, "profile spacing h must be > 0");
  return AX_OK;
}

struct DevBuf {
  double *p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
};

}  // namespace

extern "C" {

void ax_sor_default_params(ax_sor_params *p) {
  if (!p) return;
  memset(p, 0, sizeof *p);
  /* singleSemiAnalytic.cpp:19-32 */
  p->nx = 30001;
  p->h = 0.01;
  p->w = 1.5;
  p->max_iter = 2000000;
  p->tol = 1e-3;
  p->n = 1;
  p->lambda = 1;
  p->eta = 1;
  p->g = 0;
}

int ax_sor_profile(const ax_sor_params *p, const double *init, double *out, int32_t *iterations, double *residual) {
  int rc = sor_check(p);
  if (rc) return rc;
  if (!out) return fail(AX_EINVAL, "NULL output");
  const int nx = p->nx;
  std::vector<double> hp(nx), ha(nx);
  if (init) {
    for (int i = 0; i < nx; ++i) {
      hp[i] = init[2 * i];
      ha[i] = init[2 * i + 1];
    }
  } else {
    for (int i = 0; i < nx; ++i) {          /* ic_type 0 (singleSemiAnalytic.cpp:56-61) */
      hp[i] = p->eta * tanh(0.5 * p->h * i);
      ha[i] = 0;
    }
  }
  hp[0] = 0;                                /* singleSemiAnalytic.cpp:76-78 */
  ha[0] = 0;

  int iters = 0;
  double tol_test = 1;                      /* singleSemiAnalytic.cpp:80 */
  if (tol_test > p->tol && p->max_iter > 0) {
    SorConsts k;
    k.nx = nx;
    k.h = p->h;
    k.w = p->w;
    k.n = p->n;
    k.lambda = p->lambda;
    k.eta = p->eta;
    k.g = p->g;
    k.hh = p->h * p->h;
    k.two_hh = 2 / (p->h * p->h);
    k.half_lam = 0.5 * p->lambda;
    k.eta2 = p->eta * p->eta;

    /* waves per launch, as many as the sweeps and the rows' memory allow (at
     * least 4, as fast as one workgroup of 16 waves would be) */
    int waves = (int)std::min<long long>(SOR_MAX_WAVES, ((long long)p->max_iter + 63) / 64);
    waves = (int)std::min<size_t>(waves, std::max<size_t>(4, SOR_ROWS_BYTES / ((size_t)16 * nx)));
    DevBuf buf, rows, dres;
    hipError_t e = hipMalloc(&buf.p, (size_t)4 * nx * sizeof(double));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc profile");
    while ((e = hipMalloc(&rows.p, (size_t)2 * waves * nx * sizeof(double))) != hipSuccess && waves > 1) {
      (void)hipGetLastError();   /* clear the sticky error of the failed call */
      waves /= 2;
    }
    if (e != hipSuccess) return hip_fail(e, "hipMalloc sweep rows");
    e = hipMalloc(&dres.p, (size_t)64 * waves * sizeof(double) + sizeof(SorControl));
    if (e != hipSuccess) return hip_fail(e, "hipMalloc residuals");
    SorControl *ctl = (SorControl *)(dres.p + (size_t)64 * waves);
    double *inp = buf.p, *ina = buf.p + nx, *outp = buf.p + 2 * (size_t)nx, *outa = buf.p + 3 * (size_t)nx;
    hipStream_t st;
    e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
    if (e != hipSuccess) return hip_fail(e, "hipStreamCreate");
    struct StreamGuard {
      hipStream_t s;
      ~StreamGuard() { (void)hipStreamDestroy(s); }
    } sg{st};
    e = hipMemcpyAsync(inp, hp.data(), nx * sizeof(double), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipMemcpyAsync(ina, ha.data(), nx * sizeof(double), hipMemcpyHostToDevice, st);
    if (e != hipSuccess) return hip_fail(e, "upload profile");
    std::vector<double> hres((size_t)64 * waves);
    const char *se = getenv("AX_SOR_SPINS");
    const unsigned spins = se ? (unsigned)atol(se) : SOR_SPINS;
    /* n sweeps from (fp, fa) into (outp, outa), their residuals into hres;
     * late: a wave waited too long and the launch has no result */
    bool late = false;
    auto sweep = [&](const double *fp, const double *fa, double *between, int n) -> int {
      const int nw = (n + 63) / 64;
      const size_t cells = (size_t)2 * (nw - 1) * nx;
      const unsigned cb = (unsigned)std::min<size_t>(2048, cells / 256 + 1);
      hipLaunchKernelGGL(sor_clear_kernel, dim3(cb), dim3(256), 0, st, (unsigned long long *)between, cells, ctl);
      hipLaunchKernelGGL(sor_kernel, dim3(nw), dim3(64), 0, st, k, p->tol, fp, fa, between, outp, outa, dres.p, n, ctl,
                         spins);
      SorControl done;
      hipError_t er = hipGetLastError();
      if (er == hipSuccess) er = hipMemcpyAsync(hres.data(), dres.p, n * sizeof(double), hipMemcpyDeviceToHost, st);
      if (er == hipSuccess) er = hipMemcpyAsync(&done, ctl, sizeof done, hipMemcpyDeviceToHost, st);
      if (er == hipSuccess) er = hipStreamSynchronize(st);
      if (er != hipSuccess) return hip_fail(er, "SOR sweeps");
      late = done.failed != 0;
      return AX_OK;
    };
    while (iters < p->max_iter) {
      const int nb = std::min(64 * waves, p->max_iter - iters);
      if ((rc = sweep(inp, ina, rows.p, nb)) != AX_OK) return rc;
      if (late) {   /* never of one wave */
        waves = 1;
        continue;
      }
      int stop = -1;
      for (int l = 0; l < nb; ++l)
        if (!(hres[l] > p->tol)) {
          stop = l;
          break;
        }
      if (stop >= 0) {
        tol_test = hres[stop];
        if (stop < nb - 1) {
          /* the stopping sweep's own wave again, from the row before it; the
           * row it was in the launch's last place for is free */
          const int w = stop / 64;
          const double *fp = w ? rows.p + (size_t)2 * (w - 1) * nx : inp, *fa = w ? fp + nx : ina;
          if ((rc = sweep(fp, fa, rows.p + (size_t)2 * w * nx, stop % 64 + 1)) != AX_OK) return rc;
        }
        iters += stop + 1;
        std::swap(inp, outp);
        std::swap(ina, outa);
        break;
      }
      iters += nb;
      tol_test = hres[nb - 1];
      std::swap(inp, outp);
      std::swap(ina, outa);
    }
    e = hipMemcpyAsync(hp.data(), inp, nx * sizeof(double), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipMemcpyAsync(ha.data(), ina, nx * sizeof(double), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_fail(e, "download profile");
  }
  for (int i = 0; i < nx; ++i) {
    out[2 * i] = hp[i];
    out[2 * i + 1] = ha[i];
  }
  if (iterations) *iterations = iters;
  if (residual) *residual = tol_test;
  return AX_OK;
}

int ax_init_straight_string(ax_lattice *L, const double *profile, int32_t nprof, double dr, double n, double g,
                            int64_t *off_grid) {
  if (!L || !profile) return fail(AX_EINVAL, "NULL argument");
  if (nprof < 2) return fail(AX_EINVAL, "profile needs at least 2 points (got %d)", nprof);
  if (!(dr > 0)) return fail(AX_EINVAL, "profile spacing must be > 0");
  const ax_params &p = lattice_params(L);
  if (p.model == AX_MODEL_MOORE) return fail(AX_EINVAL, "straight-string initial condition: AH or global model only");
  StraightArgs a;
  a.nx = p.nx;
  a.ny = p.ny;
  a.nz = p.nz;
  a.nprof = nprof;
  a.global = p.model == AX_MODEL_GLOBAL;
  a.dx = p.dx;
  a.dy = p.dy;
  a.dz = p.dz;
  a.dr = dr;
  a.nw = n;
  a.g = g;
  a.pitch = lattice_pitch(L);
  const size_t V = lattice_sites(L);
  hipStream_t st = lattice_stream(L);
  DevBuf prof, cnt;
  hipError_t e = hipMalloc(&prof.p, (size_t)2 * nprof * sizeof(double) + 256);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc profile");
  unsigned long long *dcount = (unsigned long long *)(prof.p + 2 * (size_t)nprof);
  unsigned long long hcount = 0;
  e = hipMemcpyAsync(prof.p, profile, (size_t)2 * nprof * sizeof(double), hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipMemsetAsync(dcount, 0, sizeof *dcount, st);
  if (e != hipSuccess) return hip_fail(e, "upload profile");
  const unsigned blocks = (unsigned)((V + 255) / 256);
  if (p.precision == 64)
    hipLaunchKernelGGL(straight_kernel<double>, dim3(blocks), dim3(256), 0, st, a, prof.p,
                       (double *)lattice_state(L), dcount);
  else
    hipLaunchKernelGGL(straight_kernel<float>, dim3(blocks), dim3(256), 0, st, a, prof.p, (float *)lattice_state(L),
                       dcount);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(&hcount, dcount, sizeof hcount, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return hip_fail(e, "straight-string initial condition");
  lattice_reset_timestep(L);
  if (off_grid) *off_grid = (int64_t)(hcount * (unsigned long long)p.nz);
  return AX_OK;
}

}  // extern "C"
