/*
 * ax_march_moore.h - the Moore-model update (mooreEvol.cpp:202-337: two
 * complex scalars with charges q1, q2 on one U(1) link field, no friction)
 * as a 64-lane wave marching along x over a 64-site chunk of the (y, z)
 * plane, like ah_march.  Same arithmetic and operand order as moore_update in
 * ax_step.hip; the cos/sin of q_f theta_x(s-x) and the plaquette sines at
 * s-x come from the previous plane of the march, y-backward values are
 * recomputed, and so are z-backward ones where ZB below does not shift them
 * over from lane - 1; the six plaquette sines at s are computed once and take
 * the short k = 0 form when the whole wave qualifies.
 */
#ifndef AXIONS_AX_MARCH_MOORE_H
#define AXIONS_AX_MARCH_MOORE_H

#include "ax_march.h"

namespace ax {

template <typename R>
struct MooreConsts {
  R dx2, dy2, dz2, dt2, m2gg;
  R hl1, hl2, hl12, eta1sq, eta2sq, q1, q2;
  R inv_dx2, inv_dy2, inv_dz2;
};

/* Division by a divisor that is the same for the whole launch, with the
 * bits of the compiler's IEEE division a / d.  That division is: y = rcp(d)
 * refined by two Newton steps, q = a*y, r = fma(-d, q, a), fma(r, y, q),
 * with range scaling (v_div_scale) and special-case repair (v_div_fixup)
 * around it that change nothing while d and a/d are far from the exponent
 * limits.  With d in [2^-100, 2^100] (checked by the launcher) and a = 0 or
 * |a| in [2^-800, 2^600] the steps after y are done here as they stand, and
 * y once per wave (+-0 take a's sign: the bare steps return +0 for -0).
 *
 * The numerators are sums of products of the current level's values and
 * their sines and cosines.  When every value of that level is 0 or has
 * magnitude in [2^-250, 2^40] (in_moore_band) and the charges satisfy
 * |q| <= 2^8 (checked by the launcher), every trig argument -- q*theta or a
 * plaquette angle, a sum of four link values -- is below 2^50 in
 * magnitude, where ax_reduce_pio2 still finds the quadrant exactly and
 * leaves |r| <~ pi/4, so every sine and cosine lies in [-1, 1] (tested on
 * the host up to 2^50).  Then every term of a numerator (a product of a
 * value and a sine or cosine, or 2 times a value) is 0 or a multiple of
 * 2^-605 and at most 2^41 in magnitude, and every numerator (at most five
 * such terms) is 0 or in [2^-605, 2^44]: the step that
 * writes a level checks its outputs against that band and ORs a per-level
 * flag, and the next step divides this way only when the flag of its
 * current level is clear. */
struct FixedDivisor {
  double d, y;
};
__device__ __forceinline__ FixedDivisor fixed_divisor(double d) {
  const double r0 = __builtin_amdgcn_rcp(d);
  const double r1 = fma(r0, fma(-d, r0, 1.0), r0);
  const double y = fma(r1, fma(-d, r1, 1.0), r1);
  /* the same on every lane: kept in scalar registers */
  const uint64_t b = __double_as_longlong(y);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return {d, __longlong_as_double((long long)(((uint64_t)hi << 32) | lo))};
}
__device__ __forceinline__ double fixed_div(double a, const FixedDivisor &v) {
  const double q = a * v.y;
  return copysign(fma(fma(-v.d, q, a), v.y, q), a);
}
inline bool fixed_divisor_range(double d) { return d >= 0x1p-100 && d <= 0x1p100; }
/* charges for which q*theta stays below 2^50 for every in-band theta */
inline bool moore_band_charge(int q) { return q >= -256 && q <= 256; }
__device__ __forceinline__ bool in_moore_band(double v) {
  const double m = fabs(v);
  return m <= 0x1p40 && (m >= 0x1p-250 || m == 0);
}

template <typename R>
inline void moore_consts_from(const StepConsts &k, MooreConsts<R> &m) {
  m.dx2 = (R)k.dx2; m.dy2 = (R)k.dy2; m.dz2 = (R)k.dz2; m.dt2 = (R)k.dt2; m.m2gg = (R)k.m2gg;
  m.hl1 = (R)k.hl1; m.hl2 = (R)k.hl2; m.hl12 = (R)k.hl12; m.eta1sq = (R)k.eta1sq; m.eta2sq = (R)k.eta2sq;
  m.q1 = (R)k.q1; m.q2 = (R)k.q2;
  m.inv_dx2 = (R)1 / m.dx2; m.inv_dy2 = (R)1 / m.dy2; m.inv_dz2 = (R)1 / m.dz2;
}

/* What the site (y, z - 1) contributes to a chunk's first lane (ZEdge in
 * ax_march.h): sin/cos of q_f theta_z there and its F_xz, F_yz plaquette
 * sines. */
template <typename R>
struct MooreEdge {
  R s[2], c[2], qxz, qyz;
};

/* BUF: the loop's loads and stores are raw buffer accesses, one resource per
 * field spanning both of its levels (planes 2c, 2c+1; the caller checks that
 * two planes fit 32-bit offsets), with the streaming hint on the previous
 * level as in ah_march; otherwise plain global accesses from each x plane's
 * 64-bit address (field planes of any size, 1001^3 FP64 included).
 * FASTDIV (FP64, divisors not powers of two): divisions by dx^2, dy^2,
 * dz^2 through FixedDivisor; the caller has checked the current level's
 * band flag.  CHECK: OR 1 into *bad when a written value lies outside the
 * band (every lane of the wave must reach the end). */
template <typename R, bool POW2, bool BUF, bool FLAT, bool FASTDIV = false, bool CHECK = false>
__device__ __forceinline__ void moore_march(const MooreConsts<R> &k, const Levels<R> &L, int NX, int NY, int NZ,
                                            uint32_t p0, int x0, int x1, bool xfix = false, bool zfix = false,
                                            int *bad = nullptr) {
  typedef TrigR<R> T;
  /* Chunks across rows in FP64 without the band check: the neighbours' phi is
   * loaded ahead of the plaquette sines, whose branch keeps the compiler from
   * moving loads over it.  us per step late / early: dx^2 no power of two,
   * faces fixed 201x201x51 155.5 / 142.8, 250^3 1023 / 899, 100^3 73.7 / 68.2,
   * 50^3 13.5 / 11.9; powers of two, periodic 250^3 952 / 817, 100^3 62.2 /
   * 55.5.  The other kernels are slower with it: whole chunks 256^3 845 / 931
   * and (powers of two) 767 / 834, with the band check 250^3 824 / 875, 256^3
   * 847 / 900; FP32 is the same. */
  /* ZB: whole chunks with the band check take the z-backward cos/sin and
   * sines from lane - 1, the chunk edge's from a pass over four planes
   * (zedge), as ah_march, instead of evaluating them again: two of ten
   * sincos and two of ten sines fewer; and the first charge's phi rows are
   * loaded ahead of the plaquette sines.  us per step 256^3 854 -> 819 ->
   * 813.5, 128^3 114 -> 111.  The other kernels lose: powers of two 256^3 766
   * -> 800, chunks across rows with the check 150^3 181 -> 184 (registers). */
  constexpr bool ZB = sizeof(R) == 8 && BUF && !FLAT && CHECK;
  constexpr bool EARLY = sizeof(R) == 8 && BUF && FLAT && !CHECK;
  const size_t NYNZ = (size_t)NY * NZ;
  const LaneSite<FLAT> ls(NY, NZ, p0);
  const int y = ls.y, z = ls.z;
  /* xfix, zfix: x and y, z not periodic; their face sites are not stepped */
  const bool act = ls.act && !(zfix && (z == 0 || z == NZ - 1)) && !(xfix && (y == 0 || y == NY - 1));
  const uint32_t E = (uint32_t)sizeof(R);
  const uint32_t PLB = (uint32_t)NYNZ * E;          /* plane bytes */
  auto row = [&](int r) { return ls.row(r, E); };
  auto col = [&](int r, int c) { return ls.col(r, c, E); };
  const uint32_t R0 = row(0), RM = row(-1), RP = row(1);
  const uint32_t oz = col(0, 0), ozp = col(0, 1), ozm = col(0, -1);   /* in row R0 */
  const uint32_t pz = col(1, 0), pzm = col(1, -1), mz = col(-1, 0), mzp = col(-1, 1);   /* in rows RP, RP, RM, RM */
  const R *F[7] = {L.cur[0], L.cur[1], L.cur[2], L.cur[3], L.cur[4], L.cur[5], L.cur[6]};
  R *O[7] = {L.prv[0], L.prv[1], L.prv[2], L.prv[3], L.prv[4], L.prv[5], L.prv[6]};
  const R *TX = F[4], *TY = F[5], *TZ = F[6];
  const R q[2] = {k.q1, k.q2};
  FixedDivisor fdx = {}, fdy = {}, fdz = {};
  if constexpr (FASTDIV) {
    fdx = fixed_divisor((double)k.dx2);
    fdy = fixed_divisor((double)k.dy2);
    fdz = fixed_divisor((double)k.dz2);
  }
  /* a / d_a for axis a (x, y, z) */
  auto dvx = [&](R a) -> R { if constexpr (FASTDIV) return fixed_div(a, fdx); else return mdiv<R, POW2>(a, k.dx2, k.inv_dx2); };
  auto dvy = [&](R a) -> R { if constexpr (FASTDIV) return fixed_div(a, fdy); else return mdiv<R, POW2>(a, k.dy2, k.inv_dy2); };
  auto dvz = [&](R a) -> R { if constexpr (FASTDIV) return fixed_div(a, fdz); else return mdiv<R, POW2>(a, k.dz2, k.inv_dz2); };
  bool inband = true;
  /* field c's lower plane, and the byte offsets of the two levels from it */
  __amdgpu_buffer_rsrc_t FR[7];
  uint32_t offC = 0, offP = 0;
  if (BUF) {
    for (int c = 0; c < 7; ++c) FR[c] = plane_rsrc(L.cur[c] < L.prv[c] ? (const void *)L.cur[c] : (const void *)L.prv[c]);
    const bool curLow = L.cur[0] < L.prv[0];
    const uint32_t lev = (uint32_t)(curLow ? (const char *)L.prv[0] - (const char *)L.cur[0]
                                           : (const char *)L.cur[0] - (const char *)L.prv[0]);
    offC = curLow ? 0u : lev;
    offP = curLow ? lev : 0u;
  }
  /* current-level value of field c in x plane x at (row byte offset ro,
   * lane offset lo); without BUF the plane's 64-bit address is formed on
   * the scalar unit, so planes of any size work */
  auto LC = [&](int c, int x, uint32_t ro, uint32_t lo) -> R {
    if (BUF) return bld<R>(FR[c], lo, offC + (uint32_t)x * PLB + ro);
    return ldo(F[c] + (size_t)x * NYNZ, ro, lo);
  };
  auto LG = [&](const R *f, int x, uint32_t ro, uint32_t lo) -> R { return ldo(f + (size_t)x * NYNZ, ro, lo); };

  /* carry from plane x-1: phi_f(s-x), cos/sin(q_f theta_x(s-x)), sines at s-x */
  const int xm0 = x0 == 0 ? NX - 1 : x0 - 1;
  R Pm[4], cxm[2], sxm[2], Qyx_m, Qzx_m;
  {
    for (int c = 0; c < 4; ++c) Pm[c] = LG(F[c], xm0, R0, oz);
    const R X = LG(TX, xm0, R0, oz), Y = LG(TY, xm0, R0, oz), Z = LG(TZ, xm0, R0, oz);
    for (int f = 0; f < 2; ++f) T::sc(q[f] * X, &sxm[f], &cxm[f]);
    Qyx_m = T::sn(Y + LG(TX, xm0, RP, pz) - LG(TY, x0, R0, oz) - X);
    Qzx_m = T::sn(Z + LG(TX, xm0, R0, ozp) - LG(TZ, x0, R0, oz) - X);
  }
  R C[7];
  for (int c = 0; c < 7; ++c) C[c] = LG(F[c], x0, R0, oz);

  /* ZB: lane j < 4 evaluates the edge of plane xb + j */
  const bool e0 = (threadIdx.x & 63) == 0;
  __shared__ MooreEdge<R> zedge[4];
  auto edge_block = [&](int xb, int xe) {
    const int j = (int)(threadIdx.x & 63), xj = min(xb + j, xe - 1);
    const uint32_t z0 = p0 % (uint32_t)NZ, zm = (z0 == 0 ? (uint32_t)NZ : z0) - 1;
    const uint32_t em = R0 + zm * E, emP = RP + zm * E, ec = R0 + z0 * E;   /* (y, z0 - 1), (y + 1, z0 - 1), (y, z0) */
    const int xjp = xj == NX - 1 ? 0 : xj + 1;
    auto at = [&](int c, int xx, uint32_t off) -> R { return bld<R>(FR[c], offC + (uint32_t)xx * PLB + off, 0); };
    const R TZe = at(6, xj, em), TXe = at(4, xj, em), TYe = at(5, xj, em);
    const R TZxe = at(6, xjp, em), TZye = at(6, xj, emP), TX0 = at(4, xj, ec), TY0 = at(5, xj, ec);
    MooreEdge<R> e;
    for (int f = 0; f < 2; ++f) T::sc(q[f] * TZe, &e.s[f], &e.c[f]);
    e.qxz = T::sn(TXe + TZxe - TX0 - TZe);   /* a_xz at (xj, y, z - 1) */
    e.qyz = T::sn(TYe + TZye - TY0 - TZe);   /* a_yz there */
    __syncthreads();   /* the previous block's values have been read */
    if (j < xe - xb) zedge[j] = e;
    __syncthreads();
  };

  for (int x = x0; x < x1; ++x) {
    if constexpr (ZB) {
      if (((x - x0) & 3) == 0) edge_block(x, min(x1, x + 4));
    }
    const MooreEdge<R> &ze = zedge[(x - x0) & 3];
    const int xp = x == NX - 1 ? 0 : x + 1;
    const uint32_t so = (uint32_t)x * PLB + R0;   /* BUF only */
    R Nx[7];
    for (int c = 0; c < 7; ++c) Nx[c] = LC(c, xp, R0, oz);
    const R X = C[4], Y = C[5], Z = C[6];
    const R TXyp = LC(4, x, RP, pz), TZyp = LC(6, x, RP, pz);
    const R TXzp = LC(4, x, R0, ozp), TYzp = LC(5, x, R0, ozp);
    const R TXym = LC(4, x, RM, mz), TYym = LC(5, x, RM, mz), TZym = LC(6, x, RM, mz);
    const R TYxpym = LC(5, xp, RM, mz), TYymzp = LC(5, x, RM, mzp);
    R TZzm = 0, b_xz = 0, b_yz = 0;
    if constexpr (!ZB) {
      const R TXzm = LC(4, x, R0, ozm), TYzm = LC(5, x, R0, ozm);
      TZzm = LC(6, x, R0, ozm);
      const R TZxpzm = LC(6, xp, R0, ozm), TZypzm = LC(6, x, RP, pzm);
      b_xz = TXzm + TZxpzm - X - TZzm;
      b_yz = TYzm + TZypzm - Y - TZzm;
    }

    R Pyp[4], Pym[4], Pzp[4], Pzm[4];
    auto phi_rows = [&](int f) {
      for (int c = 2 * f; c < 2 * f + 2; ++c) {
        Pyp[c] = LC(c, x, RP, pz); Pym[c] = LC(c, x, RM, mz);
        Pzp[c] = LC(c, x, R0, ozp); Pzm[c] = LC(c, x, R0, ozm);
      }
    };
    if (EARLY || ZB)
      for (int f = 0; f < (EARLY ? 2 : 1); ++f) phi_rows(f);

    /* plaquette sines (mooreEvol.cpp:310-333 operand order) */
    const R a_xy = X + Nx[5] - TXyp - Y;
    const R a_xz = X + Nx[6] - TXzp - Z;
    const R a_yx = Y + TXyp - Nx[5] - X;
    const R a_yz = Y + TZyp - TYzp - Z;
    const R a_zx = Z + TXzp - Nx[6] - X;
    const R a_zy = Z + TYzp - TZyp - Y;
    const R b_xy = TXym + TYxpym - X - TYym;
    const R b_zy = TZym + TYymzp - Z - TYym;
    R Qxy, Qxz, Qyx, Qyz, Qzx, Qzy, Qxy_m, Qzy_m, Qxz_m, Qyz_m;
    const uint64_t small = small_lanes(a_xy) & small_lanes(a_xz) & small_lanes(a_yx) & small_lanes(a_yz) &
                           small_lanes(a_zx) & small_lanes(a_zy) & small_lanes(b_xy) & small_lanes(b_zy) &
                           (ZB ? ~0ull : small_lanes(b_xz) & small_lanes(b_yz));
    if (small == __builtin_amdgcn_read_exec()) {
      Qxy = T::sn_small(a_xy); Qxz = T::sn_small(a_xz); Qyx = T::sn_small(a_yx);
      Qyz = T::sn_small(a_yz); Qzx = T::sn_small(a_zx); Qzy = T::sn_small(a_zy);
      Qxy_m = T::sn_small(b_xy); Qzy_m = T::sn_small(b_zy);
      if constexpr (!ZB) { Qxz_m = T::sn_small(b_xz); Qyz_m = T::sn_small(b_yz); }
    } else {
      Qxy = T::sn(a_xy); Qxz = T::sn(a_xz); Qyx = T::sn(a_yx);
      Qyz = T::sn(a_yz); Qzx = T::sn(a_zx); Qzy = T::sn(a_zy);
      Qxy_m = T::sn(b_xy); Qzy_m = T::sn(b_zy);
      if constexpr (!ZB) { Qxz_m = T::sn(b_xz); Qyz_m = T::sn(b_yz); }
    }
    if constexpr (ZB) {   /* the second sines of F_xz, F_yz are lane - 1's first ones */
      Qxz_m = z_back<false, R>(Qxz, ze.qxz, e0);
      Qyz_m = z_back<false, R>(Qyz, ze.qyz, e0);
    }
    const R fxy = dvy(Qxy - Qxy_m);
    const R fxz = dvz(Qxz - Qxz_m);
    const R fyx = dvx(Qyx - Qyx_m);
    const R fyz = dvz(Qyz - Qyz_m);
    const R fzx = dvx(Qzx - Qzx_m);
    const R fzy = dvy(Qzy - Qzy_m);

    const R m1 = C[0] * C[0] + C[1] * C[1];
    const R m2 = C[2] * C[2] + C[3] * C[3];
    const R pot[2] = {k.hl1 * (m1 - k.eta1sq) + k.hl12 * (m2 - k.eta2sq),
                      k.hl2 * (m2 - k.eta2sq) + k.hl12 * (m1 - k.eta1sq)};
    R cur[2][3], acc[2][2], cxs[2], sxs[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int cr = 2 * f, ci = 2 * f + 1;
      R sx, cx, sy, cy, sz, cz, sym_, cym, szm, czm;
      T::sc(q[f] * X, &sx, &cx);
      T::sc(q[f] * Y, &sy, &cy);
      T::sc(q[f] * Z, &sz, &cz);
      T::sc(q[f] * TYym, &sym_, &cym);
      if constexpr (ZB) {
        szm = z_back<false, R>(sz, ze.s[f], e0);
        czm = z_back<false, R>(cz, ze.c[f], e0);
      } else {
        T::sc(q[f] * TZzm, &szm, &czm);
      }
      const R ar = C[cr], ai = C[ci];
      const R rxp = Nx[cr], ixp = Nx[ci];
      if (!EARLY && !(ZB && f == 0)) phi_rows(f);
      const R ryp = Pyp[cr], iyp = Pyp[ci], rym = Pym[cr], iym = Pym[ci];
      const R rzp = Pzp[cr], izp = Pzp[ci], rzm = Pzm[cr], izm = Pzm[ci];
      {
        R lxx = dvx(cx * rxp + sx * ixp - 2 * ar + cxm[f] * Pm[cr] - sxm[f] * Pm[ci]);
        R lyy = dvy(cy * ryp + sy * iyp - 2 * ar + cym * rym - sym_ * iym);
        R lzz = dvz(cz * rzp + sz * izp - 2 * ar + czm * rzm - szm * izm);
        acc[f][0] = lxx + lyy + lzz - pot[f] * ar;
      }
      {
        R lxx = dvx(cx * ixp + (-sx) * rxp - 2 * ai + cxm[f] * Pm[ci] - (-sxm[f]) * Pm[cr]);
        R lyy = dvy(cy * iyp + (-sy) * ryp - 2 * ai + cym * iym - (-sym_) * rym);
        R lzz = dvz(cz * izp + (-sz) * rzp - 2 * ai + czm * izm - (-szm) * rzm);
        acc[f][1] = lxx + lyy + lzz - pot[f] * ai;
      }
      cur[f][0] = q[f] * (cx * (ai * rxp - ar * ixp) + sx * (ar * rxp + ai * ixp));
      cur[f][1] = q[f] * (cy * (ai * ryp - ar * iyp) + sy * (ar * ryp + ai * iyp));
      cur[f][2] = q[f] * (cz * (ai * rzp - ar * izp) + sz * (ar * rzp + ai * izp));
      cxs[f] = cx;
      sxs[f] = sx;
    }
    const R atx = k.m2gg * (cur[0][0] + cur[1][0]) - fxy - fxz;
    const R aty = k.m2gg * (cur[0][1] + cur[1][1]) - fyx - fyz;
    const R atz = k.m2gg * (cur[0][2] + cur[1][2]) - fzx - fzy;
    /* previous level at s: read once, overwritten with level n+1 */
    auto LP = [&](int c) -> R {
      if (BUF) return bld<R, kStream>(FR[c], oz, offP + so);
      return ldo((const R *)O[c] + (size_t)x * NYNZ, R0, oz);
    };
    R Onew[7];
#pragma unroll
    for (int c = 0; c < 4; ++c) Onew[c] = 2 * C[c] - LP(c) + k.dt2 * acc[c >> 1][c & 1];
    Onew[4] = 2 * X - LP(4) + k.dt2 * atx;
    Onew[5] = 2 * Y - LP(5) + k.dt2 * aty;
    Onew[6] = 2 * Z - LP(6) + k.dt2 * atz;
    if (act) {
      for (int c = 0; c < 7; ++c) {
        if (BUF) bst<R, kStream>(FR[c], oz, offP + so, Onew[c]);
        else sto(O[c] + (size_t)x * NYNZ, R0, oz, Onew[c]);
      }
      if constexpr (CHECK)
        for (int c = 0; c < 7; ++c) inband = inband && in_moore_band((double)Onew[c]);
    }
    /* carry */
    for (int c = 0; c < 4; ++c) Pm[c] = C[c];
    for (int f = 0; f < 2; ++f) { cxm[f] = cxs[f]; sxm[f] = sxs[f]; }
    Qyx_m = Qyx;
    Qzx_m = Qzx;
    for (int c = 0; c < 7; ++c) C[c] = Nx[c];
  }
  if constexpr (CHECK) {
    /* one store is enough, and the waves of a launch would queue up for the
     * flag's cache line (a diverged state, 128^3, 11008 waves: 517 us a step,
     * 127 with this; 256^3 1290, 943) */
    if (__builtin_amdgcn_ballot_w64(!inband) != 0 && (threadIdx.x & 63) == 0 &&
        __hip_atomic_load(bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
      __hip_atomic_store(bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

}  // namespace ax

#endif
