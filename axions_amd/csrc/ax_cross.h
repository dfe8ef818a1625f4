/*
 * ax_cross.h - the zeros of phi on one face of the lattice: the FP64 equations
 * of the reference and the FP32 classification that settles most faces before
 * them (cross_kernel, ax_diag.hip).
 */
#ifndef AXIONS_AX_CROSS_H
#define AXIONS_AX_CROSS_H

#include <math.h>

#include <algorithm>

#if defined(__HIPCC__) || defined(__HIP__)
#include <hip/hip_runtime.h>
#endif

namespace ax {

/* How many roots face_roots finds on the face with corners v.. of Re phi
 * and Im phi: 0, 1 or 2, or 3 if FP32 cannot tell, or 4: none if the corners
 * of Re phi or of Im phi, zero in FP32, are zero, else 3.  (With four zeros
 * every coefficient is 0 or not a number, and with a NaN a and disc are NaN:
 * face_roots finds no root.)
 *
 * In coordinates p, q in [0, 1] of the face, phi_c = A + B p + C q + D p q;
 * the roots have a q^2 + b q + c = 0 with a = D1 C0 - D0 C1, b = D1 A0 - D0 A1
 * + B1 C0 - B0 C1, c = B1 A0 - B0 A1, and p = -(A0 + C0 q)/(B0 + D0 q): these
 * are face_roots' equations scaled and shifted.  A value within a bound of a
 * decision is left undecided, and so is a face out of FP32's middle range or
 * not finite: 2e-2 of the faces of random phases, 3e-3 of a damped network's.
 *
 * The bound.  m0, m1: the largest |Re phi|, |Im phi| of the corners, S = m0 m1;
 * u = 2^-24, e = 2^-53; |A| <= m, |B|, |C| <= 2 m, |D| <= 4 m, so |a|, |b| <=
 * 16 S.  To first order, every operation at its largest:
 *   FP32   B, C off by 4 u m, D by 12 u m; a and b by 112 u S, c by 20 u S.
 *   FP64   face_roots works in lattice coordinates; h >= 3.5 is their largest
 *          value in spacings.  Its c1 is off by 9 e m, c2 and c3 by 16 e h m,
 *          c4 by 22 e h^2 m; a by 285 e h S, b by 837 e h^2 S, c by 464 e h^3 S
 *          (coefficients of the coordinate itself, |b| <= |b| + 2 h |a| there).
 *   E = k S with k = max(2^-16, 2^10 e h^3) (cross_bound).
 *   disc   FP32 is off by u S (256 |b| + 80 |a| + 576 |c|), FP64 by e S (3050
 *          h^2 |b| + 6400 h^3 |a| + 1250 h |c|): together below 0.82 F, F = E
 *          (4 |b| + 8 (|a| + |c|) + 16 E).  disc < -F has no root, also where
 *          FP64 finds a = 0 (|a| < E then).  disc > 2 F, |a| > 16 E has two,
 *          and their difference from FP64's is below 0.46 F / root.
 *   q      the numerator over 2 |a|: 0.7 E (FP32's b, its two sums, FP64's a
 *          and b over h) and 0.46 F / root; a's own 0.9 E / |a| for |q| <= 2;
 *          rounding 8 u.  eq = (3 E + F / root) / |a| + 1e-5 holds them.
 *   p      A + C q off by 10 u m0 + 2 m0 eq, FP64's numerator and denominator
 *          by 95 e h^2 m0; en = m0 (2 k + 2 eq), and for B + D q ed = 2 en.
 *
 * Re phi of one sign settles a face by itself: a point is kept only where
 * p = -(A0 + C0 q)/(B0 + D0 q) lies on it, that is where Re phi, a mean of
 * the corners there, vanishes; it is at least lo, and FP64 is off by at most
 * 101 e h^2 hi. */
__device__ __forceinline__ bool one_sign(float a, float b, float c, float d, float k) {
  const float lo = fminf(fminf(a, b), fminf(c, d)), hi = fmaxf(fmaxf(a, b), fmaxf(c, d));
  return (lo > 1e-6f && lo > k * hi && hi < 1e6f) || (hi < -1e-6f && hi < k * lo && lo > -1e6f);
}
__device__ __forceinline__ int face_class(float r00, float r10, float r01, float r11, float i00, float i10, float i01,
                                          float i11, float k) {
  const float m0 = fmaxf(fmaxf(fabsf(r00), fabsf(r10)), fmaxf(fabsf(r01), fabsf(r11)));
  const float m1 = fmaxf(fmaxf(fabsf(i00), fabsf(i10)), fmaxf(fabsf(i01), fabsf(i11)));
  const float B0 = r10 - r00, C0 = r01 - r00, D0 = (r11 - r10) - C0;
  const float B1 = i10 - i00, C1 = i01 - i00, D1 = (i11 - i10) - C1;
  const float a = D1 * C0 - D0 * C1;
  const float b = (D1 * r00 - D0 * i00) + (B1 * C0 - B0 * C1);
  const float c = B1 * r00 - B0 * i00;
  const float E = k * (m0 * m1);
  const float disc = b * b - 4 * (a * c);
  const float F = E * (4 * fabsf(b) + 8 * (fabsf(a) + fabsf(c)) + 16 * E);
  /* not finite makes disc + F NaN or infinite and the tests below fail */
  const bool sane = m0 > 1e-6f && m1 > 1e-6f && m0 < 1e6f && m1 < 1e6f && fabsf(disc) < 1e30f && k < 1;
  if (sane && disc < -F) return 0;
  if (!(sane && disc > 2 * F && fabsf(a) > 16 * E)) {
    if (sane) return 3;
    const bool nan = __builtin_isunordered(r00, r10) || __builtin_isunordered(r01, r11) ||
                     __builtin_isunordered(i00, i10) || __builtin_isunordered(i01, i11);
    return nan ? 0 : m0 == 0 || m1 == 0 ? 4 : 3;
  }
  const float root = __builtin_amdgcn_sqrtf(disc), inv = __builtin_amdgcn_rcpf(2 * a);
  const float eq = (3 * E + F * __builtin_amdgcn_rcpf(root)) * fabsf(2 * inv) * 1.01f + 1e-5f;
  const float en = m0 * (2 * k + 2 * eq), ed = 2 * en;
  int n = 0;
  bool sure = true;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float q = ((s ? -root : root) - b) * inv;
    const float num = -(r00 + C0 * q), den = B0 + D0 * q;
    const float t0 = den < 0 ? -num : num, t1 = fabsf(den) - t0;
    const bool in = q > eq && q < 1 - eq && t0 > en && t1 > en + ed;
    const bool out = q < -eq || q > 1 + eq || (fabsf(den) > ed && (t0 < -en || t1 < -(en + ed)));
    n += in ? 1 : 0;
    sure = sure && (in || out);
  }
  return sure ? n : 3;
}

/* Solve the face of mpi_evolution.cpp:552-623: its roots inside the face
 * (0..2), the + root before the - root. */
__device__ __forceinline__ int face_roots(const double v00[2], const double v10[2], const double v01[2],
                                          const double v11[2], double u, double du, double w, double dw,
                                          double &r1, double &r2, double &q1, double &q2) {
  double c1[2], c2[2], c3[2], c4[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    c1[c] = v11[c] - v10[c] - v01[c] + v00[c];
    c2[c] = (w + dw) * (v10[c] - v00[c]) + w * (v01[c] - v11[c]);
    c3[c] = (u + du) * (v01[c] - v00[c]) + u * (v10[c] - v11[c]);
    c4[c] = (u + du) * ((w + dw) * v00[c] - w * v01[c]) - u * ((w + dw) * v10[c] - w * v11[c]);
  }
  const double a = c1[1] * c3[0] - c1[0] * c3[1];
  const double b = c1[1] * c4[0] + c2[1] * c3[0] - c1[0] * c4[1] - c2[0] * c3[1];
  const double c = c2[1] * c4[0] - c2[0] * c4[1];
  const double disc = b * b - 4 * a * c;
  auto inside = [&](double s2, double &s1) {
    s1 = 0;
    if (!(s2 >= w && s2 <= w + dw)) return false;
    s1 = -(c3[0] * s2 + c4[0]) / (c1[0] * s2 + c2[0]);
    return s1 >= u && s1 <= u + du;
  };
  int n = 0;
  if (a == 0) {
    if (b != 0) {
      r2 = -c / b;
      n = inside(r2, r1) ? 1 : 0;
    }
  } else if (disc >= 0) {
    const double root = sqrt(disc);
    double s1, s2 = (-b + root) / (2 * a);
    if (inside(s2, s1)) {
      r1 = s1;
      r2 = s2;
      n = 1;
    }
    s2 = (-b - root) / (2 * a);
    if (inside(s2, s1)) {
      if (n) {
        q1 = s1;
        q2 = s2;
      } else {
        r1 = s1;
        r2 = s2;
      }
      ++n;
    }
  }
  return n;
}

/* face_class's k for a lattice; 2 (every face in FP64) where it would decide
 * little, or where face_roots' products, up to the fourth power of a spacing,
 * leave FP64's range. */
inline float cross_bound(int nx, int ny, int nz, double dx, double dy, double dz) {
  const double h = 0.5 * std::max(nx, std::max(ny, nz)) + 2;
  const double k = std::max(0x1p-16, 0x1p-43 * h * h * h);
  const double lo = std::min(dx, std::min(dy, dz)), hi = std::max(dx, std::max(dy, dz));
  return k < 0x1p-8 && lo > 1e-60 && hi < 1e60 ? (float)k : 2.0f;
}

}  // namespace ax

#endif
