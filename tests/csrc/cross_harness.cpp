// Test harness: the face classification of the crossings
// (axions_amd/csrc/ax_cross.h) on the CPU, its device square root and
// reciprocal replaced by values up to one unit in the last place off; built by
// tests/test_face_class.py with g++ -ffp-contract=off.
#include <math.h>
#include <stdint.h>

#include <random>

#define __device__
#define __forceinline__ inline
static thread_local uint32_t ulp_state = 1;
static float off_by_an_ulp(float v) {
  ulp_state = ulp_state * 1664525u + 1013904223u;
  const uint32_t r = ulp_state >> 30;
  return r == 0 ? nextafterf(v, INFINITY) : r == 1 ? nextafterf(v, -INFINITY) : v;
}
#define __builtin_amdgcn_sqrtf(x) off_by_an_ulp(sqrtf(x))
#define __builtin_amdgcn_rcpf(x) off_by_an_ulp(1.0f / (x))
#include "../../axions_amd/csrc/ax_cross.h"

// Corners 00, 10, 01, 11 of one face.
struct Face {
  double r[4], i[4];
};

static Face draw(std::mt19937_64 &g, int kind) {
  std::uniform_real_distribution<double> u(-1, 1), w(0, 1);
  std::normal_distribution<double> n;
  Face f;
  auto bilinear = [](double A, double B, double C, double D, double *v) {
    v[0] = A;
    v[1] = A + B;
    v[2] = A + C;
    v[3] = A + B + C + D;
  };
  if (kind == 0) {                       // random phases
    for (int c = 0; c < 4; ++c) {
      const double a = 3.14159265358979 * u(g);
      f.r[c] = cos(a);
      f.i[c] = sin(a);
    }
  } else if (kind == 1) {                // every corner by itself, scales apart
    const double s = exp(9 * u(g)), t = exp(9 * u(g));
    for (int c = 0; c < 4; ++c) {
      f.r[c] = s * n(g);
      f.i[c] = t * n(g);
    }
  } else if (kind == 2) {                // smooth, with a zero near or on the face
    const double e = pow(10, -4 * w(g)), p = 1.2 * w(g) - 0.1, q = 1.2 * w(g) - 0.1;
    for (double *v : {f.r, f.i}) {
      const double B = u(g), C = u(g), D = e * u(g);
      bilinear(-(B * p + C * q + D * p * q), B, C, D, v);
    }
  } else if (kind == 3) {                // a zero within rounding of an edge or a corner
    const double d = pow(10, -2 - 14 * w(g)) * u(g);
    const double p = w(g) < 0.5 ? (w(g) < 0.5 ? d : 1 + d) : w(g), q = w(g) < 0.7 ? (w(g) < 0.5 ? d : 1 + d) : w(g);
    for (double *v : {f.r, f.i}) {
      const double B = n(g), C = n(g), D = n(g);
      bilinear(-(B * p + C * q + D * p * q), B, C, D, v);
    }
  } else if (kind == 4) {                // two zeros close together
    const double p = w(g), q = w(g), d = pow(10, -1 - 8 * w(g));
    const double p2 = p + d * u(g), q2 = q + d * u(g);
    for (double *v : {f.r, f.i}) {
      // A + B p + C q + D p q = 0 at (p, q) and (p2, q2), for given C, D
      const double C = n(g), D = n(g);
      const double B = p2 == p ? n(g) : -(C * (q2 - q) + D * (p2 * q2 - p * q)) / (p2 - p);
      bilinear(-(B * p + C * q + D * p * q), B, C, D, v);
    }
  } else if (kind == 5) {                // Re phi barely of one sign
    const double s = u(g) < 0 ? -1 : 1;
    for (int c = 0; c < 4; ++c) {
      f.r[c] = s * w(g);
      f.i[c] = n(g);
    }
    f.r[(int)(4 * w(g)) & 3] = s * pow(10, -7 * w(g)) * (w(g) < 0.3 ? -1 : 1);
  } else if (kind == 7) {                // zeros, NaNs, infinities, values FP32 does not hold
    const double odd[6] = {0, -0.0, NAN, INFINITY, 1e-200, 1e200};
    for (int c = 0; c < 4; ++c) {
      f.r[c] = n(g);
      f.i[c] = n(g);
    }
    const int every = (int)(g() % 3);    // one corner; all of Re phi; all of Im phi
    const double v = odd[g() % 6], s = w(g) < 0.5 ? 1 : 1 + w(g);
    if (every == 0) (g() & 1 ? f.r : f.i)[g() & 3] = v;
    else
      for (int c = 0; c < 4; ++c) (every == 1 ? f.r : f.i)[c] = v * (c & 1 ? s : 1);
  } else {                               // q's equation nearly linear
    const double t = pow(10, -1 - 12 * w(g));
    double B0 = n(g), C0 = n(g), D0 = n(g), k = n(g), p = w(g), q = w(g);
    bilinear(-(B0 * p + C0 * q + D0 * p * q), B0, C0, D0, f.r);
    const double B1 = n(g), C1 = k * C0, D1 = k * D0 * (1 + t * u(g));
    bilinear(-(B1 * p + C1 * q + D1 * p * q), B1, C1, D1, f.i);
  }
  return f;
}

extern "C" {
// n faces of one kind at random places of an nx x ny x nz lattice, as the
// count pass treats them: out[0] undecided, out[1] settled with another number
// of roots than face_roots finds, out[2] settled by the sign of Re phi.
// fp32: the corners hold FP32 values.
void check_faces(int kind, long long n, unsigned seed, int nx, int ny, int nz, double d, int fp32, float k,
                 long long *out) {
  std::mt19937_64 g(seed);
  if (k == 0) k = ax::cross_bound(nx, ny, nz, d, d, d);
  const int dims[3] = {nx, ny, nz};
  for (long long s = 0; s < n; ++s) {
    Face f = draw(g, kind);
    if (fp32)
      for (int c = 0; c < 4; ++c) {
        f.r[c] = (float)f.r[c];
        f.i[c] = (float)f.i[c];
      }
    const int a = (int)(g() % 3), b = (a + 1 + (int)(g() % 2)) % 3;
    // half of the faces at the lattice's ends, where coordinates are largest
    auto at = [&](int m) { return g() & 1 ? (g() & 1 ? 0 : m - 1) : (int)(g() % m); };
    const double x = (at(dims[a]) - int(0.5 * (dims[a] - 1))) * d, y = (at(dims[b]) - int(0.5 * (dims[b] - 1))) * d;
    int got = 0;
    const float r[4] = {(float)f.r[0], (float)f.r[1], (float)f.r[2], (float)f.r[3]};
    if (ax::one_sign(r[0], r[1], r[2], r[3], k)) {
      ++out[2];
    } else {
      got = ax::face_class(r[0], r[1], r[2], r[3], (float)f.i[0], (float)f.i[1], (float)f.i[2], (float)f.i[3], k);
      auto zero = [](const double *v) { return v[0] == 0 && v[1] == 0 && v[2] == 0 && v[3] == 0; };
      if (got == 4) got = zero(f.r) || zero(f.i) ? 0 : 3;
    }
    if (got == 3) {
      ++out[0];
      continue;
    }
    double p0, p1, p2, p3;
    const double v00[2] = {f.r[0], f.i[0]}, v10[2] = {f.r[1], f.i[1]}, v01[2] = {f.r[2], f.i[2]}, v11[2] = {f.r[3], f.i[3]};
    if (ax::face_roots(v00, v10, v01, v11, x, d, y, d, p0, p1, p2, p3) != got) ++out[1];
  }
}
float cross_bound(int nx, int ny, int nz, double dx, double dy, double dz) {
  return ax::cross_bound(nx, ny, nz, dx, dy, dz);
}
}
