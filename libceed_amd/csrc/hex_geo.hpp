// Geometric factors of a trilinear hex, recomputed from the element's vertices.
//
// With the mesh basis of two nodes per direction the map of an element is
//   x(xi, eta, zeta) = sum_{ijk in {0,1}} c_ijk xi^i eta^j zeta^k,
// 21 numbers per element that matter to the Jacobian (c_000 does not), against
// 6 Q^3 stored factors: at Q = 6 the stored factors are 10.4 kB per element and
// seven tenths of the diffusion apply's bytes, the coefficients 0.2 kB.  On
// the column (xi, eta) of quadrature points the three columns of the Jacobian
// are linear in zeta (and the third constant), so a point costs two vector
// fmas, three cross products, one division and the six dot products of
//   (w / det J) adj(J) adj(J)^T.
//
// Every kernel that needs the factors (the stored q_data of the plan and the
// fused kernels that recompute them) calls the functions below, in which each
// rounding is written out, so the values are the same bits everywhere.
#pragma once

#include <hip/hip_runtime.h>

namespace mi355 {

// doubles per element: the vectors c_100, c_010, c_001, c_110, c_101, c_011, c_111, and 3 unused (192 bytes)
constexpr int kGeoStride = 24;
// and in LDS, where a multiple of 8 would put the elements of a wavefront on the same banks
constexpr int kGeoLds = 26;

// Jacobian columns on one column of quadrature points: d/dxi = p0 + zeta q0,
// d/deta = p1 + zeta q1, d/dzeta = c
struct GeoColumn {
  double p0[3], q0[3], p1[3], q1[3], c[3];
  __device__ __forceinline__ void load(const double *g, double xi, double eta) {
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const double c100 = g[d], c010 = g[3 + d], c001 = g[6 + d], c110 = g[9 + d], c101 = g[12 + d], c011 = g[15 + d], c111 = g[18 + d];
      p0[d] = __builtin_fma(eta, c110, c100);
      q0[d] = __builtin_fma(eta, c111, c101);
      p1[d] = __builtin_fma(xi, c110, c010);
      q1[d] = __builtin_fma(xi, c111, c011);
      c[d]  = __builtin_fma(eta, q1[d], __builtin_fma(xi, c101, c001));
    }
  }
};

// a x b, each entry rounded as fma(a, b, -round(a b))
__device__ __forceinline__ void geo_cross(const double (&a)[3], const double (&b)[3], double (&r)[3]) {
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int i = (d + 1) % 3, j = (d + 2) % 3;
    r[d] = __builtin_fma(a[i], b[j], -(a[j] * b[i]));
  }
}
__device__ __forceinline__ double geo_dot(const double (&a)[3], const double (&b)[3]) {
  return __builtin_fma(a[2], b[2], __builtin_fma(a[1], b[1], a[0] * b[0]));
}

// w / x with 1 / x to within two units in the last place: the hardware's
// reciprocal and two Newton steps, which turn the infinite reciprocal of 0 into
// NaN, so the last instruction puts the division's own result where x or w is 0,
// infinite or NaN (7 instructions; the IEEE division takes 11).  An element of
// no volume then has the factors the division gives it, infinite or NaN
// (without that instruction NaN throughout, and at 8M DoFs p=1 0.965 ms
// against 0.979, p=2 0.408 against 0.417, p=4 0.2420 against 0.2426).
__device__ __forceinline__ double geo_div(double w, double x) {
  double r = __builtin_amdgcn_rcp(x);
  r        = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  r        = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_amdgcn_div_fixup(w * r, x, w);
}

// w (d/dxi x d/deta) . d/dzeta = w det J  (Mass3DBuild)
__device__ __forceinline__ double geo_mass(const GeoColumn &k, double zeta, double w) {
  double a[3], b[3], n[3];
#pragma unroll
  for (int d = 0; d < 3; d++) a[d] = __builtin_fma(zeta, k.q0[d], k.p0[d]), b[d] = __builtin_fma(zeta, k.q1[d], k.p1[d]);
  geo_cross(a, b, n);
  return w * geo_dot(n, k.c);
}

// (w / det J) adj(J) adj(J)^T in Voigt order {xx, yy, zz, yz, xz, xy}  (Poisson3DBuild), J = (a b c)
__device__ __forceinline__ void geo_poisson(const double (&a)[3], const double (&b)[3], const double (&c)[3], double w, double (&s)[6]) {
  double A0[3], A1[3], A2[3];
  geo_cross(b, c, A0);
  geo_cross(c, a, A1);
  geo_cross(a, b, A2);
  const double qw = geo_div(w, geo_dot(a, A0));
  s[0] = qw * geo_dot(A0, A0);
  s[1] = qw * geo_dot(A1, A1);
  s[2] = qw * geo_dot(A2, A2);
  s[3] = qw * geo_dot(A1, A2);
  s[4] = qw * geo_dot(A0, A2);
  s[5] = qw * geo_dot(A0, A1);
}
__device__ __forceinline__ void geo_poisson(const GeoColumn &k, double zeta, double w, double (&s)[6]) {
  double a[3], b[3];
#pragma unroll
  for (int d = 0; d < 3; d++) a[d] = __builtin_fma(zeta, k.q0[d], k.p0[d]), b[d] = __builtin_fma(zeta, k.q1[d], k.p1[d]);
  geo_poisson(a, b, k.c, w, s);
}

}  // namespace mi355
