/*
 * User QFunctions for operators whose output stays at the quadrature points,
 * and for several passive fields: every kind of input the run-time compiled
 * kernels take, in an order that is not theirs.
 */
#include <ceed/types.h>

struct PointsContext {
  double a, b;
};

/* w (a |u|^2 + b sum_dc du_dc f_(dc mod 2)) + g, and a second value, of a field
 * of NC components: inputs f (2), du, w, u, g (1) */
#define MIXED_AT_POINTS(name, NC)                                                                                     \
  CEED_QFUNCTION(name)(void *ctx, const CeedInt Q, const CeedScalar *const *in, CeedScalar *const *out) {             \
    const struct PointsContext *c = (const struct PointsContext *)ctx;                                                \
    const CeedScalar           *f = in[0], *du = in[1], *w = in[2], *u = in[3], *g = in[4];                           \
    for (CeedInt i = 0; i < Q; i++) {                                                                                 \
      CeedScalar s = 0, t = 0;                                                                                        \
      for (CeedInt k = 0; k < NC; k++) s += u[k * Q + i] * u[k * Q + i];                                              \
      for (CeedInt k = 0; k < 3 * NC; k++) t += du[k * Q + i] * f[(k % 2) * Q + i] * (k + 1);                         \
      out[0][0 * Q + i] = w[i] * (c->a * s + c->b * t) + g[i];                                                        \
      out[0][1 * Q + i] = u[(NC - 1) * Q + i] - 2 * du[(3 * NC - 1) * Q + i];                                         \
    }                                                                                                                 \
    return 0;                                                                                                         \
  }
MIXED_AT_POINTS(mixed_at_points_1, 1)
MIXED_AT_POINTS(mixed_at_points_2, 2)
MIXED_AT_POINTS(mixed_at_points_3, 3)

/* values only, no gradient: out = (u + 1) f */
CEED_QFUNCTION(values_at_points)(void *ctx, const CeedInt Q, const CeedScalar *const *in, CeedScalar *const *out) {
  for (CeedInt i = 0; i < Q; i++) out[0][i] = (in[0][i] + 1) * in[1][i];
  return 0;
}

/* three passive fields around the active ones: v = f u + g0, dv = h du */
CEED_QFUNCTION(three_passive)(void *ctx, const CeedInt Q, const CeedScalar *const *in, CeedScalar *const *out) {
  const CeedScalar *f = in[0], *u = in[1], *g = in[2], *du = in[3], *h = in[4];
  for (CeedInt i = 0; i < Q; i++) {
    out[1][i] = f[i] * u[i] + g[0 * Q + i] * g[1 * Q + i];
    for (CeedInt d = 0; d < 3; d++) out[0][d * Q + i] = h[d * Q + i] * du[d * Q + i];
  }
  return 0;
}
