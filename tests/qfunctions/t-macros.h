/*
 * User QFunctions whose source defines macros with short names, among them
 * names that the run-time compiled kernels use for their template parameters
 * and variables.
 */
#include <ceed/types.h>

#define E 2.5
#define P 0.25
#define X(a) (E * (a))
#define NC 3

/* out = w E |u|^2 + P f, of a field of three components: inputs u, w, f */
CEED_QFUNCTION(macros_at_points)(void *ctx, const CeedInt Q, const CeedScalar *const *in, CeedScalar *const *out) {
  for (CeedInt i = 0; i < Q; i++) {
    CeedScalar s = 0;
    for (CeedInt k = 0; k < NC; k++) s += in[0][k * Q + i] * in[0][k * Q + i];
    out[0][i] = X(in[1][i] * s) + P * in[2][i];
  }
  return 0;
}

/* dv = E f du, v = P g u: inputs du, u, f, g */
CEED_QFUNCTION(macros_two_passive)(void *ctx, const CeedInt Q, const CeedScalar *const *in, CeedScalar *const *out) {
  for (CeedInt i = 0; i < Q; i++) {
    for (CeedInt d = 0; d < 3; d++) out[0][d * Q + i] = X(in[2][i] * in[0][d * Q + i]);
    out[1][i] = P * in[3][i] * in[1][i];
  }
  return 0;
}

/* v = P q u: inputs u, q */
CEED_QFUNCTION(macros_mass)(void *ctx, const CeedInt Q, const CeedScalar *const *in, CeedScalar *const *out) {
  for (CeedInt i = 0; i < Q; i++) out[0][i] = P * in[1][i] * in[0][i];
  return 0;
}
