/*
 * The backend's choice between its paths, on the CPU: the core, the backend
 * and the CPU stand-in for the kernel library (tests/c/plugin) in one program.
 * CeedElemRestrictionHasBackendStrides is wrapped to answer as libCEED's core
 * does: an error for a restriction without strides.
 *
 * The operators are those of tests/qfunctions/t-points.h on two trilinear
 * hexes: values at the quadrature points (mixed_at_points_3), and a nodal
 * result with three passive fields, one of them on an offset restriction
 * (three_passive); each also with an output that is one of its inputs.
 * Usage: points-backend <t-points.h>; prints the sums of Apply and of ApplyAdd
 * of each.
 */
#include <ceed.h>
#include <ceed/backend.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define CHECK(call)                                                       \
  do {                                                                    \
    int ierr_ = (call);                                                   \
    if (ierr_) {                                                          \
      printf("FAIL: %s returned %d (line %d)\n", #call, ierr_, __LINE__); \
      exit(1);                                                            \
    }                                                                     \
  } while (0)

int __real_CeedElemRestrictionHasBackendStrides(CeedElemRestriction rstr, bool *has_backend_strides);
int __wrap_CeedElemRestrictionHasBackendStrides(CeedElemRestriction rstr, bool *has_backend_strides) {
  CeedRestrictionType type;
  CHECK(CeedElemRestrictionGetType(rstr, &type));
  if (type != CEED_RESTRICTION_STRIDED) {
    printf("CeedElemRestriction has no stride data\n");
    return CEED_ERROR_MINOR;
  }
  return __real_CeedElemRestrictionHasBackendStrides(rstr, has_backend_strides);
}

enum { E = 2, P = 2, Q = 3, NQ = Q * Q * Q, NN = 12 };
static Ceed        ceed;
static const char *qf_file;

static double value(unsigned *s) {
  *s = *s * 1664525u + 1013904223u;
  return (*s >> 8) / 16777216.0;
}

static CeedVector vector(CeedSize n, unsigned seed) {
  CeedVector  v;
  CeedScalar *a;
  CHECK(CeedVectorCreate(ceed, n, &v));
  CHECK(CeedVectorGetArrayWrite(v, CEED_MEM_HOST, &a));
  for (CeedSize i = 0; i < n; i++) a[i] = value(&seed);
  CHECK(CeedVectorRestoreArray(v, &a));
  return v;
}

static void report(const char *what, CeedVector v) {
  CeedSize          n;
  const CeedScalar *a;
  double            s = 0;
  CHECK(CeedVectorGetLength(v, &n));
  CHECK(CeedVectorGetArrayRead(v, CEED_MEM_HOST, &a));
  for (CeedSize i = 0; i < n; i++) s += a[i] * (1 + i % 13);
  CHECK(CeedVectorRestoreArrayRead(v, &a));
  printf("%s %.17g\n", what, s);
}

static CeedQFunction qfunction(const char *name) {
  char          source[4096];
  CeedQFunction qf;
  snprintf(source, sizeof(source), "%s:%s", qf_file, name);
  CHECK(CeedQFunctionCreateInterior(ceed, 1, NULL, source, &qf));
  return qf;
}

static CeedElemRestriction strided(CeedInt nc) {
  CeedElemRestriction r;
  CHECK(CeedElemRestrictionCreateStrided(ceed, E, NQ, nc, (CeedSize)E * NQ * nc, CEED_STRIDES_BACKEND, &r));
  return r;
}

static void apply_both(const char *what, CeedOperator op, CeedVector in, CeedVector out) {
  char name[100];
  CHECK(CeedOperatorApply(op, in, out, CEED_REQUEST_IMMEDIATE));
  snprintf(name, sizeof(name), "%s-apply", what);
  report(name, out);
  CHECK(CeedOperatorApplyAdd(op, in, out, CEED_REQUEST_IMMEDIATE));
  snprintf(name, sizeof(name), "%s-add", what);
  report(name, out);
}

int main(int argc, char **argv) {
  CeedInt off[E * P * P * P], point_off[E * NQ];
  if (argc < 2) return 2;
  qf_file = argv[1];
  CHECK(CeedInit("/gpu/hip/mi355", &ceed));
  for (int e = 0, i = 0; e < E; e++)
    for (int z = 0; z < 2; z++)
      for (int y = 0; y < 2; y++)
        for (int x = 0; x < 2; x++) off[i++] = (z * 2 + y) * 3 + x + e;
  for (int i = 0; i < E * NQ; i++) point_off[i] = (i * 5) % (E * NQ);

  { /* values at the quadrature points: f, du, w, u, g -> 2 values */
    double               ctx_data[2] = {0.7, -0.3};
    CeedQFunction        qf          = qfunction("mixed_at_points_3");
    CeedQFunctionContext ctx;
    CeedElemRestriction  ru, rf = strided(2), rg = strided(1);
    CeedBasis            basis;
    CeedOperator         op;
    CeedVector           u = vector(3 * NN, 1), f = vector(E * NQ * 2, 2), g = vector(E * NQ, 3), out = vector(E * NQ * 2, 4);
    CHECK(CeedElemRestrictionCreate(ceed, E, P * P * P, 3, NN, 3 * NN, CEED_MEM_HOST, CEED_COPY_VALUES, off, &ru));
    CHECK(CeedBasisCreateTensorH1Lagrange(ceed, 3, 3, P, Q, CEED_GAUSS, &basis));
    CHECK(CeedQFunctionContextCreate(ceed, &ctx));
    CHECK(CeedQFunctionContextSetData(ctx, CEED_MEM_HOST, CEED_COPY_VALUES, sizeof(ctx_data), ctx_data));
    CHECK(CeedQFunctionSetContext(qf, ctx));
    CHECK(CeedQFunctionAddInput(qf, "f", 2, CEED_EVAL_NONE));
    CHECK(CeedQFunctionAddInput(qf, "du", 9, CEED_EVAL_GRAD));
    CHECK(CeedQFunctionAddInput(qf, "w", 1, CEED_EVAL_WEIGHT));
    CHECK(CeedQFunctionAddInput(qf, "u", 3, CEED_EVAL_INTERP));
    CHECK(CeedQFunctionAddInput(qf, "g", 1, CEED_EVAL_NONE));
    CHECK(CeedQFunctionAddOutput(qf, "out", 2, CEED_EVAL_NONE));
    CHECK(CeedOperatorCreate(ceed, qf, CEED_QFUNCTION_NONE, CEED_QFUNCTION_NONE, &op));
    CHECK(CeedOperatorSetField(op, "f", rf, CEED_BASIS_NONE, f));
    CHECK(CeedOperatorSetField(op, "du", ru, basis, CEED_VECTOR_ACTIVE));
    CHECK(CeedOperatorSetField(op, "w", CEED_ELEMRESTRICTION_NONE, basis, CEED_VECTOR_NONE));
    CHECK(CeedOperatorSetField(op, "u", ru, basis, CEED_VECTOR_ACTIVE));
    CHECK(CeedOperatorSetField(op, "g", rg, CEED_BASIS_NONE, g));
    CHECK(CeedOperatorSetField(op, "out", rf, CEED_BASIS_NONE, CEED_VECTOR_ACTIVE));
    apply_both("points", op, u, out);
    apply_both("points-in-place", op, u, f); /* the output is also a passive input */
    CHECK(CeedOperatorDestroy(&op));
    CHECK(CeedQFunctionContextDestroy(&ctx));
    CHECK(CeedQFunctionDestroy(&qf));
    CHECK(CeedBasisDestroy(&basis));
    CHECK(CeedElemRestrictionDestroy(&ru));
    CHECK(CeedElemRestrictionDestroy(&rf));
    CHECK(CeedElemRestrictionDestroy(&rg));
    CHECK(CeedVectorDestroy(&u));
    CHECK(CeedVectorDestroy(&f));
    CHECK(CeedVectorDestroy(&g));
    CHECK(CeedVectorDestroy(&out));
  }

  { /* three passive fields: f, u, g, du, h -> dv, v */
    CeedQFunction       qf = qfunction("three_passive");
    CeedElemRestriction ru, rf, rg = strided(2), rh = strided(3);
    CeedBasis           basis;
    CeedOperator        op;
    CeedVector          u = vector(NN, 1), f = vector(E * NQ, 2), g = vector(E * NQ * 2, 3), h = vector(E * NQ * 3, 4), out = vector(NN, 5);
    CHECK(CeedElemRestrictionCreate(ceed, E, P * P * P, 1, 1, NN, CEED_MEM_HOST, CEED_COPY_VALUES, off, &ru));
    CHECK(CeedElemRestrictionCreate(ceed, E, NQ, 1, 1, E * NQ, CEED_MEM_HOST, CEED_COPY_VALUES, point_off, &rf));
    CHECK(CeedBasisCreateTensorH1Lagrange(ceed, 3, 1, P, Q, CEED_GAUSS, &basis));
    CHECK(CeedQFunctionAddInput(qf, "f", 1, CEED_EVAL_NONE));
    CHECK(CeedQFunctionAddInput(qf, "u", 1, CEED_EVAL_INTERP));
    CHECK(CeedQFunctionAddInput(qf, "g", 2, CEED_EVAL_NONE));
    CHECK(CeedQFunctionAddInput(qf, "du", 3, CEED_EVAL_GRAD));
    CHECK(CeedQFunctionAddInput(qf, "h", 3, CEED_EVAL_NONE));
    CHECK(CeedQFunctionAddOutput(qf, "dv", 3, CEED_EVAL_GRAD));
    CHECK(CeedQFunctionAddOutput(qf, "v", 1, CEED_EVAL_INTERP));
    CHECK(CeedOperatorCreate(ceed, qf, CEED_QFUNCTION_NONE, CEED_QFUNCTION_NONE, &op));
    CHECK(CeedOperatorSetField(op, "f", rf, CEED_BASIS_NONE, f));
    CHECK(CeedOperatorSetField(op, "u", ru, basis, CEED_VECTOR_ACTIVE));
    CHECK(CeedOperatorSetField(op, "g", rg, CEED_BASIS_NONE, g));
    CHECK(CeedOperatorSetField(op, "du", ru, basis, CEED_VECTOR_ACTIVE));
    CHECK(CeedOperatorSetField(op, "h", rh, CEED_BASIS_NONE, h));
    CHECK(CeedOperatorSetField(op, "dv", ru, basis, CEED_VECTOR_ACTIVE));
    CHECK(CeedOperatorSetField(op, "v", ru, basis, CEED_VECTOR_ACTIVE));
    apply_both("passive", op, u, out);
    apply_both("passive-in-place", op, out, out);
    CHECK(CeedOperatorDestroy(&op));
    CHECK(CeedQFunctionDestroy(&qf));
    CHECK(CeedBasisDestroy(&basis));
    CHECK(CeedElemRestrictionDestroy(&ru));
    CHECK(CeedElemRestrictionDestroy(&rf));
    CHECK(CeedElemRestrictionDestroy(&rg));
    CHECK(CeedElemRestrictionDestroy(&rh));
    CHECK(CeedVectorDestroy(&u));
    CHECK(CeedVectorDestroy(&f));
    CHECK(CeedVectorDestroy(&g));
    CHECK(CeedVectorDestroy(&h));
    CHECK(CeedVectorDestroy(&out));
  }
  CHECK(CeedDestroy(&ceed));
  return 0;
}
