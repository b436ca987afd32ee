/*
 * CeedOperator for /gpu/hip/mi355.
 *
 * Fused path: an operator made of one gallery pointwise operator
 * (MassApply, Vector3MassApply, Poisson3DApply, Vector3Poisson3DApply), an
 * active field with a standard restriction and a 3D tensor basis used for both
 * input and output, and passive geometric factors (EVAL_NONE), runs as one
 * fused kernel: v (+)= E^T B^T D B E u, whose E^T is completed without
 * atomics by an ordered gather over the transpose offset map (see the
 * CeedMi355OperatorCreateHex plan).  This is the path of the reference's
 * fused GPU backends (backends/hip-gen/ceed-hip-gen-operator.c:52-258),
 * rebuilt for gfx950.
 *
 * Fused path, run-time compiled: an operator whose pointwise function is a
 * user (or any non-inlined) QFunction, with scalar active fields on one
 * standard restriction and one 3D tensor basis (inputs INTERP and/or GRAD,
 * outputs INTERP and/or GRAD) and passive EVAL_NONE inputs, runs as one fused
 * kernel too: the QFunction source is compiled with hipRTC into
 * the line-layout kernel (CeedMi355OperatorCreateHexJit), the role of the
 * reference's hip-gen backend (backends/hip-gen/ceed-hip-gen-operator-build.cpp).
 * So does one whose output stays at the quadrature points (geometric factors
 * from coordinates: CeedMi355PointOperatorCreate).
 * CEED_MI355_FUSE_QFUNCTIONS=0 keeps such operators on the generic path.
 *
 * Generic path (any other operator): the staged apply of the reference
 * backends (backends/hip-ref/ceed-hip-ref-operator.c:258-638 and
 * backends/ref/ceed-ref-operator.c:145-500): E-vectors for all elements,
 * basis apply, the run-time compiled QFunction over every point, transposed
 * basis, and the ordered E^T.  Passive inputs are restricted again only when
 * their vector's state changes.
 */
#include <stdlib.h>
#include <string.h>

#include "ceed-mi355-backend.h"

typedef struct {
  bool     is_set_up, fused, jit;
  /* fused path */
  CeedMi355Operator hex;
  CeedSize          l_size;
  CeedInt           num_passive; /* passive inputs held in the plan: their fields, in order, and sizes */
  CeedInt           passive_field[CEED_FIELD_MAX], passive_size[CEED_FIELD_MAX];
  uint64_t          passive_state[CEED_FIELD_MAX];
  bool              passive_valid[CEED_FIELD_MAX];
  /* values at the quadrature points (CeedMi355PointOperator) */
  CeedMi355PointOperator points;
  CeedSize               points_size; /* E-vector length of the output */
  /* generic path */
  bool     is_staged; /* generic_setup has run */
  CeedInt  num_in, num_out, num_elem, Q;
  double  *e_in[CEED_FIELD_MAX], *q_in[CEED_FIELD_MAX];
  double  *e_out[CEED_FIELD_MAX], *q_out[CEED_FIELD_MAX];
  bool     q_in_is_e[CEED_FIELD_MAX], q_out_is_e[CEED_FIELD_MAX];
  uint64_t in_state[CEED_FIELD_MAX];
  bool     in_valid[CEED_FIELD_MAX];
} OperatorData;

/* Whether a restriction has the backend's strides; libCEED answers
 * CeedElemRestrictionHasBackendStrides for strided restrictions only and
 * raises an error for the others. */
static int has_backend_strides(CeedElemRestriction rstr, bool *backend) {
  CeedRestrictionType type;
  *backend = false;
  CeedCallBackend(CeedElemRestrictionGetType(rstr, &type));
  if (type == CEED_RESTRICTION_STRIDED) CeedCallBackend(CeedElemRestrictionHasBackendStrides(rstr, backend));
  return CEED_ERROR_SUCCESS;
}

/* E-vector of qdata in [elem][comp][qpt]: the field's L-vector itself when its
 * restriction has the backend strides, else a temporary restricted copy. */
static int qdata_evector(Ceed ceed, CeedElemRestriction rstr, CeedVector vec, const double **e, double **temp) {
  bool        backend;
  CeedScalar *dl;
  *temp = NULL;
  CeedCallBackend(CeedMi355VectorDevice(vec, false, &dl));
  CeedCallBackend(has_backend_strides(rstr, &backend));
  if (backend) {
    *e = dl;
    return CEED_ERROR_SUCCESS;
  }
  RestrictionData *rd;
  CeedSize         e_size;
  CeedCallBackend(CeedElemRestrictionGetData(rstr, &rd));
  CeedCallBackend(CeedElemRestrictionGetEVectorSize(rstr, &e_size));
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355Malloc(sizeof(double) * (size_t)e_size, (void **)temp)));
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355RestrictionApply(rd->handle, CEED_NOTRANSPOSE, dl, *temp, NULL)));
  *e = *temp;
  return CEED_ERROR_SUCCESS;
}

/* ------------------------------------------------------------------------ */
/* fused path                                                                */
/* ------------------------------------------------------------------------ */
static bool ends_with(const char *s, const char *suffix) {
  const size_t ls = s ? strlen(s) : 0, lx = strlen(suffix);
  return ls >= lx && !strcmp(s + ls - lx, suffix);
}

/* Gallery pointwise operators the fused kernel inlines, recognised by kernel
 * name and source file: this library's gallery header, or the reference
 * gallery's files when the backend is built into a libCEED library
 * (include/ceed/jit-source/gallery/ceed-{massapply,vectormassapply,
 * poisson3dapply,vectorpoisson3dapply}.h). */
static int fused_kind(const char *path, const char *name, int *qf_kind, CeedInt *num_comp) {
  *qf_kind = -1;
  if (!path || !name) return 0;
  const bool own = ends_with(path, "ceed-mi355-gallery.h");
  if (!own && !ends_with(path, "ceed-massapply.h") && !ends_with(path, "ceed-vectormassapply.h") && !ends_with(path, "ceed-poisson3dapply.h") &&
      !ends_with(path, "ceed-vectorpoisson3dapply.h"))
    return 0;
  if (!strcmp(name, "MassApply")) *qf_kind = CEED_MI355_QF_MASS, *num_comp = 1;
  else if (!strcmp(name, "Vector3MassApply")) *qf_kind = CEED_MI355_QF_MASS, *num_comp = 3;
  else if (!strcmp(name, "Poisson3DApply")) *qf_kind = CEED_MI355_QF_DIFFUSION, *num_comp = 1;
  else if (!strcmp(name, "Vector3Poisson3DApply")) *qf_kind = CEED_MI355_QF_DIFFUSION, *num_comp = 3;
  return 0;
}

/* Build the fused plan when the operator has the supported shape; leaves
 * d->fused false otherwise. */
static int try_fused(CeedOperator op, OperatorData *d) {
  Ceed                ceed;
  CeedQFunction       qf;
  CeedInt             num_in, num_out, num_comp = 0, dim, P, Q, rstr_comp, comp_stride, elem_size;
  CeedOperatorField  *in, *out;
  CeedQFunctionContext ctx;
  const char         *path, *name;
  int                 kind;
  CeedElemRestriction ru = NULL, rv = NULL, rq = NULL;
  CeedBasis           bu = NULL, bv = NULL;
  CeedVector          vu = NULL, vv = NULL, vq = NULL;
  CeedRestrictionType type;
  int                 ok = 0;

  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
  CeedCallBackend(CeedQFunctionGetSourcePath(qf, &path));
  CeedCallBackend(CeedQFunctionGetKernelName(qf, &name));
  CeedCallBackend(CeedQFunctionGetContext(qf, &ctx));
  CeedCallBackend(fused_kind(path, name, &kind, &num_comp));
  CeedCallBackend(CeedOperatorGetFields(op, &num_in, &in, &num_out, &out));
  if (kind < 0 || ctx || num_in != 2 || num_out != 1) goto done;
  CeedCallBackend(CeedOperatorFieldGetElemRestriction(in[0], &ru));
  CeedCallBackend(CeedOperatorFieldGetBasis(in[0], &bu));
  CeedCallBackend(CeedOperatorFieldGetVector(in[0], &vu));
  CeedCallBackend(CeedOperatorFieldGetElemRestriction(in[1], &rq));
  CeedCallBackend(CeedOperatorFieldGetVector(in[1], &vq));
  CeedCallBackend(CeedOperatorFieldGetElemRestriction(out[0], &rv));
  CeedCallBackend(CeedOperatorFieldGetBasis(out[0], &bv));
  CeedCallBackend(CeedOperatorFieldGetVector(out[0], &vv));
  if (vu != CEED_VECTOR_ACTIVE || vv != CEED_VECTOR_ACTIVE || ru != rv || bu != bv) goto done;
  if (vq == CEED_VECTOR_ACTIVE || vq == CEED_VECTOR_NONE) goto done;
  CeedCallBackend(CeedElemRestrictionGetType(ru, &type));
  if (type != CEED_RESTRICTION_STANDARD) goto done;
  CeedCallBackend(CeedBasisGetDimension(bu, &dim));
  CeedCallBackend(CeedBasisGetNumNodes1D(bu, &P));
  CeedCallBackend(CeedBasisGetNumQuadraturePoints1D(bu, &Q));
  CeedCallBackend(CeedElemRestrictionGetNumComponents(ru, &rstr_comp));
  if (dim != 3 || rstr_comp != num_comp) goto done;
  {
    CeedInt q_comp, q_elem;
    CeedCallBackend(CeedElemRestrictionGetNumComponents(rq, &q_comp));
    CeedCallBackend(CeedElemRestrictionGetElementSize(rq, &q_elem));
    if (q_comp != (kind == CEED_MI355_QF_MASS ? 1 : 6) || q_elem != Q * Q * Q) goto done;
  }
  {
    const CeedScalar *interp, *grad;
    const CeedInt    *offsets;
    CeedInt           num_elem;
    CeedCallBackend(CeedBasisGetInterp1D(bu, &interp));
    CeedCallBackend(CeedBasisGetGrad1D(bu, &grad));
    CeedCallBackend(CeedElemRestrictionGetNumElements(ru, &num_elem));
    CeedCallBackend(CeedElemRestrictionGetElementSize(ru, &elem_size));
    CeedCallBackend(CeedElemRestrictionGetCompStride(ru, &comp_stride));
    CeedCallBackend(CeedElemRestrictionGetLVectorSize(ru, &d->l_size));
    CeedCallBackend(CeedElemRestrictionGetOffsets(ru, CEED_MEM_HOST, &offsets));
    /* shapes the fused kernels are instantiated for; anything else takes the generic path */
    int ierr = CEED_MI355_ERROR_UNSUPPORTED;
    if (elem_size == P * P * P && P >= 2 && P <= 9 && (Q == P || Q == P + 1))
      ierr = CeedMi355OperatorCreateHex(kind, CEED_MI355_FP64, num_comp, num_elem, P, Q, interp, grad, offsets, comp_stride, d->l_size, 0,
                                        &d->hex);
    CeedCallBackend(CeedElemRestrictionRestoreOffsets(ru, &offsets));
    if (ierr != CEED_MI355_ERROR_UNSUPPORTED) {
      CeedCallBackend(CeedMi355Check(ceed, ierr));
      ok = 1;
    }
  }
done:
  d->fused            = ok;
  d->num_passive      = 1;
  d->passive_field[0] = 1;
  CeedCallBackend(CeedElemRestrictionDestroy(&ru));
  CeedCallBackend(CeedElemRestrictionDestroy(&rv));
  CeedCallBackend(CeedElemRestrictionDestroy(&rq));
  CeedCallBackend(CeedBasisDestroy(&bu));
  CeedCallBackend(CeedBasisDestroy(&bv));
  CeedCallBackend(CeedVectorDestroy(&vu));
  CeedCallBackend(CeedVectorDestroy(&vv));
  CeedCallBackend(CeedVectorDestroy(&vq));
  CeedCallBackend(CeedQFunctionContextDestroy(&ctx));
  CeedCallBackend(CeedQFunctionDestroy(&qf));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

/* Fused plan with a run-time compiled QFunction, when the operator has the
 * supported shape; leaves d->fused false otherwise. */
static int try_fused_jit(CeedOperator op, OperatorData *d) {
  Ceed                 ceed;
  CeedQFunction        qf;
  CeedInt              num_in, num_out, q_comp = 0, num_passive = 0, P = 0, Q = 0;
  CeedOperatorField   *in, *out;
  CeedQFunctionField  *qf_in, *qf_out;
  const char          *path, *name;
  CeedElemRestriction  ru = NULL;
  CeedBasis            bu = NULL;
  int32_t              in_kinds[CEED_FIELD_MAX], in_sizes[CEED_FIELD_MAX], out_kinds[2];
  int                  ok = 1;
  const char          *env = getenv("CEED_MI355_FUSE_QFUNCTIONS");

  d->fused = false;
  if (env && !strcmp(env, "0")) return CEED_ERROR_SUCCESS;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
  CeedCallBackend(CeedQFunctionGetSourcePath(qf, &path));
  CeedCallBackend(CeedQFunctionGetKernelName(qf, &name));
  CeedCallBackend(CeedOperatorGetFields(op, &num_in, &in, &num_out, &out));
  CeedCallBackend(CeedQFunctionGetFields(qf, NULL, &qf_in, NULL, &qf_out));
  if (!path || !name || num_in < 1 || num_in > 10 || num_out < 1 || num_out > 2) ok = 0;
  for (CeedInt f = 0; ok && f < num_in + num_out; f++) {
    const bool          is_in = f < num_in;
    const CeedInt       i     = is_in ? f : f - num_in;
    CeedElemRestriction rstr;
    CeedBasis           basis;
    CeedVector          vec;
    CeedEvalMode        mode;
    CeedInt             size;
    CeedCallBackend(CeedOperatorFieldGetElemRestriction(is_in ? in[i] : out[i], &rstr));
    CeedCallBackend(CeedOperatorFieldGetBasis(is_in ? in[i] : out[i], &basis));
    CeedCallBackend(CeedOperatorFieldGetVector(is_in ? in[i] : out[i], &vec));
    CeedCallBackend(CeedQFunctionFieldGetEvalMode(is_in ? qf_in[i] : qf_out[i], &mode));
    CeedCallBackend(CeedQFunctionFieldGetSize(is_in ? qf_in[i] : qf_out[i], &size));
    if (vec == CEED_VECTOR_ACTIVE) {
      /* all active fields: the same restriction and basis, scalar */
      if ((mode != CEED_EVAL_INTERP && mode != CEED_EVAL_GRAD) || (ru && (rstr != ru || basis != bu)) || size != (mode == CEED_EVAL_GRAD ? 3 : 1))
        ok = 0;
      if (ok && !ru) {
        CeedCallBackend(CeedElemRestrictionReferenceCopy(rstr, &ru));
        CeedCallBackend(CeedBasisReferenceCopy(basis, &bu));
      }
      const int32_t kind = mode == CEED_EVAL_GRAD ? CEED_MI355_FIELD_GRAD : CEED_MI355_FIELD_INTERP;
      if (is_in) in_kinds[i] = kind;
      else out_kinds[i] = kind;
    } else if (is_in && vec != CEED_VECTOR_NONE && mode == CEED_EVAL_NONE && rstr != CEED_ELEMRESTRICTION_NONE) {
      in_kinds[i]                     = CEED_MI355_FIELD_PASSIVE;
      in_sizes[i]                     = size;
      d->passive_field[num_passive]   = i;
      d->passive_size[num_passive++]  = size;
      q_comp += size;
    } else {
      ok = 0;
    }
    CeedCallBackend(CeedVectorDestroy(&vec));
    CeedCallBackend(CeedBasisDestroy(&basis));
    CeedCallBackend(CeedElemRestrictionDestroy(&rstr));
  }
  if (ok && ru) {
    CeedRestrictionType type;
    CeedInt             dim, nc, rc, elem_size, num_elem;
    CeedCallBackend(CeedElemRestrictionGetType(ru, &type));
    CeedCallBackend(CeedBasisGetDimension(bu, &dim));
    CeedCallBackend(CeedBasisGetNumComponents(bu, &nc));
    CeedCallBackend(CeedElemRestrictionGetNumComponents(ru, &rc));
    CeedCallBackend(CeedBasisGetNumNodes1D(bu, &P));
    CeedCallBackend(CeedBasisGetNumQuadraturePoints1D(bu, &Q));
    CeedCallBackend(CeedElemRestrictionGetElementSize(ru, &elem_size));
    CeedCallBackend(CeedElemRestrictionGetNumElements(ru, &num_elem));
    ok = type == CEED_RESTRICTION_STANDARD && dim == 3 && nc == 1 && rc == 1 && elem_size == P * P * P && P >= 2 && P <= 9 && Q >= P && Q <= 10;
    for (CeedInt k = 0; ok && k < num_passive; k++) {  /* a passive field: Q^3 points per element, its size per point */
      CeedElemRestriction rq;
      CeedInt             q_elem, q_nc, q_ne;
      CeedCallBackend(CeedOperatorFieldGetElemRestriction(in[d->passive_field[k]], &rq));
      CeedCallBackend(CeedElemRestrictionGetElementSize(rq, &q_elem));
      CeedCallBackend(CeedElemRestrictionGetNumComponents(rq, &q_nc));
      CeedCallBackend(CeedElemRestrictionGetNumElements(rq, &q_ne));
      ok = q_elem == Q * Q * Q && q_nc == d->passive_size[k] && q_ne == num_elem;
      CeedCallBackend(CeedElemRestrictionDestroy(&rq));
    }
    if (ok) {
      const CeedScalar *interp, *grad;
      const CeedInt    *offsets;
      CeedCallBackend(CeedBasisGetInterp1D(bu, &interp));
      CeedCallBackend(CeedBasisGetGrad1D(bu, &grad));
      CeedCallBackend(CeedElemRestrictionGetLVectorSize(ru, &d->l_size));
      CeedCallBackend(CeedElemRestrictionGetOffsets(ru, CEED_MEM_HOST, &offsets));
      int ierr = num_passive > 1 ? CeedMi355OperatorCreateHexJitFields(path, name, num_in, in_kinds, in_sizes, num_out, out_kinds, num_elem, P, Q,
                                                                       interp, grad, offsets, d->l_size, 0, &d->hex)
                                 : CeedMi355OperatorCreateHexJit(path, name, num_in, in_kinds, num_out, out_kinds, q_comp, num_elem, P, Q, interp,
                                                                 grad, offsets, d->l_size, 0, &d->hex);
      CeedCallBackend(CeedElemRestrictionRestoreOffsets(ru, &offsets));
      /* a QFunction that does not compile within the fused kernel (a macro of
       * its source named like something there) may still compile by itself:
       * the staged path, which reports what is wrong where it is not that */
      if (ierr == CEED_MI355_ERROR_UNSUPPORTED || ierr == CEED_MI355_ERROR_BACKEND) ok = 0;
      else CeedCallBackend(CeedMi355Check(ceed, ierr));
    }
  } else {
    ok = 0;
  }
  d->fused       = ok;
  d->jit         = ok;
  d->num_passive = num_passive;
  CeedCallBackend(CeedElemRestrictionDestroy(&ru));
  CeedCallBackend(CeedBasisDestroy(&bu));
  CeedCallBackend(CeedQFunctionDestroy(&qf));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

/* reload the passive values into the plan whose vector changed, and (run-time
 * compiled plans) hand over the current device context */
static int fused_sync_qdata(CeedOperator op, OperatorData *d) {
  Ceed               ceed;
  CeedOperatorField *in;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  if (d->jit) {
    CeedQFunction qf;
    void         *ctx;
    CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
    CeedCallBackend(CeedMi355QFunctionContextDevice(qf, &ctx));
    CeedCallBackend(CeedMi355Check(ceed, CeedMi355OperatorSetContext(d->hex, ctx)));
    CeedCallBackend(CeedQFunctionDestroy(&qf));
  }
  CeedCallBackend(CeedOperatorGetFields(op, NULL, &in, NULL, NULL));
  for (CeedInt k = 0, first = 0; k < d->num_passive; first += d->passive_size[k++]) {
    CeedElemRestriction rq;
    CeedVector          vq;
    uint64_t            state;
    CeedCallBackend(CeedOperatorFieldGetVector(in[d->passive_field[k]], &vq));
    CeedCallBackend(CeedVectorGetState(vq, &state));
    if (!d->passive_valid[k] || state != d->passive_state[k]) {
      const double *e;
      double       *temp;
      CeedCallBackend(CeedOperatorFieldGetElemRestriction(in[d->passive_field[k]], &rq));
      CeedCallBackend(qdata_evector(ceed, rq, vq, &e, &temp));
      if (d->num_passive > 1) CeedCallBackend(CeedMi355Check(ceed, CeedMi355OperatorSetQDataComponents(d->hex, first, d->passive_size[k], e, NULL)));
      else CeedCallBackend(CeedMi355Check(ceed, CeedMi355OperatorSetQData(d->hex, e, NULL)));
      if (temp) CeedMi355Free(temp);
      CeedCallBackend(CeedElemRestrictionDestroy(&rq));
      d->passive_state[k] = state;
      d->passive_valid[k] = true;
    }
    CeedCallBackend(CeedVectorDestroy(&vq));
  }
  return CeedDestroy(&ceed);
}

/* ------------------------------------------------------------------------ */
/* values at the quadrature points                                           */
/* ------------------------------------------------------------------------ */
/* Set up CeedMi355PointOperator when the operator has its shape: one active
 * field of up to three components on a standard restriction and a 3D tensor
 * basis (INTERP and/or GRAD), any of quadrature weights and passive EVAL_NONE
 * fields with backend strides, and one active EVAL_NONE output with backend
 * strides; leaves d->points NULL otherwise. */
static int try_points(CeedOperator op, OperatorData *d) {
  Ceed                ceed;
  CeedQFunction       qf;
  CeedInt             num_in, num_out, num_elem, num_qpts, num_comp = 0, num_passive = 0, P = 0, Q = 0, out_size = 0;
  CeedOperatorField  *in, *out;
  CeedQFunctionField *qf_in, *qf_out;
  const char         *path, *name, *env = getenv("CEED_MI355_FUSE_QFUNCTIONS");
  CeedElemRestriction ru = NULL;
  CeedBasis           bu = NULL, bw = NULL;
  int32_t             in_kinds[CEED_FIELD_MAX], in_sizes[CEED_FIELD_MAX];
  bool                ok;

  if (env && !strcmp(env, "0")) return CEED_ERROR_SUCCESS;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
  CeedCallBackend(CeedQFunctionGetSourcePath(qf, &path));
  CeedCallBackend(CeedQFunctionGetKernelName(qf, &name));
  CeedCallBackend(CeedOperatorGetFields(op, &num_in, &in, &num_out, &out));
  CeedCallBackend(CeedQFunctionGetFields(qf, NULL, &qf_in, NULL, &qf_out));
  CeedCallBackend(CeedOperatorGetNumElements(op, &num_elem));
  CeedCallBackend(CeedOperatorGetNumQuadraturePoints(op, &num_qpts));
  ok = path && name && num_in >= 1 && num_in <= 10 && num_out == 1;
  for (CeedInt f = 0; ok && f < num_in + num_out; f++) {
    const bool          is_in = f < num_in;
    const CeedInt       i     = is_in ? f : f - num_in;
    CeedElemRestriction rstr;
    CeedBasis           basis;
    CeedVector          vec;
    CeedEvalMode        mode;
    CeedInt             size, elem_size = 0, rstr_comp = 0;
    bool                backend = false;
    CeedCallBackend(CeedOperatorFieldGetElemRestriction(is_in ? in[i] : out[i], &rstr));
    CeedCallBackend(CeedOperatorFieldGetBasis(is_in ? in[i] : out[i], &basis));
    CeedCallBackend(CeedOperatorFieldGetVector(is_in ? in[i] : out[i], &vec));
    CeedCallBackend(CeedQFunctionFieldGetEvalMode(is_in ? qf_in[i] : qf_out[i], &mode));
    CeedCallBackend(CeedQFunctionFieldGetSize(is_in ? qf_in[i] : qf_out[i], &size));
    if (rstr != CEED_ELEMRESTRICTION_NONE) {
      CeedCallBackend(has_backend_strides(rstr, &backend));
      CeedCallBackend(CeedElemRestrictionGetElementSize(rstr, &elem_size));
      CeedCallBackend(CeedElemRestrictionGetNumComponents(rstr, &rstr_comp));
    }
    const bool at_points = mode == CEED_EVAL_NONE && backend && elem_size == num_qpts && rstr_comp == size;
    if (!is_in) {
      ok       = vec == CEED_VECTOR_ACTIVE && at_points;
      out_size = size;
      if (ok) CeedCallBackend(CeedElemRestrictionGetEVectorSize(rstr, &d->points_size));
    } else if (vec == CEED_VECTOR_ACTIVE) {
      ok = (mode == CEED_EVAL_INTERP || mode == CEED_EVAL_GRAD) && (!ru || (rstr == ru && basis == bu));
      if (ok && !ru) {
        CeedCallBackend(CeedElemRestrictionReferenceCopy(rstr, &ru));
        CeedCallBackend(CeedBasisReferenceCopy(basis, &bu));
      }
      in_kinds[i] = mode == CEED_EVAL_GRAD ? CEED_MI355_FIELD_GRAD : CEED_MI355_FIELD_INTERP;
    } else if (mode == CEED_EVAL_WEIGHT && basis != CEED_BASIS_NONE) {
      ok          = !bw || basis == bw;
      in_kinds[i] = CEED_MI355_FIELD_WEIGHT;
      if (ok && !bw) CeedCallBackend(CeedBasisReferenceCopy(basis, &bw));
    } else {
      ok                            = vec != CEED_VECTOR_NONE && at_points;
      in_kinds[i]                   = CEED_MI355_FIELD_PASSIVE;
      d->passive_field[num_passive] = i;
      d->passive_size[num_passive++] = size;
    }
    if (is_in) in_sizes[i] = size;
    CeedCallBackend(CeedVectorDestroy(&vec));
    CeedCallBackend(CeedBasisDestroy(&basis));
    CeedCallBackend(CeedElemRestrictionDestroy(&rstr));
  }
  if (ok && ru && bu != CEED_BASIS_NONE) {
    CeedRestrictionType type;
    CeedInt             dim, rc, elem_size, re, Qw = 0, dim_w = 3;
    CeedCallBackend(CeedElemRestrictionGetType(ru, &type));
    CeedCallBackend(CeedBasisGetDimension(bu, &dim));
    CeedCallBackend(CeedBasisGetNumComponents(bu, &num_comp));
    CeedCallBackend(CeedElemRestrictionGetNumComponents(ru, &rc));
    CeedCallBackend(CeedBasisGetNumNodes1D(bu, &P));
    CeedCallBackend(CeedBasisGetNumQuadraturePoints1D(bu, &Q));
    CeedCallBackend(CeedElemRestrictionGetElementSize(ru, &elem_size));
    CeedCallBackend(CeedElemRestrictionGetNumElements(ru, &re));
    if (bw) {
      CeedCallBackend(CeedBasisGetDimension(bw, &dim_w));
      CeedCallBackend(CeedBasisGetNumQuadraturePoints1D(bw, &Qw));
    }
    ok = type == CEED_RESTRICTION_STANDARD && dim == 3 && dim_w == 3 && rc == num_comp && elem_size == P * P * P && re == num_elem &&
         num_qpts == Q * Q * Q && (!bw || Qw == Q) && P >= 2 && P <= Q && Q <= 10;
    if (ok) {
      const CeedScalar *interp, *grad, *weights = NULL;
      const CeedInt    *offsets;
      CeedInt           comp_stride;
      CeedSize          l_size;
      CeedCallBackend(CeedBasisGetInterp1D(bu, &interp));
      CeedCallBackend(CeedBasisGetGrad1D(bu, &grad));
      if (bw) CeedCallBackend(CeedBasisGetQWeights(bw, &weights));
      CeedCallBackend(CeedElemRestrictionGetCompStride(ru, &comp_stride));
      CeedCallBackend(CeedElemRestrictionGetLVectorSize(ru, &l_size));
      CeedCallBackend(CeedElemRestrictionGetOffsets(ru, CEED_MEM_HOST, &offsets));
      const int ierr = CeedMi355PointOperatorCreate(path, name, num_in, in_kinds, in_sizes, out_size, num_comp, num_elem, P, Q, interp, grad, weights,
                                                    offsets, comp_stride, l_size, &d->points);
      CeedCallBackend(CeedElemRestrictionRestoreOffsets(ru, &offsets));
      /* (as for fused plans: where it does not compile, the staged path) */
      if (ierr != CEED_MI355_ERROR_UNSUPPORTED && ierr != CEED_MI355_ERROR_BACKEND) CeedCallBackend(CeedMi355Check(ceed, ierr));
    }
  }
  d->num_passive = num_passive;
  CeedCallBackend(CeedElemRestrictionDestroy(&ru));
  CeedCallBackend(CeedBasisDestroy(&bu));
  CeedCallBackend(CeedBasisDestroy(&bw));
  CeedCallBackend(CeedQFunctionDestroy(&qf));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

/* out (= or +=) the values at the quadrature points */
static int points_apply(CeedOperator op, OperatorData *d, CeedVector in_vec, CeedVector out_vec, bool add) {
  Ceed               ceed;
  CeedQFunction      qf;
  CeedOperatorField *in;
  CeedScalar        *du, *dv;
  const double      *passive[CEED_FIELD_MAX];
  void              *ctx;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
  CeedCallBackend(CeedMi355QFunctionContextDevice(qf, &ctx));
  CeedCallBackend(CeedOperatorGetFields(op, NULL, &in, NULL, NULL));
  for (CeedInt k = 0; k < d->num_passive; k++) {
    CeedVector  vec;
    CeedScalar *dp;
    CeedCallBackend(CeedOperatorFieldGetVector(in[d->passive_field[k]], &vec));
    CeedCallBackend(CeedMi355VectorDevice(vec, false, &dp));
    passive[k] = dp;
    CeedCallBackend(CeedVectorDestroy(&vec));
  }
  CeedCallBackend(CeedMi355VectorDevice(in_vec, false, &du));
  if (add) CeedCallBackend(CeedVectorGetArray(out_vec, CEED_MEM_DEVICE, &dv));
  else CeedCallBackend(CeedVectorGetArrayWrite(out_vec, CEED_MEM_DEVICE, &dv));
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355PointOperatorApply(d->points, ctx, du, passive, dv, add, NULL)));
  CeedCallBackend(CeedVectorRestoreArray(out_vec, &dv));
  CeedCallBackend(CeedQFunctionDestroy(&qf));
  return CeedDestroy(&ceed);
}

/* ------------------------------------------------------------------------ */
/* generic path                                                              */
/* ------------------------------------------------------------------------ */
static int field_size(CeedBasis basis, CeedElemRestriction rstr, CeedEvalMode mode, CeedInt *per_point) {
  CeedInt nc = 1, dim = 1;
  if (basis != CEED_BASIS_NONE) {
    CeedCallBackend(CeedBasisGetNumComponents(basis, &nc));
    CeedCallBackend(CeedBasisGetDimension(basis, &dim));
  } else if (rstr != CEED_ELEMRESTRICTION_NONE) {
    CeedCallBackend(CeedElemRestrictionGetNumComponents(rstr, &nc));
  }
  *per_point = mode == CEED_EVAL_GRAD ? nc * dim : (mode == CEED_EVAL_WEIGHT ? 1 : nc);
  return CEED_ERROR_SUCCESS;
}

static int generic_setup(CeedOperator op, OperatorData *d) {
  Ceed               ceed;
  CeedQFunction      qf;
  CeedInt            num_in, num_out;
  CeedOperatorField *in, *out;
  CeedQFunctionField *qf_in, *qf_out;
  if (d->is_staged) return CEED_ERROR_SUCCESS;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
  CeedCallBackend(CeedOperatorGetFields(op, &num_in, &in, &num_out, &out));
  CeedCallBackend(CeedQFunctionGetFields(qf, NULL, &qf_in, NULL, &qf_out));
  CeedCallBackend(CeedOperatorGetNumElements(op, &d->num_elem));
  CeedCallBackend(CeedOperatorGetNumQuadraturePoints(op, &d->Q));
  d->num_in  = num_in;
  d->num_out = num_out;
  const size_t points = (size_t)d->num_elem * (size_t)d->Q;
  for (CeedInt f = 0; f < num_in + num_out; f++) {
    const bool          is_in = f < num_in;
    const CeedInt       i     = is_in ? f : f - num_in;
    CeedElemRestriction rstr;
    CeedBasis           basis;
    CeedEvalMode        mode;
    CeedInt             per_point = 0;
    CeedCallBackend(CeedOperatorFieldGetElemRestriction(is_in ? in[i] : out[i], &rstr));
    CeedCallBackend(CeedOperatorFieldGetBasis(is_in ? in[i] : out[i], &basis));
    CeedCallBackend(CeedQFunctionFieldGetEvalMode(is_in ? qf_in[i] : qf_out[i], &mode));
    CeedCallBackend(field_size(basis, rstr, mode, &per_point));
    double **e = is_in ? &d->e_in[i] : &d->e_out[i], **q = is_in ? &d->q_in[i] : &d->q_out[i];
    bool    *same = is_in ? &d->q_in_is_e[i] : &d->q_out_is_e[i];
    if (rstr != CEED_ELEMRESTRICTION_NONE) {
      CeedSize e_size;
      CeedCallBackend(CeedElemRestrictionGetEVectorSize(rstr, &e_size));
      CeedCallBackend(CeedMi355Check(ceed, CeedMi355Malloc(sizeof(double) * (size_t)(e_size > 0 ? e_size : 1), (void **)e)));
    }
    if (mode == CEED_EVAL_NONE) {
      *q    = *e;
      *same = true;
    } else {
      CeedCallBackend(CeedMi355Check(ceed, CeedMi355Malloc(sizeof(double) * (points * (size_t)per_point + 1), (void **)q)));
    }
    if (is_in && mode == CEED_EVAL_WEIGHT) {
      BasisData *bd;
      CeedCallBackend(CeedBasisGetData(basis, &bd));
      CeedCallBackend(CeedMi355Check(ceed, CeedMi355BasisApply(bd->handle, d->num_elem, CEED_NOTRANSPOSE, CEED_EVAL_WEIGHT, 0, NULL, *q, NULL)));
    }
    CeedCallBackend(CeedElemRestrictionDestroy(&rstr));
    CeedCallBackend(CeedBasisDestroy(&basis));
  }
  d->is_staged = true;
  CeedCallBackend(CeedQFunctionDestroy(&qf));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

static int generic_apply_add(CeedOperator op, OperatorData *d, CeedVector in_vec, CeedVector out_vec) {
  Ceed               ceed;
  CeedQFunction      qf;
  CeedOperatorField *in, *out;
  CeedQFunctionField *qf_in, *qf_out;
  CeedMi355QFunction kernel;
  void              *ctx;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorGetQFunction(op, &qf));
  CeedCallBackend(CeedOperatorGetFields(op, NULL, &in, NULL, &out));
  CeedCallBackend(CeedQFunctionGetFields(qf, NULL, &qf_in, NULL, &qf_out));
  CeedCallBackend(CeedMi355QFunctionKernel(qf, &kernel));
  CeedCallBackend(CeedMi355QFunctionContextDevice(qf, &ctx));

  /* inputs: E then B */
  for (CeedInt i = 0; i < d->num_in; i++) {
    CeedElemRestriction rstr;
    CeedBasis           basis;
    CeedVector          vec;
    CeedEvalMode        mode;
    CeedCallBackend(CeedQFunctionFieldGetEvalMode(qf_in[i], &mode));
    if (mode == CEED_EVAL_WEIGHT) continue; /* filled once at set-up */
    CeedCallBackend(CeedOperatorFieldGetElemRestriction(in[i], &rstr));
    CeedCallBackend(CeedOperatorFieldGetBasis(in[i], &basis));
    CeedCallBackend(CeedOperatorFieldGetVector(in[i], &vec));
    const bool active = vec == CEED_VECTOR_ACTIVE;
    CeedVector l_vec  = active ? in_vec : vec;
    bool       fresh  = true;
    if (!active) {
      uint64_t state;
      CeedCallBackend(CeedVectorGetState(l_vec, &state));
      fresh          = !d->in_valid[i] || state != d->in_state[i];
      d->in_state[i] = state;
      d->in_valid[i] = true;
    }
    if (fresh) {
      RestrictionData *rd;
      CeedScalar      *dl;
      CeedCallBackend(CeedElemRestrictionGetData(rstr, &rd));
      CeedCallBackend(CeedMi355VectorDevice(l_vec, false, &dl));
      CeedCallBackend(CeedMi355Check(ceed, CeedMi355RestrictionApply(rd->handle, CEED_NOTRANSPOSE, dl, d->e_in[i], NULL)));
      if (mode != CEED_EVAL_NONE) {
        BasisData *bd;
        CeedCallBackend(CeedBasisGetData(basis, &bd));
        CeedCallBackend(
            CeedMi355Check(ceed, CeedMi355BasisApply(bd->handle, d->num_elem, CEED_NOTRANSPOSE, mode, 0, d->e_in[i], d->q_in[i], NULL)));
      }
    }
    CeedCallBackend(CeedVectorDestroy(&vec));
    CeedCallBackend(CeedBasisDestroy(&basis));
    CeedCallBackend(CeedElemRestrictionDestroy(&rstr));
  }

  /* D at every quadrature point */
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355QFunctionApply(kernel, d->num_elem, d->Q, ctx, (const double *const *)d->q_in, d->q_out, NULL)));

  /* outputs: B^T then E^T (summed into the L-vector) */
  for (CeedInt i = 0; i < d->num_out; i++) {
    CeedElemRestriction rstr;
    CeedBasis           basis;
    CeedVector          vec;
    CeedEvalMode        mode;
    RestrictionData    *rd;
    CeedScalar         *dl;
    CeedCallBackend(CeedQFunctionFieldGetEvalMode(qf_out[i], &mode));
    CeedCallBackend(CeedOperatorFieldGetElemRestriction(out[i], &rstr));
    CeedCallBackend(CeedOperatorFieldGetBasis(out[i], &basis));
    CeedCallBackend(CeedOperatorFieldGetVector(out[i], &vec));
    if (mode != CEED_EVAL_NONE) {
      BasisData *bd;
      CeedCallBackend(CeedBasisGetData(basis, &bd));
      CeedCallBackend(CeedMi355Check(ceed, CeedMi355BasisApply(bd->handle, d->num_elem, CEED_TRANSPOSE, mode, 0, d->q_out[i], d->e_out[i], NULL)));
    }
    CeedVector l_vec = vec == CEED_VECTOR_ACTIVE ? out_vec : vec;
    if (l_vec != CEED_VECTOR_NONE) {
      CeedCallBackend(CeedElemRestrictionGetData(rstr, &rd));
      CeedCallBackend(CeedVectorGetArray(l_vec, CEED_MEM_DEVICE, &dl));
      CeedCallBackend(CeedMi355Check(ceed, CeedMi355RestrictionApply(rd->handle, CEED_TRANSPOSE, d->e_out[i], dl, NULL)));
      CeedCallBackend(CeedVectorRestoreArray(l_vec, &dl));
    }
    CeedCallBackend(CeedVectorDestroy(&vec));
    CeedCallBackend(CeedBasisDestroy(&basis));
    CeedCallBackend(CeedElemRestrictionDestroy(&rstr));
  }
  CeedCallBackend(CeedQFunctionDestroy(&qf));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

/* ------------------------------------------------------------------------ */
/* slots                                                                     */
/* ------------------------------------------------------------------------ */
static int setup(CeedOperator op, OperatorData *d) {
  if (d->is_set_up) return CEED_ERROR_SUCCESS;
  CeedCallBackend(try_fused(op, d));
  if (!d->fused) CeedCallBackend(try_fused_jit(op, d));
  if (!d->fused) CeedCallBackend(try_points(op, d));
  if (!d->fused && !d->points) CeedCallBackend(generic_setup(op, d));
  d->is_set_up = true;
  return CEED_ERROR_SUCCESS;
}

/* Whether this apply is staged: no kernel has the operator's shape, or (values
 * at the quadrature points, several passive fields) the output is also an
 * input, all of which the staged path reads before it writes. */
static int runs_staged(CeedOperator op, OperatorData *d, CeedVector in, CeedVector out, bool *staged) {
  CeedOperatorField *fields;
  *staged = !d->fused && !d->points;
  if (*staged || (!d->points && d->num_passive < 2)) return CEED_ERROR_SUCCESS;
  *staged = out == CEED_VECTOR_NONE || out == in;
  CeedCallBackend(CeedOperatorGetFields(op, NULL, &fields, NULL, NULL));
  for (CeedInt k = 0; !*staged && k < d->num_passive; k++) {
    CeedVector vec;
    CeedCallBackend(CeedOperatorFieldGetVector(fields[d->passive_field[k]], &vec));
    *staged = vec == out;
    CeedCallBackend(CeedVectorDestroy(&vec));
  }
  if (*staged) CeedCallBackend(generic_setup(op, d));
  return CEED_ERROR_SUCCESS;
}

static int OperatorApplyAdd(CeedOperator op, CeedVector in, CeedVector out, CeedRequest *request) {
  OperatorData *d;
  Ceed          ceed;
  bool          staged;
  (void)request;
  CeedCallBackend(CeedOperatorGetData(op, &d));
  CeedCallBackend(setup(op, d));
  CeedCallBackend(runs_staged(op, d, in, out, &staged));
  if (staged) return generic_apply_add(op, d, in, out);
  if (d->points) return points_apply(op, d, in, out, true);
  CeedScalar *du, *dv;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(fused_sync_qdata(op, d));
  CeedCallBackend(CeedMi355VectorDevice(in, false, &du));
  CeedCallBackend(CeedVectorGetArray(out, CEED_MEM_DEVICE, &dv));
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355OperatorApplyAdd(d->hex, du, dv, NULL)));
  CeedCallBackend(CeedVectorRestoreArray(out, &dv));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

static int OperatorApply(CeedOperator op, CeedVector in, CeedVector out, CeedRequest *request) {
  OperatorData *d;
  Ceed          ceed;
  CeedSize      out_len;
  bool          staged;
  CeedCallBackend(CeedOperatorGetData(op, &d));
  CeedCallBackend(setup(op, d));
  CeedCallBackend(runs_staged(op, d, in, out, &staged));
  if (out != CEED_VECTOR_NONE) CeedCallBackend(CeedVectorGetLength(out, &out_len));
  if (d->points && !staged && out_len == d->points_size) return points_apply(op, d, in, out, false);
  /* the fused plan overwrites its whole L-vector; a longer output (or the
   * generic path) is zeroed first and accumulated into */
  if (staged || d->points || out == CEED_VECTOR_NONE || out_len != d->l_size) {
    if (out != CEED_VECTOR_NONE) CeedCallBackend(CeedVectorSetValue(out, 0.0));
    return OperatorApplyAdd(op, in, out, request);
  }
  CeedScalar *du, *dv;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(fused_sync_qdata(op, d));
  CeedCallBackend(CeedMi355VectorDevice(in, false, &du));
  CeedCallBackend(CeedVectorGetArrayWrite(out, CEED_MEM_DEVICE, &dv));
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355OperatorApply(d->hex, du, dv, NULL)));
  CeedCallBackend(CeedVectorRestoreArray(out, &dv));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

/* Name of the path the operator's applies take (include/ceed-mi355.h) */
int CeedMi355OperatorGetPath(CeedOperator op, const char **path) {
  OperatorData *d;
  Ceed          ceed;
  bool          is_composite;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCallBackend(CeedOperatorIsComposite(op, &is_composite));
  CeedCheck(!is_composite, ceed, CEED_ERROR_MINOR, "a composite operator has a path for each of its sub-operators");
  CeedCallBackend(CeedDestroy(&ceed));
  CeedCallBackend(CeedOperatorCheckReady(op));
  CeedCallBackend(CeedOperatorGetData(op, &d));
  CeedCallBackend(setup(op, d));
  *path = d->jit ? "fused-qfunction" : d->fused ? "fused" : d->points ? "points" : "staged";
  return CEED_ERROR_SUCCESS;
}

/* Diagonal of the operator (Jacobi preconditioning): the fused plan's
 * diagonal kernel; the staged path has no diagonal assembly. */
static int assemble_diagonal(CeedOperator op, CeedVector assembled, bool add) {
  OperatorData *d;
  Ceed          ceed;
  CeedScalar   *da;
  CeedCallBackend(CeedOperatorGetData(op, &d));
  CeedCallBackend(setup(op, d));
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  CeedCheck(d->fused && !d->jit, ceed, CEED_ERROR_UNSUPPORTED, "diagonal assembly needs a gallery mass or diffusion operator on 3D tensor hexes");
  CeedCallBackend(fused_sync_qdata(op, d));
  CeedCallBackend(CeedVectorGetArray(assembled, CEED_MEM_DEVICE, &da));
  CeedCallBackend(CeedMi355Check(ceed, CeedMi355OperatorAssembleDiagonal(d->hex, da, add, NULL)));
  CeedCallBackend(CeedVectorRestoreArray(assembled, &da));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}

static int OperatorLinearAssembleDiagonal(CeedOperator op, CeedVector assembled, CeedRequest *request) {
  (void)request;
  return assemble_diagonal(op, assembled, false);
}

static int OperatorLinearAssembleAddDiagonal(CeedOperator op, CeedVector assembled, CeedRequest *request) {
  (void)request;
  return assemble_diagonal(op, assembled, true);
}

static int OperatorDestroy(CeedOperator op) {
  OperatorData *d;
  CeedCallBackend(CeedOperatorGetData(op, &d));
  if (d->hex) CeedMi355OperatorDestroy(&d->hex);
  if (d->points) CeedMi355PointOperatorDestroy(&d->points);
  for (CeedInt i = 0; i < CEED_FIELD_MAX; i++) {
    if (d->q_in[i] && !d->q_in_is_e[i]) CeedMi355Free(d->q_in[i]);
    if (d->e_in[i]) CeedMi355Free(d->e_in[i]);
    if (d->q_out[i] && !d->q_out_is_e[i]) CeedMi355Free(d->q_out[i]);
    if (d->e_out[i]) CeedMi355Free(d->e_out[i]);
  }
  free(d);
  return CEED_ERROR_SUCCESS;
}

int CeedOperatorCreate_Mi355(CeedOperator op) {
  Ceed ceed;
  CeedCallBackend(CeedOperatorGetCeed(op, &ceed));
  OperatorData *d = calloc(1, sizeof(OperatorData));
  CeedCheck(d, ceed, CEED_ERROR_MAJOR, "host allocation failed");
  CeedCallBackend(CeedOperatorSetData(op, d));
  CeedCallBackend(CeedSetBackendFunction(ceed, "Operator", op, "Apply", OperatorApply));
  CeedCallBackend(CeedSetBackendFunction(ceed, "Operator", op, "ApplyAdd", OperatorApplyAdd));
  CeedCallBackend(CeedSetBackendFunction(ceed, "Operator", op, "LinearAssembleDiagonal", OperatorLinearAssembleDiagonal));
  CeedCallBackend(CeedSetBackendFunction(ceed, "Operator", op, "LinearAssembleAddDiagonal", OperatorLinearAssembleAddDiagonal));
  CeedCallBackend(CeedSetBackendFunction(ceed, "Operator", op, "Destroy", OperatorDestroy));
  CeedCallBackend(CeedDestroy(&ceed));
  return CEED_ERROR_SUCCESS;
}
