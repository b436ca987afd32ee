// Fused hex operator plans whose pointwise operator is a user QFunction,
// compiled at run time with hipRTC into the line-layout kernel: E, the
// sum-factorised interpolation and collocated gradient, the QFunction at
// every quadrature point, the transposes and the plan's E^T in one kernel.
// This is what the reference's hip-gen backend does for arbitrary
// QFunctions (backends/hip-gen/ceed-hip-gen-operator-build.cpp generates a
// fused kernel around the QFunction source); here the generated part is only
// the per-point glue that hands the QFunction its field arrays in field
// order, the kernel body is fixed (the line layout of hex_lines.hpp).
//
// Supported shape: scalar (1-component) active fields on one basis and one
// restriction, active inputs with INTERP and/or GRAD, active outputs with
// INTERP and/or GRAD, passive EVAL_NONE inputs (at most 32 values per point
// together, the plan's q_data), and the QFunction context.  FP64.
//
// A second body serves operators whose output stays at the quadrature points
// (geometric factors from coordinates): E, B and the QFunction of a field of
// one to three components, quadrature weights and passive fields among the
// inputs, the values stored where the next operator reads them.
#include <math.h>
#include <string.h>

#include <sstream>
#include <string>
#include <vector>

#include "hex_plan.hpp"
#include "mi355_common.h"

int mi355_jit_user_source(const char *source_path, std::string &out);
int mi355_jit_build(const std::string &code, const char *what, const char *kernel_name, hipModule_t *module, hipFunction_t *fn);

struct CeedMi355JitKernel {
  hipModule_t   module = nullptr;
  hipFunction_t kernel = nullptr;
  void         *ctx    = nullptr;  // device copy of the QFunction context (owned by the caller)
};

void mi355_jit_kernel_destroy(CeedMi355JitKernel *k) {
  if (!k) return;
  if (k->module) (void)hipModuleUnload(k->module);
  delete k;
}

namespace mi355 {
void collocated_grad(int P, int Q, const double *interp, const double *grad, double *collo);
}  // namespace mi355

namespace {

// The kernel bodies, compiled by hipRTC after the user's QFunction source and
// the generated glue (mi355_point).  Lines are contracted in place (a line's
// thread reads all of it before it writes), slabs [z][y][x] with the padded
// strides of the line kernel (RS, PS).  Q >= 7: a phase's matrix does not fit
// the SGPRs and is read row by row.
const char *kCommon = R"(
template <typename T> using mi355_cptr = const __attribute__((address_space(4))) T *;
template <typename T> __device__ __forceinline__ mi355_cptr<T> mi355_phase(const T *p) { asm volatile("" : "+s"(p)); return (mi355_cptr<T>)p; }
__device__ __forceinline__ long mi355_xcd_chunk(long b, long grid) {
  const long x = b % 8, k = b / 8, q = grid / 8, r = grid % 8;
  return x * q + (x < r ? x : r) + k;
}
// out_i = sum_j m[i][j] in_j at S[i * step]
template <int I, int J, bool ROWS>
__device__ __forceinline__ void mi355_line(const double *mats, const double (&in)[J], double *S, int step) {
  const auto g = mi355_phase(mats);
#pragma unroll
  for (int i = 0; i < I; i++) {
    const auto m = ROWS ? mi355_phase(mats + i * J) : g + i * J;
    double     s = 0;
#pragma unroll
    for (int j = 0; j < J; j++) s += m[j] * in[j];
    S[i * step] = s;
  }
}
// acc_i += sum_j m[j][i] in_j, each sum in ascending j
template <int I, int J, bool ROWS>
__device__ __forceinline__ void mi355_line_t(const double *mats, const double (&in)[J], double (&acc)[I]) {
  if (ROWS) {
#pragma unroll
    for (int j = 0; j < J; j++) {
      const auto m = mi355_phase(mats + j * I);
#pragma unroll
      for (int i = 0; i < I; i++) acc[i] += m[i] * in[j];
    }
  } else {
    const auto m = mi355_phase(mats);
#pragma unroll
    for (int i = 0; i < I; i++)
#pragma unroll
      for (int j = 0; j < J; j++) acc[i] += m[j * I + i] * in[j];
  }
}
)";

// E, B, the QFunction and the transposes of scalar fields.  Template
// parameters: P, Q, slab strides, which active input/output evaluations the
// QFunction uses, QC passive values per point.  Two slabs per element.
const char *kFused = R"(
enum { kAdd = 0, kOverwrite = 1, kAtomic = 2, kEvec = 3, kSplit = 4 };

template <int P, int Q, int RS, int PS, bool IN_U, bool IN_G, bool OUT_U, bool OUT_G, int QC>
__device__ __forceinline__ void mi355_fused(long elem_begin, long elem_end, int scatter, const int *__restrict__ offsets,
                                            const double *__restrict__ q_data, const double *__restrict__ mats, const double *__restrict__ u,
                                            double *__restrict__ v, double *__restrict__ evec, const int *__restrict__ tpos, const int *__restrict__ elem_sys,
                                            const int *__restrict__ sys_active, void *ctx, double *lds) {
  constexpr int  NT = Q * Q, SLAB = Q * PS, P3 = P * P * P, Q3 = Q * Q * Q;
  constexpr bool ROWS = Q >= 7;
  const int epb = blockDim.x / NT;
  const int le = threadIdx.x / NT, t = threadIdx.x - le * NT;
  double   *X = lds + (long)le * 2 * SLAB, *Y = X + SLAB;
  auto      at = [](int z, int y, int x) { return z * PS + y * RS + x; };
  const long e    = elem_begin + mi355_xcd_chunk(blockIdx.x, gridDim.x) * epb + le;
  const bool live = le < epb && e < elem_end && (!elem_sys || sys_active[elem_sys[e]]);
  if (elem_sys && !__syncthreads_or(live)) return;
  const int  cx = t % Q, cy = t / Q, ny = t % P, nz = t / P;  // column, also x-line (qy, qz) and y-line (qx, qz); x-line of nodes
  const bool xline = t < P * P, node = live && cx < P && cy < P;
  int off[P];
  if (node) {
#pragma unroll
    for (int z = 0; z < P; z++) off[z] = offsets[e * P3 + (z * P + cy) * P + cx];
  }
  const double *qd = q_data + (live ? e : 0) * (long)(QC > 0 ? QC : 1) * Q3 + (cy * Q + cx);
  // up to 7 passive values per point: the column's values all loaded at the
  // element start, in flight together while E and the interpolation run
  constexpr bool kEarly = QC > 0 && QC <= 7;
  double         sq[kEarly ? Q : 1][kEarly ? QC : 1];
  if (kEarly) {
#pragma unroll
    for (int qz = 0; qz < Q; qz++)
#pragma unroll
      for (int k = 0; k < QC; k++) sq[qz][k] = __builtin_nontemporal_load(&qd[k * Q3 + qz * Q * Q]);
  }
  // ---- E, then B_x, B_y by lines and B_z on the column
  if (node) {
#pragma unroll
    for (int z = 0; z < P; z++) X[at(z, cy, cx)] = u[off[z] >> 1];
  }
  __syncthreads();
  if (xline) {
    double in[P];
#pragma unroll
    for (int x = 0; x < P; x++) in[x] = X[at(nz, ny, x)];
    mi355_line<Q, P, ROWS>(mats, in, X + at(nz, ny, 0), 1);
  }
  __syncthreads();
  if (t < Q * P) {
    double in[P];
#pragma unroll
    for (int b = 0; b < P; b++) in[b] = X[at(cy, b, cx)];
    mi355_line<Q, P, ROWS>(mats, in, X + at(cy, 0, cx), RS);
  }
  __syncthreads();
  double uq[Q];
  {
    double col[P];
#pragma unroll
    for (int b = 0; b < P; b++) col[b] = X[at(b, cy, cx)];
    mi355_line<Q, P, ROWS>(mats, col, uq, 1);
  }
  // ---- collocated gradient: z on the column, x (into Y) and y (in place) by lines of X
  double dz[Q];
  if (IN_G) {
    mi355_line<Q, Q, ROWS>(mats + Q * P, uq, dz, 1);
#pragma unroll
    for (int qz = 0; qz < Q; qz++) X[at(qz, cy, cx)] = uq[qz];
    __syncthreads();
    double in[Q];
#pragma unroll
    for (int c = 0; c < Q; c++) in[c] = X[at(cy, cx, c)];
    mi355_line<Q, Q, ROWS>(mats + Q * P, in, Y + at(cy, cx, 0), 1);
#pragma unroll
    for (int c = 0; c < Q; c++) in[c] = X[at(cy, c, cx)];
    __syncthreads();
    mi355_line<Q, Q, ROWS>(mats + Q * P, in, X + at(cy, 0, cx), RS);
    __syncthreads();
  }
  // ---- the QFunction at every point of the column
  double wu[Q], vz[Q];
#pragma unroll
  for (int qz = 0; qz < Q; qz++) {
    double fu[1] = {uq[qz]}, fg[3] = {0, 0, 0}, fq[QC > 0 ? QC : 1], ou[1] = {0}, og[3] = {0, 0, 0};
    if (IN_G) {
      fg[0] = Y[at(qz, cy, cx)];
      fg[1] = X[at(qz, cy, cx)];
      fg[2] = dz[qz];
    }
#pragma unroll
    for (int k = 0; k < QC; k++) fq[k] = kEarly ? sq[kEarly ? qz : 0][kEarly ? k : 0] : __builtin_nontemporal_load(&qd[k * Q3 + qz * Q * Q]);
    mi355_point(ctx, fu, fg, fq, ou, og);
    wu[qz] = ou[0];
    if (OUT_G) {
      Y[at(qz, cy, cx)] = og[0];
      X[at(qz, cy, cx)] = og[1];
      vz[qz]            = og[2];
    }
  }
  // ---- transposes: D_x^T and D_y^T by lines in place, then the column sum and B_z^T into X
  double w[Q];
  if (OUT_G) {
    __syncthreads();
    {
      double in[Q], out[Q];
#pragma unroll
      for (int c = 0; c < Q; c++) in[c] = Y[at(cy, cx, c)], out[c] = 0;
      mi355_line_t<Q, Q, ROWS>(mats + Q * P, in, out);
#pragma unroll
      for (int c = 0; c < Q; c++) Y[at(cy, cx, c)] = out[c];
#pragma unroll
      for (int c = 0; c < Q; c++) in[c] = X[at(cy, c, cx)], out[c] = 0;
      mi355_line_t<Q, Q, ROWS>(mats + Q * P, in, out);
#pragma unroll
      for (int c = 0; c < Q; c++) X[at(cy, c, cx)] = out[c];
    }
    __syncthreads();
#pragma unroll
    for (int qz = 0; qz < Q; qz++) w[qz] = Y[at(qz, cy, cx)] + X[at(qz, cy, cx)];
    mi355_line_t<Q, Q, ROWS>(mats + Q * P, vz, w);
    if (OUT_U) {
#pragma unroll
      for (int qz = 0; qz < Q; qz++) w[qz] += wu[qz];
    }
  } else {
#pragma unroll
    for (int qz = 0; qz < Q; qz++) w[qz] = wu[qz];
  }
  {
    double out[P] = {};
    mi355_line_t<P, Q, ROWS>(mats, w, out);
#pragma unroll
    for (int b = 0; b < P; b++) X[at(b, cy, cx)] = out[b];
  }
  __syncthreads();
  if (t < Q * P) {
    double in[Q], out[P] = {};
#pragma unroll
    for (int a = 0; a < Q; a++) in[a] = X[at(cy, a, cx)];
    mi355_line_t<P, Q, ROWS>(mats, in, out);
#pragma unroll
    for (int y = 0; y < P; y++) X[at(cy, y, cx)] = out[y];
  }
  __syncthreads();
  if (xline) {
    double in[Q], out[P] = {};
#pragma unroll
    for (int a = 0; a < Q; a++) in[a] = X[at(nz, ny, a)];
    mi355_line_t<P, Q, ROWS>(mats, in, out);
#pragma unroll
    for (int x = 0; x < P; x++) X[at(nz, ny, x)] = out[x];
  }
  __syncthreads();
  if (node) {  // E^T from the node columns
    double s[P];
#pragma unroll
    for (int z = 0; z < P; z++) s[z] = X[at(z, cy, cx)];
    if (scatter == kEvec) {
#pragma unroll
      for (int z = 0; z < P; z++) evec[tpos[e * (long)P3 + (z * P + cy) * P + cx]] = s[z];
    } else if (scatter == kSplit) {  // shared entries to their E-vector slot, the rest onto the zeroed target
#pragma unroll
      for (int z = 0; z < P; z++) {
        if (off[z] & 1) evec[tpos[e * (long)P3 + (z * P + cy) * P + cx]] = s[z];
        else atomicAdd(&v[off[z] >> 1], s[z]);
      }
    } else if (scatter == kAtomic) {
#pragma unroll
      for (int z = 0; z < P; z++) atomicAdd(&v[off[z] >> 1], s[z]);
    } else {
      const bool overwrite = scatter == kOverwrite;
      double     old[P];
#pragma unroll
      for (int z = 0; z < P; z++) old[z] = (overwrite && (off[z] & 1)) ? 0.0 : v[off[z] >> 1];
#pragma unroll
      for (int z = 0; z < P; z++) v[off[z] >> 1] = (overwrite && (off[z] & 1)) ? s[z] : old[z] + s[z];
    }
  }
}
)";

// E, B and the QFunction of a field of NC components, the values stored at the
// quadrature points: [elem][component][Q^3], the layout of CEED_STRIDES_BACKEND.
// A slab per component, two with a gradient; all components pass each barrier
// together.
const char *kPoint = R"(
struct mi355_fields { const double *p[MI355_NPASSIVE > 0 ? MI355_NPASSIVE : 1]; };

template <int P, int Q, int RS, int PS, int NC, bool IN_G, int OC>
__device__ __forceinline__ void mi355_at_points(long num_elem, const int *__restrict__ offsets, long comp_stride, const double *__restrict__ mats,
                                                const double *__restrict__ q_weight, const double *__restrict__ u, mi355_fields passive,
                                                double *__restrict__ v, int add, void *ctx, double *lds) {
  constexpr int  NT = Q * Q, SLAB = Q * PS, P3 = P * P * P, Q3 = Q * Q * Q, NS = IN_G ? 2 : 1;
  constexpr bool ROWS = Q >= 7;
  const int epb = blockDim.x / NT;
  const int le = threadIdx.x / NT, t = threadIdx.x - le * NT;
  double   *S = lds + (long)le * NC * NS * SLAB;  // component c: X at c * SLAB, Y at (NC + c) * SLAB
  auto      at = [](int z, int y, int x) { return z * PS + y * RS + x; };
  const long e    = mi355_xcd_chunk(blockIdx.x, gridDim.x) * epb + le;
  const bool live = le < epb && e < num_elem;
  const int  cx = t % Q, cy = t / Q, ny = t % P, nz = t / P;
  if (live && cx < P && cy < P) {
#pragma unroll
    for (int z = 0; z < P; z++) {
      const long o = offsets[e * P3 + (z * P + cy) * P + cx];
#pragma unroll
      for (int c = 0; c < NC; c++) S[c * SLAB + at(z, cy, cx)] = u[o + c * comp_stride];
    }
  }
  __syncthreads();
  if (t < P * P) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      double *X = S + c * SLAB, in[P];
#pragma unroll
      for (int x = 0; x < P; x++) in[x] = X[at(nz, ny, x)];
      mi355_line<Q, P, ROWS>(mats, in, X + at(nz, ny, 0), 1);
    }
  }
  __syncthreads();
  if (t < Q * P) {
#pragma unroll
    for (int c = 0; c < NC; c++) {
      double *X = S + c * SLAB, in[P];
#pragma unroll
      for (int b = 0; b < P; b++) in[b] = X[at(cy, b, cx)];
      mi355_line<Q, P, ROWS>(mats, in, X + at(cy, 0, cx), RS);
    }
  }
  __syncthreads();
  double uq[NC][Q], dz[IN_G ? NC : 1][Q];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    double *X = S + c * SLAB, col[P];
#pragma unroll
    for (int b = 0; b < P; b++) col[b] = X[at(b, cy, cx)];
    mi355_line<Q, P, ROWS>(mats, col, uq[c], 1);
    if (IN_G) {
      mi355_line<Q, Q, ROWS>(mats + Q * P, uq[c], dz[IN_G ? c : 0], 1);
#pragma unroll
      for (int qz = 0; qz < Q; qz++) X[at(qz, cy, cx)] = uq[c][qz];
    }
  }
  if (IN_G) {
    __syncthreads();
    double in[NC][Q];
#pragma unroll
    for (int c = 0; c < NC; c++) {
      double *X = S + c * SLAB, *Y = S + (NC + c) * SLAB;
#pragma unroll
      for (int k = 0; k < Q; k++) in[c][k] = X[at(cy, cx, k)];
      mi355_line<Q, Q, ROWS>(mats + Q * P, in[c], Y + at(cy, cx, 0), 1);
#pragma unroll
      for (int k = 0; k < Q; k++) in[c][k] = X[at(cy, k, cx)];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NC; c++) mi355_line<Q, Q, ROWS>(mats + Q * P, in[c], S + c * SLAB + at(cy, 0, cx), RS);
    __syncthreads();
  }
  if (!live) return;
  const double wx = q_weight[cx], wy = q_weight[cy];
  const auto   wz = mi355_phase(q_weight);
#pragma unroll
  for (int qz = 0; qz < Q; qz++) {
    double fu[NC], fg[3 * NC], fw[1] = {wz[qz] * (wy * wx)}, out[OC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
      fu[c] = uq[c][qz];
      if (IN_G) {
        fg[c]          = S[(NC + c) * SLAB + at(qz, cy, cx)];
        fg[NC + c]     = S[c * SLAB + at(qz, cy, cx)];
        fg[2 * NC + c] = dz[IN_G ? c : 0][qz];
      }
    }
#pragma unroll
    for (int k = 0; k < OC; k++) out[k] = 0;
    mi355_point(ctx, fu, fg, fw, passive, e, Q3, (qz * Q + cy) * Q + cx, out);
    double *o = v + e * (long)OC * Q3 + (qz * Q + cy) * Q + cx;
    if (add) {
#pragma unroll
      for (int k = 0; k < OC; k++) o[k * (long)Q3] += out[k];
    } else {
#pragma unroll
      for (int k = 0; k < OC; k++) o[k * (long)Q3] = out[k];
    }
  }
}
)";

// The declarations the bodies start with and the strides of their slabs
std::string slab_strides(int Q) {
  using std::to_string;
  return to_string(mi355::line_row_stride(Q, 8)) + ", " + to_string(mi355::line_plane_stride(Q, 8));
}

int launch_jit(const CeedMi355Operator_private *op, const void *u, void *v, int overwrite, const mi355::ApplyExtras &x, hipStream_t s) {
  const int    Q = op->Q, nt = Q * Q, epb = op->epb;
  const size_t lds  = sizeof(double) * (size_t)epb * 2 * mi355::line_slab_entries(Q, 8);
  const bool   tmap = op->scatter == 0, split = op->scatter == CEED_MI355_PLAN_SPLIT;
  // the split mode's atomic adds land on a zeroed target: v in Apply, the scratch vector in ApplyAdd
  double *target = split && !overwrite ? (double *)op->d_scratch : (double *)v;
  if (split && !overwrite) {
    const int err = mi355::fill_zero(op, target, s);
    if (err) return err;
  }
  for (size_t c = 0; c + 1 < op->color_start.size(); c++) {
    const int64_t b = op->color_start[c], e = op->color_start[c + 1];
    if (e <= b) continue;
    const int64_t grid    = (e - b + epb - 1) / epb;
    int           scatter = tmap ? 3 : split ? 4 : (op->scatter == CEED_MI355_PLAN_ATOMIC ? 2 : (overwrite ? 1 : 0));
    long          eb = (long)b, ee = (long)e;
    const int32_t *offsets = op->d_offsets, *tpos = op->d_tpos, *elem_sys = op->d_elem_sys, *sys_active = op->d_sys_active;
    const double  *q_data = (const double *)op->d_qdata, *mats = (const double *)op->d_mats, *uu = (const double *)u;
    double        *vv = target, *evec = (double *)op->d_evec;
    void          *ctx    = op->jit->ctx;
    void          *args[] = {&eb, &ee, &scatter, &offsets, &q_data, &mats, &uu, &vv, &evec, &tpos, &elem_sys, &sys_active, &ctx};
    MI355_HIP(hipModuleLaunchKernel(op->jit->kernel, (unsigned)grid, 1, 1, epb * nt, 1, 1, (unsigned)lds, s, args, nullptr));
  }
  if (tmap) return mi355::transpose_gather(op, v, overwrite, x.dot, s);
  if (split) return mi355::split_finish(op, v, overwrite, s);
  return CEED_MI355_SUCCESS;
}

}  // namespace

extern "C" int CeedMi355OperatorCreateHexJit(const char *source_path, const char *function_name, int32_t num_in, const int32_t *in_kinds,
                                             int32_t num_out, const int32_t *out_kinds, int32_t q_comp, int32_t num_elem, int32_t P_1d,
                                             int32_t Q_1d, const double *interp_1d_host, const double *grad_1d_host, const int32_t *offsets_host,
                                             int64_t l_size, int flags, CeedMi355Operator *op_out) {
  *op_out = nullptr;
  MI355_CHECK(num_in >= 1 && num_in <= 3, CEED_MI355_ERROR_UNSUPPORTED, "%d inputs", num_in);
  int32_t sizes[3] = {0, 0, 0};
  int     passive  = 0;
  for (int i = 0; i < num_in; i++)
    if (in_kinds[i] == CEED_MI355_FIELD_PASSIVE) sizes[i] = q_comp, passive++;
  MI355_CHECK(passive <= 1, CEED_MI355_ERROR_UNSUPPORTED, "two input fields of kind %d", CEED_MI355_FIELD_PASSIVE);
  MI355_CHECK(passive || q_comp == 0, CEED_MI355_ERROR_UNSUPPORTED, "passive field of %d values per point", q_comp);
  return CeedMi355OperatorCreateHexJitFields(source_path, function_name, num_in, in_kinds, sizes, num_out, out_kinds, num_elem, P_1d, Q_1d,
                                             interp_1d_host, grad_1d_host, offsets_host, l_size, flags, op_out);
}

extern "C" int CeedMi355OperatorCreateHexJitFields(const char *source_path, const char *function_name, int32_t num_in, const int32_t *in_kinds,
                                                   const int32_t *in_sizes, int32_t num_out, const int32_t *out_kinds, int32_t num_elem,
                                                   int32_t P_1d, int32_t Q_1d, const double *interp_1d_host, const double *grad_1d_host,
                                                   const int32_t *offsets_host, int64_t l_size, int flags, CeedMi355Operator *op_out) {
  *op_out = nullptr;
  MI355_CHECK(source_path && function_name, CEED_MI355_ERROR_MAJOR, "null QFunction source or name");
  MI355_CHECK(P_1d >= 2 && P_1d <= 9 && Q_1d >= P_1d && Q_1d <= 10, CEED_MI355_ERROR_UNSUPPORTED, "fused run-time kernel for P=%d Q=%d", P_1d, Q_1d);
  MI355_CHECK(num_in >= 1 && num_in <= 10 && num_out >= 1 && num_out <= 2, CEED_MI355_ERROR_UNSUPPORTED, "%d inputs / %d outputs", num_in, num_out);
  bool in_u = false, in_g = false, out_u = false, out_g = false;
  int  passive = 0, q_comp = 0;
  for (int i = 0; i < num_in; i++) {
    const int k = in_kinds[i];
    MI355_CHECK(k == CEED_MI355_FIELD_INTERP || k == CEED_MI355_FIELD_GRAD || k == CEED_MI355_FIELD_PASSIVE, CEED_MI355_ERROR_UNSUPPORTED,
                "input field kind %d", k);
    MI355_CHECK(!(k == CEED_MI355_FIELD_INTERP && in_u) && !(k == CEED_MI355_FIELD_GRAD && in_g), CEED_MI355_ERROR_UNSUPPORTED,
                "two input fields of kind %d", k);
    in_u |= k == CEED_MI355_FIELD_INTERP;
    in_g |= k == CEED_MI355_FIELD_GRAD;
    if (k == CEED_MI355_FIELD_PASSIVE) {
      MI355_CHECK(in_sizes[i] >= 1 && in_sizes[i] <= 32, CEED_MI355_ERROR_UNSUPPORTED, "passive field of %d values per point", in_sizes[i]);
      passive++;
      q_comp += in_sizes[i];
    }
  }
  for (int i = 0; i < num_out; i++) {
    const int k = out_kinds[i];
    MI355_CHECK(k == CEED_MI355_FIELD_INTERP || k == CEED_MI355_FIELD_GRAD, CEED_MI355_ERROR_UNSUPPORTED, "output field kind %d", k);
    MI355_CHECK(!(k == CEED_MI355_FIELD_INTERP && out_u) && !(k == CEED_MI355_FIELD_GRAD && out_g), CEED_MI355_ERROR_UNSUPPORTED,
                "two output fields of kind %d", k);
    out_u |= k == CEED_MI355_FIELD_INTERP;
    out_g |= k == CEED_MI355_FIELD_GRAD;
  }
  MI355_CHECK(in_u || in_g, CEED_MI355_ERROR_UNSUPPORTED, "no active input");
  MI355_CHECK(q_comp <= 32, CEED_MI355_ERROR_UNSUPPORTED, "passive fields of %d values per point", q_comp);

  std::string src;
  int         ierr = mi355_jit_user_source(source_path, src);
  if (ierr) return ierr;
  std::ostringstream code;
  // mi355_point, the per-point glue, is used in the body and defined after it
  code << src << "__device__ __forceinline__ void mi355_point(void *ctx, const double *fu, const double *fg, const double *fq, double *ou, double *og);\n"
       << kCommon << kFused;
  // the QFunction's field arrays in its field order, the passive fields one after the other in fq
  code << "__device__ __forceinline__ void mi355_point(void *ctx, const double *fu, const double *fg, const double *fq, double *ou, double *og) {\n";
  code << "  (void)fu; (void)fg; (void)fq; (void)ou; (void)og;\n";
  code << "  const CeedScalar *in[" << num_in << "] = {";
  for (int i = 0, at = 0; i < num_in; i++) {
    code << (i ? ", " : "");
    if (in_kinds[i] == CEED_MI355_FIELD_PASSIVE) code << "fq + " << at, at += in_sizes[i];
    else code << (in_kinds[i] == CEED_MI355_FIELD_INTERP ? "fu" : "fg");
  }
  code << "};\n  CeedScalar *out[" << num_out << "] = {";
  for (int i = 0; i < num_out; i++) code << (i ? ", " : "") << (out_kinds[i] == CEED_MI355_FIELD_INTERP ? "ou" : "og");
  code << "};\n  " << function_name << "(ctx, 1, in, out);\n}\n";
  code << "extern \"C\" __global__ void __launch_bounds__(256) CeedMi355FusedJit(long eb, long ee, int scatter, const int *offsets, "
          "const double *q_data, const double *mats, const double *u, double *v, double *evec, const int *tpos, const int *elem_sys, "
          "const int *sys_active, "
          "void *ctx) {\n  extern __shared__ double mi355_lds[];\n";
  code << "  mi355_fused<" << P_1d << ", " << Q_1d << ", " << slab_strides(Q_1d) << ", " << (in_u ? "true" : "false") << ", "
       << (in_g ? "true" : "false") << ", " << (out_u ? "true" : "false") << ", " << (out_g ? "true" : "false") << ", " << q_comp
       << ">(eb, ee, scatter, offsets, q_data, mats, u, v, evec, tpos, elem_sys, sys_active, ctx, mi355_lds);\n}\n";

  CeedMi355JitKernel *k = new CeedMi355JitKernel();
  ierr                  = mi355_jit_build(code.str(), function_name, "CeedMi355FusedJit", &k->module, &k->kernel);
  if (ierr) {
    delete k;
    return ierr;
  }
  CeedMi355Operator op = nullptr;
  ierr = mi355::create_plan(mi355::kQfJit, CEED_MI355_FP64, 1, num_elem, P_1d, Q_1d, interp_1d_host, grad_1d_host, offsets_host, 1, l_size, flags,
                            q_comp, launch_jit, &op);
  if (ierr) {
    mi355_jit_kernel_destroy(k);
    return ierr;
  }
  op->jit  = k;
  *op_out  = op;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorSetContext(CeedMi355Operator op, void *ctx_device) {
  MI355_CHECK(op && op->jit, CEED_MI355_ERROR_BACKEND, "the context belongs to plans of run-time compiled QFunctions");
  op->jit->ctx = ctx_device;
  return CEED_MI355_SUCCESS;
}

// ---------------------------------------------------------------------------
// A QFunction's values at the quadrature points
// ---------------------------------------------------------------------------
struct CeedMi355PointOperator_private {
  int32_t            num_elem = 0, P = 0, Q = 0, num_comp = 0, num_passive = 0, comp_stride = 0, epb = 1;
  size_t             lds = 0;
  int32_t           *d_offsets = nullptr;
  double            *d_mats    = nullptr;  // B (Q x P), D (Q x Q), weights (Q)
  CeedMi355JitKernel kernel;
};

extern "C" int CeedMi355PointOperatorCreate(const char *source_path, const char *function_name, int32_t num_in, const int32_t *in_kinds,
                                            const int32_t *in_sizes, int32_t out_size, int32_t num_comp, int32_t num_elem, int32_t P_1d,
                                            int32_t Q_1d, const double *interp_1d_host, const double *grad_1d_host,
                                            const double *q_weight_1d_host, const int32_t *offsets_host, int32_t comp_stride, int64_t l_size,
                                            CeedMi355PointOperator *op_out) {
  *op_out = nullptr;
  MI355_CHECK(source_path && function_name, CEED_MI355_ERROR_MAJOR, "null QFunction source or name");
  MI355_CHECK(P_1d >= 2 && P_1d <= Q_1d && Q_1d <= 10 && num_comp >= 1 && num_comp <= 3, CEED_MI355_ERROR_UNSUPPORTED,
              "point operator for P=%d Q=%d num_comp=%d", P_1d, Q_1d, num_comp);
  MI355_CHECK(num_in >= 1 && num_in <= 10 && out_size >= 1 && out_size <= 32 && num_elem >= 0, CEED_MI355_ERROR_UNSUPPORTED,
              "%d inputs / %d output values", num_in, out_size);
  bool in_u = false, in_g = false;
  int  num_passive = 0, passive_size = 0;
  for (int i = 0; i < num_in; i++) {
    const int k = in_kinds[i];
    MI355_CHECK((k == CEED_MI355_FIELD_INTERP && !in_u && in_sizes[i] == num_comp) || (k == CEED_MI355_FIELD_GRAD && !in_g && in_sizes[i] == 3 * num_comp) ||
                    (k == CEED_MI355_FIELD_PASSIVE && in_sizes[i] >= 1) || (k == CEED_MI355_FIELD_WEIGHT && in_sizes[i] == 1),
                CEED_MI355_ERROR_UNSUPPORTED, "input field of kind %d, size %d", k, in_sizes[i]);
    MI355_CHECK(k != CEED_MI355_FIELD_WEIGHT || q_weight_1d_host, CEED_MI355_ERROR_UNSUPPORTED, "quadrature weights without a rule");
    in_u |= k == CEED_MI355_FIELD_INTERP;
    in_g |= k == CEED_MI355_FIELD_GRAD;
    if (k == CEED_MI355_FIELD_PASSIVE) num_passive++, passive_size += in_sizes[i];
  }
  MI355_CHECK(in_u || in_g, CEED_MI355_ERROR_UNSUPPORTED, "no active input");
  MI355_CHECK(passive_size <= 32, CEED_MI355_ERROR_UNSUPPORTED, "passive fields of %d values per point", passive_size);
  const int64_t n = (int64_t)num_elem * P_1d * P_1d * P_1d;
  for (int64_t i = 0; i < n; i++)
    MI355_CHECK(offsets_host[i] >= 0 && offsets_host[i] + (int64_t)(num_comp - 1) * comp_stride < l_size, CEED_MI355_ERROR_DIMENSION,
                "offset %d outside L-vector of size %lld", offsets_host[i], (long long)l_size);

  std::string src;
  int         ierr = mi355_jit_user_source(source_path, src);
  if (ierr) return ierr;
  const std::string  sig = "__device__ __forceinline__ void mi355_point(void *ctx, const double *fu, const double *fg, const double *fw, "
                           "const mi355_fields &passive, long e, int q3, int pt, double *res)";
  std::ostringstream code;
  std::string        body = kPoint;
  const size_t       head = body.find('\n', body.find("struct mi355_fields")) + 1;
  code << src << "#define MI355_NPASSIVE " << num_passive << "\n" << kCommon << body.substr(0, head) << sig << ";\n" << body.substr(head);
  code << sig << " {\n  (void)fu; (void)fg; (void)fw; (void)passive; (void)e; (void)q3; (void)pt;\n";
  for (int i = 0, p = 0; i < num_in; i++)
    if (in_kinds[i] == CEED_MI355_FIELD_PASSIVE) {
      code << "  double p" << i << "[" << in_sizes[i] << "];\n  for (int k = 0; k < " << in_sizes[i] << "; k++) p" << i << "[k] = passive.p[" << p
           << "][(e * " << in_sizes[i] << " + k) * q3 + pt];\n";
      p++;
    }
  code << "  const CeedScalar *in[" << num_in << "] = {";
  for (int i = 0; i < num_in; i++) {
    code << (i ? ", " : "");
    switch (in_kinds[i]) {
      case CEED_MI355_FIELD_INTERP: code << "fu"; break;
      case CEED_MI355_FIELD_GRAD: code << "fg"; break;
      case CEED_MI355_FIELD_WEIGHT: code << "fw"; break;
      default: code << "p" << i;
    }
  }
  code << "};\n  CeedScalar *out[1] = {res};\n  " << function_name << "(ctx, 1, in, out);\n}\n";
  code << "extern \"C\" __global__ void __launch_bounds__(256) CeedMi355AtPoints(long num_elem, const int *offsets, long comp_stride, const double *mats, "
          "const double *q_weight, const double *u, mi355_fields passive, double *v, int add, void *ctx) {\n  extern __shared__ double mi355_lds[];\n"
       << "  mi355_at_points<" << P_1d << ", " << Q_1d << ", " << slab_strides(Q_1d) << ", " << num_comp << ", " << (in_g ? "true" : "false") << ", "
       << out_size << ">(num_elem, offsets, comp_stride, mats, q_weight, u, passive, v, add, ctx, mi355_lds);\n}\n";

  CeedMi355PointOperator op = new CeedMi355PointOperator_private();
  op->num_elem = num_elem, op->P = P_1d, op->Q = Q_1d, op->num_comp = num_comp, op->num_passive = num_passive, op->comp_stride = comp_stride;
  // whole wavefronts of elements within the default LDS budget
  const size_t per = sizeof(double) * num_comp * (in_g ? 2 : 1) * mi355::line_slab_entries(Q_1d, 8);
  op->epb          = mi355::geo_default_epb(Q_1d);
  while (op->epb > 1 && (op->epb * Q_1d * Q_1d > 256 || op->epb * per > (size_t)mi355::kDefaultLdsBytes)) op->epb--;
  op->lds = op->epb * per;
  ierr    = mi355_jit_build(code.str(), function_name, "CeedMi355AtPoints", &op->kernel.module, &op->kernel.kernel);
  const int           QP = Q_1d * P_1d, QQ = Q_1d * Q_1d;
  std::vector<double> mats(QP + QQ + Q_1d, 0.0);
  memcpy(mats.data(), interp_1d_host, sizeof(double) * QP);
  mi355::collocated_grad(P_1d, Q_1d, interp_1d_host, grad_1d_host, &mats[QP]);
  if (q_weight_1d_host) memcpy(&mats[QP + QQ], q_weight_1d_host, sizeof(double) * Q_1d);
  if (!ierr && (hipMalloc(&op->d_offsets, sizeof(int32_t) * (n + 1)) != hipSuccess || hipMalloc(&op->d_mats, sizeof(double) * mats.size()) != hipSuccess ||
                hipMemcpy(op->d_offsets, offsets_host, sizeof(int32_t) * n, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(op->d_mats, mats.data(), sizeof(double) * mats.size(), hipMemcpyHostToDevice) != hipSuccess)) {
    mi355::set_error("point operator: device memory for %lld offsets", (long long)n);
    ierr = CEED_MI355_ERROR_BACKEND;
  }
  if (ierr) {
    CeedMi355PointOperatorDestroy(&op);
    return ierr;
  }
  *op_out = op;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355PointOperatorApply(CeedMi355PointOperator op, void *ctx_device, const double *u, const double *const *passive_host, double *v,
                                           int add, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null point operator");
  if (op->num_elem == 0) return CEED_MI355_SUCCESS;
  struct {
    const double *p[10];
  } passive = {};
  for (int i = 0; i < op->num_passive; i++) passive.p[i] = passive_host[i];
  long          num_elem = op->num_elem, comp_stride = op->comp_stride;
  const int     Q        = op->Q;
  const double *mats = op->d_mats, *q_weight = op->d_mats + Q * op->P + Q * Q;
  void         *args[]   = {&num_elem, &op->d_offsets, &comp_stride, &mats, &q_weight, &u, &passive, &v, &add, &ctx_device};
  MI355_HIP(hipModuleLaunchKernel(op->kernel.kernel, (unsigned)((num_elem + op->epb - 1) / op->epb), 1, 1, op->epb * Q * Q, 1, 1, (unsigned)op->lds,
                                  (hipStream_t)stream, args, nullptr));
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355PointOperatorDestroy(CeedMi355PointOperator *op) {
  if (!op || !*op) return CEED_MI355_SUCCESS;
  if ((*op)->kernel.module) (void)hipModuleUnload((*op)->kernel.module);
  (void)hipFree((*op)->d_offsets);
  (void)hipFree((*op)->d_mats);
  delete *op;
  *op = nullptr;
  return CEED_MI355_SUCCESS;
}
