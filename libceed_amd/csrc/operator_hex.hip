// Fused hex operator plans: element colouring, colour-ordered data layout,
// geometric factors on the GPU, and the apply entry points.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "hex_plan.hpp"

namespace mi355 {
void collocated_grad(int P, int Q, const double *interp, const double *grad, double *collo);

int lds_bytes(int P, int Q, int qf, int num_comp, int epb, int scalar_bytes, int layout) {
  if (layout == kLayoutLines) return (int)line_lds_bytes(Q, num_comp, qf, scalar_bytes, false, epb);
  if (layout == kLayoutPoints) return scalar_bytes * (Q * P + Q * Q + epb * (qf == kQfMass ? 3 : 4) * Q * Q * Q);
  const int slabs = qf == kQfMass ? 2 : 3;
  return scalar_bytes * (Q * P + Q * Q + epb * slabs * Q * Q * Q);
}

int64_t brick_threads(int Q, int64_t ns) {
  const int nt = Q * Q;
  if (nt > 64) return ns * nt;
  const int epw = 64 / nt;
  return 64 * ((ns + epw - 1) / epw);
}

int64_t brick_lds_bytes(int P, int Q, int qf, int scalar_bytes, const int *shape) {
  const int64_t ns = (int64_t)shape[0] * shape[1] * shape[2];
  const int64_t nb = (int64_t)(shape[0] * (P - 1) + 1) * (shape[1] * (P - 1) + 1) * (shape[2] * (P - 1) + 1);
  return (int64_t)scalar_bytes * ns * (qf == kQfMass ? 2 : 3) * Q * Q * Q + 4 * nb;
}

// Recomputing pays for diffusion, where it replaces 6 values per point: at
// every order in FP64 with one component (1.4-1.9x).  Exceptions, all
// measured on MI355X at 4M DoFs (ms per apply, stored / recomputed): mass
// replaces one value (p=2 0.135 / 0.161, p=4 0.068 / 0.065, p=6 0.057 /
// 0.058); FP32 reads half the bytes but computes the factors in FP64 all the
// same, which costs as much as it saves at Q = 8 (0.069 / 0.069) and Q = 10
// (0.084 / 0.082), not at Q = 7 (0.093 / 0.082) or Q = 9 (0.087 / 0.077),
// whose elements fill the wavefronts less well; three components share one
// read of the factors: in FP64 only Q = 4 gains nothing (0.203 / 0.204; Q = 3
// 0.657 / 0.579, Q = 5 0.143 / 0.127, Q = 7 0.130 / 0.114, Q = 8 0.119 / 0.105),
// in FP32 (us, P = Q - 1, at 0.5M, 4M and 24M DoFs in their default E^T) Q = 3
// 471 / 417 (4M), Q = 5 19.5 / 20.8, 88 / 93, 448 / 447, Q = 6 20.8 / 21.8, 76 /
// 77, 394 / 400, Q = 7 21.9 / 25.8, 82 / 84, 441 / 433, Q = 8 23.8 / 24.6, 71 / 70,
// 369 / 377, Q = 9 27.2 / 27.6, 85 / 82, 417 / 398, Q = 10 30.8 / 31.6, 94 / 92,
// 477 / 465, and with P = Q (4M and 24M) Q = 5 58 / 55, 306 / 280, Q = 6 59 / 57,
// 350 / 328, Q = 7 60 / 63, 327 / 323, Q = 8 58 / 56 (4M).
bool geo_pays(int P, int Q, int qf, int num_comp, int scalar_bytes) {
  if (qf != kQfDiffusion && qf != kQfDiffusionKappa) return false;
  if (scalar_bytes == 8) return num_comp == 1 || Q != 4;
  if (num_comp == 1) return Q != 8 && Q != 10;
  return Q <= 3 || Q >= 9 || (P == Q && (Q == 5 || Q == 6));
}

// Elements per workgroup with recomputed factors: the count of at most 256
// threads that leaves the fewest lanes of its wavefronts idle (Q = 3 63 of 64,
// 4 64, 5 125 of 128, 6 252 of 256, 7 245 of 256, 9 243 of 256, 10 200 of 256)
// with no more wavefronts than that takes, the fastest measured at Q = 3..7
// and 9 (8M DoFs, p=4: 0.222 ms, the next best, 5, 0.234); whole
// wavefronts at Q = 2 and 8 share the barriers best at 128 and 256 threads
// (p=6: 4 elements 0.182 ms, 1 element 0.197).
int geo_default_epb(int Q) {
  static const int table[11] = {0, 0, 32, 7, 4, 5, 7, 5, 4, 3, 2};
  return Q >= 2 && Q <= 10 ? table[Q] : 1;
}

int default_epb(int P, int Q, int qf, int num_comp, int scalar_bytes, int layout) {
  if (layout == kLayoutLines && qf != kQfMass && Q >= 2 && Q <= 10) {
    // diffusion in the line layout: the autotuner's choices for FP64 at ~8M
    // DoFs on MI355X (Q = 2..10); within a few percent of the best for FP32
    static const int table[11] = {0, 0, 8, 6, 4, 2, 3, 1, 4, 3, 2};
    int              epb = table[Q];
    while (epb > 1 && (epb * Q * Q > 256 || lds_bytes(P, Q, qf, num_comp, epb, scalar_bytes, layout) > kMaxLdsBytes)) epb--;
    return epb;
  }
  // as many elements as fit 256 threads and the default LDS budget
  int epb = 256 / layout_threads(Q, layout);
  if (epb < 1) epb = 1;
  while (epb > 1 && lds_bytes(P, Q, qf, num_comp, epb, scalar_bytes, layout) > kDefaultLdsBytes) epb--;
  return epb;
}
}  // namespace mi355

namespace {

using mi355::kQfDiffusion;
using mi355::kQfDiffusionKappa;
using mi355::kQfMass;
using mi355::kQfJit;

template <typename T>
__global__ void __launch_bounds__(256) fill_kernel(int64_t n, T value, T *__restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) x[i] = value;
}

// Set entries [slot, slot + per) of every element block (block stride `stride`) to `value`.
template <typename T>
__global__ void __launch_bounds__(256) fill_slot(int64_t num_elem, int64_t per, int64_t stride, int64_t slot, T value, T *__restrict__ x) {
  const int64_t n = num_elem * per;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = i / per;
    x[p * stride + slot + (i - p * per)] = value;
  }
}

// Copy per-element blocks of `per` entries between the caller's element order
// and the plan's colour order.  to_packed: dst[p] = src[perm[p]].
template <typename TS, typename TD>
__global__ void __launch_bounds__(256) permute_elements(int64_t num_elem, int64_t per, const int32_t *__restrict__ perm, int to_packed,
                                                        const TS *__restrict__ src, TD *__restrict__ dst) {
  const int64_t n = num_elem * per;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = i / per, r = i - p * per, o = perm[p];
    if (to_packed) dst[i] = (TD)src[o * per + r];
    else dst[o * per + r] = (TD)src[i];
  }
}

// Geometric factors from coordinates, FP64 arithmetic.  One Q x Q thread slab
// per element; mesh basis has PM <= Q nodes per direction (runtime).
// Mass3DBuild:    q = w det J                    (gallery/ceed-mass3dbuild.h)
// Poisson3DBuild: q = Voigt of (w/det J) adj(J) adj(J)^T (gallery/ceed-poisson3dbuild.h)
template <int Q, int BUILD, typename TOUT>
__global__ void __launch_bounds__(1024) hex_build_kernel(int64_t num_elem, int PM, const int32_t *__restrict__ mesh_offsets,
                                                         int32_t mesh_comp_stride, const double *__restrict__ coords,
                                                         const double *__restrict__ mats, int64_t out_elem_stride,
                                                         TOUT *__restrict__ q_data) {
  constexpr int T1 = Q, NT = Q * Q, SLAB = Q * Q * Q, QC = BUILD == 0 ? 1 : 6;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double *sB = reinterpret_cast<double *>(lds_raw);  // Q x PM
  double *sD = sB + Q * PM;                          // Q x Q
  double *sW = sD + Q * Q;                           // Q
  const int epb = blockDim.x / NT, le = threadIdx.x / NT, t = threadIdx.x - le * NT, tx = t % T1, ty = t / T1;
  double   *S0 = sW + Q + (size_t)le * 5 * SLAB, *S1 = S0 + SLAB, *X = S1 + SLAB;  // X: 3 slabs of coordinates at qpts
  for (int i = threadIdx.x; i < Q * PM + Q * Q + Q; i += blockDim.x) sB[i] = mats[i];
  const int64_t e    = (int64_t)blockIdx.x * epb + le;
  const bool    live = e < num_elem;
  const int     PM3  = PM * PM * PM;
  auto sidx = [](int z, int y, int x) { return (z * T1 + y) * T1 + x; };
  __syncthreads();
  for (int c = 0; c < 3; c++) {
    if (live && tx < PM && ty < PM)
      for (int z = 0; z < PM; z++) S0[sidx(z, ty, tx)] = coords[mesh_offsets[e * PM3 + (z * PM + ty) * PM + tx] + (int64_t)c * mesh_comp_stride];
    __syncthreads();
    if (ty < PM) {
      for (int z = 0; z < PM; z++) {
        double s = 0;
        for (int b = 0; b < PM; b++) s += sB[tx * PM + b] * S0[sidx(z, ty, b)];
        S1[sidx(z, ty, tx)] = s;
      }
    }
    __syncthreads();
    double acc[Q];
    for (int z = 0; z < PM; z++) {
      double s = 0;
      for (int b = 0; b < PM; b++) s += sB[ty * PM + b] * S1[sidx(z, b, tx)];
      acc[z] = s;
    }
    double *Xc = X + c * SLAB;
    for (int qz = 0; qz < Q; qz++) {
      double s = 0;
      for (int b = 0; b < PM; b++) s += sB[qz * PM + b] * acc[b];
      Xc[sidx(qz, ty, tx)] = s;
    }
  }
  __syncthreads();
  if (!live) return;
  const int64_t Q3 = SLAB;
  for (int qz = 0; qz < Q; qz++) {
    double J[3][3];  // J[d][c] = d x_c / d X_d
    for (int c = 0; c < 3; c++) {
      const double *Xc = X + c * SLAB;
      double        d0 = 0, d1 = 0, d2 = 0;
      for (int k = 0; k < Q; k++) {
        d0 += sD[tx * Q + k] * Xc[sidx(qz, ty, k)];
        d1 += sD[ty * Q + k] * Xc[sidx(qz, k, tx)];
        d2 += sD[qz * Q + k] * Xc[sidx(k, ty, tx)];
      }
      J[0][c] = d0;
      J[1][c] = d1;
      J[2][c] = d2;
    }
    const double  w   = sW[qz] * (sW[ty] * sW[tx]);
    const int64_t pt  = (qz * Q + ty) * Q + tx;
    TOUT         *out = q_data + e * out_elem_stride + pt;
    if (BUILD == 0) {
      const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) - J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                         J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
      out[0] = (TOUT)(det * w);
    } else {
      double A[3][3];
      for (int j = 0; j < 3; j++)
        for (int k = 0; k < 3; k++)
          A[k][j] = J[(k + 1) % 3][(j + 1) % 3] * J[(k + 2) % 3][(j + 2) % 3] - J[(k + 2) % 3][(j + 1) % 3] * J[(k + 1) % 3][(j + 2) % 3];
      const double qw = w / (J[0][0] * A[0][0] + J[0][1] * A[0][1] + J[0][2] * A[0][2]);
      out[0 * Q3] = (TOUT)(qw * (A[0][0] * A[0][0] + A[0][1] * A[0][1] + A[0][2] * A[0][2]));
      out[1 * Q3] = (TOUT)(qw * (A[1][0] * A[1][0] + A[1][1] * A[1][1] + A[1][2] * A[1][2]));
      out[2 * Q3] = (TOUT)(qw * (A[2][0] * A[2][0] + A[2][1] * A[2][1] + A[2][2] * A[2][2]));
      out[3 * Q3] = (TOUT)(qw * (A[1][0] * A[2][0] + A[1][1] * A[2][1] + A[1][2] * A[2][2]));
      out[4 * Q3] = (TOUT)(qw * (A[0][0] * A[2][0] + A[0][1] * A[2][1] + A[0][2] * A[2][2]));
      out[5 * Q3] = (TOUT)(qw * (A[0][0] * A[1][0] + A[0][1] * A[1][1] + A[0][2] * A[1][2]));
    }
  }
}

template <int Q, typename TOUT>
int launch_build(int build, int64_t num_elem, int PM, const int32_t *mesh_offsets, int32_t mcs, const double *coords, const double *mats,
                 int64_t stride, TOUT *q_data, hipStream_t s) {
  const int nt = Q * Q;
  int       epb = std::max(1, 256 / nt);
  while (epb > 1 && sizeof(double) * (Q * PM + Q * Q + Q + (size_t)epb * 5 * Q * Q * Q) > 64 * 1024) epb--;
  const size_t lds = sizeof(double) * (Q * PM + Q * Q + Q + (size_t)epb * 5 * Q * Q * Q);
  const int64_t grid = (num_elem + epb - 1) / epb;
  if (build == 0)
    hex_build_kernel<Q, 0, TOUT><<<(unsigned)grid, epb * nt, lds, s>>>(num_elem, PM, mesh_offsets, mcs, coords, mats, stride, q_data);
  else hex_build_kernel<Q, 1, TOUT><<<(unsigned)grid, epb * nt, lds, s>>>(num_elem, PM, mesh_offsets, mcs, coords, mats, stride, q_data);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

// The trilinear map of every element (hex_geo.hpp) from its 8 vertices.  Each
// coefficient takes its differences before its sums, so that the cancellation
// between neighbouring vertices happens on the coordinates themselves.
__global__ void __launch_bounds__(256) geo_coefficients(int64_t num_elem, const int32_t *__restrict__ mesh_offsets, int32_t mesh_comp_stride,
                                                        const double *__restrict__ coords, double *__restrict__ geo) {
  const int64_t n = num_elem * 3;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = i / 3;
    const int     d = (int)(i - e * 3);
    double        x[8];
    for (int k = 0; k < 8; k++) x[k] = coords[mesh_offsets[e * 8 + k] + (int64_t)d * mesh_comp_stride];
    double *g = geo + e * mi355::kGeoStride + d;
    const double x0 = x[1] - x[0], x1 = x[3] - x[2], x2 = x[5] - x[4], x3 = x[7] - x[6];  // differences along xi
    const double y0 = x[2] - x[0], y1 = x[3] - x[1], y2 = x[6] - x[4], y3 = x[7] - x[5];  // along eta
    const double z0 = x[4] - x[0], z1 = x[5] - x[1], z2 = x[6] - x[2], z3 = x[7] - x[3];  // along zeta
    g[0]  = 0.125 * ((x0 + x1) + (x2 + x3));
    g[3]  = 0.125 * ((y0 + y1) + (y2 + y3));
    g[6]  = 0.125 * ((z0 + z1) + (z2 + z3));
    g[9]  = 0.125 * ((x1 - x0) + (x3 - x2));
    g[12] = 0.125 * ((x2 - x0) + (x3 - x1));
    g[15] = 0.125 * ((y2 - y0) + (y3 - y1));
    g[18] = 0.125 * ((x3 - x2) - (x1 - x0));
    g[21] = 0;
  }
}

// The plan's stored factors of a trilinear geometry: a thread per quadrature point
template <typename T>
__global__ void __launch_bounds__(256) geo_qdata(int64_t num_elem, int Q, int qf_mass, int64_t elem_stride, const double *__restrict__ geo,
                                                 const double *__restrict__ pts, T *__restrict__ q_data) {
  const int64_t q3 = (int64_t)Q * Q * Q, n = num_elem * q3;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = i / q3;
    const int     r = (int)(i - e * q3), qx = r % Q, qy = (r / Q) % Q, qz = r / (Q * Q);
    mi355::GeoColumn c;
    c.load(geo + e * mi355::kGeoStride, pts[qx], pts[qy]);
    const double w = pts[Q + qz] * (pts[Q + qy] * pts[Q + qx]);
    T           *o = q_data + e * elem_stride + r;
    if (qf_mass) {
      o[0] = (T)mi355::geo_mass(c, pts[qz], w);
    } else {
      double s[6];
      mi355::geo_poisson(c, pts[qz], w, s);
      for (int k = 0; k < 6; k++) o[k * q3] = (T)s[k];
    }
  }
}

// Device memory of one call
struct TempBuffer {
  void *p = nullptr;
  ~TempBuffer() { (void)hipFree(p); }
};

// The plan's stored factors are no longer its trilinear geometry's: for the graphs captured while they were
__global__ void mark_replaced(int32_t *turn) { turn[0] = 0, turn[1] = 1; }

int factors_replaced(CeedMi355Operator op, hipStream_t s) {
  if (!op->d_geo_turn) return CEED_MI355_SUCCESS;
  mark_replaced<<<1, 1, 0, s>>>(op->d_geo_turn);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

bool is_capturing(hipStream_t s) {
  if (!s) return false;  // the null stream cannot be captured (and the query is 0.1 us of a small apply's 4.5 on the host)
  hipStreamCaptureStatus st;
  if (hipStreamIsCapturing(s, &st) == hipSuccess) return st == hipStreamCaptureStatusActive;
  (void)hipGetLastError();
  return false;
}

// Whether a mesh basis of two nodes is the linear one, (1 -+ xi)/2 at every point with slopes -+1/2
bool linear_mesh_basis(int Q, const double *B, const double *G) {
  for (int q = 0; q < Q; q++)
    if (!(std::fabs(B[2 * q] + B[2 * q + 1] - 1) <= 1e-14 && std::fabs(G[2 * q] + 0.5) <= 1e-14 && std::fabs(G[2 * q + 1] - 0.5) <= 1e-14)) return false;
  return true;
}

template <typename TOUT>
int dispatch_build(int Q, int build, int64_t num_elem, int PM, const int32_t *mo, int32_t mcs, const double *coords, const double *mats,
                   int64_t st, TOUT *q_data, hipStream_t s) {
  switch (Q) {
    case 2: return launch_build<2, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 3: return launch_build<3, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 4: return launch_build<4, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 5: return launch_build<5, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 6: return launch_build<6, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 7: return launch_build<7, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 8: return launch_build<8, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 9: return launch_build<9, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
    case 10: return launch_build<10, TOUT>(build, num_elem, PM, mo, mcs, coords, mats, st, q_data, s);
  }
  MI355_CHECK(false, CEED_MI355_ERROR_UNSUPPORTED, "geometric factors: Q=%d outside 2..10", Q);
}

// Greedy colouring in ascending element order over every L index an element
// touches: an element takes the smallest colour none of its entries carries.
int color_elements(const int32_t *offsets, int64_t num_elem, int es, int nc, int64_t cs, int64_t l_size, std::vector<int32_t> &color,
                   int &num_colors) {
  std::vector<uint64_t> mask((size_t)l_size, 0);
  color.assign((size_t)num_elem, 0);
  num_colors = 0;
  for (int64_t e = 0; e < num_elem; e++) {
    uint64_t used = 0;
    for (int i = 0; i < es; i++)
      for (int k = 0; k < nc; k++) {
        const int64_t l = (int64_t)offsets[e * es + i] + k * cs;
        MI355_CHECK(l >= 0 && l < l_size, CEED_MI355_ERROR_DIMENSION, "offset %lld outside L-vector of size %lld", (long long)l,
                    (long long)l_size);
        used |= mask[l];
      }
    MI355_CHECK(~used != 0, CEED_MI355_ERROR_UNSUPPORTED, "element colouring needs more than 64 colours");
    int c = 0;
    while (used & (1ull << c)) c++;
    color[e] = c;
    num_colors = std::max(num_colors, c + 1);
    for (int i = 0; i < es; i++)
      for (int k = 0; k < nc; k++) mask[(int64_t)offsets[e * es + i] + k * cs] |= 1ull << c;
  }
  return CEED_MI355_SUCCESS;
}

// Autotuner results by (P, Q, num_comp, pointwise operator, scalar type, E^T
// mode, recomputed factors).
struct Launch {
  int  layout, epb;
  bool line_only;
};
std::mutex                                                       g_tune_mutex;
std::map<std::tuple<int, int, int, int, int, int, bool>, Launch> g_tuned;

std::tuple<int, int, int, int, int, int, bool> tune_key(const CeedMi355Operator op) {
  return std::make_tuple(op->P, op->Q, op->num_comp, op->qf, op->scalar_type, op->scatter, op->geo_valid);
}

void set_launch(CeedMi355Operator op, const Launch &l) { op->layout = l.layout, op->epb = l.epb, op->line_only = l.line_only; }

// Take the autotuner's launch for plans of this kind, if there is one
void tuned_launch(CeedMi355Operator op) {
  std::lock_guard<std::mutex> lock(g_tune_mutex);
  auto                        it = g_tuned.find(tune_key(op));
  if (it != g_tuned.end()) set_launch(op, it->second);
}

// A known layout the plan's kernels exist in (run-time compiled QFunctions:
// the line layout only; the point layout up to Q^3 = 256 threads)
bool layout_exists(int Q, int qf, int layout) {
  return layout == mi355::kLayoutLines || (qf != kQfJit && (layout == mi355::kLayoutColumns || (layout == mi355::kLayoutPoints && Q * Q * Q <= 256)));
}

bool admissible(int P, int Q, int qf, int num_comp, int scalar_bytes, int layout, int epb) {
  return layout_exists(Q, qf, layout) && epb >= 1 && epb * mi355::layout_threads(Q, layout) <= mi355::max_threads(layout) &&
         mi355::lds_bytes(P, Q, qf, num_comp, epb, scalar_bytes, layout) <= mi355::kMaxLdsBytes;
}

int plan_default_epb(const CeedMi355Operator op, int layout) {
  if (layout == mi355::kLayoutLines && op->geo_valid) return mi355::geo_default_epb(op->Q);
  // three components work three times as long on an element's factors: at
  // Q = 5 with the transpose map, once its one launch fills the GPU several
  // times over, full wavefronts beat small workgroups (MI355X, us per apply, 2
  // elements / 5: P = 4 2197 elements 16.8 / 16.7, 12167 46.5 / 48.6, 17576 63.3
  // / 63.0, 24389 82.3 / 78.5, 46656 146 / 131, 110592 327 / 320; P = 5 2744
  // elements 23.1 / 24.6, 10648 54.3 / 54.0, 19683 85.6 / 85.1; in colours two are
  // better).  Not at Q = 7 (one / 5: 512 elements 21.9 / 25.7, 2744 42.5 / 48.5,
  // 8000 103 / 108, 10648 130 / 127, 24389 292 / 296).
  if (layout == mi355::kLayoutLines && op->num_comp == 3 && op->scalar_bytes == 8 && op->qf == kQfDiffusion && op->scatter == 0 && op->Q == 5 &&
      op->num_elem >= 16384)
    return 5;
  return mi355::default_epb(op->P, op->Q, op->qf, op->num_comp, op->scalar_bytes, layout);
}

// The factors of the plan are from now on a trilinear geometry's (valid) or
// the caller's; a launch nobody chose follows.
void set_geo_valid(CeedMi355Operator op, bool valid) {
  valid = valid && !op->qdata_in_graph;
  if (op->geo_valid == valid) return;
  op->geo_valid = valid;
  if (op->own_launch || op->scatter == CEED_MI355_PLAN_SEGMENT) return;
  op->layout    = mi355::kLayoutLines;
  op->epb       = plan_default_epb(op, op->layout);
  op->line_only = false;
  tuned_launch(op);
}

// A launch the plan can take: segment plans have one (the line layout with an
// element slot for each element of the longest segment)
bool plan_admissible(const CeedMi355Operator op, int layout, int epb) {
  if (op->scatter == CEED_MI355_PLAN_SEGMENT) return layout == mi355::kLayoutLines && epb == op->seg_max;
  return admissible(op->P, op->Q, op->qf, op->num_comp, op->scalar_bytes, layout, epb);
}

// Resident workgroups of a launch shape on the current device, cached by
// (kernel, threads, LDS bytes, device).

int64_t elem_block(const CeedMi355Operator op) {
  return (int64_t)op->q_comp * op->Q * op->Q * op->Q;
}

// Transpose offset map of the E-vector (element order = caller order): the
// slot of every contribution (elem, comp, node) in an E-vector sorted by L
// entry, contributions of one L entry in ascending (elem, comp, node) order.
int build_transpose_map(CeedMi355Operator op, const int32_t *offsets) {
  const int64_t es = (int64_t)op->P * op->P * op->P, nnz = (int64_t)op->num_elem * op->num_comp * es;
  MI355_CHECK(nnz < INT32_MAX && op->l_size < INT32_MAX, CEED_MI355_ERROR_UNSUPPORTED,
              "transpose map needs fewer than 2^31 E-vector entries (have %lld); use CEED_MI355_PLAN_COLOR", (long long)nnz);
  std::vector<int32_t> row((size_t)op->l_size + 1, 0), pos((size_t)nnz + 1);
  for (int64_t e = 0; e < op->num_elem; e++)
    for (int64_t k = 0; k < op->num_comp; k++)
      for (int64_t i = 0; i < es; i++) row[(size_t)(offsets[e * es + i] + k * op->comp_stride) + 1]++;
  for (int64_t t = 0; t < op->l_size; t++) row[t + 1] += row[t];
  std::vector<int32_t> cursor(row.begin(), row.end() - 1);
  for (int64_t e = 0; e < op->num_elem; e++)
    for (int64_t k = 0; k < op->num_comp; k++)
      for (int64_t i = 0; i < es; i++) pos[(size_t)((e * op->num_comp + k) * es + i)] = cursor[offsets[e * es + i] + k * op->comp_stride]++;
  MI355_HIP(hipMalloc(&op->d_trow, sizeof(int32_t) * row.size()));
  MI355_HIP(hipMalloc(&op->d_tpos, sizeof(int32_t) * pos.size()));
  MI355_HIP(hipMalloc(&op->d_evec, (size_t)op->scalar_bytes * (nnz + 1)));
  MI355_HIP(hipMemcpy(op->d_trow, row.data(), sizeof(int32_t) * row.size(), hipMemcpyHostToDevice));
  MI355_HIP(hipMemcpy(op->d_tpos, pos.data(), sizeof(int32_t) * pos.size(), hipMemcpyHostToDevice));
  // line_last: every L entry has a contribution (the gather also zeroes the
  // others), and the elements fit its workgroups at the most there can be in one
  bool last = op->qf != kQfJit && mi355::line_takes_last(op->P, op->num_comp) && op->num_elem <= mi355::kLastWorkgroups * (256 / (op->Q * op->Q));
  for (int64_t t = 0; t < op->l_size && last; t++) last = row[t] < row[t + 1];
  if (last) {
    MI355_HIP(hipMalloc(&op->d_tcount, sizeof(int32_t) * (size_t)op->l_size));
    // (a copy: done when it returns, also for a stream that does not wait for the null stream)
    const std::vector<int32_t> zero((size_t)op->l_size, 0);
    MI355_HIP(hipMemcpy(op->d_tcount, zero.data(), sizeof(int32_t) * zero.size(), hipMemcpyHostToDevice));
  }
  return CEED_MI355_SUCCESS;
}

// The split mode's maps (element order = caller order, packed offsets with
// the shared bit): slots in the shared E-vector for shared contributions
// only, sorted by L entry and, within one entry, ascending (elem, comp, node);
// row runs for shared entries; the list of shared entries; ApplyAdd's target.
int build_split_map(CeedMi355Operator op, const int32_t *packed) {
  const int64_t es = (int64_t)op->P * op->P * op->P, nnz = (int64_t)op->num_elem * op->num_comp * es;
  MI355_CHECK(nnz < INT32_MAX && op->l_size < INT32_MAX, CEED_MI355_ERROR_UNSUPPORTED,
              "the split E^T needs fewer than 2^31 E-vector entries (have %lld); use CEED_MI355_PLAN_COLOR", (long long)nnz);
  std::vector<int32_t> row((size_t)op->l_size + 1, 0), pos((size_t)nnz + 1, -1), srows;
  for (int64_t e = 0; e < op->num_elem; e++)
    for (int64_t k = 0; k < op->num_comp; k++)
      for (int64_t i = 0; i < es; i++) {
        const int32_t o = packed[e * es + i];
        if (o & 1) row[(size_t)((o >> 1) + k * op->comp_stride) + 1]++;
      }
  for (int64_t t = 0; t < op->l_size; t++) {
    if (row[t + 1] > 0) srows.push_back((int32_t)t);
    row[t + 1] += row[t];
  }
  std::vector<int32_t> cursor(row.begin(), row.end() - 1);
  for (int64_t e = 0; e < op->num_elem; e++)
    for (int64_t k = 0; k < op->num_comp; k++)
      for (int64_t i = 0; i < es; i++) {
        const int32_t o = packed[e * es + i];
        if (o & 1) pos[(size_t)((e * op->num_comp + k) * es + i)] = cursor[(o >> 1) + k * op->comp_stride]++;
      }
  const int64_t nshared = row[(size_t)op->l_size];
  op->num_shared        = (int64_t)srows.size();
  MI355_HIP(hipMalloc(&op->d_trow, sizeof(int32_t) * row.size()));
  MI355_HIP(hipMalloc(&op->d_tpos, sizeof(int32_t) * pos.size()));
  MI355_HIP(hipMalloc(&op->d_srows, sizeof(int32_t) * (srows.size() + 1)));
  MI355_HIP(hipMalloc(&op->d_evec, (size_t)op->scalar_bytes * (nshared + 1)));
  MI355_HIP(hipMalloc(&op->d_scratch, (size_t)op->scalar_bytes * (op->l_size + 1)));
  MI355_HIP(hipMemcpy(op->d_trow, row.data(), sizeof(int32_t) * row.size(), hipMemcpyHostToDevice));
  MI355_HIP(hipMemcpy(op->d_tpos, pos.data(), sizeof(int32_t) * pos.size(), hipMemcpyHostToDevice));
  if (!srows.empty()) MI355_HIP(hipMemcpy(op->d_srows, srows.data(), sizeof(int32_t) * srows.size(), hipMemcpyHostToDevice));
  return CEED_MI355_SUCCESS;
}

// split mode, Apply: each shared entry = the ordered sum of its run
template <typename T>
__global__ void __launch_bounds__(256) split_gather_kernel(int64_t num_shared, const int32_t *__restrict__ srows, const int32_t *__restrict__ row,
                                                           const T *__restrict__ evec, T *__restrict__ v) {
  for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < num_shared; j += (int64_t)gridDim.x * blockDim.x) {
    const int32_t t   = srows[j];
    T             acc = 0;
    for (int32_t m = row[t]; m < row[t + 1]; m++) acc += evec[m];
    v[t] = acc;
  }
}

// split mode, ApplyAdd: v += (the ordered run of a shared entry, else the atomic target w)
template <typename T>
__global__ void __launch_bounds__(256) split_add_kernel(int64_t l_size, const int32_t *__restrict__ row, const T *__restrict__ evec,
                                                        const T *__restrict__ w, T *__restrict__ v) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < l_size; t += (int64_t)gridDim.x * blockDim.x) {
    const int32_t b = row[t], e = row[t + 1];
    T             a = 0;
    if (b == e) a = w[t];
    for (int32_t m = b; m < e; m++) a += evec[m];
    v[t] += a;
  }
}

// v[t] (= or +=) the sum of t's contiguous run of the sorted E-vector, in order
template <typename T>
__global__ void __launch_bounds__(256) transpose_gather_kernel(int64_t l_size, const int32_t *__restrict__ row, const T *__restrict__ evec,
                                                               T *__restrict__ v, int overwrite) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < l_size; t += (int64_t)gridDim.x * blockDim.x) {
    T acc = overwrite ? T(0) : v[t];
    for (int32_t m = row[t]; m < row[t + 1]; m++) acc += evec[m];
    v[t] = acc;
  }
}

// The gather with the partial sums of u . v, in a fixed order: the blocks'
// strides, then a tree over the block (CeedMi355CG: p . Ap while Ap is in
// registers, instead of a kernel that reads both vectors again)
template <typename T>
__global__ void __launch_bounds__(256) transpose_gather_dot_kernel(int64_t l_size, const int32_t *__restrict__ row, const T *__restrict__ evec,
                                                                   const T *__restrict__ u, T *__restrict__ v, double *__restrict__ partial,
                                                                   double *__restrict__ to, const double *__restrict__ from) {
  __shared__ double sum[256];
  if (blockIdx.x == 0 && threadIdx.x == 0) *to = *from;
  double dot = 0;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < l_size; t += (int64_t)gridDim.x * blockDim.x) {
    T acc = 0;
    for (int32_t m = row[t]; m < row[t + 1]; m++) acc += evec[m];
    v[t] = acc;
    dot += (double)u[t] * (double)acc;
  }
  sum[threadIdx.x] = dot;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) sum[threadIdx.x] += sum[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = sum[0];
}

// The same over chunks of L entries, one block per chunk; chunks of inactive
// systems (batched solvers) are left out
template <typename T>
__global__ void __launch_bounds__(256) transpose_gather_chunks_kernel(const int64_t *__restrict__ chunk_begin, const int32_t *__restrict__ chunk_sys,
                                                                      const int32_t *__restrict__ active, const int32_t *__restrict__ row,
                                                                      const T *__restrict__ evec, T *__restrict__ v, int overwrite) {
  const int64_t c = blockIdx.x;
  if (!active[chunk_sys[c]]) return;  // uniform over the block
  for (int64_t t = chunk_begin[c] + threadIdx.x; t < chunk_begin[c + 1]; t += blockDim.x) {
    T acc = overwrite ? T(0) : v[t];
    for (int32_t m = row[t]; m < row[t + 1]; m++) acc += evec[m];
    v[t] = acc;
  }
}

}  // namespace

namespace mi355 {
int fill_zero(const CeedMi355Operator_private *op, void *x, hipStream_t s) {
  if (op->scalar_type == CEED_MI355_FP64) fill_kernel<double><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, 0.0, (double *)x);
  else fill_kernel<float><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, 0.0f, (float *)x);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

int split_finish(const CeedMi355Operator_private *op, void *v, int overwrite, hipStream_t s) {
  if (overwrite) {
    if (op->num_shared == 0) return CEED_MI355_SUCCESS;
    const int nb = mi355_blocks(op->num_shared, 256, 1 << 20);
    if (op->scalar_type == CEED_MI355_FP64)
      split_gather_kernel<double><<<nb, 256, 0, s>>>(op->num_shared, op->d_srows, op->d_trow, (const double *)op->d_evec, (double *)v);
    else split_gather_kernel<float><<<nb, 256, 0, s>>>(op->num_shared, op->d_srows, op->d_trow, (const float *)op->d_evec, (float *)v);
  } else {
    const int nb = mi355_blocks(op->l_size, 256, 1 << 20);
    if (op->scalar_type == CEED_MI355_FP64)
      split_add_kernel<double><<<nb, 256, 0, s>>>(op->l_size, op->d_trow, (const double *)op->d_evec, (const double *)op->d_scratch, (double *)v);
    else
      split_add_kernel<float><<<nb, 256, 0, s>>>(op->l_size, op->d_trow, (const float *)op->d_evec, (const float *)op->d_scratch, (float *)v);
  }
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

int transpose_gather(const CeedMi355Operator_private *op, void *v, int overwrite, GatherDot *dot, hipStream_t s) {
  if (op->d_gather_chunk_begin && op->d_sys_active && op->gather_num_chunks > 0) {
    const unsigned nb = (unsigned)op->gather_num_chunks;
    if (op->scalar_type == CEED_MI355_FP64)
      transpose_gather_chunks_kernel<double><<<nb, 256, 0, s>>>(op->d_gather_chunk_begin, op->d_gather_chunk_sys, op->d_sys_active, op->d_trow,
                                                                (const double *)op->d_evec, (double *)v, overwrite);
    else
      transpose_gather_chunks_kernel<float><<<nb, 256, 0, s>>>(op->d_gather_chunk_begin, op->d_gather_chunk_sys, op->d_sys_active, op->d_trow,
                                                               (const float *)op->d_evec, (float *)v, overwrite);
    MI355_LAUNCH_CHECK();
    return CEED_MI355_SUCCESS;
  }
  if (dot && overwrite) {
    GatherDot &d = *dot;
    d.nb         = mi355_blocks(op->l_size, 256, kDotBlocks);
    if (op->scalar_type == CEED_MI355_FP64)
      transpose_gather_dot_kernel<double><<<d.nb, 256, 0, s>>>(op->l_size, op->d_trow, (const double *)op->d_evec, (const double *)d.u, (double *)v,
                                                               d.partial, d.to, d.from);
    else
      transpose_gather_dot_kernel<float><<<d.nb, 256, 0, s>>>(op->l_size, op->d_trow, (const float *)op->d_evec, (const float *)d.u, (float *)v,
                                                              d.partial, d.to, d.from);
    MI355_LAUNCH_CHECK();
    return CEED_MI355_SUCCESS;
  }
  const int nb = mi355_blocks(op->l_size, 256, 1 << 20);
  if (op->scalar_type == CEED_MI355_FP64)
    transpose_gather_kernel<double><<<nb, 256, 0, s>>>(op->l_size, op->d_trow, (const double *)op->d_evec, (double *)v, overwrite);
  else transpose_gather_kernel<float><<<nb, 256, 0, s>>>(op->l_size, op->d_trow, (const float *)op->d_evec, (float *)v, overwrite);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}
}  // namespace mi355

extern "C" int CeedMi355OperatorCreateHex(int qf, int scalar_type, int32_t num_comp, int32_t num_elem, int32_t P_1d, int32_t Q_1d,
                                          const double *interp_1d_host, const double *grad_1d_host, const int32_t *offsets_host,
                                          int32_t comp_stride, int64_t l_size, int flags, CeedMi355Operator *op_out) {
  *op_out = nullptr;
  MI355_CHECK(qf == kQfMass || qf == kQfDiffusion || qf == kQfDiffusionKappa, CEED_MI355_ERROR_UNSUPPORTED, "unknown pointwise operator %d", qf);
  MI355_CHECK(scalar_type == CEED_MI355_FP64 || scalar_type == CEED_MI355_FP32, CEED_MI355_ERROR_UNSUPPORTED, "unknown scalar type");
  MI355_CHECK(num_elem >= 0 && l_size > 0, CEED_MI355_ERROR_DIMENSION, "invalid operator sizes");
  mi355::ApplyFn fn = scalar_type == CEED_MI355_FP64 ? mi355::pick_apply_f64(P_1d, Q_1d, num_comp, qf)
                                                     : mi355::pick_apply_f32(P_1d, Q_1d, num_comp, qf);
  MI355_CHECK(fn, CEED_MI355_ERROR_UNSUPPORTED, "no fused kernel for P=%d Q=%d num_comp=%d qf=%d", P_1d, Q_1d, num_comp, qf);
  return mi355::create_plan(qf, scalar_type, num_comp, num_elem, P_1d, Q_1d, interp_1d_host, grad_1d_host, offsets_host, comp_stride, l_size,
                            flags, qf == kQfMass ? 1 : (qf == kQfDiffusion ? 6 : 7), fn, op_out);
}

int mi355::create_plan(int qf, int scalar_type, int32_t num_comp, int32_t num_elem, int32_t P_1d, int32_t Q_1d, const double *interp_1d_host,
                       const double *grad_1d_host, const int32_t *offsets_host, int32_t comp_stride, int64_t l_size, int flags, int q_comp,
                       mi355::ApplyFn fn, CeedMi355Operator *op_out) {
  *op_out = nullptr;
  CeedMi355Operator op = new CeedMi355Operator_private();
  op->qf = qf;
  op->scalar_type = scalar_type;
  op->scalar_bytes = scalar_type == CEED_MI355_FP64 ? 8 : 4;
  op->num_comp = num_comp;
  op->P = P_1d;
  op->Q = Q_1d;
  op->q_comp = q_comp;
  op->num_elem = num_elem;
  op->comp_stride = comp_stride;
  op->l_size = l_size;
  op->apply = fn;
  // E^T mode; by default colours only where they are faster than the
  // transpose map on MI355X: below P = 6 (FP64 and FP32; FP32 at P = 6, 8M
  // DoFs: map 0.169 ms, colours 0.200), where the
  // E-vector round trip of the map costs more than the colour launches, and
  // from 10M E-vector entries, where each of the (about 8) colour launches
  // still fills the GPU (at 2M DoFs, p = 4, the map is 1.33x faster; at 8M,
  // colours are 1.07x faster).  From 10M entries at P = 7 and 8 in FP64 the
  // multiplicity split (same Apply bits as the map) is faster still for one
  // component: 1.08x at p = 6, 1.03x at p = 7, 8M DoFs; with three
  // components the map is (8M nodes: p = 6 0.691 vs 0.803 ms, p = 7 0.727
  // vs 0.831 ms).
  const int64_t evec_entries = (int64_t)num_elem * P_1d * P_1d * P_1d * num_comp;
  const bool    big          = evec_entries >= 10000000;
  if (flags & CEED_MI355_PLAN_SEGMENT) op->scatter = CEED_MI355_PLAN_SEGMENT;
  else if (flags & CEED_MI355_PLAN_BRICK) op->scatter = CEED_MI355_PLAN_BRICK;
  else if (flags & CEED_MI355_PLAN_SPLIT) op->scatter = CEED_MI355_PLAN_SPLIT;
  else if (flags & CEED_MI355_PLAN_ATOMIC) op->scatter = CEED_MI355_PLAN_ATOMIC;
  else if (flags & CEED_MI355_PLAN_COLOR) op->scatter = CEED_MI355_PLAN_COLOR;
  else if (flags & CEED_MI355_PLAN_TMAP) op->scatter = 0;
  else if (big && scalar_type == CEED_MI355_FP64 && num_comp == 1 && (P_1d == 7 || P_1d == 8)) op->scatter = CEED_MI355_PLAN_SPLIT;
  else op->scatter = P_1d >= 6 || !big ? 0 : CEED_MI355_PLAN_COLOR;
  const int explicit_modes =
      CEED_MI355_PLAN_ATOMIC | CEED_MI355_PLAN_COLOR | CEED_MI355_PLAN_TMAP | CEED_MI355_PLAN_SPLIT | CEED_MI355_PLAN_BRICK | CEED_MI355_PLAN_SEGMENT;
  const int default_scatter = op->scatter;
  if (!(flags & explicit_modes))
    if (const char *env = getenv("CEED_MI355_SCATTER")) {  // color | tmap | split | atomic | brick | segment replaces the default
      if (!strcmp(env, "color")) op->scatter = CEED_MI355_PLAN_COLOR;
      else if (!strcmp(env, "tmap")) op->scatter = 0;
      else if (!strcmp(env, "split")) op->scatter = CEED_MI355_PLAN_SPLIT;
      else if (!strcmp(env, "atomic")) op->scatter = CEED_MI355_PLAN_ATOMIC;
      else if (!strcmp(env, "brick")) op->scatter = CEED_MI355_PLAN_BRICK;
      else if (!strcmp(env, "segment")) op->scatter = CEED_MI355_PLAN_SEGMENT;
      else {
        delete op;
        MI355_CHECK(false, CEED_MI355_ERROR_BACKEND, "CEED_MI355_SCATTER=%s: expected color, tmap, split, atomic, brick or segment", env);
      }
    }
  // the brick and segment E^T exist for the gallery mass and diffusion
  // kernels; a plan of another kind asked for one by flag is an error, by the
  // environment it keeps its default
  if ((op->scatter == CEED_MI355_PLAN_BRICK || op->scatter == CEED_MI355_PLAN_SEGMENT) && !(qf == kQfMass || qf == kQfDiffusion)) {
    if (flags & (CEED_MI355_PLAN_BRICK | CEED_MI355_PLAN_SEGMENT)) {
      delete op;
      MI355_CHECK(false, CEED_MI355_ERROR_UNSUPPORTED, "the brick and segment E^T support mass and diffusion plans only");
    }
    op->scatter = default_scatter;
  }
  // launch: the tuned (layout, elements per workgroup) of this kind of plan if the
  // autotuner has run on one in this process, else the line layout (faster
  // than the column layout at every order measured on MI355X, equal at p <= 2)
  // with its default workgroup size; CEED_MI355_LAYOUT / CEED_MI355_EPB override
  op->layout = mi355::kLayoutLines;
  op->epb    = plan_default_epb(op, op->layout);
  tuned_launch(op);
  if (const char *env = getenv("CEED_MI355_LAYOUT")) {
    const int l = atoi(env);
    if (layout_exists(Q_1d, qf, l)) op->own_launch = true, op->layout = l, op->epb = mi355::default_epb(P_1d, Q_1d, qf, num_comp, op->scalar_bytes, l);
  }
  if (qf == kQfJit && op->layout != mi355::kLayoutLines)  // run-time compiled kernels exist in the line layout only
    op->layout = mi355::kLayoutLines, op->epb = mi355::default_epb(P_1d, Q_1d, qf, num_comp, op->scalar_bytes, op->layout);
  if (const char *env = getenv("CEED_MI355_EPB")) {
    const int v = atoi(env);
    if (admissible(P_1d, Q_1d, qf, num_comp, op->scalar_bytes, op->layout, v)) op->own_launch = op->line_only = true, op->epb = v;
  }

  const int            es = P_1d * P_1d * P_1d;
  std::vector<int32_t> color;
  int                  num_colors = 0;
  int                  ierr       = CEED_MI355_SUCCESS;
  if (op->scatter == CEED_MI355_PLAN_BRICK) {
    // bricks of face-sharing elements, one workgroup each: the largest of
    // 2x2x2, 2x2x1, 2x1x1, 1x1x1 whose workgroup fits 512 threads and the
    // CU's LDS; CEED_MI355_BRICK="bx,by,bz" replaces it
    static const int candidates[4][3] = {{2, 2, 2}, {2, 2, 1}, {2, 1, 1}, {1, 1, 1}};
    int              shape[3]         = {1, 1, 1};
    auto             fits             = [&](const int *sh) {
      const int64_t ns = (int64_t)sh[0] * sh[1] * sh[2];
      return mi355::brick_threads(Q_1d, ns) <= 512 && mi355::brick_lds_bytes(P_1d, Q_1d, qf, op->scalar_bytes, sh) <= mi355::kMaxLdsBytes;
    };
    for (const auto &c : candidates)
      if (fits(c)) {
        shape[0] = c[0], shape[1] = c[1], shape[2] = c[2];
        break;
      }
    if (const char *env = getenv("CEED_MI355_BRICK")) {
      int a, b, c;
      if (sscanf(env, "%d,%d,%d", &a, &b, &c) == 3 && a >= 1 && b >= 1 && c >= 1 && a * b * c <= 8) shape[0] = a, shape[1] = b, shape[2] = c;
    }
    if (!fits(shape)) {
      CeedMi355OperatorDestroy(&op);
      MI355_CHECK(false, CEED_MI355_ERROR_UNSUPPORTED, "brick %dx%dx%d needs more than 512 threads or %d bytes of LDS", shape[0], shape[1],
                  shape[2], mi355::kMaxLdsBytes);
    }
    ierr = num_elem > 0 ? mi355::build_bricks(op, offsets_host, shape[0], shape[1], shape[2], op->perm) : CEED_MI355_SUCCESS;
    if (ierr == CEED_MI355_ERROR_UNSUPPORTED && !(flags & CEED_MI355_PLAN_BRICK)) {  // no bricks in this mesh: the default mode
      for (void *d : {(void *)op->d_brick_start, (void *)op->d_brick_mask, (void *)op->d_bnode, (void *)op->d_blist, (void *)op->d_brow,
                      (void *)op->d_bslot, op->d_partials})
        (void)hipFree(d);
      op->d_brick_start = op->d_brick_mask = op->d_bnode = op->d_blist = op->d_brow = op->d_bslot = nullptr;
      op->d_partials = nullptr;
      op->num_bricks = op->num_bound = 0;
      op->scatter    = default_scatter == CEED_MI355_PLAN_BRICK ? 0 : default_scatter;
      ierr           = CEED_MI355_SUCCESS;
    }
    if (ierr) {
      CeedMi355OperatorDestroy(&op);
      return ierr;
    }
  }
  const bool colored  = op->scatter == CEED_MI355_PLAN_COLOR;
  const bool bricks   = op->scatter == CEED_MI355_PLAN_BRICK;
  const bool segments = op->scatter == CEED_MI355_PLAN_SEGMENT;
  std::vector<uint8_t> seg_first;  // segments: packed element starts its segment
  if (segments) {
    // a workgroup per segment in the line layout, as many element slots as
    // 256 threads hold (within the CU's LDS), no other launch
    int max_len = 256 / (Q_1d * Q_1d);
    if (const char *env = getenv("CEED_MI355_SEGMENT_MAX")) max_len = std::max(1, std::min(max_len, atoi(env)));
    while (max_len > 1 && mi355::lds_bytes(P_1d, Q_1d, qf, num_comp, max_len, op->scalar_bytes, mi355::kLayoutLines) > mi355::kMaxLdsBytes) max_len--;
    mi355::SegmentLayout L;
    ierr = mi355::segment_layout(offsets_host, num_elem, P_1d, max_len, L);
    if (ierr) {
      delete op;
      return ierr;
    }
    op->perm      = std::move(L.perm);
    op->seg_color = std::move(L.color);
    op->seg_max   = std::max(1, L.max_len);  // (1 for a plan without elements)
    op->layout    = mi355::kLayoutLines;
    op->epb       = op->seg_max;
    op->color_start.assign(op->seg_color.size(), 0);
    for (size_t c = 0; c < op->seg_color.size(); c++) op->color_start[c] = L.start[op->seg_color[c]];
    seg_first.assign((size_t)num_elem, 0);
    for (size_t g = 0; g + 1 < L.start.size(); g++) seg_first[L.start[g]] = 1;
    MI355_HIP(hipMalloc(&op->d_seg_start, sizeof(int32_t) * L.start.size()));
    MI355_HIP(hipMemcpy(op->d_seg_start, L.start.data(), sizeof(int32_t) * L.start.size(), hipMemcpyHostToDevice));
  } else if (colored) ierr = color_elements(offsets_host, num_elem, es, num_comp, comp_stride, l_size, color, num_colors);
  else {  // one launch over all elements in element order (brick order for bricks)
    color.assign((size_t)num_elem, 0);
    num_colors = num_elem > 0 ? 1 : 0;
  }
  if (ierr) {
    delete op;
    return ierr;
  }
  if (bricks) {
    op->color_start.assign(2, 0);
    op->color_start[1] = num_elem;
    if (num_elem == 0) op->color_start.resize(1);
  } else if (!segments) {  // (segments: packed order and colours from the segment layout)
    // packed order: by colour, ascending element index inside a colour
    op->color_start.assign(num_colors + 1, 0);
    for (int64_t e = 0; e < num_elem; e++) op->color_start[color[e] + 1]++;
    for (int c = 0; c < num_colors; c++) op->color_start[c + 1] += op->color_start[c];
    op->perm.resize(num_elem);
    std::vector<int64_t> cursor(op->color_start.begin(), op->color_start.end() - 1);
    for (int64_t e = 0; e < num_elem; e++) op->perm[cursor[color[e]]++] = (int32_t)e;
  }
  // offsets in colour order, encoded 2 * node + bit: with colours (and segments) the bit marks
  // the first element (in launch order) writing a node, which may overwrite v in CeedOperatorApply
  // instead of accumulating; in the split mode it marks nodes of more than two contributions.
  // In a segment, the x = 0 face of every element but the first is written by the element
  // before it, so it neither writes nor counts as reaching the node.
  std::vector<int32_t> packed((size_t)num_elem * es);
  const bool           split = op->scatter == CEED_MI355_PLAN_SPLIT;
  {
    int64_t n_nodes = 0;
    for (int64_t i = 0; i < (int64_t)num_elem * es; i++) n_nodes = std::max<int64_t>(n_nodes, (int64_t)offsets_host[i] + 1);
    if (n_nodes >= (1ll << 30)) {
      CeedMi355OperatorDestroy(&op);
      MI355_CHECK(false, CEED_MI355_ERROR_UNSUPPORTED, "more than 2^30 nodes");
    }
    std::vector<char>    touched(n_nodes, 0);
    std::vector<int32_t> mult(split ? n_nodes : 0, 0);
    if (split)
      for (int64_t i = 0; i < (int64_t)num_elem * es; i++) mult[offsets_host[i]]++;
    for (int64_t p = 0; p < num_elem; p++)
      for (int i = 0; i < es; i++) {
        const int32_t node     = offsets_host[(int64_t)op->perm[p] * es + i];
        const bool    absorbed = segments && !seg_first[p] && i % P_1d == 0;
        packed[p * es + i]     = 2 * node + (((colored || segments) && !absorbed && !touched[node]) || (split && mult[node] > 2) ? 1 : 0);
        if (!absorbed) touched[node] = 1;
      }
    std::vector<uint8_t> hit(l_size, 0);
    for (int64_t n = 0; n < n_nodes; n++)
      if (touched[n])
        for (int k = 0; k < num_comp; k++) {
          uint8_t &h = hit[n + (int64_t)k * comp_stride];
          if (h) {
            CeedMi355OperatorDestroy(&op);
            MI355_CHECK(false, CEED_MI355_ERROR_UNSUPPORTED, "components overlap at L index %lld", (long long)(n + (int64_t)k * comp_stride));
          }
          h = 1;
        }
    // the transpose map writes every L entry; atomics need a zeroed v; colours and bricks overwrite what they reach
    op->covers_all = op->scatter == 0 || ((colored || bricks || segments) && std::all_of(hit.begin(), hit.end(), [](uint8_t h) { return h != 0; }));
  }
  if (split) {
    ierr = build_split_map(op, packed.data());
    if (ierr) {
      CeedMi355OperatorDestroy(&op);
      return ierr;
    }
  }
  if (op->scatter == 0) {
    ierr = build_transpose_map(op, offsets_host);
    if (ierr) {
      CeedMi355OperatorDestroy(&op);
      return ierr;
    }
  }

  // B and the collocated derivative D = G pinv(B), then (for the diagonal) the
  // entrywise products B B, B G, G G with G = D B, in the plan's scalar type
  const int           QP = Q_1d * P_1d, QQ = Q_1d * Q_1d;
  std::vector<double> mats(QP + QQ + 3 * QP);
  memcpy(mats.data(), interp_1d_host, sizeof(double) * Q_1d * P_1d);
  mi355::collocated_grad(P_1d, Q_1d, interp_1d_host, grad_1d_host, &mats[Q_1d * P_1d]);
  for (int q = 0; q < Q_1d; q++)
    for (int a = 0; a < P_1d; a++) {
      double g = 0;
      for (int c = 0; c < Q_1d; c++) g += mats[QP + q * Q_1d + c] * mats[c * P_1d + a];
      const double b = mats[q * P_1d + a];
      const int    i = QP + QQ + q * P_1d + a;
      mats[i] = b * b, mats[i + QP] = b * g, mats[i + 2 * QP] = g * g;
    }

  MI355_HIP(hipMalloc(&op->d_offsets, sizeof(int32_t) * (packed.size() + 1)));
  MI355_HIP(hipMemcpy(op->d_offsets, packed.data(), sizeof(int32_t) * packed.size(), hipMemcpyHostToDevice));
  MI355_HIP(hipMalloc(&op->d_perm, sizeof(int32_t) * (num_elem + 1)));
  MI355_HIP(hipMemcpy(op->d_perm, op->perm.data(), sizeof(int32_t) * num_elem, hipMemcpyHostToDevice));
  MI355_HIP(hipMalloc(&op->d_mats, op->scalar_bytes * mats.size()));
  if (scalar_type == CEED_MI355_FP64) {
    MI355_HIP(hipMemcpy(op->d_mats, mats.data(), sizeof(double) * mats.size(), hipMemcpyHostToDevice));
  } else {
    std::vector<float> m32(mats.begin(), mats.end());
    MI355_HIP(hipMemcpy(op->d_mats, m32.data(), sizeof(float) * m32.size(), hipMemcpyHostToDevice));
  }
  MI355_HIP(hipMalloc(&op->d_qdata, (size_t)op->scalar_bytes * ((size_t)num_elem * elem_block(op) + 1)));
  MI355_HIP(hipMemset(op->d_qdata, 0, (size_t)op->scalar_bytes * ((size_t)num_elem * elem_block(op) + 1)));
  *op_out = op;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorBuildQData(CeedMi355Operator op, int build, int32_t mesh_P_1d, const double *mesh_interp_1d_host,
                                           const double *mesh_grad_1d_host, const double *q_weight_1d_host, const int32_t *mesh_offsets_host,
                                           int32_t mesh_comp_stride, const double *coords, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  MI355_CHECK((build == 0 && op->qf == kQfMass) || (build == 1 && (op->qf == kQfDiffusion || op->qf == kQfDiffusionKappa)),
              CEED_MI355_ERROR_BACKEND, "geometric factor kind %d does not match the operator", build);
  MI355_CHECK(mesh_P_1d >= 2 && mesh_P_1d <= op->Q, CEED_MI355_ERROR_UNSUPPORTED, "mesh P_1d=%d must be in 2..Q=%d", mesh_P_1d, op->Q);
  hipStream_t s = (hipStream_t)stream;
  const int   Q = op->Q, PM = mesh_P_1d, PM3 = PM * PM * PM;
  // mesh offsets in the plan's colour order
  std::vector<int32_t> mo((size_t)op->num_elem * PM3);
  for (int64_t p = 0; p < op->num_elem; p++) memcpy(&mo[p * PM3], &mesh_offsets_host[(int64_t)op->perm[p] * PM3], sizeof(int32_t) * PM3);
  std::vector<double> mats(Q * PM + Q * Q + Q);
  memcpy(mats.data(), mesh_interp_1d_host, sizeof(double) * Q * PM);
  mi355::collocated_grad(PM, Q, mesh_interp_1d_host, mesh_grad_1d_host, &mats[Q * PM]);
  memcpy(&mats[Q * PM + Q * Q], q_weight_1d_host, sizeof(double) * Q);
  const int64_t blk = elem_block(op);
  // a linear mesh basis: the elements' trilinear maps, kept where the plan's applies recompute the factors from them
  const bool            linear    = PM == 2 && linear_mesh_basis(Q, mesh_interp_1d_host, mesh_grad_1d_host);
  mi355::GeoLinesFn     geo_lines = op->scalar_type == CEED_MI355_FP64 ? mi355::pick_geo_f64(op->P, Q, op->num_comp, op->qf)
                                                                       : mi355::pick_geo_f32(op->P, Q, op->num_comp, op->qf);
  const bool            trilinear = linear && geo_lines && mi355::geo_pays(op->P, Q, op->qf, op->num_comp, op->scalar_bytes);
  std::vector<double>   pts(2 * Q);  // pts, turn: read by the copies below until the synchronisation
  const int32_t         turn[2] = {1, 0};
  const size_t          geo_bytes = sizeof(double) * mi355::kGeoStride * ((size_t)op->num_elem + 1), pts_bytes = sizeof(double) * pts.size();
  TempBuffer            mo_buf, mats_buf, geo_buf, pts_buf;
  // from here on a failure leaves a plan that reads whatever factors it holds, not one that recomputes half-written ones
  const bool was_valid = op->geo_valid;
  op->geo_valid        = false;
  MI355_HIP(hipMalloc(&mo_buf.p, sizeof(int32_t) * (mo.size() + 1)));
  MI355_HIP(hipMemcpyAsync(mo_buf.p, mo.data(), sizeof(int32_t) * mo.size(), hipMemcpyHostToDevice, s));
  const int32_t *d_mo = (const int32_t *)mo_buf.p;
  if (linear) {
    for (int q = 0; q < Q; q++) pts[q] = mesh_interp_1d_host[2 * q + 1] - mesh_interp_1d_host[2 * q], pts[Q + q] = q_weight_1d_host[q];
    if (trilinear) {
      if (!op->d_geo) MI355_HIP(hipMalloc(&op->d_geo, geo_bytes));
      if (!op->d_geo_pts) MI355_HIP(hipMalloc(&op->d_geo_pts, pts_bytes));
      if (!op->d_geo_turn) MI355_HIP(hipMalloc(&op->d_geo_turn, sizeof(turn)));
      MI355_HIP(hipMemcpyAsync(op->d_geo_turn, turn, sizeof(turn), hipMemcpyHostToDevice, s));
      op->geo_lines = geo_lines;
    } else {
      MI355_HIP(hipMalloc(&geo_buf.p, geo_bytes));
      MI355_HIP(hipMalloc(&pts_buf.p, pts_bytes));
    }
    double *d_geo = trilinear ? op->d_geo : (double *)geo_buf.p, *d_pts = trilinear ? op->d_geo_pts : (double *)pts_buf.p;
    MI355_HIP(hipMemcpyAsync(d_pts, pts.data(), pts_bytes, hipMemcpyHostToDevice, s));
    const int64_t q3 = (int64_t)Q * Q * Q;
    geo_coefficients<<<mi355_blocks(op->num_elem * 3, 256), 256, 0, s>>>(op->num_elem, d_mo, mesh_comp_stride, coords, d_geo);
    if (op->scalar_type == CEED_MI355_FP64)
      geo_qdata<double><<<mi355_blocks(op->num_elem * q3, 256), 256, 0, s>>>(op->num_elem, Q, build == 0, blk, d_geo, d_pts, (double *)op->d_qdata);
    else geo_qdata<float><<<mi355_blocks(op->num_elem * q3, 256), 256, 0, s>>>(op->num_elem, Q, build == 0, blk, d_geo, d_pts, (float *)op->d_qdata);
    MI355_LAUNCH_CHECK();
  } else {
    MI355_HIP(hipMalloc(&mats_buf.p, sizeof(double) * mats.size()));
    MI355_HIP(hipMemcpyAsync(mats_buf.p, mats.data(), sizeof(double) * mats.size(), hipMemcpyHostToDevice, s));
    const double *d_mats = (const double *)mats_buf.p;
    const int     ierr   = op->scalar_type == CEED_MI355_FP64
                               ? dispatch_build<double>(Q, build, op->num_elem, PM, d_mo, mesh_comp_stride, coords, d_mats, blk, (double *)op->d_qdata, s)
                               : dispatch_build<float>(Q, build, op->num_elem, PM, d_mo, mesh_comp_stride, coords, d_mats, blk, (float *)op->d_qdata, s);
    if (ierr) return ierr;
  }
  if (!trilinear) {
    const int ierr = factors_replaced(op, s);
    if (ierr) return ierr;
  }
  MI355_HIP(hipStreamSynchronize(s));
  op->geo_valid = was_valid;
  set_geo_valid(op, trilinear);
  if (op->qf == kQfDiffusionKappa) {
    // kappa slot defaults to 1 until CeedMi355OperatorSetKappa
    const int64_t Q3 = (int64_t)Q * Q * Q, n = op->num_elem * Q3;
    if (op->scalar_type == CEED_MI355_FP64)
      fill_slot<double><<<mi355_blocks(n, 256), 256, 0, s>>>(op->num_elem, Q3, 7 * Q3, 6 * Q3, 1.0, (double *)op->d_qdata);
    else fill_slot<float><<<mi355_blocks(n, 256), 256, 0, s>>>(op->num_elem, Q3, 7 * Q3, 6 * Q3, 1.0f, (float *)op->d_qdata);
    MI355_LAUNCH_CHECK();
  }
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorSetQData(CeedMi355Operator op, const void *q_data, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  const int64_t per = (int64_t)(op->qf == kQfDiffusionKappa ? 6 : op->q_comp) * op->Q * op->Q * op->Q;
  const int64_t blk = elem_block(op);
  hipStream_t   s   = (hipStream_t)stream;
  MI355_CHECK(per == blk || op->qf == kQfDiffusionKappa, CEED_MI355_ERROR_BACKEND, "layout mismatch");
  if (op->qf != kQfDiffusionKappa) {  // the caller's factors from here on
    if (is_capturing(s)) op->qdata_in_graph = true;
    set_geo_valid(op, false);
    const int err = factors_replaced(op, s);
    if (err) return err;
    if (op->scalar_type == CEED_MI355_FP64)
      permute_elements<double, double><<<mi355_blocks(op->num_elem * per, 256), 256, 0, s>>>(op->num_elem, per, op->d_perm, 1,
                                                                                             (const double *)q_data, (double *)op->d_qdata);
    else
      permute_elements<float, float><<<mi355_blocks(op->num_elem * per, 256), 256, 0, s>>>(op->num_elem, per, op->d_perm, 1,
                                                                                           (const float *)q_data, (float *)op->d_qdata);
    MI355_LAUNCH_CHECK();
    return CEED_MI355_SUCCESS;
  }
  MI355_CHECK(false, CEED_MI355_ERROR_UNSUPPORTED, "SetQData for the kappa operator: build the 6 Voigt entries with BuildQData");
}

namespace {
// components [first, first + nc) of every element block of q_comp components, from src [elem][nc][q3] in the caller's order
__global__ void __launch_bounds__(256) scatter_components(int64_t num_elem, int32_t q3, int32_t q_comp, int32_t first, int32_t nc,
                                                          const int32_t *__restrict__ perm, const double *__restrict__ src,
                                                          double *__restrict__ q_data) {
  const int64_t per = (int64_t)nc * q3, n = num_elem * per;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = i / per, r = i - p * per;
    q_data[(p * q_comp + first) * q3 + r] = src[perm[p] * per + r];
  }
}
}  // namespace

extern "C" int CeedMi355OperatorSetQDataComponents(CeedMi355Operator op, int32_t first, int32_t num, const void *q_data, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  MI355_CHECK(op->qf == kQfJit && op->scalar_type == CEED_MI355_FP64, CEED_MI355_ERROR_UNSUPPORTED,
              "components of the passive fields belong to plans of run-time compiled QFunctions");
  MI355_CHECK(first >= 0 && num >= 1 && first + num <= op->q_comp, CEED_MI355_ERROR_DIMENSION, "components %d..%d of %d", first, first + num, op->q_comp);
  const int32_t q3 = op->Q * op->Q * op->Q;
  if (op->num_elem > 0)
    scatter_components<<<mi355_blocks((int64_t)op->num_elem * num * q3, 256), 256, 0, (hipStream_t)stream>>>(
        op->num_elem, q3, op->q_comp, first, num, op->d_perm, (const double *)q_data, (double *)op->d_qdata);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorGetQData(CeedMi355Operator op, void *q_data, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  const int64_t blk = elem_block(op);
  hipStream_t   s   = (hipStream_t)stream;
  if (op->scalar_type == CEED_MI355_FP64)
    permute_elements<double, double><<<mi355_blocks(op->num_elem * blk, 256), 256, 0, s>>>(op->num_elem, blk, op->d_perm, 0,
                                                                                           (const double *)op->d_qdata, (double *)q_data);
  else
    permute_elements<float, float><<<mi355_blocks(op->num_elem * blk, 256), 256, 0, s>>>(op->num_elem, blk, op->d_perm, 0,
                                                                                         (const float *)op->d_qdata, (float *)q_data);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

namespace {
// kappa [elem][Q^3] (caller order, FP64) into q_data slot 6 of each element block
template <typename T>
__global__ void __launch_bounds__(256) scatter_kappa(int64_t num_elem, int64_t q3, const int32_t *__restrict__ perm,
                                                     const double *__restrict__ kappa, T *__restrict__ q_data) {
  const int64_t n = num_elem * q3;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t p = i / q3, r = i - p * q3;
    q_data[p * 7 * q3 + 6 * q3 + r] = (T)kappa[(int64_t)perm[p] * q3 + r];
  }
}
}  // namespace

extern "C" int CeedMi355OperatorSetKappa(CeedMi355Operator op, const double *kappa, void *stream) {
  MI355_CHECK(op && op->qf == kQfDiffusionKappa, CEED_MI355_ERROR_BACKEND, "SetKappa needs a kappa-diffusion operator");
  const int64_t q3 = (int64_t)op->Q * op->Q * op->Q;
  hipStream_t   s  = (hipStream_t)stream;
  if (op->scalar_type == CEED_MI355_FP64)
    scatter_kappa<double><<<mi355_blocks(op->num_elem * q3, 256), 256, 0, s>>>(op->num_elem, q3, op->d_perm, kappa, (double *)op->d_qdata);
  else scatter_kappa<float><<<mi355_blocks(op->num_elem * q3, 256), 256, 0, s>>>(op->num_elem, q3, op->d_perm, kappa, (float *)op->d_qdata);
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

namespace {
int apply_overwrite(CeedMi355Operator op, const void *u, void *v, const mi355::ApplyExtras &x, hipStream_t s) {
  mi355::touch_thread_storage();
  // first-touch entries are overwritten by the kernel; entries no element reaches are zeroed here
  if (!op->covers_all || op->num_elem == 0) {
    if (op->scalar_type == CEED_MI355_FP64)
      fill_kernel<double><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, 0.0, (double *)v);
    else fill_kernel<float><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, 0.0f, (float *)v);
    MI355_LAUNCH_CHECK();
  }
  if (op->num_elem == 0) return CEED_MI355_SUCCESS;
  return op->apply(op, u, v, 1, x, s);
}
}  // namespace

extern "C" int CeedMi355OperatorApply(CeedMi355Operator op, const void *u, void *v, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  return apply_overwrite(op, u, v, {}, (hipStream_t)stream);
}

int mi355::apply_dot(CeedMi355Operator op, const void *u, void *v, double *partial, double *to, const double *from, int *nb, hipStream_t s) {
  GatherDot d;
  d.u = u, d.partial = partial, d.to = to, d.from = from;
  ApplyExtras x;
  x.dot          = &d;
  const int ierr = apply_overwrite(op, u, v, x, s);
  *nb            = d.nb;
  return ierr;
}

bool mi355::into_callers_graph(const CeedMi355Operator_private *op, hipStream_t s) { return !op->solver_graph && is_capturing(s); }

extern "C" int CeedMi355OperatorApplyKappa(CeedMi355Operator op, const double *kappa, const void *u, void *v, void *stream) {
  MI355_CHECK(op && op->qf == kQfDiffusionKappa && (kappa || op->num_elem == 0), CEED_MI355_ERROR_BACKEND,
              "ApplyKappa needs a kappa-diffusion operator and kappa");
  // the line kernel that recomputes the factors takes kappa from the caller
  // and keeps it on the way, unless it may skip elements (stopped systems) or
  // is one of two kernels in a caller's graph
  if (!mi355::plan_recomputes(op) || op->d_elem_sys || mi355::into_callers_graph(op, (hipStream_t)stream)) {
    const int err = CeedMi355OperatorSetKappa(op, kappa, stream);
    return err ? err : CeedMi355OperatorApply(op, u, v, stream);
  }
  mi355::ApplyExtras x;
  x.kappa = kappa;
  return apply_overwrite(op, u, v, x, (hipStream_t)stream);
}

extern "C" int CeedMi355OperatorApplyAdd(CeedMi355Operator op, const void *u, void *v, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  if (op->num_elem == 0) return CEED_MI355_SUCCESS;
  mi355::touch_thread_storage();
  return op->apply(op, u, v, 0, {}, (hipStream_t)stream);
}

extern "C" int CeedMi355OperatorSetLaunch(CeedMi355Operator op, int32_t elems_per_block) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  MI355_CHECK(plan_admissible(op, op->layout, elems_per_block), CEED_MI355_ERROR_BACKEND,
              "%d elements per workgroup do not fit (at most 256 threads and 160 KiB of LDS for P=%d Q=%d)", elems_per_block, op->P, op->Q);
  op->epb        = elems_per_block;
  op->own_launch = op->line_only = true;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorSetLayout(CeedMi355Operator op, int32_t layout, int32_t elems_per_block) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  MI355_CHECK(layout == mi355::kLayoutColumns || layout == mi355::kLayoutLines || layout == mi355::kLayoutPoints, CEED_MI355_ERROR_BACKEND,
              "unknown thread layout %d", layout);
  MI355_CHECK(layout == mi355::kLayoutLines || op->qf != kQfJit, CEED_MI355_ERROR_UNSUPPORTED,
              "plans of run-time compiled QFunctions have the line layout only");
  MI355_CHECK(layout_exists(op->Q, op->qf, layout), CEED_MI355_ERROR_UNSUPPORTED, "the point layout needs Q^3 <= 256 (Q = %d)", op->Q);
  const int epb = elems_per_block > 0                       ? elems_per_block
                  : op->scatter == CEED_MI355_PLAN_SEGMENT ? op->seg_max
                                                           : plan_default_epb(op, layout);
  MI355_CHECK(plan_admissible(op, layout, epb), CEED_MI355_ERROR_BACKEND,
              "%d elements per workgroup do not fit layout %d (at most 256 threads and 160 KiB of LDS for P=%d Q=%d)", epb, layout, op->P, op->Q);
  op->layout     = layout;
  op->epb        = epb;
  op->own_launch = true;
  op->line_only  = elems_per_block > 0;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorRecomputesFactors(CeedMi355Operator op, int32_t *yes) {
  MI355_CHECK(op && yes, CEED_MI355_ERROR_MAJOR, "null argument");
  *yes = mi355::plan_recomputes(op);
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorGetLaunch(CeedMi355Operator op, int32_t *layout, int32_t *elems_per_block) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  if (layout) *layout = op->layout;
  if (elems_per_block) *elems_per_block = op->epb;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorGetKernel(CeedMi355Operator op, int32_t *kernel, int32_t *gather) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  int64_t most = 0;  // elements of the largest launch
  for (size_t c = 0; c + 1 < op->color_start.size(); c++) most = std::max<int64_t>(most, op->color_start[c + 1] - op->color_start[c]);
  if (kernel)
    *kernel = op->scatter == CEED_MI355_PLAN_BRICK                             ? CEED_MI355_KERNEL_BRICK
              : mi355::plan_recomputes(op) && mi355::elements_take(op, most) ? CEED_MI355_KERNEL_ELEMENTS
              : op->layout == mi355::kLayoutLines                             ? CEED_MI355_KERNEL_LINES
              : op->layout == mi355::kLayoutPoints                            ? CEED_MI355_KERNEL_POINTS
                                                                              : CEED_MI355_KERNEL_COLUMNS;
  if (gather)
    *gather = (op->scatter == 0 && !mi355::plan_sums_last(op)) || op->scatter == CEED_MI355_PLAN_SPLIT || op->scatter == CEED_MI355_PLAN_BRICK;
  return CEED_MI355_SUCCESS;
}

namespace {
template <typename T>
__global__ void __launch_bounds__(256) tune_fill(int64_t n, T *__restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) x[i] = T(1) + T(i % 7) * T(0.125);
}
}  // namespace

extern "C" int CeedMi355OperatorAutotune(CeedMi355Operator op, int32_t reps, int32_t *best_epb, double *best_ms, void *stream) {
  MI355_CHECK(op && reps >= 1, CEED_MI355_ERROR_MAJOR, "bad autotune arguments");
  hipStream_t s = (hipStream_t)stream;
  void       *u = nullptr, *v = nullptr;
  hipEvent_t  t0 = nullptr, t1 = nullptr;
  auto        release = [&]() {
    if (t0) (void)hipEventDestroy(t0);
    if (t1) (void)hipEventDestroy(t1);
    (void)hipFree(u);
    (void)hipFree(v);
  };
  const size_t bytes = (size_t)op->scalar_bytes * (op->l_size + 1);
  if (hipMalloc(&u, bytes) != hipSuccess || hipMalloc(&v, bytes) != hipSuccess || hipEventCreate(&t0) != hipSuccess ||
      hipEventCreate(&t1) != hipSuccess) {
    release();
    MI355_CHECK(false, CEED_MI355_ERROR_BACKEND, "autotune: scratch vectors or events could not be created (%zu bytes)", bytes);
  }
  if (op->scalar_type == CEED_MI355_FP64) tune_fill<double><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, (double *)u);
  else tune_fill<float><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, (float *)u);
  const Launch start{op->layout, op->epb, op->line_only};
  Launch       best = start;
  float        bms  = 1e30f;
  int       err  = hipGetLastError() == hipSuccess ? CEED_MI355_SUCCESS : CEED_MI355_ERROR_BACKEND;
  if (err) mi355::set_error("autotune: the fill of the scratch input failed to launch");
  // ms per apply of one launch shape: a warm-up apply, then n timed applies
  auto time_launch = [&](const Launch &l, int n, float *ms) -> int {
    set_launch(op, l);
    int e      = CeedMi355OperatorApply(op, u, v, s);
    if (e) return e;
    MI355_HIP(hipEventRecord(t0, s));
    for (int r = 0; r < n && !e; r++) e = CeedMi355OperatorApply(op, u, v, s);
    if (e) return e;
    MI355_HIP(hipEventRecord(t1, s));
    MI355_HIP(hipEventSynchronize(t1));
    MI355_HIP(hipEventElapsedTime(ms, t0, t1));
    *ms /= n;
    return CEED_MI355_SUCCESS;
  };
  struct Cand {
    float  ms;
    Launch l;
  };
  std::vector<Cand> cands;
  auto try_launch = [&](const Launch &l) {
    float ms = 0;
    err = time_launch(l, reps, &ms);
    if (!err) cands.push_back({ms, l});
  };
  // one thread per element where it may take the plan's launches, beside the
  // line kernel with each count (a smaller plan leaves it open for larger ones)
  set_launch(op, {mi355::kLayoutLines, op->scatter == CEED_MI355_PLAN_SEGMENT ? op->seg_max : plan_default_epb(op, mi355::kLayoutLines), false});
  int32_t kernel = 0;
  if (!err) err = CeedMi355OperatorGetKernel(op, &kernel, nullptr);
  const bool elements = kernel == CEED_MI355_KERNEL_ELEMENTS;
  if (!err && elements) try_launch({op->layout, op->epb, false});
  for (int layout = mi355::kLayoutColumns; layout <= mi355::kLayoutPoints && !err; layout++) {
    for (int epb = 1; epb * mi355::layout_threads(op->Q, layout) <= mi355::max_threads(layout) && !err; epb++) {
      if (plan_admissible(op, layout, epb)) try_launch({layout, epb, elements});
    }
  }
  // launches within a few per cent of each other swap places from one timing
  // to the next: the three fastest are timed again, twice each, interleaved,
  // with twice the applies, and each keeps its best time
  std::sort(cands.begin(), cands.end(), [](const Cand &a, const Cand &b) { return a.ms < b.ms; });
  if (cands.size() > 3) cands.resize(3);
  for (int round = 0; round < 2 && cands.size() > 1 && !err; round++)
    for (Cand &c : cands) {
      float ms = 0;
      err = time_launch(c.l, 2 * reps, &ms);
      if (err) break;
      c.ms = std::min(c.ms, ms);
    }
  for (const Cand &c : cands)
    if (c.ms < bms) bms = c.ms, best = c.l;
  set_launch(op, err ? start : best);
  release();
  if (err) return err;
  {
    std::lock_guard<std::mutex> lock(g_tune_mutex);
    g_tuned[tune_key(op)] = best;
  }
  if (best_epb) *best_epb = best.epb;
  if (best_ms) *best_ms = bms;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorGetScatter(CeedMi355Operator op, int32_t *mode) {
  MI355_CHECK(op && mode, CEED_MI355_ERROR_MAJOR, "null argument");
  *mode = op->scatter == 0 ? CEED_MI355_PLAN_TMAP : op->scatter;
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorGetColors(CeedMi355Operator op, int32_t *num_colors, int32_t *color_sizes_host) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  *num_colors = (int32_t)op->color_start.size() - 1;
  if (color_sizes_host)
    for (int c = 0; c < *num_colors; c++) color_sizes_host[c] = (int32_t)(op->color_start[c + 1] - op->color_start[c]);
  return CEED_MI355_SUCCESS;
}

extern "C" int CeedMi355OperatorDestroy(CeedMi355Operator *op) {
  if (!op || !*op) return CEED_MI355_SUCCESS;
  if ((*op)->jit) mi355_jit_kernel_destroy((*op)->jit);
  (void)hipFree((*op)->d_offsets);
  (void)hipFree((*op)->d_perm);
  (void)hipFree((*op)->d_mats);
  (void)hipFree((*op)->d_qdata);
  (void)hipFree((*op)->d_trow);
  (void)hipFree((*op)->d_tcount);
  (void)hipFree((*op)->d_tpos);
  (void)hipFree((*op)->d_evec);
  (void)hipFree((*op)->d_srows);
  (void)hipFree((*op)->d_scratch);
  (void)hipFree((*op)->d_brick_start);
  (void)hipFree((*op)->d_brick_mask);
  (void)hipFree((*op)->d_bnode);
  (void)hipFree((*op)->d_blist);
  (void)hipFree((*op)->d_brow);
  (void)hipFree((*op)->d_bslot);
  (void)hipFree((*op)->d_partials);
  (void)hipFree((*op)->d_seg_start);
  (void)hipFree((*op)->d_geo);
  (void)hipFree((*op)->d_geo_pts);
  (void)hipFree((*op)->d_geo_turn);
  delete *op;
  *op = nullptr;
  return CEED_MI355_SUCCESS;
}
