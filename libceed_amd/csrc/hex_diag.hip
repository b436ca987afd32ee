// Diagonal of a fused hex plan's operator, assembled on the GPU: the input of
// Jacobi preconditioning (the reference's CeedOperatorLinearAssembleDiagonal,
// interface/ceed-preconditioning.c:2395, used by examples/petsc/src/matops.c:54).
//
// Element diagonal of node i = (a, b, c) (x fastest):
//   mass:       sum_q (B_a(qx) B_b(qy) B_c(qz))^2 qd(q)
//   diffusion:  sum_q g_i(q)^T S(q) g_i(q),  g_i = (G_a B_b B_c, B_a G_b B_c, B_a B_b G_c)
//               (times kappa(q) for the kappa-weighted operator),
// with G = D B, D the plan's collocated derivative; every component of a
// vector operator has the same diagonal.  Written out, each of the six entries
// of S meets a tensor product of three of the matrices BB = B o B, BG = B o G,
// GG = G o G (entrywise products), so the diagonal is six sum-factorised
// transposes that share their last steps:
//   z:  A0 = BB S00, A1 = BB S11, A2 = GG S22, A3 = 2 BG S12, A4 = 2 BG S02, A5 = 2 BB S01
//   y:  R0 = BB A0,  R1 = GG A1 + BB A2 + BG A3,  R2 = BB A4 + BG A5
//   x:  GG R0 + BB R1 + BG R2
// 6 Q^3 P + 6 Q^2 P^2 + 3 Q P^3 multiply-adds per element instead of the
// P^3 Q^3 terms of the sum itself (27 thousand against 74 thousand terms of 20
// operations each at P = 6, Q = 7).
//
// One Q x Q slab of threads per element: the z step on the columns (factors
// read, or recomputed where the plan's apply does), the y step on the lines
// (qx, z) and the x step on the rows (y, z), in place in the slabs.  The
// element diagonals are summed into the L-vector by the plan's E^T mode.
// MI355X, FP64 diffusion, p=5, 1.1M DoFs: 592 us with the P^3 Q^3 loop, 40 us
// now; its 0.5 GFLOP take 7 us at the FP64 rate, and what bounds it is latency
// at the three or four waves per SIMD that 6 P accumulators leave.
#include "hex_plan.hpp"

namespace mi355 {
namespace {

// The products' slabs: mass one, diffusion three, which take the six products
// in two turns (with six slabs LDS held a CU to 9 wavefronts at P = 6; p=5,
// 1.1M DoFs, us per assembly: 48.7 with six, 42.5 with three).
__host__ __device__ constexpr int diag_slabs(int qf) { return qf == kQfMass ? 1 : 3; }

// Four waves per SIMD where the accumulators fit 128 VGPRs without spills
// (P <= 5; at P = 6 the bound spills 92 bytes: 47 us against 40).
template <int P, int Q, int QF, bool kGeo, typename T>
__global__ void __launch_bounds__(256, (P <= 5 ? 4 : 1)) hex_diag_kernel(int64_t elem_begin, int64_t elem_end, int scatter, int num_comp,
                                                       const int32_t *__restrict__ offsets, int32_t comp_stride, const T *__restrict__ q_data,
                                                       const T *__restrict__ mats, const double *__restrict__ geo,
                                                       const double *__restrict__ geo_pts, T *__restrict__ v, T *__restrict__ evec,
                                                       const int32_t *__restrict__ tpos) {
  constexpr int NT = Q * Q, P3 = P * P * P, Q3 = Q * Q * Q, QP = Q * P, QC = QfTraits<QF>::kComps, NS = diag_slabs(QF), NA = QF == kQfMass ? 1 : 6;
  constexpr int SR = line_row_stride(Q, sizeof(T)), SP = line_plane_stride(Q, sizeof(T)), SLAB = P * SP;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int     epb = blockDim.x / NT, le = threadIdx.x / NT, t = threadIdx.x - le * NT;
  T            *A  = reinterpret_cast<T *>(lds_raw) + (size_t)le * NS * SLAB;
  auto          at = [](int k, int z, int y, int x) { return k * SLAB + z * SP + y * SR + x; };
  const int64_t e    = elem_begin + xcd_chunk(blockIdx.x, gridDim.x) * epb + le;
  const bool    live = le < epb && e < elem_end;
  const int64_t ec   = live ? e : elem_begin;  // lanes without an element work on the first one's factors and write nothing
  const int     cx = t % Q, cy = t / Q;
  const T      *sq = mats + QP + Q * Q;  // BB, BG, GG (Q x P each) behind B and D

  // ---- z on the column (cx, cy): acc[k][b] = A_k at (b, cy, cx), b < P
  T acc[NA][P];
#pragma unroll
  for (int k = 0; k < NA; k++)
#pragma unroll
    for (int b = 0; b < P; b++) acc[k][b] = 0;
  {
    const T  *qd = q_data + ec * (int64_t)QC * Q3 + cy * Q + cx;
    GeoColumn col;
    double    wxy = 0;
    if constexpr (kGeo) {
      col.load(geo + ec * kGeoStride, geo_pts[cx], geo_pts[cy]);
      wxy = geo_pts[Q + cy] * geo_pts[Q + cx];
    }
#pragma unroll
    for (int qz = 0; qz < Q; qz++) {
      T s[QC];
      if constexpr (kGeo) {
        const auto gp = phase_ptr(geo_pts);
        double     g6[6];
        __builtin_amdgcn_sched_barrier(0);  // one point's factors at a time in registers
        geo_poisson(col, gp[qz], gp[Q + qz] * wxy, g6);
#pragma unroll
        for (int k = 0; k < 6; k++) s[k] = (T)g6[k];
        if constexpr (QF == kQfDiffusionKappa) s[6] = __builtin_nontemporal_load(qd + 6 * Q3 + qz * Q * Q);
      } else {
#pragma unroll
        for (int k = 0; k < QC; k++) s[k] = __builtin_nontemporal_load(qd + k * Q3 + qz * Q * Q);
      }
      const auto bb = phase_ptr(sq + qz * P), bg = phase_ptr(sq + QP + qz * P), gg = phase_ptr(sq + 2 * QP + qz * P);
      if constexpr (QF == kQfMass) {
#pragma unroll
        for (int b = 0; b < P; b++) acc[0][b] += bb[b] * s[0];
      } else {
        if constexpr (QF == kQfDiffusionKappa) {
#pragma unroll
          for (int k = 0; k < 6; k++) s[k] *= s[6];
        }
        const T s3 = 2 * s[3], s4 = 2 * s[4], s5 = 2 * s[5];
#pragma unroll
        for (int b = 0; b < P; b++) {
          acc[0][b] += bb[b] * s[0];
          acc[1][b] += bb[b] * s[1];
          acc[2][b] += gg[b] * s[2];
          acc[3][b] += bg[b] * s3;
          acc[4][b] += bg[b] * s4;
          acc[5][b] += bb[b] * s5;
        }
      }
    }
  }
  // the products are complete here: without this the compiler sinks half of
  // their sums behind the first barrier and spills the matrices to carry them
#pragma unroll
  for (int k = 0; k < NA; k++)
#pragma unroll
    for (int b = 0; b < P; b++) asm volatile("" : "+v"(acc[k][b]));
  const bool yline = t < QP, xline = t < P * P;
  const int  ny = t % P, nz = t / P;
  // ---- y on the lines (qx = cx, z = cy < P), then x on the rows (y, z)
  if constexpr (QF == kQfMass) {
#pragma unroll
    for (int b = 0; b < P; b++) A[at(0, b, cy, cx)] = acc[0][b];
    __syncthreads();
    if (yline) {
      T r[P] = {};
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const auto bb = phase_ptr(sq + q * P);
        const T    a0 = A[at(0, cy, q, cx)];
#pragma unroll
        for (int b = 0; b < P; b++) r[b] += bb[b] * a0;
      }
#pragma unroll
      for (int b = 0; b < P; b++) A[at(0, cy, b, cx)] = r[b];
    }
    __syncthreads();
    if (xline) {
      T r[P] = {};
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const auto bb = phase_ptr(sq + q * P);
        const T    a0 = A[at(0, nz, ny, q)];
#pragma unroll
        for (int x = 0; x < P; x++) r[x] += bb[x] * a0;
      }
#pragma unroll
      for (int x = 0; x < P; x++) A[at(0, nz, ny, x)] = r[x];
    }
  } else {
#pragma unroll
    for (int b = 0; b < P; b++) A[at(0, b, cy, cx)] = acc[1][b], A[at(1, b, cy, cx)] = acc[2][b], A[at(2, b, cy, cx)] = acc[3][b];
    __syncthreads();
    T r1[P] = {};
    if (yline) {
#pragma unroll
      for (int q = 0; q < Q; q++) {
        if (q % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // two rows of each matrix in SGPRs at a time
        const auto bb = phase_ptr(sq + q * P), bg = phase_ptr(sq + QP + q * P), gg = phase_ptr(sq + 2 * QP + q * P);
        const T    a1 = A[at(0, cy, q, cx)], a2 = A[at(1, cy, q, cx)], a3 = A[at(2, cy, q, cx)];
#pragma unroll
        for (int b = 0; b < P; b++) {
          r1[b] += gg[b] * a1;
          r1[b] += bb[b] * a2;
          r1[b] += bg[b] * a3;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < P; b++) A[at(0, b, cy, cx)] = acc[0][b], A[at(1, b, cy, cx)] = acc[4][b], A[at(2, b, cy, cx)] = acc[5][b];
    __syncthreads();
    if (yline) {
      T r0[P] = {}, r2[P] = {};
#pragma unroll
      for (int q = 0; q < Q; q++) {
        if (q % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // two rows of each matrix in SGPRs at a time
        const auto bb = phase_ptr(sq + q * P), bg = phase_ptr(sq + QP + q * P);
        const T    a0 = A[at(0, cy, q, cx)], a4 = A[at(1, cy, q, cx)], a5 = A[at(2, cy, q, cx)];
#pragma unroll
        for (int b = 0; b < P; b++) {
          r0[b] += bb[b] * a0;
          r2[b] += bb[b] * a4;
          r2[b] += bg[b] * a5;
        }
      }
#pragma unroll
      for (int b = 0; b < P; b++) A[at(0, cy, b, cx)] = r0[b], A[at(1, cy, b, cx)] = r1[b], A[at(2, cy, b, cx)] = r2[b];
    }
    __syncthreads();
    if (xline) {
      T r[P] = {};
#pragma unroll
      for (int q = 0; q < Q; q++) {
        if (q % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // two rows of each matrix in SGPRs at a time
        const auto bb = phase_ptr(sq + q * P), bg = phase_ptr(sq + QP + q * P), gg = phase_ptr(sq + 2 * QP + q * P);
        const T    a0 = A[at(0, nz, ny, q)], a1 = A[at(1, nz, ny, q)], a2 = A[at(2, nz, ny, q)];
#pragma unroll
        for (int x = 0; x < P; x++) {
          r[x] += gg[x] * a0;
          r[x] += bb[x] * a1;
          r[x] += bg[x] * a2;
        }
      }
#pragma unroll
      for (int x = 0; x < P; x++) A[at(0, nz, ny, x)] = r[x];
    }
  }
  __syncthreads();
  // ---- E^T from the node columns, as the fused apply
  if (live && cx < P && cy < P) {
#pragma unroll
    for (int z = 0; z < P; z++) {
      const int     i   = (z * P + cy) * P + cx;
      const T       acc = A[at(0, z, cy, cx)];
      const int32_t o   = offsets[e * P3 + i];
      for (int k = 0; k < num_comp; k++) {
        if (scatter == kScatterElem) {  // element-major E-vector (brick plans)
          evec[(e * num_comp + k) * (int64_t)P3 + i] = acc;
          continue;
        }
        if (scatter == kScatterEvec || (scatter == kScatterSplit && (o & 1))) {  // L-entry-sorted E-vector
          evec[tpos[(e * num_comp + k) * (int64_t)P3 + i]] = acc;
          continue;
        }
        T *dst = &v[(o >> 1) + (int64_t)k * comp_stride];
        if (scatter == kScatterSplit) {  // at most two contributions: onto the zeroed target
          unsafeAtomicAdd(dst, acc);
          continue;
        }
        if (scatter == kScatterAtomic) unsafeAtomicAdd(dst, acc);
        else if (scatter == kScatterOverwrite && (o & 1)) *dst = acc;
        else *dst += acc;
      }
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) diag_zero(int64_t n, T *__restrict__ x) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) x[i] = T(0);
}

// Element diagonals of packed elements [b, e), added or stored by `scatter`
template <int P, int Q, typename T>
int launch_diag_elements(const CeedMi355Operator_private *op, int64_t b, int64_t e, int scatter, T *v, hipStream_t s) {
  // as many elements as fit 256 threads and the default LDS budget (at least
  // one: 44 kB at P = 9, Q = 10 in FP64)
  const size_t per = sizeof(T) * (size_t)diag_slabs(op->qf) * P * line_plane_stride(Q, sizeof(T));
  int          epb = 256 / (Q * Q);
  while (epb > 1 && epb * per > (size_t)kDefaultLdsBytes) epb--;
  const unsigned grid = (unsigned)((e - b + epb - 1) / epb), nt = (unsigned)(epb * Q * Q);
#define MI355_DIAG_LAUNCH(QF, GEO)                                                                                                        \
  hex_diag_kernel<P, Q, QF, GEO, T><<<grid, nt, epb * per, s>>>(b, e, scatter, op->num_comp, op->d_offsets, op->comp_stride,              \
                                                                (const T *)op->d_qdata, (const T *)op->d_mats, op->d_geo, op->d_geo_pts, v, \
                                                                (T *)op->d_evec, op->d_tpos)
  // (a graph of the caller's may be replayed after the plan's factors have changed kind: it takes the kernel that
  // reads them, which are the geometry's while that is the plan's, and every replay follows the plan; two kernels by
  // turns as in the apply cost the calls outside graphs 0.2 us of 13 at p=6, 48 elements, one more test in each.
  // MI355X, FP64, 1M DoFs, us recomputed / read: p=1 208 / 504, p=2 60 / 83, p=4 40 / 53, p=8 45 / 46)
  const bool geo = op->geo_valid && !into_callers_graph(op, s);
  if (op->qf == kQfMass) MI355_DIAG_LAUNCH(kQfMass, false);
  else if (op->qf == kQfDiffusion && geo) MI355_DIAG_LAUNCH(kQfDiffusion, true);
  else if (op->qf == kQfDiffusion) MI355_DIAG_LAUNCH(kQfDiffusion, false);
  else if (geo) MI355_DIAG_LAUNCH(kQfDiffusionKappa, true);
  else MI355_DIAG_LAUNCH(kQfDiffusionKappa, false);
#undef MI355_DIAG_LAUNCH
  MI355_LAUNCH_CHECK();
  return CEED_MI355_SUCCESS;
}

template <int P, int Q, typename T>
int launch_diag(const CeedMi355Operator_private *op, void *v, int add, hipStream_t s) {
  const bool tmap  = op->scatter == 0;
  const bool split = op->scatter == CEED_MI355_PLAN_SPLIT;
  const bool brick = op->scatter == CEED_MI355_PLAN_BRICK;
  MI355_CHECK(op->scatter != CEED_MI355_PLAN_SEGMENT, CEED_MI355_ERROR_UNSUPPORTED,
              "diagonal assembly does not take segment plans (elements of a colour share segment faces)");
  if (brick) {  // element diagonals into the element-major E-vector, then the brick E^T
    if (!add && !op->covers_all) {
      diag_zero<T><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, (T *)v);
      MI355_LAUNCH_CHECK();
    }
    const int err = launch_diag_elements<P, Q, T>(op, 0, op->num_elem, kScatterElem, (T *)v, s);
    return err ? err : brick_evec(op, op->d_evec, v, !add, s);
  }
  // the split mode's atomic adds land on a zeroed target: v, or with add the scratch vector
  T *target = split && add ? (T *)op->d_scratch : (T *)v;
  if ((!add && !tmap && !op->covers_all) || (split && add)) {
    diag_zero<T><<<mi355_blocks(op->l_size, 256, 4096), 256, 0, s>>>(op->l_size, target);
    MI355_LAUNCH_CHECK();
  }
  for (size_t c = 0; c + 1 < op->color_start.size(); c++) {
    const int64_t b = op->color_start[c], e = op->color_start[c + 1];
    if (e <= b) continue;
    const int scatter = tmap ? kScatterEvec
                        : split ? kScatterSplit
                                : (op->scatter == CEED_MI355_PLAN_ATOMIC ? kScatterAtomic : (add ? kScatterAdd : kScatterOverwrite));
    const int err = launch_diag_elements<P, Q, T>(op, b, e, scatter, target, s);
    if (err) return err;
  }
  if (tmap) return transpose_gather(op, v, !add, nullptr, s);
  if (split) return split_finish(op, v, !add, s);
  return CEED_MI355_SUCCESS;
}
using DiagFn = int (*)(const CeedMi355Operator_private *, void *, int, hipStream_t);

template <typename T>
DiagFn pick_diag(int P, int Q) {
#define MI355_DIAG_CASE(PP, QQ) \
  if (P == PP && Q == QQ) return launch_diag<PP, QQ, T>;
  MI355_DIAG_CASE(2, 2) MI355_DIAG_CASE(2, 3) MI355_DIAG_CASE(3, 3) MI355_DIAG_CASE(3, 4) MI355_DIAG_CASE(4, 4) MI355_DIAG_CASE(4, 5)
  MI355_DIAG_CASE(5, 5) MI355_DIAG_CASE(5, 6) MI355_DIAG_CASE(6, 6) MI355_DIAG_CASE(6, 7) MI355_DIAG_CASE(7, 7) MI355_DIAG_CASE(7, 8)
  MI355_DIAG_CASE(8, 8) MI355_DIAG_CASE(8, 9) MI355_DIAG_CASE(9, 9) MI355_DIAG_CASE(9, 10)
#undef MI355_DIAG_CASE
  return nullptr;
}

}  // namespace
}  // namespace mi355

extern "C" int CeedMi355OperatorAssembleDiagonal(CeedMi355Operator op, void *diag, int add, void *stream) {
  MI355_CHECK(op, CEED_MI355_ERROR_MAJOR, "null operator");
  MI355_CHECK(op->qf == mi355::kQfMass || op->qf == mi355::kQfDiffusion || op->qf == mi355::kQfDiffusionKappa, CEED_MI355_ERROR_UNSUPPORTED,
              "diagonal assembly needs a mass or diffusion plan");
  if (op->num_elem == 0) return CEED_MI355_SUCCESS;
  mi355::touch_thread_storage();
  if (op->scatter == CEED_MI355_PLAN_BRICK && !op->d_evec)  // element-major E-vector of the brick plan's diagonal, made once
    MI355_HIP(hipMalloc(&op->d_evec, (size_t)op->scalar_bytes * ((size_t)op->num_elem * op->num_comp * op->P * op->P * op->P + 1)));
  auto fn = op->scalar_type == CEED_MI355_FP64 ? mi355::pick_diag<double>(op->P, op->Q) : mi355::pick_diag<float>(op->P, op->Q);
  MI355_CHECK(fn, CEED_MI355_ERROR_UNSUPPORTED, "no diagonal kernel for P=%d Q=%d", op->P, op->Q);
  return fn(op, diag, add, (hipStream_t)stream);
}
