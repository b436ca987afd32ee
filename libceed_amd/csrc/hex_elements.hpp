// One thread per element, for the lowest order: with two nodes per direction
// an element's whole diffusion apply fits one thread's registers, so there is
// nothing to exchange through LDS and nothing to wait for (the line kernel at
// Q = 3 runs nine threads per element through eleven barriers and issues 4400
// instructions per element, this one 2900).  The geometric factors come from
// the element's trilinear map, whose coefficients a wavefront stages through
// LDS (coalesced; a thread's own 21 then lie on an odd stride).  Bound by FP64
// issue at Q = 3 (252 registers, two waves per SIMD) and by memory at Q = 2.
// Every value is computed by the operations of the line kernel in its order,
// so the results are the same bits.
// MI355X, line kernel / this one, us per apply with the E^T pass:
//   970k elements: FP64 Q=2 131 / 107, Q=3 212 / 162; FP32 Q=2 99 / 74, Q=3 175 / 141
//   3.9M elements: FP64 Q=2 493 / 427, Q=3 778 / 569
#pragma once

#include "hex_geo.hpp"
#include "hex_lines.hpp"

namespace mi355 {

// Elements of a launch from which this kernel takes it: its wavefronts are few
// and long, and the line kernel is the better one until the SIMDs have more
// than one of them each.  us, line / this: FP64 Q=2 36k elements 11.1 / 11.0, 74k
// 16.4 / 13.7; FP64 Q=3 74k 20.8 / 21.0, 125k 30.3 / 25.5; FP32 Q=2 74k 12.2 /
// 12.2, 125k 17.2 / 15.0; FP32 Q=3 74k 17.5 / 19.7, 125k 25.9 / 23.2; eight
// colours, each a launch: FP64 Q=3 71k each 133 / 139, 121k each 202 / 164, and
// FP64 Q=2 23k each 51 / 50, 47k each 77 / 60.
constexpr int64_t elements_min(int Q, int sb) { return Q == 2 && sb == 8 ? 32768 : 98304; }
constexpr int kElemThreads = 64;
constexpr int kElemGeo     = kGeoStride + 1;  // an odd stride in LDS

template <int P, int Q, typename T>
__global__ void __launch_bounds__(kElemThreads, 2) hex_apply_elements_kernel(int64_t elem_begin, int64_t elem_end, int scatter,
                                                                             const int32_t *__restrict__ offsets, const T *__restrict__ mats,
                                                                             const T *__restrict__ u, T *__restrict__ v, T *__restrict__ evec,
                                                                             const int32_t *__restrict__ tpos, const int32_t *__restrict__ elem_sys,
                                                                             const int32_t *__restrict__ sys_active, const double *__restrict__ geo,
                                                                             const double *__restrict__ geo_pts) {
  constexpr int P3 = P * P * P;
  static_assert(P3 % 4 == 0, "offsets are read four at a time");
  __shared__ double sgeo[kElemThreads * kElemGeo];

  const int64_t first = elem_begin + xcd_chunk(blockIdx.x, gridDim.x) * kElemThreads;
  const int     lane = threadIdx.x, n = (int)(elem_end - first < kElemThreads ? elem_end - first : kElemThreads);
  const int64_t e    = first + lane;
  bool          live = lane < n;
  if (elem_sys) {
    if (elem_sys == sys_active) {
      if (!*sys_active) return;
    } else {
      live = live && sys_active[elem_sys[e]];
    }
  }

  // (lanes past the end read the last element and store nothing)
  const int64_t er = lane < n ? e : elem_end - 1;
  int           off[P3];  // 2 * node + first_touch
  T             x[P3];
#pragma unroll
  for (int i = 0; i < P3; i += 4) *reinterpret_cast<int4 *>(&off[i]) = *reinterpret_cast<const int4 *>(&offsets[er * P3 + i]);
  {
    const double2 *src  = reinterpret_cast<const double2 *>(geo + first * kGeoStride);
    const int      last = n * (kGeoStride / 2) - 1;
    double2        c[kGeoStride / 2];
#pragma unroll
    for (int k = 0; k < kGeoStride / 2; k++) {
      const int i = k * kElemThreads + lane;
      c[k]        = src[i < last ? i : last];
    }
#pragma unroll
    for (int i = 0; i < P3; i++) x[i] = u[off[i] >> 1];
#pragma unroll
    for (int k = 0; k < kGeoStride / 2; k++) {
      const int i = k * kElemThreads + lane, row = i / (kGeoStride / 2), col = i - row * (kGeoStride / 2);
      sgeo[row * kElemGeo + 2 * col]     = c[k].x;
      sgeo[row * kElemGeo + 2 * col + 1] = c[k].y;
    }
  }
  __syncthreads();
  const double *g  = sgeo + lane * kElemGeo;
  const auto    B  = phase_ptr(mats);
  const auto    D  = phase_ptr(mats + Q * P);
  const auto    gp = phase_ptr(geo_pts);

  // ---- interpolation to the quadrature points, x then y then z
  T xq[Q][Q][Q];
  {
    T a[P][P][Q], b[P][Q][Q];
#pragma unroll
    for (int z = 0; z < P; z++)
#pragma unroll
      for (int y = 0; y < P; y++)
#pragma unroll
        for (int q = 0; q < Q; q++) {
          T s = 0;
#pragma unroll
          for (int i = 0; i < P; i++) s += B[q * P + i] * x[(z * P + y) * P + i];
          a[z][y][q] = s;
        }
#pragma unroll
    for (int z = 0; z < P; z++)
#pragma unroll
      for (int q = 0; q < Q; q++)
#pragma unroll
        for (int qx = 0; qx < Q; qx++) {
          T s = 0;
#pragma unroll
          for (int i = 0; i < P; i++) s += B[q * P + i] * a[z][i][qx];
          b[z][q][qx] = s;
        }
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int qy = 0; qy < Q; qy++)
#pragma unroll
        for (int qx = 0; qx < Q; qx++) {
          T s = 0;
#pragma unroll
          for (int i = 0; i < P; i++) s += B[q * P + i] * b[i][qy][qx];
          xq[q][qy][qx] = s;
        }
  }
  // ---- plane by plane: collocated derivatives, the pointwise operator, the
  // x and y transposes; the z parts wait for the last plane
  T w[Q][Q][Q], vz[Q][Q][Q];
#pragma unroll
  for (int qz = 0; qz < Q; qz++) {
    T dx[Q][Q], dy[Q][Q];
#pragma unroll
    for (int qy = 0; qy < Q; qy++)
#pragma unroll
      for (int qx = 0; qx < Q; qx++) {
        T sx = 0, sy = 0, sz = 0;
#pragma unroll
        for (int c = 0; c < Q; c++) {
          sx += D[qx * Q + c] * xq[qz][qy][c];
          sy += D[qy * Q + c] * xq[qz][c][qx];
          sz += D[qz * Q + c] * xq[c][qy][qx];
        }
        dx[qy][qx] = sx, dy[qy][qx] = sy, vz[qz][qy][qx] = sz;
      }
    // The Jacobian's columns as GeoColumn has them, each computed once per
    // plane: d/dxi depends on (eta, zeta) alone, d/deta on (xi, zeta)
    __builtin_amdgcn_sched_barrier(0);  // (also: the coefficients are read again for each plane, not kept in registers)
    const double zeta = gp[qz];
    double       ja[Q][3];
#pragma unroll
    for (int qy = 0; qy < Q; qy++)
#pragma unroll
      for (int d = 0; d < 3; d++)
        ja[qy][d] = __builtin_fma(zeta, __builtin_fma(gp[qy], g[18 + d], g[12 + d]), __builtin_fma(gp[qy], g[9 + d], g[d]));
#pragma unroll
    for (int qx = 0; qx < Q; qx++) {
      double jb[3], q1[3], r[3];
#pragma unroll
      for (int d = 0; d < 3; d++) {
        q1[d] = __builtin_fma(gp[qx], g[18 + d], g[15 + d]);
        jb[d] = __builtin_fma(zeta, q1[d], __builtin_fma(gp[qx], g[9 + d], g[3 + d]));
        r[d]  = __builtin_fma(gp[qx], g[12 + d], g[6 + d]);
      }
#pragma unroll
      for (int qy = 0; qy < Q; qy++) {
        double jc[3], s6[6];
        T      s[6], wx, wy, wz;
#pragma unroll
        for (int d = 0; d < 3; d++) jc[d] = __builtin_fma(gp[qy], q1[d], r[d]);
        geo_poisson(ja[qy], jb, jc, gp[Q + qz] * (gp[Q + qy] * gp[Q + qx]), s6);
#pragma unroll
        for (int i = 0; i < 6; i++) s[i] = (T)s6[i];
        poisson_regs<T>(s, dx[qy][qx], dy[qy][qx], vz[qz][qy][qx], wx, wy, wz);
        dx[qy][qx] = wx, dy[qy][qx] = wy, vz[qz][qy][qx] = wz;
        __builtin_amdgcn_sched_barrier(0);  // one point's factors at a time in registers
      }
    }
#pragma unroll
    for (int qy = 0; qy < Q; qy++)
#pragma unroll
      for (int qx = 0; qx < Q; qx++) {
        T sx = 0, sy = 0;
#pragma unroll
        for (int j = 0; j < Q; j++) {
          sx += D[j * Q + qx] * dx[qy][j];
          sy += D[j * Q + qy] * dy[j][qx];
        }
        w[qz][qy][qx] = sx + sy;
      }
  }
  // ---- z transposes and back to the nodes, z then y then x
  T b[P][Q][Q];
#pragma unroll
  for (int qy = 0; qy < Q; qy++)
#pragma unroll
    for (int qx = 0; qx < Q; qx++) {
      T col[Q];
#pragma unroll
      for (int i = 0; i < Q; i++) {
        T s = w[i][qy][qx];
#pragma unroll
        for (int j = 0; j < Q; j++) s += D[j * Q + i] * vz[j][qy][qx];
        col[i] = s;
      }
#pragma unroll
      for (int i = 0; i < P; i++) {
        T s = 0;
#pragma unroll
        for (int j = 0; j < Q; j++) s += B[j * P + i] * col[j];
        b[i][qy][qx] = s;
      }
    }
#pragma unroll
  for (int z = 0; z < P; z++) {
    T a[P][Q];
#pragma unroll
    for (int y = 0; y < P; y++)
#pragma unroll
      for (int qx = 0; qx < Q; qx++) {
        T s = 0;
#pragma unroll
        for (int j = 0; j < Q; j++) s += B[j * P + y] * b[z][j][qx];
        a[y][qx] = s;
      }
#pragma unroll
    for (int y = 0; y < P; y++)
#pragma unroll
      for (int i = 0; i < P; i++) {
        T s = 0;
#pragma unroll
        for (int j = 0; j < Q; j++) s += B[j * P + i] * a[y][j];
        x[(z * P + y) * P + i] = s;
      }
  }
  // computed here, not where the stores need it: the compiler would move all of
  // the above behind the branch, except the reads of the map, and spill
#pragma unroll
  for (int i = 0; i < P3; i++) asm volatile("" : "+v"(x[i]));
  if (!live) return;
  // ---- E^T
  if (scatter == kScatterEvec || scatter == kScatterSplit) {
    int pos[P3];
#pragma unroll
    for (int i = 0; i < P3; i += 4) *reinterpret_cast<int4 *>(&pos[i]) = *reinterpret_cast<const int4 *>(&tpos[e * P3 + i]);
#pragma unroll
    for (int i = 0; i < P3; i++) {  // split: shared entries to their E-vector slot, the rest onto the zeroed v
      if (scatter == kScatterEvec || (off[i] & 1)) evec[pos[i]] = x[i];
      else unsafeAtomicAdd(&v[off[i] >> 1], x[i]);
    }
  } else if (scatter == kScatterAtomic) {
#pragma unroll
    for (int i = 0; i < P3; i++) unsafeAtomicAdd(&v[off[i] >> 1], x[i]);
  } else {  // colour-exclusive; kScatterOverwrite: the first element to reach a node writes it
#pragma unroll
    for (int i = 0; i < P3; i++) {
      T *dst = &v[off[i] >> 1];
      *dst   = scatter == kScatterOverwrite && (off[i] & 1) ? x[i] : *dst + x[i];
    }
  }
}

}  // namespace mi355
