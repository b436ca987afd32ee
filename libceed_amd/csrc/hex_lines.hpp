// Fused per-element hex operator, "line" thread layout.
//
// Same operator as hex_apply_kernel (gather E, sum-factorised interp and
// collocated gradient B, pointwise D, transposes, E^T), with a different
// assignment of work to threads.  The column-slab kernel gives thread (x, y)
// the z-column of its point and contracts x and y through LDS, so every
// output point reads Q values back from LDS (Q-fold redundant reads of the
// same slab row by the Q threads of that row).  Here, for each x- or
// y-contraction, a thread owns one whole 1D line of the slab: it reads the
// line's Q (or P) inputs once, computes all of the line's outputs with the
// 1D matrix entries (wave-uniform: scalar loads, no LDS), and writes them
// back.  Per element and component this reads and writes each slab entry
// about once per contraction instead of Q times, so the LDS traffic, which
// bounds the column-slab kernel at p >= 3, drops about threefold.  The
// z-contractions and the pointwise operator stay in registers on the
// (x, y) columns, as in the column-slab kernel.
//
// kGeo: on a trilinear geometry the factors are not read but recomputed from
// the element's map (hex_geo.hpp).  With the 48 bytes per point gone (1.30 of
// the 1.49 GB of an apply at p=4, 8M DoFs) what bounds the kernel is its own
// issue rate and the latency between its barriers, so whole wavefronts of
// elements (geo_default_epb) and the in-place slabs count: MI355X, FP64
// diffusion, 8M DoFs, ms per apply, stored factors / recomputed / recomputed
// with the lines in place: p=2 0.621 / 0.462 / 0.445, p=4 0.357 / 0.254 /
// 0.222, p=6 0.252 / 0.229 / 0.180, p=8 0.283 / 0.231 / 0.199 (applies one after
// the other on one pair of vectors, with a spread of 3% between machines; on vectors and
// plans that change from apply to apply p=4 takes 0.232 to 0.243).
//
// Thread t of an element's Q*Q threads plays these roles:
//   column (qx, qy) = (t % Q, t / Q)                     z-contractions, pointwise D
//   node column (x, y) = (t % Q, t / Q), x, y < P      gather E, scatter E^T (coalesced)
//   x-line of nodes (y, z) = (t % P, t / P), t < P*P     B_x, B_x^T
//   y-line (qx, z) = (t % Q, t / Q), t < Q*P              B_y, B_y^T
//   x-line (qy, qz) and y-line (qx, qz) = (t % Q, t / Q)  the collocated derivatives
// Slabs are [z][y][x] with strides (Q*Q, Q, 1), padded against LDS bank
// conflicts in FP64 at Q = 3, 4, 7 and 8 and in FP32 at Q = 8 (line_row_stride,
// line_plane_stride, line_elem_pad).  A line's thread reads
// all of it before it writes and no other thread touches it in that phase, so
// lines are contracted in place: mass needs one slab per element, diffusion
// two (the y-lines of the derivative are read before and written after the
// barrier that ends the x-lines' reads), against two and three with separate
// source and target, and eleven barriers against thirteen.
#pragma once

#include "hex_fused.hpp"
#include "hex_geo.hpp"

namespace mi355 {

// The 1D matrices are read with wave-uniform addresses (scalar loads into
// SGPRs).  Loaded once for the whole kernel they would need ~2(QP + Q^2)
// SGPRs, far more than a wave has, and the compiler would spill them to VGPR
// lanes (a v_writelane/v_readlane pair per use).  Re-deriving the pointer
// through an empty asm at the start of each phase keeps the loads inside the
// phase that uses them, so only that phase's entries are live.
// The pointer is returned in the constant address space (read-only for the
// kernel's lifetime, which the matrices are), so the loads stay scalar.
template <typename T>
using const_ptr = const __attribute__((address_space(4))) T *;

template <typename T>
__device__ __forceinline__ const_ptr<T> phase_ptr(const T *p) {
  asm volatile("" : "+s"(p));
  return (const_ptr<T>)p;
}

// Lanes 2m and 2m+1 of a wave hold the columns (cx, cy) and (cx+1, cy), cx
// even: each loads q_data for both columns, half of the components each, with
// 16-byte loads (half the load instructions), and they swap halves with a DPP
// quad permutation [1, 0, 3, 2] when the values are used.
template <typename T>
using line_v2 = T __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double pair_swap(double x) {
  const long long b  = __double_as_longlong(x);
  const int       lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xF, 0xF, false);
  const int       hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Slabs per element: the line kernel contracts its lines in place (mass one,
// diffusion two, and a third where the z-derivatives wait in LDS:
// line_dz_in_lds); the shared pipeline below (line_element) goes back and forth.
__host__ __device__ constexpr bool line_dz_in_lds(int Q, int ncomp, int qf, int sb, bool geo) {
  return !geo && (qf == kQfDiffusion || qf == kQfDiffusionKappa) && ncomp == 1 && sb == 8 && Q >= 10;
}
__host__ __device__ constexpr int line_kernel_slabs(int Q, int ncomp, int qf, int sb, bool geo) {
  return qf == kQfMass ? 1 : line_dz_in_lds(Q, ncomp, qf, sb, geo) ? 3 : 2;
}
template <int QF>
struct LineSlabs {
  static constexpr int kSlabs = QF == kQfMass ? 2 : 3;
};

// Row and plane strides (entries) of the line kernel's slabs, for entries of
// sb bytes.  At Q = 8 the natural strides (8, 64) are powers of two: the
// entries an x-line, y-line or x-node-line phase touches in one wavefront
// then fall into a few LDS bank groups (SQ_LDS_BANK_CONFLICT 32% of the
// cycles at p=6, 39% with 3 components).  Rows of 9 and planes of 72 (FP64),
// planes of 73 (FP32) spread them (a bank model of the phases' access
// patterns: 2.1x fewer conflict cycles in FP64, 3.8x in FP32).  Measured on
// MI355X, 8M DoFs, ms per apply: FP32 p=6 0.136-0.139 vs 0.148, 3-component
// FP64 p=6 0.648-0.650 vs 0.689-0.691, scalar FP64 p=6 unchanged within run
// to run noise.  At Q = 7 (FP64) planes of 58 model 10% fewer conflict
// cycles: 3-component p=5 0.783-0.784 vs 0.794-0.796 ms, scalar p=5
// unchanged.  With the factors recomputed LDS weighs more (conflicts 38% of
// the cycles at p=1, 14% at p=4), and planes of 18 at Q = 4 and 5 entries
// between elements at Q = 3, which model 44% and 19% fewer passes, measure
// 0.245 vs 0.256 (p=2) and 0.770 vs 0.790 ms (p=1, 4M DoFs, two interleaved
// runs); the same search changed nothing at Q = 2, 5 and 10 and cost 2% at
// Q = 6 (planes of 37 and 39).
__host__ __device__ constexpr int line_row_stride(int Q, int sb) { return sb == 8 && Q == 8 ? 9 : Q; }
__host__ __device__ constexpr int line_plane_stride(int Q, int sb) {
  if (sb == 8) return Q == 4 ? 18 : Q == 7 ? 58 : Q == 8 ? 72 : Q * Q;
  return Q == 8 ? 73 : Q * Q;
}
// entries between the slabs of one element and the next
__host__ __device__ constexpr int line_elem_pad(int Q, int sb) { return sb == 8 && Q == 3 ? 5 : 0; }
__host__ __device__ constexpr int line_slab_entries(int Q, int sb) { return Q * line_plane_stride(Q, sb); }

// Entries from one element's slabs to the next one's in the line kernel
__host__ __device__ constexpr int line_elem_entries(int Q, int ncomp, int qf, int sb, bool geo) {
  return line_kernel_slabs(Q, ncomp, qf, sb, geo) * line_slab_entries(Q, sb) + line_elem_pad(Q, sb);
}

// LDS bytes of a workgroup of epb elements: the slabs and, where the factors
// are recomputed, the elements' trilinear maps behind them
__host__ __device__ constexpr size_t line_lds_bytes(int Q, int ncomp, int qf, int sb, bool geo, int epb) {
  const size_t slabs = (size_t)sb * epb * line_elem_entries(Q, ncomp, qf, sb, geo);
  return geo ? ((slabs + 15) & ~(size_t)15) + sizeof(double) * kGeoLds * (size_t)epb : slabs;
}

// Where the factors are recomputed (kGeo): once per element into the registers
// the stored ones would be loaded into, or point by point in every component.
// One component: at the point, the registers are worth more.  Three: once
// where 6 Q doubles fit beside the pipeline (Q <= 7, and FP32), per component
// above (MI355X, 4M DoFs, ms per apply, once / per component: FP64 Q=4 0.214 /
// 0.239, Q=6 0.098 / 0.106, Q=8 0.110 / 0.104, Q=10 0.149 / 0.133).
__host__ __device__ constexpr bool line_geo_once(int Q, int ncomp, int sb) { return ncomp > 1 && (Q <= 7 || sb == 4); }

// The column's geometric factors (QC values at each of its Q points) and how
// they are loaded: all loads issued at once and shared by the components, at
// the element start (in flight during E and the interpolation), or for
// scalar FP64 diffusion from Q = 9 just before the pointwise operator, where
// 6Q doubles held through the whole element cost a wave per SIMD (191 -> 137
// VGPRs at Q = 9; measured on MI355X, 8M DoFs: p=7 26.6 -> 27.6 GDoF/s, p=8
// 26.2 -> 27.5; later loads lose at Q <= 8 and in FP32, where the exposed
// latency costs more than the occupancy gains).  FP64 scalar diffusion with
// early loads and Q even loads them in lane pairs with 16-byte loads
// (interleaved A/B on MI355X, 8M DoFs: p=4 +0.7% with colours, +3.7% with the
// map, p=6 +0-4% with the split; with the late loads at Q = 10 the swap in the
// pointwise loop cost 15%; FP32 pairs of 8-byte loads were 3-5% slower).
template <int Q, int NCOMP, int QF, typename T>
struct LineQData {
  static constexpr int  QC     = QfTraits<QF>::kComps, Q3 = Q * Q * Q, QH = QC / 2;
  static constexpr bool kEarly = QF == kQfMass || NCOMP > 1 || Q < 9 || sizeof(T) < 8;
  static constexpr bool kPair  = kEarly && sizeof(T) == 8 && QF == kQfDiffusion && NCOMP == 1 && Q % 2 == 0;
  T                     sq[kPair ? 1 : Q][QC];
  line_v2<T>            sp[kPair ? Q : 1][kPair ? QH : 1];

  // qe: the element's block [QC][Q^3]; (cx, cy) the column
  __device__ __forceinline__ void load(const T *qe, int cx, int cy) {
    if constexpr (kPair) {  // 16-byte aligned: Q even, so (cy * Q + cx - odd) and every stride are even
      const T *pb = qe + (cy * Q + (cx & ~1)) + ((cx & 1) ? QH : 0) * Q3;
#pragma unroll
      for (int qz = 0; qz < Q; qz++)
#pragma unroll
        for (int kk = 0; kk < QH; kk++) sp[qz][kk] = __builtin_nontemporal_load((const line_v2<T> *)(pb + kk * Q3 + qz * Q * Q));
    } else {
      const T *qd = qe + (cy * Q + cx);
#pragma unroll
      for (int qz = 0; qz < Q; qz++)
#pragma unroll
        for (int k = 0; k < QC; k++) sq[qz][k] = __builtin_nontemporal_load(&qd[k * Q3 + qz * Q * Q]);
    }
  }
  // the QC values of point qz of the column (with the pairs: this column's
  // half from the own load, the other half from the partner lane)
  __device__ __forceinline__ void point(int qz, int cx, T (&s)[QC]) const {
    if constexpr (kPair) {
      const bool odd = cx & 1;
#pragma unroll
      for (int kk = 0; kk < QH; kk++) {
        const line_v2<T> d = sp[qz][kk];
        const T       keep = odd ? d.y : d.x, got = pair_swap(odd ? d.x : d.y);
        s[kk]              = odd ? got : keep;
        s[QH + kk]         = odd ? keep : got;
      }
    } else {
#pragma unroll
      for (int k = 0; k < QC; k++) s[k] = sq[qz][k];
    }
  }
};

// acc[i] += sum_j M[j][i] in[j] for a row-major J x I matrix at m: the sums in
// ascending j, as a line contraction with the transposed matrix forms them.
// By rows (from Q = 7, where the matrix does not fit the SGPRs) a row of I
// contiguous entries is loaded for each j; column by column it is I J scalar
// loads of one entry each (705 against 255 scalar loads per wave at p=8; MI355X,
// FP64 diffusion, us per apply, columns / rows: stored factors 8M DoFs p=6 252
// / 246, p=8 299 / 278, three components 4M DoFs p=5 168 / 125, p=7 145 / 132;
// recomputed 8M DoFs p=8 199 / 187).
template <int I, int J, typename T>
__device__ __forceinline__ void transposed_line(const T *m, const T (&in)[J], T (&acc)[I]) {
#pragma unroll
  for (int j = 0; j < J; j++) {
    const auto r = phase_ptr(m + j * I);
#pragma unroll
    for (int i = 0; i < I; i++) acc[i] += r[i] * in[j];
  }
}

// Synchronisation of one element's threads between the phases of the line
// pipeline: the whole workgroup, or the wavefront alone when an element never
// spans two wavefronts (a wavefront's LDS operations are performed in the
// order it issues them; the fences keep the compiler from moving them).
struct SyncBlock {
  __device__ __forceinline__ void operator()() const { __syncthreads(); }
};
struct SyncWave {
  __device__ __forceinline__ void operator()() const {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
};

// One element and component through B, D and B^T in the line layout.  On
// entry S0 holds the element's nodal values at (z, y, x), x, y, z < P, and
// the element's threads are synchronised; on return S0 holds the nodal
// results there, synchronised again.  t is the thread's index among the
// element's Q*Q threads; threads with active false (lanes of a wavefront
// that hold no element) only take part in the synchronisations.  qd holds
// the column's geometric factors (loaded here first when they are late,
// from qe); live false zeroes the pointwise output.
template <int P, int Q, int NCOMP, int QF, typename T, typename Sync>
__device__ __forceinline__ void line_element(T *S0, T *S1, T *S2, int t, bool active, bool live, const T *__restrict__ mats,
                                             LineQData<Q, NCOMP, QF, T> &qd, const T *qe, Sync sync) {
  constexpr int QC = QfTraits<QF>::kComps;
  // from Q = 7 one phase's matrix entries no longer fit the SGPRs: load them
  // per output row (or column) instead of per phase
  constexpr bool kRowWise = Q >= 7;
  // B (Q x P) then D (Q x Q), row-major, at mats
  auto       at = [](int z, int y, int x) { return (z * Q + y) * Q + x; };
  const int  cx = t % Q, cy = t / Q;  // column
  const int  ny = t % P, nz = t / P;  // x-line of nodes
  const bool xline = active && t < P * P;
  // ---- B_x: x-line (ny, nz) of nodes, Q interpolated values into S1
  if (xline) {
    const auto gB = phase_ptr(mats);
    T          in[P];
#pragma unroll
    for (int x = 0; x < P; x++) in[x] = S0[at(nz, ny, x)];
#pragma unroll
    for (int qx = 0; qx < Q; qx++) {
      const auto m = kRowWise ? phase_ptr(mats + qx * P) : gB + qx * P;
      T          s = 0;
#pragma unroll
      for (int b = 0; b < P; b++) s += m[b] * in[b];
      S1[at(nz, ny, qx)] = s;
    }
  }
  sync();
  // ---- B_y: y-line (qx, z), z < P
  if (active && t < Q * P) {
    const auto gB = phase_ptr(mats);
    const int  qx = t % Q, z = t / Q;
    T          in[P];
#pragma unroll
    for (int b = 0; b < P; b++) in[b] = S1[at(z, b, qx)];
#pragma unroll
    for (int qy = 0; qy < Q; qy++) {
      const auto m = kRowWise ? phase_ptr(mats + qy * P) : gB + qy * P;
      T          s = 0;
#pragma unroll
      for (int b = 0; b < P; b++) s += m[b] * in[b];
      S0[at(z, qy, qx)] = s;
    }
  }
  sync();
  // ---- B_z on the column (cx, cy): uq[qz]
  T uq[Q];
  if (active) {
    const auto gB = phase_ptr(mats);
    T          col[P];
#pragma unroll
    for (int b = 0; b < P; b++) col[b] = S0[at(b, cy, cx)];
#pragma unroll
    for (int qz = 0; qz < Q; qz++) {
      const auto m = kRowWise ? phase_ptr(mats + qz * P) : gB + qz * P;
      T          s = 0;
#pragma unroll
      for (int b = 0; b < P; b++) s += m[b] * col[b];
      uq[qz] = s;
    }
  }
  if constexpr (QF == kQfMass) {
    // ---- D, then B_z^T back into the column's own S0 entries (read only by this thread)
    if (active) {
      const auto gB = phase_ptr(mats);
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        T s[QC];
        qd.point(qz, cx, s);
        uq[qz] *= live ? s[0] : T(0);
      }
#pragma unroll
      for (int b = 0; b < P; b++) {
        const auto m = kRowWise ? phase_ptr(mats + b) : gB + b;
        T          s = 0;
#pragma unroll
        for (int qz = 0; qz < Q; qz++) s += m[qz * P] * uq[qz];
        S0[at(b, cy, cx)] = s;
      }
    }
  } else {
    // ---- collocated derivatives: z on the column, x and y by lines through S1
    T dz[Q];
    if (active) {
      const auto gD = phase_ptr(mats + Q * P);
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        const auto m = kRowWise ? phase_ptr(mats + Q * P + qz * Q) : gD + qz * Q;
        T          s = 0;
#pragma unroll
        for (int c = 0; c < Q; c++) s += m[c] * uq[c];
        dz[qz]             = s;
        S1[at(qz, cy, cx)] = uq[qz];
      }
    }
    sync();
    if (active) {
      const auto gD = phase_ptr(mats + Q * P);
      const int  a = t % Q, qz = t / Q;  // x-line (qy = a, qz) and y-line (qx = a, qz)
      T          in[Q];
#pragma unroll
      for (int c = 0; c < Q; c++) in[c] = S1[at(qz, a, c)];
#pragma unroll
      for (int qx = 0; qx < Q; qx++) {
        const auto m = kRowWise ? phase_ptr(mats + Q * P + qx * Q) : gD + qx * Q;
        T          s = 0;
#pragma unroll
        for (int c = 0; c < Q; c++) s += m[c] * in[c];
        S2[at(qz, a, qx)] = s;
      }
#pragma unroll
      for (int c = 0; c < Q; c++) in[c] = S1[at(qz, c, a)];
#pragma unroll
      for (int qy = 0; qy < Q; qy++) {
        const auto m = kRowWise ? phase_ptr(mats + Q * P + qy * Q) : gD + qy * Q;
        T          s = 0;
#pragma unroll
        for (int c = 0; c < Q; c++) s += m[c] * in[c];
        S0[at(qz, qy, a)] = s;
      }
    }
    sync();
    // ---- pointwise (Poisson3DApply, times kappa for the kappa-weighted operator) on the column
    if constexpr (!LineQData<Q, NCOMP, QF, T>::kEarly) {
      if (active) qd.load(qe, cx, cy);
    }
    T vz[Q];
    if (active) {
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        T vx, vy, vzz;
        T s[QC];
        qd.point(qz, cx, s);
        poisson_regs<T>(s, S2[at(qz, cy, cx)], S0[at(qz, cy, cx)], dz[qz], vx, vy, vzz);
        if constexpr (QF == kQfDiffusionKappa) {
          vx *= s[6];
          vy *= s[6];
          vzz *= s[6];
        }
        if (!live) vx = vy = vzz = 0;
        S2[at(qz, cy, cx)] = vx;
        S0[at(qz, cy, cx)] = vy;
        vz[qz]             = vzz;
      }
    }
    sync();
    // ---- D_x^T by x-lines into S1; D_y^T by y-lines, held in registers
    // until every x-line has read S2, then written over it
    {
      const int a = t % Q, qz = t / Q;
      T         ty[Q];
      if (active) {
        {
          const auto gD = phase_ptr(mats + Q * P);
          T          in[Q];
#pragma unroll
          for (int c = 0; c < Q; c++) in[c] = S2[at(qz, a, c)];
#pragma unroll
          for (int qx = 0; qx < Q; qx++) {
            const auto m = kRowWise ? phase_ptr(mats + Q * P + qx) : gD + qx;
            T          s = 0;
#pragma unroll
            for (int c = 0; c < Q; c++) s += m[c * Q] * in[c];
            S1[at(qz, a, qx)] = s;
          }
        }
        {
          const auto gD = phase_ptr(mats + Q * P);
          T          in[Q];
#pragma unroll
          for (int c = 0; c < Q; c++) in[c] = S0[at(qz, c, a)];
#pragma unroll
          for (int qy = 0; qy < Q; qy++) {
            const auto m = kRowWise ? phase_ptr(mats + Q * P + qy) : gD + qy;
            T          s = 0;
#pragma unroll
            for (int c = 0; c < Q; c++) s += m[c * Q] * in[c];
            ty[qy] = s;
          }
        }
      }
      sync();
      if (active) {
#pragma unroll
        for (int qy = 0; qy < Q; qy++) S2[at(qz, qy, a)] = ty[qy];
      }
    }
    sync();
    // ---- sum of the three transposes on the column, then B_z^T into S0
    if (active) {
      const auto gDz = phase_ptr(mats + Q * P);
      T          w[Q];
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        const auto m = kRowWise ? phase_ptr(mats + Q * P + qz) : gDz + qz;
        T          s = S1[at(qz, cy, cx)] + S2[at(qz, cy, cx)];
#pragma unroll
        for (int c = 0; c < Q; c++) s += m[c * Q] * vz[c];
        w[qz] = s;
      }
      const auto gBz = phase_ptr(mats);
#pragma unroll
      for (int b = 0; b < P; b++) {
        const auto m = kRowWise ? phase_ptr(mats + b) : gBz + b;
        T          s = 0;
#pragma unroll
        for (int qz = 0; qz < Q; qz++) s += m[qz * P] * w[qz];
        S0[at(b, cy, cx)] = s;
      }
    }
  }
  sync();
  // ---- B_y^T: y-line (qx, z), z < P, into S1
  if (active && t < Q * P) {
    const auto gB = phase_ptr(mats);
    const int  qx = t % Q, z = t / Q;
    T          in[Q];
#pragma unroll
    for (int a = 0; a < Q; a++) in[a] = S0[at(z, a, qx)];
#pragma unroll
    for (int y = 0; y < P; y++) {
      const auto m = kRowWise ? phase_ptr(mats + y) : gB + y;
      T          s = 0;
#pragma unroll
      for (int a = 0; a < Q; a++) s += m[a * P] * in[a];
      S1[at(z, y, qx)] = s;
    }
  }
  sync();
  // ---- B_x^T: x-line (ny, nz) of nodes, into S0 (last read by B_y^T)
  if (xline) {
    const auto gB = phase_ptr(mats);
    T          in[Q];
#pragma unroll
    for (int a = 0; a < Q; a++) in[a] = S1[at(nz, ny, a)];
#pragma unroll
    for (int x = 0; x < P; x++) {
      const auto m   = kRowWise ? phase_ptr(mats + x) : gB + x;
      T          acc = 0;
#pragma unroll
      for (int a = 0; a < Q; a++) acc += m[a * P] * in[a];
      S0[at(nz, ny, x)] = acc;
    }
  }
  sync();
}

// E^T in the apply's own launch, for the node column of one thread: each
// contribution goes to its slot in the E-vector sorted by L entry, and the
// last of an entry's contributions to arrive (tcount) forms the entry's sum in
// the slots' order: the bits of the gather that otherwise follows.  The slots
// are written and read at agent scope, the release before the count and the
// acquire after it order them across the XCDs' caches; nobody waits.  The last
// contribution takes the count back by the number of contributions.
// Only for launches of at most one workgroup per CU: every wavefront's release
// writes its XCD's L2 back, and these serialise (MI355X, FP64 diffusion, us per
// apply, gather launch / this: 54 workgroups, p=2 11.2 / 8.9; 183, p=2 11.0 /
// 9.7; 247, p=1 11.4 / 9.5; 1229, p=2 12.6 / 26.5); only below P = 5: the
// nodes of a column follow one another (p=4 11.6 / 11.3, p=7 13.9 / 16.9); only
// one component: a release each (three, p=2 12.2 / 21.6).
__host__ __device__ constexpr bool line_takes_last(int P, int ncomp) { return P <= 4 && ncomp == 1; }
constexpr int64_t kLastWorkgroups = 256;
template <int P, typename T>
__device__ __forceinline__ void line_last(bool overwrite, const int (&off)[P], const int32_t *__restrict__ tpos, int tstride, const T (&s)[P],
                                          T *__restrict__ v, T *__restrict__ evec, const int32_t *__restrict__ trow, int32_t *__restrict__ tcount) {
  int32_t beg[P], num[P], old[P];
#pragma unroll
  for (int z = 0; z < P; z++) {
    const int32_t n = off[z] >> 1;
    beg[z]          = trow[n];
    num[z]          = trow[n + 1] - beg[z];
    __hip_atomic_store(&evec[tpos[z * tstride]], s[z], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
#pragma unroll
  for (int z = 0; z < P; z++) old[z] = __hip_atomic_fetch_add(&tcount[off[z] >> 1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
  for (int z = 0; z < P; z++) {
    if ((old[z] + 1) % num[z]) continue;
    const int32_t n = off[z] >> 1;
    T             c[8], acc = overwrite ? T(0) : v[n];
    (void)__hip_atomic_fetch_sub(&tcount[n], num[z], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int m = 0; m < 8; m++) c[m] = __hip_atomic_load(&evec[beg[z] + (m < num[z] ? m : 0)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int m = 0; m < 8; m++) {
      if (m < num[z]) acc += c[m];
    }
    for (int m = 8; m < num[z]; m++) acc += __hip_atomic_load(&evec[beg[z] + m], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v[n] = acc;
  }
}

// The line kernel keeps the pipeline written out in its own body rather than
// calling line_element: the same code through the shared function compiles
// to a different register allocation here (P=7, Q=8 diffusion: 186 against
// 162 VGPRs, a wave per SIMD fewer, 20% slower on MI355X at 8M DoFs; P=5,
// Q=6: 133 against 127).  Both compute every value with the same operations
// in the same order (tests/test_gpu_brick.py::test_brick_single_brick_bitwise).
// kSeg: the workgroup runs one segment of elements chained along x
// (seg_start), summing the face between consecutive elements in LDS before
// E^T; a template parameter so that the other modes keep their registers.
// No bound on the registers: four waves per SIMD forced on FP64 3-component
// diffusion at P = 4, Q = 5 were 5% faster with three slabs per element and are
// 0 to 1% slower with lines in place (MI355X, us per apply, bound / without:
// 2.3M DoFs 85.3 / 84.7, 24M 745-756 / 736-738); FP64 P = 5, Q = 6 spills and
// FP32 P = 6, Q = 7 (5 waves) is 4% slower.
template <int P, int Q, int NCOMP, int QF, typename T, bool kSeg = false, bool kGeo = false>
__global__ void __launch_bounds__(256) hex_apply_lines_kernel(int64_t elem_begin, int64_t elem_end, int scatter,
                                                               const int32_t *__restrict__ offsets, int32_t comp_stride,
                                                               const T *__restrict__ q_data, const T *__restrict__ mats,
                                                               const T *__restrict__ u, T *__restrict__ v, T *__restrict__ evec,
                                                               const int32_t *__restrict__ tpos,
                                                               const int32_t *__restrict__ elem_sys, const int32_t *__restrict__ sys_active,
                                                               const int32_t *__restrict__ seg_start, const double *__restrict__ geo,
                                                               const double *__restrict__ geo_pts,
                                                               const int32_t *__restrict__ perm, const double *__restrict__ kappa_src,
                                                               T *__restrict__ kappa_keep, const int32_t *__restrict__ trow,
                                                               int32_t *__restrict__ tcount) {
  constexpr int NT = Q * Q, P3 = P * P * P, Q3 = Q * Q * Q, QC = QfTraits<QF>::kComps;
  constexpr int SR = line_row_stride(Q, sizeof(T)), SP = line_plane_stride(Q, sizeof(T)), SLAB = Q * SP;
  static_assert(SR >= Q && SP >= Q * SR, "slab rows and planes must not overlap");
  constexpr int ES = line_elem_entries(Q, NCOMP, QF, sizeof(T), kGeo);
  constexpr bool kDzLds = line_dz_in_lds(Q, NCOMP, QF, sizeof(T), kGeo);
  constexpr bool kOnce = line_geo_once(Q, NCOMP, sizeof(T));
  // from Q = 7 one phase's matrix entries no longer fit the SGPRs: load them
  // per output row (or column) instead of per phase
  constexpr bool kRowWise = Q >= 7;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  // B (Q x P) then D (Q x Q), row-major, at mats

  const int epb = blockDim.x / NT;
  const int le = threadIdx.x / NT, t = threadIdx.x - le * NT;
  T        *X = reinterpret_cast<T *>(lds_raw) + le * ES;
  T        *Y = X + SLAB;  // diffusion only
  T        *Z = Y + SLAB;  // kDzLds only
  auto      at = [](int z, int y, int x) { return z * SP + y * SR + x; };
  // kGeo: the element's trilinear map behind the slabs
  double *sgeo = reinterpret_cast<double *>(lds_raw + (((size_t)epb * ES * sizeof(T) + 15) & ~(size_t)15)) + le * kGeoLds;

  // the workgroup's elements: epb consecutive packed elements, or (kSeg)
  // segment elem_begin + chunk, whose consecutive elements share x-faces
  const int64_t chunk = xcd_chunk(blockIdx.x, gridDim.x);
  const int32_t sbeg  = kSeg ? seg_start[elem_begin + chunk] : 0;
  const int32_t slen  = kSeg ? seg_start[elem_begin + chunk + 1] - sbeg : 0;
  const int64_t e     = kSeg ? (int64_t)sbeg + le : elem_begin + chunk * epb + le;
  bool          live  = le < epb && (kSeg ? le < slen : e < elem_end);
  // elem_sys: the system of each element, where some are frozen; the same
  // pointer as sys_active: one entry for all, in a caller's graph (into_callers_graph)
  if (elem_sys) {
    if (elem_sys == sys_active) {
      if (!*sys_active) return;
    } else {
      live = live && sys_active[elem_sys[e]];
      if (!__syncthreads_or(live)) return;  // every element of the workgroup is frozen (uniform exit)
    }
  }

  const int  cx = t % Q, cy = t / Q;  // column; also the x-line (qy = cx, qz = cy) and the y-line (qx = cx, qz = cy)
  const int  ny = t % P, nz = t / P;  // x-line of nodes
  const bool xline = t < P * P;
  // E and E^T run on the node columns (cx, cy < P), like the column layout, so
  // that a wave's loads and stores of u and v are coalesced along x
  const bool node = live && cx < P && cy < P;
  int        off[P];  // 2 * node + first_touch, nodes (cx, cy, z)
  if (node) {
#pragma unroll
    for (int z = 0; z < P; z++) off[z] = offsets[e * P3 + (z * P + cy) * P + cx];
  }
  // the column's geometric factors (LineQData; kGeo: recomputed at the
  // pointwise operator from the element's map, staged in LDS here)
  LineQData<Q, NCOMP, QF, T> qd;
  constexpr bool             kEarly = LineQData<Q, NCOMP, QF, T>::kEarly;
  const T                   *qe     = q_data + (live ? e : 0) * (int64_t)QC * Q3;
  double                     xi = 0, eta = 0, wxy = 0;
  T                          kappa[kGeo && QF == kQfDiffusionKappa ? Q : 1];
  if constexpr (kGeo && kOnce) {
    GeoColumn k;
    k.load(geo + (live ? e : 0) * kGeoStride, geo_pts[cx], geo_pts[cy]);
    wxy = geo_pts[Q + cy] * geo_pts[Q + cx];
    const auto gp = phase_ptr(geo_pts);
#pragma unroll
    for (int qz = 0; qz < Q; qz++) {
      double g6[6];
      __builtin_amdgcn_sched_barrier(0);
      geo_poisson(k, gp[qz], gp[Q + qz] * wxy, g6);
#pragma unroll
      for (int i = 0; i < 6; i++) qd.sq[qz][i] = (T)g6[i];
    }
  } else if constexpr (kGeo) {
    for (int i = t; i < kGeoStride; i += NT) sgeo[i] = geo[(live ? e : 0) * kGeoStride + i];
    xi  = geo_pts[cx];
    eta = geo_pts[cy];
    wxy = geo_pts[Q + cy] * geo_pts[Q + cx];
    if constexpr (QF == kQfDiffusionKappa) {
      // from the caller's array, kept in the plan (kappa_keep, its q_data) on
      // the way: p=4, Q=5, 3.9M DoFs 84 us, against 22..32 for the copy alone
      // and 70 for the kernel after it
      if (kappa_src) {
        if (live) {
          const double *src  = kappa_src + (int64_t)perm[e] * Q3 + cy * Q + cx;
          T            *keep = kappa_keep + e * (int64_t)QC * Q3 + 6 * Q3 + cy * Q + cx;
#pragma unroll
          for (int qz = 0; qz < Q; qz++) kappa[qz] = (T)__builtin_nontemporal_load(src + qz * Q * Q);
#pragma unroll
          for (int qz = 0; qz < Q; qz++) keep[qz * Q * Q] = kappa[qz];
        }
      } else {
#pragma unroll
        for (int qz = 0; qz < Q; qz++) kappa[qz] = __builtin_nontemporal_load(&qe[6 * Q3 + (qz * Q + cy) * Q + cx]);
      }
    }
  } else if constexpr (kEarly) {
    qd.load(qe, cx, cy);
  }

  // A line contraction in place needs no second slab and no synchronisation:
  // the line's thread reads all of it before it writes, and owns it.
  // The short phases between barriers issue before the wavefronts that are in
  // the long pointwise phase, which fill the gaps (MI355X, FP64 diffusion, us
  // per apply, without / with: p=3 1M DoFs 44.9 / 44.0, p=4 1M 37.3 / 36.5, 8M
  // 243 / 239, p=6 4M 101 / 98, p=7 4M 107 / 104, p=8 4M 112 / 109; p=2 no
  // change; the other way round 1-3% slower; nothing where the factors are
  // read, whose pointwise phase is short).
  if constexpr (kGeo && !kOnce) __builtin_amdgcn_s_setprio(1);
  for (int comp = 0; comp < NCOMP; comp++) {
    const int64_t coff = (int64_t)comp * comp_stride;
    if (comp > 0) __syncthreads();  // the previous component's E^T still reads X
    // ---- E: the node column gathers its P nodes into X
    if (node) {
#pragma unroll
      for (int z = 0; z < P; z++) X[at(z, cy, cx)] = u[(off[z] >> 1) + coff];
    }
    __syncthreads();
    // ---- B_x on the x-line (ny, nz) of nodes, in place
    if (xline) {
      const auto gB = phase_ptr(mats);
      T          in[P];
#pragma unroll
      for (int x = 0; x < P; x++) in[x] = X[at(nz, ny, x)];
#pragma unroll
      for (int qx = 0; qx < Q; qx++) {
        const auto m = kRowWise ? phase_ptr(mats + qx * P) : gB + qx * P;
        T          s = 0;
#pragma unroll
        for (int b = 0; b < P; b++) s += m[b] * in[b];
        X[at(nz, ny, qx)] = s;
      }
    }
    __syncthreads();
    // ---- B_y on the y-line (qx = cx, z = cy < P), in place
    if (t < Q * P) {
      const auto gB = phase_ptr(mats);
      T          in[P];
#pragma unroll
      for (int b = 0; b < P; b++) in[b] = X[at(cy, b, cx)];
#pragma unroll
      for (int qy = 0; qy < Q; qy++) {
        const auto m = kRowWise ? phase_ptr(mats + qy * P) : gB + qy * P;
        T          s = 0;
#pragma unroll
        for (int b = 0; b < P; b++) s += m[b] * in[b];
        X[at(cy, qy, cx)] = s;
      }
    }
    __syncthreads();
    // ---- B_z on the column (cx, cy): uq[qz]
    T uq[Q];
    {
      const auto gB = phase_ptr(mats);
      T          col[P];
#pragma unroll
      for (int b = 0; b < P; b++) col[b] = X[at(b, cy, cx)];
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        const auto m = kRowWise ? phase_ptr(mats + qz * P) : gB + qz * P;
        T          s = 0;
#pragma unroll
        for (int b = 0; b < P; b++) s += m[b] * col[b];
        uq[qz] = s;
      }
    }
    if constexpr (QF == kQfMass) {
      // ---- D, then B_z^T back into the column's own entries
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        T s[QC];
        qd.point(qz, cx, s);
        uq[qz] *= s[0];
      }
      if constexpr (kRowWise) {
        T out[P];
#pragma unroll
        for (int i = 0; i < P; i++) out[i] = 0;
        transposed_line(mats, uq, out);
#pragma unroll
        for (int i = 0; i < P; i++) X[at(i, cy, cx)] = out[i];
      } else {
        const auto m = phase_ptr(mats);
#pragma unroll
        for (int i = 0; i < P; i++) {
          T s = 0;
#pragma unroll
          for (int j = 0; j < Q; j++) s += m[j * P + i] * uq[j];
          X[at(i, cy, cx)] = s;
        }
      }
    } else {
      // ---- collocated derivatives: z on the column; x by x-lines of X into Y,
      // y by y-lines of X in place once every x-line has been read
      T dz[Q];
      {
        const auto gD = phase_ptr(mats + Q * P);
#pragma unroll
        for (int qz = 0; qz < Q; qz++) {
          const auto m = kRowWise ? phase_ptr(mats + Q * P + qz * Q) : gD + qz * Q;
          T          s = 0;
#pragma unroll
          for (int c = 0; c < Q; c++) s += m[c] * uq[c];
          dz[qz]            = s;
          X[at(qz, cy, cx)] = uq[qz];
        }
      }
      __syncthreads();
      {
        T in[Q];
#pragma unroll
        for (int c = 0; c < Q; c++) in[c] = X[at(cy, cx, c)];
        {
          const auto gD = phase_ptr(mats + Q * P);
#pragma unroll
          for (int qx = 0; qx < Q; qx++) {
            const auto m = kRowWise ? phase_ptr(mats + Q * P + qx * Q) : gD + qx * Q;
            T          s = 0;
#pragma unroll
            for (int c = 0; c < Q; c++) s += m[c] * in[c];
            Y[at(cy, cx, qx)] = s;
          }
        }
#pragma unroll
        for (int c = 0; c < Q; c++) in[c] = X[at(cy, c, cx)];
        __syncthreads();
        const auto gD = phase_ptr(mats + Q * P);
#pragma unroll
        for (int qy = 0; qy < Q; qy++) {
          const auto m = kRowWise ? phase_ptr(mats + Q * P + qy * Q) : gD + qy * Q;
          T          s = 0;
#pragma unroll
          for (int c = 0; c < Q; c++) s += m[c] * in[c];
          X[at(cy, qy, cx)] = s;
        }
      }
      __syncthreads();
      // ---- pointwise (Poisson3DApply, times kappa for the kappa-weighted operator) on the column, in place
      // From Q = 10 the column's z-derivatives wait in a third slab (only this
      // thread's entries) rather than in registers beside the late q_data
      // loads (interleaved A/B on MI355X, 8M DoFs: p=8 0.283 vs 0.293 ms; at
      // Q = 9, p=7, 0.280 vs 0.274, so not there).
      if constexpr (kDzLds) {
#pragma unroll
        for (int qz = 0; qz < Q; qz++) Z[at(qz, cy, cx)] = dz[qz];
      }
      if constexpr (!kGeo && !kEarly) qd.load(qe, cx, cy);
      GeoColumn  k;
      const auto gp = phase_ptr(geo_pts);
      if constexpr (kGeo && !kOnce) __builtin_amdgcn_s_setprio(0);
      if constexpr (kGeo && !kOnce) k.load(sgeo, xi, eta);
      T vz[Q];
#pragma unroll
      for (int qz = 0; qz < Q; qz++) {
        T s[QC], vx, vy, vzz;
        if constexpr (kGeo && !kOnce) {
          double g6[6];
          __builtin_amdgcn_sched_barrier(0);  // one point's factors at a time in registers (Q = 6: 92 VGPRs against 99, five waves per SIMD)
          geo_poisson(k, gp[qz], gp[Q + qz] * wxy, g6);
#pragma unroll
          for (int i = 0; i < 6; i++) s[i] = (T)g6[i];
          if constexpr (QF == kQfDiffusionKappa) s[6] = kappa[qz];
        } else {
          qd.point(qz, cx, s);
        }
        poisson_regs<T>(s, Y[at(qz, cy, cx)], X[at(qz, cy, cx)], kDzLds ? Z[at(qz, cy, cx)] : dz[qz], vx, vy, vzz);
        if constexpr (QF == kQfDiffusionKappa) {
          vx *= s[6];
          vy *= s[6];
          vzz *= s[6];
        }
        Y[at(qz, cy, cx)] = vx;
        X[at(qz, cy, cx)] = vy;
        vz[qz]            = vzz;
      }
      if constexpr (kGeo && !kOnce) __builtin_amdgcn_s_setprio(1);
      __syncthreads();
      // ---- D_x^T by x-lines of Y, D_y^T by y-lines of X, both in place
      {
        T in[Q];
#pragma unroll
        for (int c = 0; c < Q; c++) in[c] = Y[at(cy, cx, c)];
        if constexpr (kRowWise) {
          T out[Q];
#pragma unroll
          for (int i = 0; i < Q; i++) out[i] = 0;
          transposed_line(mats + Q * P, in, out);
#pragma unroll
          for (int i = 0; i < Q; i++) Y[at(cy, cx, i)] = out[i];
        } else {
          const auto m = phase_ptr(mats + Q * P);
#pragma unroll
          for (int i = 0; i < Q; i++) {
            T s = 0;
#pragma unroll
            for (int j = 0; j < Q; j++) s += m[j * Q + i] * in[j];
            Y[at(cy, cx, i)] = s;
          }
        }
#pragma unroll
        for (int c = 0; c < Q; c++) in[c] = X[at(cy, c, cx)];
        if constexpr (kRowWise) {
          T out[Q];
#pragma unroll
          for (int i = 0; i < Q; i++) out[i] = 0;
          transposed_line(mats + Q * P, in, out);
#pragma unroll
          for (int i = 0; i < Q; i++) X[at(cy, i, cx)] = out[i];
        } else {
          const auto m = phase_ptr(mats + Q * P);
#pragma unroll
          for (int i = 0; i < Q; i++) {
            T s = 0;
#pragma unroll
            for (int j = 0; j < Q; j++) s += m[j * Q + i] * in[j];
            X[at(cy, i, cx)] = s;
          }
        }
      }
      __syncthreads();
      // ---- sum of the three transposes on the column, then B_z^T into X
      T w[Q];
      if constexpr (kRowWise) {
        T out[Q];
#pragma unroll
        for (int i = 0; i < Q; i++) out[i] = Y[at(i, cy, cx)] + X[at(i, cy, cx)];
        transposed_line(mats + Q * P, vz, out);
#pragma unroll
        for (int i = 0; i < Q; i++) w[i] = out[i];
      } else {
        const auto m = phase_ptr(mats + Q * P);
#pragma unroll
        for (int i = 0; i < Q; i++) {
          T s = Y[at(i, cy, cx)] + X[at(i, cy, cx)];
#pragma unroll
          for (int j = 0; j < Q; j++) s += m[j * Q + i] * vz[j];
          w[i] = s;
        }
      }
      if constexpr (kRowWise) {
        T out[P];
#pragma unroll
        for (int i = 0; i < P; i++) out[i] = 0;
        transposed_line(mats, w, out);
#pragma unroll
        for (int i = 0; i < P; i++) X[at(i, cy, cx)] = out[i];
      } else {
        const auto m = phase_ptr(mats);
#pragma unroll
        for (int i = 0; i < P; i++) {
          T s = 0;
#pragma unroll
          for (int j = 0; j < Q; j++) s += m[j * P + i] * w[j];
          X[at(i, cy, cx)] = s;
        }
      }
    }
    __syncthreads();
    // ---- B_y^T on the y-line (qx = cx, z = cy < P), in place
    if (t < Q * P) {
      T in[Q];
#pragma unroll
      for (int a = 0; a < Q; a++) in[a] = X[at(cy, a, cx)];
      if constexpr (kRowWise) {
        T out[P];
#pragma unroll
        for (int i = 0; i < P; i++) out[i] = 0;
        transposed_line(mats, in, out);
#pragma unroll
        for (int i = 0; i < P; i++) X[at(cy, i, cx)] = out[i];
      } else {
        const auto m = phase_ptr(mats);
#pragma unroll
        for (int i = 0; i < P; i++) {
          T s = 0;
#pragma unroll
          for (int j = 0; j < Q; j++) s += m[j * P + i] * in[j];
          X[at(cy, i, cx)] = s;
        }
      }
    }
    __syncthreads();
    // ---- B_x^T on the x-line (ny, nz) of nodes, in place
    if (xline) {
      T in[Q];
#pragma unroll
      for (int a = 0; a < Q; a++) in[a] = X[at(nz, ny, a)];
      if constexpr (kRowWise) {
        T out[P];
#pragma unroll
        for (int i = 0; i < P; i++) out[i] = 0;
        transposed_line(mats, in, out);
#pragma unroll
        for (int i = 0; i < P; i++) X[at(nz, ny, i)] = out[i];
      } else {
        const auto m = phase_ptr(mats);
#pragma unroll
        for (int i = 0; i < P; i++) {
          T s = 0;
#pragma unroll
          for (int j = 0; j < Q; j++) s += m[j * P + i] * in[j];
          X[at(nz, ny, i)] = s;
        }
      }
    }
    __syncthreads();
    // ---- E^T from the node columns
    if (node) {
      T s[P];
#pragma unroll
      for (int z = 0; z < P; z++) s[z] = X[at(z, cy, cx)];
      if (line_takes_last(P, NCOMP) && !kSeg && scatter >= kScatterLast) {
        if constexpr (line_takes_last(P, NCOMP)) line_last<P>(scatter == kScatterLast, off, &tpos[e * P3 + cy * P + cx], P * P, s, v, evec, trow, tcount);
      } else if (!kSeg && scatter == kScatterEvec) {  // tpos gives each contribution's slot in the E-vector sorted by L entry
        int32_t pos[P];
#pragma unroll
        for (int z = 0; z < P; z++) pos[z] = tpos[(e * NCOMP + comp) * (int64_t)P3 + (z * P + cy) * P + cx];
#pragma unroll
        for (int z = 0; z < P; z++) evec[pos[z]] = s[z];
      } else if (!kSeg && scatter == kScatterAtomic) {
#pragma unroll
        for (int z = 0; z < P; z++) unsafeAtomicAdd(&v[(off[z] >> 1) + coff], s[z]);
      } else if (!kSeg && scatter == kScatterSplit) {  // shared entries to their E-vector slot, the rest onto the zeroed target
#pragma unroll
        for (int z = 0; z < P; z++) {
          if (off[z] & 1) evec[tpos[(e * NCOMP + comp) * (int64_t)P3 + (z * P + cy) * P + cx]] = s[z];
          else unsafeAtomicAdd(&v[(off[z] >> 1) + coff], s[z]);
        }
      } else {
        // segments: the face x = P-1 also holds the next element's x = 0 face
        // (its X is final after the barrier above), added after the own value;
        // the next element's threads of that face write nothing
        bool write = true;
        if constexpr (kSeg) {
          if (cx == P - 1 && le + 1 < slen) {
            const T *Sn = X + ES;
#pragma unroll
            for (int z = 0; z < P; z++) s[z] += Sn[at(z, cy, 0)];
          }
          write = cx > 0 || le == 0;
        }
        if (write) {
          const bool overwrite = scatter == kScatterOverwrite;
          T          old[P];
#pragma unroll
          for (int z = 0; z < P; z++) old[z] = (overwrite && (off[z] & 1)) ? T(0) : v[(off[z] >> 1) + coff];
#pragma unroll
          for (int z = 0; z < P; z++) v[(off[z] >> 1) + coff] = (overwrite && (off[z] & 1)) ? s[z] : old[z] + s[z];
        }
      }
    }
  }
}

}  // namespace mi355
