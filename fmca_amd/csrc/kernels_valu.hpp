// Vector-ALU forms of the two kernel-entry phases: fewer than kMfmaMinRhs
// right-hand sides, geodesic entries, and shapes whose staging does not fit
// the matrix-core forms.  Included by one translation unit per precision.
//
//   leaf output   y_t = V_t^T l_t + sum_{s in near(t)} K(P_t, P_s) x_s
//   coupling      l_t = sum_{s in far(t)} K(xi_t, xi_s) m_s
//
// One workgroup serves one task of a target (leaf or cluster).  Its threads
// are numbered through (slice, row): with R target rows and k rows per
// thread, ceil(R / k) threads cover the rows and the workgroup holds
// S = threads / ceil(R / k) slices of the sources, whose sums are added in LDS
// at the end in slice order.  So the lanes stay busy whatever the leaf size:
// at 39 rows 234 of 256 lanes, at 78 rows 234, at 122 rows 244 (one slice
// of one thread per row left 39, 78 and 122).
//
// What bounds them: vector issue.  An FP32 Matern-3/2 entry takes 11
// operations of 4.7 cycles and two transcendentals of 8.5 (69 cycles per 64
// entries of a SIMD), an FP64 one 27 operations of 4.9 and one v_rsq_f64 of 16.
// Measured before -> now (ms): n = 1e6, 3-D, degree 4, 1 rhs FP32: leaf output
// 7.2 -> 6.3, coupling 4.6 -> 3.3; n = 1e4, degree 3, 1 rhs FP64: 1.15 -> 0.07,
// 0.36 -> 0.04; n = 123457, degree 3, 5 rhs FP32: 2.08 -> 0.85, 1.09 -> 0.55.
//
// Few targets (small point sets) would leave most of the 256 CUs idle, so a
// task's source list is also cut into grid.y contiguous parts; each part
// writes its sums to its own slab and k_add_parts / k_add_parts_out add the
// slabs in part order (no atomics: results do not depend on scheduling).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "device.hpp"
#include "device_math.hpp"

namespace fmca_amd {
namespace {

using namespace dev;

constexpr int kAlphaTile = 128;  // far-field coefficients staged per step
// Nodes of a source from which the coupling stages one source at a time; below,
// all sources of a tile at once, as most threads would idle and a list of a few
// nodes wait for a loop over the tile's sources (coupling, FP32, 1 rhs, n = 2e5:
// 1-D degree 1 247 -> 142 us, 2-D degree 1 228 -> 100, degree 3 120 -> 91).
constexpr int kWholeSources = 32;

// Rows per thread, while the accumulators are few.  More rows share a source's
// LDS reads and, in the coupling, the setup of a line; one row leaves the FP64
// leaf output more waves.  Measured (us): FP64 leaf output n = 1e4, 1 rhs: 72
// with one row, 79 with two; FP64 leaf output, 8 rhs, n = 2e5: 3-D degree 3
// EXPONENTIAL 3600 / 2433 with one / two rows, degree 4 MATERN32 6497 / 5863,
// but 2-D degree 5 333 / 362 (small leaves); FP32 leaf output n = 123457,
// 5 rhs: 848 / 857 with two / one, 892 with four; FP32 coupling there: 547
// with four, 608 with two.
template <typename T, int D, int NR, bool OUTPUT>
constexpr int kRowsPerThread = NR > 8 ? 1
                               : OUTPUT ? (sizeof(T) == 8 && !(NR == 8 && D == 3) ? 1 : 2)
                                        : (sizeof(T) == 4 && NR <= 6 ? 4 : 2);

// elements of a staged source (D coordinates, NR values), a multiple of 16 bytes
template <typename T, int D, int NR>
constexpr int kRecord = (D + NR + (16 / (int)sizeof(T)) - 1) / (16 / (int)sizeof(T)) *
                        (16 / (int)sizeof(T));

template <typename T, int N>
__device__ __forceinline__ void load_record(const T *p, T (&v)[N]) {
  constexpr int VL = 16 / (int)sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(VL)));
#pragma unroll
  for (int k = 0; k < N / VL; ++k) {
    const vec_t x = reinterpret_cast<const vec_t *>(p)[k];
#pragma unroll
    for (int i = 0; i < VL; ++i) v[k * VL + i] = x[i];
  }
}

// Adds the slices' accumulators in slice order; the sums end in slice 0.
template <typename T, int RPT, int NR>
__device__ __forceinline__ void add_slices(T (&acc)[RPT][NR], T *red, int slice, int tr, int nh,
                                           int S, int nr) {
  const int nt = blockDim.x;
  if (S == 1) return;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r >= nr) break;
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RPT; ++rt) red[rt * nt + threadIdx.x] = acc[rt][r];
    __syncthreads();
    if (slice == 0) {
      for (int s = 1; s < S; ++s)
#pragma unroll
        for (int rt = 0; rt < RPT; ++rt) acc[rt][r] += red[rt * nt + s * nh + tr];
    }
  }
}

// ---------------------------------------------------------------------------
// Leaf output.  LDS: one region used first for the 1-D basis factors of the
// rows with the far-field coefficients, then for the staged sources, then for
// the slice sums.
template <typename T, int D, int KT, int NR, bool GEO>
__global__ __launch_bounds__(256) void k_leaf_output(DevTreeView<T> rows, DevTreeView<T> cols,
                                                     DevPatternView pat, InterpParams<T> ip,
                                                     KernelParams<T> kp, int nrhs,
                                                     const T *__restrict__ xs,
                                                     const T *__restrict__ tlhs,
                                                     double *__restrict__ out, int64_t ldo,
                                                     int natural, int smax,
                                                     T *__restrict__ part) {
  constexpr int RPT = kRowsPerThread<T, D, NR, true>;
  constexpr int RS = kRecord<T, D, NR>;
  constexpr bool TAB = !GEO && kTableEntry<KT, T>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double tab[TAB ? 64 : 1];
  const int nt = blockDim.x;
  const int P1 = ip.P1, q = ip.q;
  T *U = reinterpret_cast<T *>(smem_raw);
  T *F = U;                                              // [D][P1][nt] basis factors
  T *Mv = F + D * P1 * nt;                               // [kAlphaTile][NR]
  int *aidx = reinterpret_cast<int *>(Mv + kAlphaTile * NR);  // [kAlphaTile]
  T *Rec = U;                                            // [nt][RS] staged sources
  T *red = U;                                            // [RPT][nt] slice sums
  const int task = pat.near_order[blockIdx.x];
  if (task < 0) return;
  const int li = pat.near_task[4 * task], flags = pat.near_task[4 * task + 3];
  int n0 = pat.near_task[4 * task + 1], n1 = pat.near_task[4 * task + 2];
  const bool split = (flags & kTaskSplit) != 0;
  const bool do_far = (flags & kTaskFar) != 0 && pat.has_far && blockIdx.y == 0;
  if (gridDim.y > 1) {
    const int64_t cnt = n1 - n0;
    n1 = n0 + (int)(cnt * (blockIdx.y + 1) / gridDim.y);
    n0 = n0 + (int)(cnt * blockIdx.y / gridDim.y);
  }
  const int c = rows.leaves[li];
  const int b0 = rows.begin[c], sz = rows.size[c];
  if constexpr (TAB) load_exp2_table(tab);
  for (int rc = 0; rc < nrhs; rc += NR) {
    const int nr = min(NR, nrhs - rc);
    for (int pbase = 0; pbase < sz; pbase += nt) {
      const int nrow = min(nt, sz - pbase);
      const int nh = (nrow + RPT - 1) / RPT;
      const int S = min(nt / nh, smax);
      const int slice = threadIdx.x / nh, tr = threadIdx.x - slice * nh;
      const bool act = slice < S;
      T x[RPT][D], acc[RPT][NR];
#pragma unroll
      for (int rt = 0; rt < RPT; ++rt) {
        const int i = pbase + min(tr + rt * nh, nrow - 1);
#pragma unroll
        for (int d = 0; d < D; ++d) x[rt][d] = rows.pts[(int64_t)d * rows.npts + b0 + i];
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[rt][r] = 0;
      }
      // far field through the leaf basis (backward_transform_impl.h:30-31),
      // applied by the first task of the leaf
      if (do_far) {
        __syncthreads();
        if ((int)threadIdx.x < nrow) {
#pragma unroll
          for (int d = 0; d < D; ++d)
            basis_1d<T>(rows.unit[(int64_t)d * rows.npts + b0 + pbase + threadIdx.x], ip,
                        F + (d * P1) * nt + threadIdx.x, nt);
        }
        for (int at = 0; at < q; at += kAlphaTile) {
          const int na = min(kAlphaTile, q - at);
          __syncthreads();
          for (int e = threadIdx.x; e < na * NR; e += nt) {
            const int al = e / NR, r = e % NR;
            Mv[e] = r < nr ? tlhs[((int64_t)c * q + at + al) * nrhs + rc + r] : T(0);
          }
          for (int e = threadIdx.x; e < na; e += nt) aidx[e] = basis_index<T, D>(at + e, ip);
          __syncthreads();
          if (act) {
            for (int al = slice; al < na; al += S) {
              const int pk = aidx[al];
#pragma unroll
              for (int rt = 0; rt < RPT; ++rt) {
                const int row = min(tr + rt * nh, nrow - 1);
                T v = F[(pk & 0xff) * nt + row];
#pragma unroll
                for (int d = 1; d < D; ++d) v *= F[(d * P1 + ((pk >> (8 * d)) & 0xff)) * nt + row];
#pragma unroll
                for (int r = 0; r < NR; ++r) acc[rt][r] += v * Mv[al * NR + r];
              }
            }
          }
        }
      }
      // near field (unsymmetricNystromEvaluator.h:63-73, H2kernelActor.h:68-69):
      // tiles of nt sources gathered across the list, thread <-> source; the
      // next tile is fetched into registers while the current one is used
      int nb = n0, joff = 0;
      T py[D], px[NR];
      auto gather = [&]() {
        int fill = 0;
        int64_t src = -1;
        while (nb < n1 && fill < nt) {
          // a run of sources with adjacent point ranges is one range
          const int run = min(pat.near_run[nb], n1 - nb);
          const int s = pat.near_src[nb], sl = pat.near_src[nb + run - 1];
          const int sb = cols.begin[s], ss = cols.begin[sl] + cols.size[sl] - sb;
          const int take = min(ss - joff, nt - fill);
          const int k = (int)threadIdx.x - fill;
          if (k >= 0 && k < take) src = (int64_t)sb + joff + k;
          fill += take;
          joff += take;
          if (joff >= ss) {
            nb += run;
            joff = 0;
          }
        }
        if (src >= 0) {
#pragma unroll
          for (int d = 0; d < D; ++d) py[d] = cols.pts[(int64_t)d * cols.npts + src];
#pragma unroll
          for (int r = 0; r < NR; ++r) px[r] = r < nr ? xs[src * nrhs + rc + r] : T(0);
        }
        return fill;
      };
      int nj = gather();
      while (nj > 0) {
        __syncthreads();
        if ((int)threadIdx.x < nj) {
#pragma unroll
          for (int d = 0; d < D; ++d) Rec[threadIdx.x * RS + d] = py[d];
#pragma unroll
          for (int r = 0; r < NR; ++r) Rec[threadIdx.x * RS + D + r] = px[r];
        }
        __syncthreads();
        const int cur = nj;
        nj = gather();
        if (act) {
#pragma unroll 2
          for (int j = slice; j < cur; j += S) {
            T v[RS];
            load_record(Rec + j * RS, v);
#pragma unroll
            for (int rt = 0; rt < RPT; ++rt) {
              T kv;
              if constexpr (GEO) {
                kv = kernel_r2<KT, T>(geodesic_r2<T, D>(x[rt], v, 1), kp);
              } else {
                T r2 = kR2Start<KT, T>;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                  const T dd = x[rt][d] - v[d];
                  r2 = fmat(dd, dd, r2);
                }
                kv = entry_value<KT, T>(r2, kp, tab);
              }
#pragma unroll
              for (int r = 0; r < NR; ++r) acc[rt][r] = fmat(kv, v[D + r], acc[rt][r]);
            }
          }
        }
      }
      add_slices<T, RPT, NR>(acc, red, slice, tr, nh, S, nr);
      if (slice == 0) {
#pragma unroll
        for (int rt = 0; rt < RPT; ++rt) {
          const int i = pbase + tr + rt * nh;
          if (tr + rt * nh >= nrow) continue;
          if (gridDim.y > 1) {
            T *p = part + ((int64_t)blockIdx.y * rows.npts + b0 + i) * nrhs + rc;
#pragma unroll
            for (int r = 0; r < NR; ++r)
              if (r < nr) p[r] = acc[rt][r];
            continue;
          }
          const int64_t row = natural ? (int64_t)rows.perm[b0 + i] : (int64_t)(b0 + i);
#pragma unroll
          for (int r = 0; r < NR; ++r)
            if (r < nr) {
              double *p = out + row + (int64_t)(rc + r) * ldo;
              if (split)
                atomic_accumulate(p, (double)acc[rt][r]);
              else
                *p = (double)acc[rt][r];
            }
        }
      }
      __syncthreads();
    }
  }
}

// Bytes of the coupling's tables before its tile: unit coordinates of the
// lines and along a line, slots of the lines.
template <typename T, int D>
__host__ __device__ inline int coupling_head(int P1, int NL, int G) {
  return ((NL * D + P1) * (int)sizeof(T) + G * NL * (int)sizeof(int) + 15) & ~15;
}

// ---------------------------------------------------------------------------
// Coupling (unsymmetricNystromEvaluator.h:42-58 with invV = I,
// H2kernelActor.h:64-66).  Tiles of G whole sources: their moments
// [G q][NR], and the node coordinates.  Tensor nodes are taken line by line
// (the P1 nodes that differ in the first axis): the squared distance of the
// other axes is formed once per line, which leaves 2 + 4 / P1 operations of
// distance per entry instead of 6 in 3-D.  Total-degree nodes and geodesic
// entries take one node at a time ("lines" of one node).
// FEW: q < kWholeSources (see there).
template <typename T, int D, int KT, int NR, bool GEO, bool FEW>
__global__ __launch_bounds__(256) void k_coupling(DevTreeView<T> rows, DevTreeView<T> cols,
                                                  DevPatternView pat, InterpParams<T> ip,
                                                  KernelParams<T> kp, int nrhs, int G, int smax,
                                                  const T *__restrict__ mom,
                                                  T *__restrict__ tlhs, T *__restrict__ part) {
  constexpr int RPT = kRowsPerThread<T, D, NR, false>;
  constexpr bool TAB = !GEO && kTableEntry<KT, T>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double tab[TAB ? 64 : 1];
  const int nt = blockDim.x;
  const int q = ip.q;
  const bool lines = !GEO && !ip.td;
  const int P1 = lines ? ip.P1 : 1;  // nodes per line
  const int NL = q / P1;             // lines per source
  T *Ul = reinterpret_cast<T *>(smem_raw);  // [NL][D] unit coordinates of the lines
  T *U0 = Ul + NL * D;                      // [P1] unit coordinates along a line
  int *gl = reinterpret_cast<int *>(U0 + P1);  // [G NL] P1 * slot of a line's source
  // [G q][NR] moments (16-byte aligned)
  T *Mv = reinterpret_cast<T *>(smem_raw + coupling_head<T, D>(P1, NL, G));
  T *Yl = Mv + G * q * NR;                  // [G NL][D] line coordinates (axis 0: single nodes)
  T *Y0 = Yl + G * NL * D;                  // [G][P1] first-axis coordinates of the lines
  T *red = Mv;                              // [RPT][nt] slice sums
  const int task = pat.far_order[blockIdx.x];
  if (task < 0) return;
  const int t = pat.far_task[4 * task];
  int f0 = pat.far_task[4 * task + 1], f1 = pat.far_task[4 * task + 2];
  const bool split = (pat.far_task[4 * task + 3] & kTaskSplit) != 0;
  if (gridDim.y > 1) {
    const int64_t cnt = f1 - f0;
    f1 = f0 + (int)(cnt * (blockIdx.y + 1) / gridDim.y);
    f0 = f0 + (int)(cnt * blockIdx.y / gridDim.y);
  }
  if constexpr (TAB) load_exp2_table(tab);
  // unit coordinate d of node a
  auto unit = [&](int a, int d) {
    return ip.td ? ip.unodes[d * q + a] : ip.xi[(basis_index<T, D>(a, ip) >> (8 * d)) & 0xff];
  };
  for (int l = threadIdx.x; l < NL; l += nt)
#pragma unroll
    for (int d = 0; d < D; ++d) Ul[l * D + d] = unit(l * P1, d);
  if (lines)
    for (int b = threadIdx.x; b < P1; b += nt) U0[b] = ip.xi[b];
  // e / q and e / NL of a tile's nodes and lines (at most 2^15)
  [[maybe_unused]] const float rq = 1.0f / (float)q, rl = 1.0f / (float)NL;
  if constexpr (FEW) {
    for (int e = threadIdx.x; e < G * NL; e += nt) gl[e] = (int)(((float)e + 0.5f) * rl) * P1;
  } else {
    for (int g = 0; g < G; ++g)
      for (int l = threadIdx.x; l < NL; l += nt) gl[g * NL + l] = g * P1;
  }
  for (int rc = 0; rc < nrhs; rc += NR) {
    const int nr = min(NR, nrhs - rc);
    for (int abase = 0; abase < q; abase += nt) {
      const int nrow = min(nt, q - abase);
      const int nh = (nrow + RPT - 1) / RPT;
      const int S = min(nt / nh, smax);
      const int slice = threadIdx.x / nh, tr = threadIdx.x - slice * nh;
      const bool act = slice < S;
      T x[RPT][D], acc[RPT][NR];
#pragma unroll
      for (int rt = 0; rt < RPT; ++rt) {
        const int al = abase + min(tr + rt * nh, nrow - 1);
#pragma unroll
        for (int d = 0; d < D; ++d)
          x[rt][d] = unit(al, d) * rows.bbsize[t * D + d] + rows.bbmin[t * D + d];
#pragma unroll
        for (int r = 0; r < NR; ++r) acc[rt][r] = 0;
      }
      for (int f = f0; f < f1; f += G) {
        const int ns = min(G, f1 - f);
        __syncthreads();
        if constexpr (FEW) {  // threads over the nodes and lines of all sources
          for (int e = threadIdx.x; e < ns * q; e += nt) {
            const int g = (int)(((float)e + 0.5f) * rq);
            const T *ms = mom + ((int64_t)pat.far_src[f + g] * q + (e - g * q)) * nrhs + rc;
#pragma unroll
            for (int r = 0; r < NR; ++r) Mv[e * NR + r] = r < nr ? ms[r] : T(0);
          }
          for (int e = threadIdx.x; e < ns * NL; e += nt) {
            const int g = (int)(((float)e + 0.5f) * rl), l = e - g * NL;
            const int64_t s = pat.far_src[f + g];
#pragma unroll
            for (int d = 0; d < D; ++d)
              Yl[e * D + d] = Ul[l * D + d] * cols.bbsize[s * D + d] + cols.bbmin[s * D + d];
            if (lines)
              for (int b = l; b < P1; b += NL)
                Y0[g * P1 + b] = U0[b] * cols.bbsize[s * D] + cols.bbmin[s * D];
          }
        } else {
          for (int g = 0; g < ns; ++g) {
            const int64_t s = pat.far_src[f + g];
            T bs[D], bm[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
              bs[d] = cols.bbsize[s * D + d];
              bm[d] = cols.bbmin[s * D + d];
            }
            const T *ms = mom + s * q * nrhs + rc;
            for (int j = threadIdx.x; j < q; j += nt)
#pragma unroll
              for (int r = 0; r < NR; ++r)
                Mv[(g * q + j) * NR + r] = r < nr ? ms[(int64_t)j * nrhs + r] : T(0);
            for (int l = threadIdx.x; l < NL; l += nt)
#pragma unroll
              for (int d = 0; d < D; ++d)
                Yl[(g * NL + l) * D + d] = Ul[l * D + d] * bs[d] + bm[d];
            if (lines)
              for (int b = threadIdx.x; b < P1; b += nt) Y0[g * P1 + b] = U0[b] * bs[0] + bm[0];
          }
        }
        __syncthreads();
        if (!act) continue;
        if (lines) {
          for (int l = slice; l < ns * NL; l += S) {
            const T *y0 = Y0 + gl[l];
            T rest[RPT];
#pragma unroll
            for (int rt = 0; rt < RPT; ++rt) {
              rest[rt] = kR2Start<KT, T>;
#pragma unroll
              for (int d = 1; d < D; ++d) {
                const T dd = x[rt][d] - Yl[l * D + d];
                rest[rt] = fmat(dd, dd, rest[rt]);
              }
            }
#pragma unroll 2
            for (int b = 0; b < P1; ++b) {
              const T y = y0[b];
              const T *m = Mv + (l * P1 + b) * NR;
#pragma unroll
              for (int rt = 0; rt < RPT; ++rt) {
                const T dd = x[rt][0] - y;
                const T kv = entry_value<KT, T>(fmat(dd, dd, rest[rt]), kp, tab);
#pragma unroll
                for (int r = 0; r < NR; ++r) acc[rt][r] = fmat(kv, m[r], acc[rt][r]);
              }
            }
          }
        } else {
#pragma unroll 2
          for (int j = slice; j < ns * NL; j += S) {
            T y[D];
#pragma unroll
            for (int d = 0; d < D; ++d) y[d] = Yl[j * D + d];
            const T *m = Mv + j * NR;
#pragma unroll
            for (int rt = 0; rt < RPT; ++rt) {
              T kv;
              if constexpr (GEO) {
                kv = kernel_r2<KT, T>(geodesic_r2<T, D>(x[rt], y, 1), kp);
              } else {
                T r2 = kR2Start<KT, T>;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                  const T dd = x[rt][d] - y[d];
                  r2 = fmat(dd, dd, r2);
                }
                kv = entry_value<KT, T>(r2, kp, tab);
              }
#pragma unroll
              for (int r = 0; r < NR; ++r) acc[rt][r] = fmat(kv, m[r], acc[rt][r]);
            }
          }
        }
      }
      add_slices<T, RPT, NR>(acc, red, slice, tr, nh, S, nr);
      if (slice == 0) {
#pragma unroll
        for (int rt = 0; rt < RPT; ++rt) {
          const int al = abase + tr + rt * nh;
          if (tr + rt * nh >= nrow) continue;
          const int64_t e = ((int64_t)t * q + al) * nrhs + rc;
          T *p = gridDim.y > 1
                     ? part + (int64_t)blockIdx.y * rows.ncl * q * nrhs + e
                     : tlhs + e;
#pragma unroll
          for (int r = 0; r < NR; ++r)
            if (r < nr) {
              if (split)
                atomic_accumulate(p + r, acc[rt][r]);
              else
                p[r] = acc[rt][r];
            }
        }
      }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
template <typename T, int D, int NR>
size_t output_lds(int P1, int nt) {
  const size_t far = ((size_t)D * P1 * nt + (size_t)kAlphaTile * NR) * sizeof(T) +
                     kAlphaTile * sizeof(int);
  const size_t near = (size_t)nt * kRecord<T, D, NR> * sizeof(T);
  const size_t red = (size_t)nt * kRowsPerThread<T, D, NR, true> * sizeof(T);
  return std::max(far, std::max(near, red));
}

// LDS of a coupling tile of G sources (td: total-degree nodes or geodesic
// entries, one node per line).
template <typename T, int D, int NR>
size_t coupling_lds(int P1, int q, bool single, int G, int nt) {
  const int p = single ? 1 : P1, nl = q / p;
  const size_t tile = (size_t)G * (q * NR + nl * D + p) * sizeof(T);
  const size_t red = (size_t)nt * kRowsPerThread<T, D, NR, false> * sizeof(T);
  return coupling_head<T, D>(p, nl, G) + std::max(tile, red);
}

constexpr size_t kValuLds = 63 * 1024;  // with the static table at most 64 KB

// Most slices of a workgroup whose list has `sources` sources: a slice of fewer
// than four costs more in add_slices than it saves (FP32 leaf output, 7 columns,
// against one row a thread: at worst 0.77 of its speed with up to 32 slices
// whatever the list, 1.07 with four sources a slice, 0.83 with sixteen).
inline int valu_slices(double sources) {
  return (int)std::max(1.0, std::min(32.0, sources / 4));
}

// Workgroup size for targets of `rows` rows: the one of 64, 128 and 256
// threads whose lanes the slices use best; of nearly equal ones (4 %) the
// smaller (cheaper barriers, finer scheduling).  `whole`: split tasks, whose
// launch is not cut into parts, take 256 threads for more than 64 rows (2-D
// degree 7, clusters, FP64 leaf output, 1 rhs: 64 threads 2.39 ms, 256 0.74).
inline int valu_threads(double rows, int rpt, int smax, bool whole) {
  int best = 256;
  double top = -1;
  for (int nt : {64, 128, 256}) {
    if (whole && nt < 256 && rows > 64) continue;
    const int r = std::max(1, (int)std::min<double>(nt, std::ceil(rows)));
    const int nh = (r + rpt - 1) / rpt;
    const int S = std::min(nt / nh, smax);
    // passes of nt rows: the last one is partly filled
    const double passes = std::ceil(std::max(1.0, rows) / nt);
    const double use = passes > 1 ? rows / (passes * nt) * ((double)S * nh / nt)
                                  : rows / rpt * S / nt;
    if (use > top + 0.04) {
      top = use;
      best = nt;
    }
  }
  return best;
}

template <typename T, int D, int KT, int NR, bool GEO>
hipError_t valu_launch(bool output, const ValuLaunch<T> &a) {
  const int q = a.ip.q, P1 = a.ip.P1;
  int parts = 1;
  T *slabs = nullptr;
  if (output) {
    if (a.pat.nnear_order <= 0) return hipSuccess;
    const int smax = valu_slices(a.pat.near_per_task);
    const int nt = valu_threads(a.rows.nleaves > 0 ? (double)a.rows.npts / a.rows.nleaves : 1,
                                kRowsPerThread<T, D, NR, true>, smax, a.pat.nnear_split > 0);
    parts = phase_parts(a.pat.nnear_order, a.pat.nnear_split, nt / 64, a.pat.near_per_task, nt,
                        a.rows.npts * a.nrhs, a.part_cap);
    if (parts > 1 && !(slabs = a.part(parts * a.rows.npts * a.nrhs))) parts = 1;
    hipLaunchKernelGGL((k_leaf_output<T, D, KT, NR, GEO>),
                       dim3(a.pat.nnear_order, (unsigned)parts), dim3(nt),
                       (output_lds<T, D, NR>(P1, nt)), a.stream, a.rows, a.cols, a.pat, a.ip,
                       a.kp, a.nrhs, a.xs, a.tlhs, a.out, a.ldo, a.natural ? 1 : 0, smax, slabs);
  } else {
    if (a.pat.nfar_order <= 0) return hipSuccess;
    const int smax = valu_slices(a.pat.far_per_task * q);
    const int nt = valu_threads(q, kRowsPerThread<T, D, NR, false>, smax, false);
    const bool single = GEO || a.ip.td;
    // whole sources per tile, up to 512 nodes of one column (fewer of more)
    const int want = NR == 1 ? 512 : (NR <= 4 ? 256 : 128);
    // (and no more than a usual list has)
    int G = std::max(1, std::min(want / std::max(1, q), 64));
    G = std::max(1, std::min(G, (int)std::ceil(2 * a.pat.far_per_task)));
    while (G > 1 && coupling_lds<T, D, NR>(P1, q, single, G, nt) > kValuLds / 2) --G;
    parts = phase_parts(a.pat.nfar_order, a.pat.nfar_split, nt / 64, a.pat.far_per_task * q, nt,
                        (int64_t)a.rows.ncl * q * a.nrhs, a.part_cap);
    if (parts > 1 && !(slabs = a.part(parts * (int64_t)a.rows.ncl * q * a.nrhs))) parts = 1;
#define FMCA_COUPLING(F)                                                                        \
  hipLaunchKernelGGL((k_coupling<T, D, KT, NR, GEO, F>), dim3(a.pat.nfar_order, (unsigned)parts), \
                     dim3(nt), (coupling_lds<T, D, NR>(P1, q, single, G, nt)), a.stream, a.rows,  \
                     a.cols, a.pat, a.ip, a.kp, a.nrhs, G, smax, a.mom, a.tlhs, slabs)
    if (q < kWholeSources)
      FMCA_COUPLING(true);
    else
      FMCA_COUPLING(false);
#undef FMCA_COUPLING
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || parts == 1) return e;
  return launch_add_parts<T>(output, a.rows, q, a.nrhs, parts, slabs, a.tlhs, a.out, a.ldo,
                             a.natural, a.stream);
}

template <typename T, int D, int NR>
hipError_t valu_kt(bool output, const ValuLaunch<T> &a) {
  if (a.kp.geodesic) {
    // geodesic entries: FP64 only, the kernel type switched at run time
    if constexpr (sizeof(T) == 8) return valu_launch<T, D, -1, NR, true>(output, a);
    return hipErrorInvalidValue;
  }
  switch (a.kp.kt) {
    case KT_EXPONENTIAL:
      return valu_launch<T, D, KT_EXPONENTIAL, NR, false>(output, a);
    case KT_MATERN32:
      return valu_launch<T, D, KT_MATERN32, NR, false>(output, a);
    case KT_MATERN52:
      return valu_launch<T, D, KT_MATERN52, NR, false>(output, a);
    case KT_GAUSSIAN:
      return valu_launch<T, D, KT_GAUSSIAN, NR, false>(output, a);
    default:
      return valu_launch<T, D, -1, NR, false>(output, a);
  }
}

// LDS of a launch with column tile NR at the largest workgroup.
template <typename T, int D, int NR>
bool valu_fits(bool output, const ValuLaunch<T> &a) {
  const bool single = a.kp.geodesic || a.ip.td;
  return (output ? output_lds<T, D, NR>(a.ip.P1, 256)
                 : coupling_lds<T, D, NR>(a.ip.P1, a.ip.q, single, 1, 256)) <= kValuLds;
}

template <typename T, int D>
hipError_t valu_d(bool output, const ValuLaunch<T> &a) {
  // the smallest column tile that holds the columns, or the largest that fits
  const int n = a.nrhs;
  if (n > 8 && valu_fits<T, D, 32>(output, a)) return valu_kt<T, D, 32>(output, a);
  if (n > 6 && valu_fits<T, D, 8>(output, a)) return valu_kt<T, D, 8>(output, a);
  if (n > 4 && valu_fits<T, D, 6>(output, a)) return valu_kt<T, D, 6>(output, a);
  if (n > 2 && valu_fits<T, D, 4>(output, a)) return valu_kt<T, D, 4>(output, a);
  if (n > 1 && valu_fits<T, D, 2>(output, a)) return valu_kt<T, D, 2>(output, a);
  if (!valu_fits<T, D, 1>(output, a)) return hipErrorInvalidConfiguration;
  return valu_kt<T, D, 1>(output, a);
}

}  // namespace

template <typename T>
hipError_t launch_valu(bool output, const ValuLaunch<T> &a) {
  // these forms evaluate one variant per launch (kp.kt)
  if ((a.kp.vmask & (a.kp.vmask - 1)) != 0) return hipErrorInvalidValue;
  switch (a.rows.dim) {
    case 1:
      return valu_d<T, 1>(output, a);
    case 2:
      return valu_d<T, 2>(output, a);
    case 3:
      return valu_d<T, 3>(output, a);
  }
  return hipErrorInvalidValue;
}

}  // namespace fmca_amd
