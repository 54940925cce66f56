// Vector kernels of the block GCR solve: blocks of up to kBlockCols columns
// that share one Krylov space (actor.cpp, block_gcr_solve).
//
// Vectors are n x nrhs column-major with a leading dimension ld that is a
// multiple of 64; the rows from n on are zero and stay zero, so the kernels
// run over whole tiles.  The columns form block_groups(nrhs) blocks of
// block_cols(nrhs) columns (the last may have fewer).  A basis
// slot holds the orthonormal block Q_j (and P_j with Q_j = (K + ridge I) P_j)
// as S, circular window as in blas1.hip.
//
// All products are tall-skinny matrix products on v_mfma_f64_16x16x4 (lane l
// supplies A[l % 16][l / 16] and B[l / 16][l % 16], result row l / 16 + 4 v):
//   dots      C_j = Q_j^T V          rows of the instruction: columns of Q_j
//   combine   out = in +- sum_j S_j C_j   rows: points
//   apply     Q_k = Y T, R -= Y (T a), and the same for P_k, X
// They read each basis block once per pass and are bound by HBM: at n = 1e6,
// 32 columns, FP32 slots, a slot costs 0.08 ms in the dots and 0.08 ms in the
// combination (about 4.7 TB/s).  One lane loads four consecutive points (16 or
// 32 bytes), which are the four k-steps (dots) or four row tiles (combine,
// apply) of its operand.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device.hpp"

namespace fmca_amd {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kBT = 256;             // threads: 4 waves
constexpr int kCols = kBlockCols;    // 32
constexpr int kMat = kCols * kCols;  // a small matrix, row-major
constexpr int kMatP = 40;            // its padded row stride in LDS

__device__ __forceinline__ d4 mma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <typename S>
__device__ __forceinline__ d4 load4(const S *p) {
  typedef S s4 __attribute__((ext_vector_type(4)));
  const s4 v = *reinterpret_cast<const s4 *>(p);
  return d4{(double)v[0], (double)v[1], (double)v[2], (double)v[3]};
}

// Y = (Y + ridge R) D, W = R D with D = diag(1 / ||r||) of the live columns
// (others become zero, whatever they hold).
__global__ __launch_bounds__(kBT) void k_block_prep(int64_t ld, double ridge,
                                                    const double *__restrict__ r,
                                                    const double *__restrict__ rr,
                                                    const int *__restrict__ live,
                                                    double *__restrict__ y,
                                                    double *__restrict__ w) {
  const int col = blockIdx.y;
  const bool on = live[col] && rr[col] > 0;
  const double d = on ? 1.0 / sqrt(rr[col]) : 0.0;
  const int64_t base = col * ld;
  for (int64_t i = (blockIdx.x * (int64_t)kBT + threadIdx.x) * 4; i < ld;
       i += (int64_t)gridDim.x * kBT * 4) {
    d4 yv = d4{0, 0, 0, 0}, wv = yv;
    if (on) {
      const d4 rv = load4(r + base + i);
      yv = (load4(y + base + i) + rv * ridge) * d;
      wv = rv * d;
    }
    *reinterpret_cast<d4 *>(y + base + i) = yv;
    *reinterpret_cast<d4 *>(w + base + i) = wv;
  }
}

// part[((g * count + j) * chunks + chunk) * kMat + a * 32 + b] = sum over the
// chunk's points of A_j(:, a) B(:, b).  A_j is window block j (tab) or, without
// a table, the FP64 vector a0; B is b1 for j = 1 where given, else b0.
template <typename S, int NT>
__global__ __launch_bounds__(kBT) void k_block_dots(int64_t ld, int nrhs,
                                                    const S *const *__restrict__ tab, int first,
                                                    int cap, const S *__restrict__ a0,
                                                    const double *__restrict__ b0,
                                                    const double *__restrict__ b1, int count,
                                                    double *__restrict__ part) {
  __shared__ double red[4][NT * NT * 256];
  const int j = blockIdx.y, g = blockIdx.z, chunks = gridDim.x;
  const int bs = block_cols(nrhs), c0 = g * bs, s = min(bs, nrhs - c0);
  const S *A = (tab ? tab[(first + j) % cap] : a0) + (int64_t)c0 * ld;
  const double *B = (j == 1 && b1 ? b1 : b0) + (int64_t)c0 * ld;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t blocks = ld / 64;
  const int64_t lo = blocks * blockIdx.x / chunks * 64, hi = blocks * (blockIdx.x + 1) / chunks * 64;
  d4 acc[NT][NT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = d4{0, 0, 0, 0};
  for (int64_t i = lo + wave * 16 + 4 * lk; i < hi; i += 64) {
    d4 av[NT], bv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = 16 * t + lr;
      av[t] = c < s ? load4(A + (int64_t)c * ld + i) : d4{0, 0, 0, 0};
      bv[t] = c < s ? load4(B + (int64_t)c * ld + i) : d4{0, 0, 0, 0};
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) acc[a][b] = mma(av[a][v], bv[b][v], acc[a][b]);
  }
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[wave][(a * 16 + lk + 4 * v) * (16 * NT) + b * 16 + lr] = acc[a][b][v];
  __syncthreads();
  double *dst = part + (((int64_t)g * count + j) * chunks + blockIdx.x) * kMat;
  for (int e = threadIdx.x; e < kMat; e += kBT) {
    const int a = e / kCols, b = e % kCols;
    double v = 0;
    if (a < 16 * NT && b < 16 * NT) {
      const int x = a * (16 * NT) + b;
      v = (red[0][x] + red[1][x]) + (red[2][x] + red[3][x]);
    }
    dst[e] = v;
  }
}

// out[(g * count + j) * kMat + e] = sum over the chunks, zero in the columns
// of inactive right-hand sides.
__global__ __launch_bounds__(kBT) void k_block_dots_final(int nrhs, int count, int chunks,
                                                          const int *__restrict__ active,
                                                          const double *__restrict__ part,
                                                          double *__restrict__ out) {
  const int64_t m = (int64_t)blockIdx.z * count + blockIdx.y;
  const int e = blockIdx.x * kBT + threadIdx.x;
  const int bs = block_cols(nrhs), b = e % kCols, col = (int)blockIdx.z * bs + b;
  double v = 0;
  if (b < bs && col < nrhs && active[col]) {
    const double *p = part + m * chunks * kMat + e;
    for (int k = 0; k < chunks; ++k) v += p[(int64_t)k * kMat];
  }
  out[m * kMat + e] = v;
}

// sq[32 g + b] = sum_j ||C_j(:, b)||^2: the part of the image's squared norm
// that lies in the window.  One workgroup per block, fixed order.
__global__ __launch_bounds__(kBT) void k_block_coef_norms(int count,
                                                          const double *__restrict__ coef,
                                                          double *__restrict__ sq) {
  __shared__ double red[kBT];
  const int g = blockIdx.x;
  const double *c = coef + (int64_t)g * count * kMat;
  double v = 0;
  for (int64_t e = threadIdx.x; e < (int64_t)count * kMat; e += kBT) v += c[e] * c[e];
  red[threadIdx.x] = v;  // column threadIdx.x % 32
  __syncthreads();
  if (threadIdx.x < kCols) {
    double t = 0;
    for (int k = threadIdx.x; k < kBT; k += kCols) t += red[k];
    sq[g * kCols + threadIdx.x] = t;
  }
}

// A tile of 64 points by 32 columns in accumulators: acc[t][b][v] is point
// i0 + 4 (lk + 4 v) + t, column 16 b + lr.
template <int NT>
__device__ __forceinline__ void mul_block(const d4 (&a)[kCols / 4], int ks,
                                          const double *__restrict__ C, int lr, int lk,
                                          d4 (&acc)[4][NT]) {
#pragma unroll
  for (int k = 0; k < kCols / 4; ++k) {
    if (k >= ks) break;
    double b[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b[nt] = C[(4 * k + lk) * kMatP + nt * 16 + lr];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[t][nt] = mma(a[k][t], b[nt], acc[t][nt]);
  }
}

// z = 0: out0 += sign0 sum_j Q_j C_j; z = 1: out1 += sign1 sum_j P_j C_j.
// Columns with active = 0 are left as they are.
template <typename S, int NT>
__global__ __launch_bounds__(kBT, 2) void k_block_combine(
    int64_t ld, int nrhs, const S *const *__restrict__ qtab, const S *const *__restrict__ ptab,
    int first, int count, int cap, const double *__restrict__ coef,
    const int *__restrict__ active, double *__restrict__ out0, double sign0,
    double *__restrict__ out1, double sign1) {
  __shared__ double C[kCols * kMatP];
  const int g = blockIdx.y, bs = block_cols(nrhs), c0 = g * bs, s = min(bs, nrhs - c0);
  const int ks = (s + 3) / 4;
  const S *const *tab = blockIdx.z ? ptab : qtab;
  double *out = (blockIdx.z ? out1 : out0) + (int64_t)c0 * ld;
  const double sign = blockIdx.z ? sign1 : sign0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + wave) * 64;
  const bool on = i0 < ld;  // whole 64-row tiles
  d4 acc[4][NT];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[t][nt] = d4{0, 0, 0, 0};
  for (int j = 0; j < count; ++j) {
    const S *A = tab[(first + j) % cap] + (int64_t)c0 * ld;
    d4 a[kCols / 4];
#pragma unroll
    for (int k = 0; k < kCols / 4; ++k) {
      const int c = 4 * k + lk;
      a[k] = on && c < s ? load4(A + (int64_t)c * ld + i0 + 4 * lr) : d4{0, 0, 0, 0};
    }
    __syncthreads();
    for (int e = threadIdx.x; e < kMat; e += kBT)
      C[(e / kCols) * kMatP + e % kCols] = coef[((int64_t)g * count + j) * kMat + e];
    __syncthreads();
    mul_block<NT>(a, ks, C, lr, lk, acc);
  }
  if (!on) return;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int c = nt * 16 + lr;
    if (c >= s || !active[c0 + c]) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      d4 *p = reinterpret_cast<d4 *>(out + (int64_t)c * ld + i0 + 4 * (lk + 4 * v));
      *p += d4{acc[0][nt][v], acc[1][nt][v], acc[2][nt][v], acc[3][nt][v]} * sign;
    }
  }
}

// mats: per block g the matrices T and T a.  z = 0: qk = Y T, r -= Y (T a);
// z = 1: pk = W T, x += W (T a).  r and x of inactive columns stay.
template <typename S, int NT>
__global__ __launch_bounds__(kBT, 2) void k_block_apply(
    int64_t ld, int nrhs, const double *__restrict__ y, const double *__restrict__ w,
    const double *__restrict__ mats, const int *__restrict__ active, S *__restrict__ qk,
    S *__restrict__ pk, double *__restrict__ r, double *__restrict__ x) {
  typedef S s4 __attribute__((ext_vector_type(4)));
  __shared__ double C[2][kCols * kMatP];
  const int g = blockIdx.y, bs = block_cols(nrhs), c0 = g * bs, s = min(bs, nrhs - c0);
  const int ks = (s + 3) / 4;
  for (int e = threadIdx.x; e < 2 * kMat; e += kBT)
    C[e / kMat][(e % kMat / kCols) * kMatP + e % kCols] = mats[(int64_t)g * 2 * kMat + e];
  const double *A = (blockIdx.z ? w : y) + (int64_t)c0 * ld;
  S *slot = (blockIdx.z ? pk : qk) + (int64_t)c0 * ld;
  double *vec = (blockIdx.z ? x : r) + (int64_t)c0 * ld;
  const double sign = blockIdx.z ? 1.0 : -1.0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + wave) * 64;
  const bool on = i0 < ld;
  d4 a[kCols / 4];
#pragma unroll
  for (int k = 0; k < kCols / 4; ++k) {
    const int c = 4 * k + lk;
    a[k] = on && c < s ? load4(A + (int64_t)c * ld + i0 + 4 * lr) : d4{0, 0, 0, 0};
  }
  __syncthreads();
  if (!on) return;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    d4 acc[4][NT];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[t][nt] = d4{0, 0, 0, 0};
    mul_block<NT>(a, ks, C[m], lr, lk, acc);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int c = nt * 16 + lr;
      if (c >= s) continue;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t at = (int64_t)c * ld + i0 + 4 * (lk + 4 * v);
        const d4 z = d4{acc[0][nt][v], acc[1][nt][v], acc[2][nt][v], acc[3][nt][v]};
        if (m == 0)
          *reinterpret_cast<s4 *>(slot + at) = s4{(S)z[0], (S)z[1], (S)z[2], (S)z[3]};
        else if (active[c0 + c])
          *reinterpret_cast<d4 *>(vec + at) += z * sign;
      }
    }
  }
}

// point chunks of a dots launch: about 2048 workgroups in all
int dot_chunks(int64_t ld, int nrhs, int count) {
  const int64_t want = std::max<int64_t>(8, 2048 / std::max(1, count * block_groups(nrhs)));
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(want, 512), ld / 64));
}

template <typename S>
hipError_t dots(int64_t ld, int nrhs, const S *const *tab, int first, int cap, const S *a0,
                const double *b0, const double *b1, int count, const int *active, double *out,
                double *scratch, hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  const int chunks = dot_chunks(ld, nrhs, count), ng = block_groups(nrhs);
  const dim3 grid(chunks, count, ng);
  if (nrhs <= 16)
    hipLaunchKernelGGL((k_block_dots<S, 1>), grid, dim3(kBT), 0, stream, ld, nrhs, tab, first, cap,
                       a0, b0, b1, count, scratch);
  else
    hipLaunchKernelGGL((k_block_dots<S, 2>), grid, dim3(kBT), 0, stream, ld, nrhs, tab, first, cap,
                       a0, b0, b1, count, scratch);
  hipLaunchKernelGGL(k_block_dots_final, dim3(kMat / kBT, count, ng), dim3(kBT), 0, stream, nrhs,
                     count, chunks, active, scratch, out);
  return hipGetLastError();
}

}  // namespace

size_t block_scratch(int64_t ld, int nrhs, int count) {
  size_t most = 0;  // over the window sizes up to `count`
  for (int k = 1; k <= std::max(2, count); ++k)
    most = std::max(most, (size_t)dot_chunks(ld, nrhs, k) * k);
  return most * block_groups(nrhs) * kMat * sizeof(double);
}

hipError_t block_prep(int64_t ld, int nrhs, double ridge, const double *r, const double *rr,
                      const int *live, double *y, double *w, hipStream_t stream) {
  const int64_t g = std::max<int64_t>(1, std::min<int64_t>((ld / 4 + kBT - 1) / kBT, 512));
  hipLaunchKernelGGL(k_block_prep, dim3((unsigned)g, nrhs), dim3(kBT), 0, stream, ld, ridge, r, rr,
                     live, y, w);
  return hipGetLastError();
}

template <typename S>
hipError_t block_dots(int64_t ld, int nrhs, const double *v, const S *const *qtab, int first,
                      int count, int cap, const int *active, double *out, double *scratch,
                      hipStream_t stream) {
  return dots<S>(ld, nrhs, qtab, first, cap, nullptr, v, nullptr, count, active, out, scratch,
                 stream);
}

hipError_t block_coef_norms(int nrhs, int count, const double *coef, double *sq,
                            hipStream_t stream) {
  hipLaunchKernelGGL(k_block_coef_norms, dim3(block_groups(nrhs)), dim3(kBT), 0, stream, count,
                     coef, sq);
  return hipGetLastError();
}

hipError_t block_gram(int64_t ld, int nrhs, const double *y, const double *r, const int *active,
                      double *out, double *scratch, hipStream_t stream) {
  return dots<double>(ld, nrhs, nullptr, 0, 1, y, y, r, 2, active, out, scratch, stream);
}

template <typename S>
hipError_t block_combine(int64_t ld, int nrhs, const S *const *qtab, const S *const *ptab,
                         int first, int count, int cap, const double *coef, const int *active,
                         double *out0, double sign0, double *out1, double sign1,
                         hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  const dim3 grid((unsigned)((ld / 64 + 3) / 4), block_groups(nrhs), 2);
  if (nrhs <= 16)
    hipLaunchKernelGGL((k_block_combine<S, 1>), grid, dim3(kBT), 0, stream, ld, nrhs, qtab, ptab,
                       first, count, cap, coef, active, out0, sign0, out1, sign1);
  else
    hipLaunchKernelGGL((k_block_combine<S, 2>), grid, dim3(kBT), 0, stream, ld, nrhs, qtab, ptab,
                       first, count, cap, coef, active, out0, sign0, out1, sign1);
  return hipGetLastError();
}

template <typename S>
hipError_t block_apply(int64_t ld, int nrhs, const double *y, const double *w, const double *mats,
                       const int *active, S *qk, S *pk, double *r, double *x, hipStream_t stream) {
  const dim3 grid((unsigned)((ld / 64 + 3) / 4), block_groups(nrhs), 2);
  if (nrhs <= 16)
    hipLaunchKernelGGL((k_block_apply<S, 1>), grid, dim3(kBT), 0, stream, ld, nrhs, y, w, mats,
                       active, qk, pk, r, x);
  else
    hipLaunchKernelGGL((k_block_apply<S, 2>), grid, dim3(kBT), 0, stream, ld, nrhs, y, w, mats,
                       active, qk, pk, r, x);
  return hipGetLastError();
}

#define FMCA_BLOCK_INST(S)                                                                      \
  template hipError_t block_dots<S>(int64_t, int, const double *, const S *const *, int, int,   \
                                    int, const int *, double *, double *, hipStream_t);         \
  template hipError_t block_combine<S>(int64_t, int, const S *const *, const S *const *, int,   \
                                       int, int, const double *, const int *, double *, double, \
                                       double *, double, hipStream_t);                          \
  template hipError_t block_apply<S>(int64_t, int, const double *, const double *,              \
                                     const double *, const int *, S *, S *, double *, double *, \
                                     hipStream_t);
FMCA_BLOCK_INST(double)
FMCA_BLOCK_INST(float)
#undef FMCA_BLOCK_INST

}  // namespace fmca_amd
