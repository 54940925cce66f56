// Matrix-core contractions of the FP32 precision form on BF16 inputs.
//
// The kernel entries are evaluated in FP32, from squared distances that the BF16
// matrix cores form from three-term splits (24 bits, see source_operand; the
// leaf output of kernels with a cusp at 0: from FP32 differences), and so are the
// right operands (rhs rows, moments).  Each
// FP32 operand v is split into two BF16 terms, hi = bf16(v) (round to nearest
// even) and lo = bf16(v - hi), and a product a.b is formed as
//     a_hi.b_hi + a_lo.b_hi + a_hi.b_lo
// with v_mfma_f32_16x16x32_bf16 and FP32 accumulation.  The dropped terms are
// of relative size 2^-16 (a_lo.b_lo and the remainders of the splits), so a
// product carries about the error of an FP32 evaluation of the entry; the sum
// accumulates in FP32 as in the FP32 forms.  One 16x16x32 BF16 instruction
// does 8 times the multiply-adds of a 16x16x4 FP32 one in half the cycles, so
// the three of them cost 3/16 of the FP32 matrix-core time per entry.  The
// squared distances come from the same instruction on three-term splits (24
// bits, see source_operand).
//
// Used where leaves and node sets are large enough (bf16_pays); the FP32 form
// takes the others.
//
// What bounds them: the vector ALU work of an entry (root, exponential,
// polynomial, split: about 60 cycles per 64 entries) plus the part of the
// matrix-core time that it does not hide.  Measured (ms, n = 1e6, MATERN32,
// degree 4; before: FP32 distance MFMAs, four row tiles on each of four waves
// at two waves per SIMD, 32 columns a pass):
//   columns            16             32             64
//   leaf output   7.29 -> 6.52   8.44 -> 7.70   16.6 -> 12.9
//   coupling      5.14 -> 4.65   6.60 -> 5.76   13.2 -> 11.0
//
// Operand layout (gfx950): lane l supplies A[l % 16][k] and B[k][l % 16] for
// the eight k of K-slot group l / 16; the two operands use the same k <-> (lane
// group, element) map, so the contraction pairs them whatever that map is.
// Lane l's eight A values are this lane's row and eight sources (or source
// nodes) of the K-step, in the order of gram_pos where the distances come from
// the matrix cores; B is read as 16 bytes from LDS, where the staged right
// operand is held transposed (column-major over sources).  The accumulator
// layout is that of the 16x16 FP32 forms: item v of lane l is
// C[4 (l / 16) + v][l % 16].
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "device.hpp"
#include "device_math.hpp"

namespace fmca_amd {

namespace {

using namespace dev;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16;

constexpr int kWaves = 8;                // waves per workgroup
constexpr int kThreads = 64 * kWaves;
// Row tiles per wave: two, so that four waves share a SIMD (128 registers).
// With four tiles and two waves the entries' transcendentals, the distance
// MFMAs and the LDS reads were exposed (n = 1e6, 32 rhs: leaf output 8.4 ms).
constexpr int kRT = 2;                   // 16-row tiles per wave -> 256 rows per pass
constexpr int kRows = kWaves * kRT * 16;
constexpr int kRowsP = kRows + 16;       // padded LDS row stride of the basis factors
constexpr int kKB = 32;                  // sources per BF16 K-step
constexpr int kChunk = 128;              // sources / nodes staged per chunk
constexpr int kChunkP = kChunk + 8;      // LDS stride of a transposed column (bf16)
constexpr int kFarChunk = 64;            // moments staged per chunk of the far output

__device__ __forceinline__ f32x4 mma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 splat4(float v) { return f32x4{v, v, v, v}; }

// The part of a task's list that this workgroup takes (grid.y parts).
__device__ __forceinline__ void list_part(int &lo, int &hi) {
  if (gridDim.y == 1) return;
  const int64_t cnt = hi - lo;
  const int lo0 = lo;
  lo = lo0 + (int)(cnt * blockIdx.y / gridDim.y);
  hi = lo0 + (int)(cnt * (blockIdx.y + 1) / gridDim.y);
}

__device__ __forceinline__ int unpack(int p, int d) { return (p >> (8 * d)) & 0xff; }

// hi = bf16(v) rounded to nearest even, lo = bf16(v - hi)
__device__ __forceinline__ void split_bf16(float v, u16 &hi, u16 &lo) {
  const __bf16 h = (__bf16)v;
  const float hf = (float)h;
  const __bf16 l = (__bf16)(v - hf);
  hi = __builtin_bit_cast(u16, h);
  lo = __builtin_bit_cast(u16, l);
}

// Pairs: one packed conversion gives both high parts, whose FP32 values are
// the two 16-bit halves shifted into place (no second conversion).
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8 &hi, bf16x8 &lo) {
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    const __bf16 h0 = (__bf16)v[i], h1 = (__bf16)v[i + 1];
    hi[i] = h0;
    hi[i + 1] = h1;
    const uint32_t u = (uint32_t)__builtin_bit_cast(u16, h0) |
                       ((uint32_t)__builtin_bit_cast(u16, h1) << 16);
    const float f0 = __builtin_bit_cast(float, u << 16);
    const float f1 = __builtin_bit_cast(float, u & 0xffff0000u);
    lo[i] = (__bf16)(v[i] - f0);
    lo[i + 1] = (__bf16)(v[i + 1] - f1);
  }
}

// Lane l of the distance MFMA's output holds sources 4 (l / 16) + v of each
// 16-source half of a K-step; the BF16 contraction reads k-slots
// 8 (l / 16) .. + 7, so source s of a 32-block is staged at this position.
__device__ __forceinline__ int gram_pos(int jj) {
  return (jj & ~31) | (((jj & 15) >> 2) << 3) | ((jj & 16) >> 2) | (jj & 3);
}

// The hi | lo << 16 words of two neighbouring sources (even position at) as one
// 32-bit store to each of the two staged halves.
__device__ __forceinline__ void store_pair(u16 *h, u16 *l, int at, float w0, float w1) {
  const uint32_t a = __builtin_bit_cast(uint32_t, w0), b = __builtin_bit_cast(uint32_t, w1);
  *reinterpret_cast<uint32_t *>(h + at) = (a & 0xffffu) | (b << 16);
  *reinterpret_cast<uint32_t *>(l + at) = (a >> 16) | (b & 0xffff0000u);
}

// the 8 bf16 values at p (16-byte aligned) as one operand
__device__ __forceinline__ bf16x8 load8(const u16 *p) {
  return *reinterpret_cast<const bf16x8 *>(p);
}

// In-place BF16 split of the right operands of one action (the permuted rhs
// before the leaf output, the source moments before the coupling): x[i]
// becomes hi | lo << 16, so the staging loops copy the two halves instead
// of splitting every value again for every target that reads it.
__global__ __launch_bounds__(256) void k_split_inplace(float *__restrict__ x, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    u16 h, l;
    split_bf16(x[i], h, l);
    x[i] = __builtin_bit_cast(float, (uint32_t)h | ((uint32_t)l << 16));
  }
}

// Waves per SIMD: 4 up to 32 columns; 64 columns hold twice the accumulators
// (leaf output n = 1e6, 64 columns: 12.9 ms at 2, 21 ms with spills at 4).
template <int NT>
constexpr int kOcc = NT <= 2 ? 4 : 2;

// K-split of R row tiles: with fewer than 9 tiles, groups of waves share the
// K-steps, at most four groups, as a chunk has four; so that no wave holds more
// than kRT row tiles, and one where there are at most two.  The groups' sums
// are added in LDS in group order.  wave = rg + wrows sg.  Against no split
// (us, 16 / 64 columns): leaf output of 49 rows (3-D degree 2, n = 2e5) 709 /
// 1945 against 878 / 2810, coupling of q = 64 (3-D degree 3, n = 2e5) 610 / 2093
// against 817 / 3080.
__device__ __forceinline__ int k_split(int R) {
  return R <= 2 * kRT ? 4 : (R <= 4 * kRT ? 2 : 1);
}

// Adds the wave groups' accumulators over LDS; the sums end in group 0.
// Red: [16 R][16 NT] (R <= 8: at most the staged right operand's room).
template <int NT>
__device__ __forceinline__ void add_groups(f32x4 (&acc)[kRT][NT], float *Red, int kspl, int wrows,
                                           int rg, int sg, const bool (&tile_on)[kRT], int lr,
                                           int lk) {
  for (int g = 1; g <= kspl; ++g) {
    __syncthreads();
    if (sg != g % kspl) continue;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        if (!tile_on[rt]) continue;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float *dst = Red + (((rg + wrows * rt) * 16 + 4 * lk + v) * NT + nt) * 16 + lr;
          const float sum = (g == 1 ? 0.f : *dst) + acc[rt][nt][v];
          if (g < kspl)
            *dst = sum;
          else
            acc[rt][nt][v] = sum;
        }
      }
  }
}

// acc += A B for one K-step: A = ah + al per row tile, B = Bh + Bl (LDS) per
// column tile, the three leading products.
template <int NT, bool ALL>
__device__ __forceinline__ void contract(const bf16x8 (&ah)[kRT], const bf16x8 (&al)[kRT],
                                         const u16 *Bh, const u16 *Bl,
                                         const bool (&tile_on)[kRT], int ntl,
                                         f32x4 (&acc)[kRT][NT]) {
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (!ALL && nt >= ntl) continue;
    const bf16x8 bh = load8(Bh + nt * 16 * kChunkP), bl = load8(Bl + nt * 16 * kChunkP);
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt)
      if (ALL || tile_on[rt]) acc[rt][nt] = mma_bf16(ah[rt], bh, acc[rt][nt]);
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt)
      if (ALL || tile_on[rt]) acc[rt][nt] = mma_bf16(al[rt], bh, acc[rt][nt]);
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt)
      if (ALL || tile_on[rt]) acc[rt][nt] = mma_bf16(ah[rt], bl, acc[rt][nt]);
  }
}

// Distance operands.  r^2 = |y|^2 - 2 x.y + |x|^2 of 16 sources and 16 targets
// comes from one v_mfma_f32_16x16x32_bf16: every coordinate and squared norm is
// split into three BF16 terms (24 bits), and its k-slots hold 24 products, per
// axis those down to 2^-16 (y1x1; y1x2 y2x1; y2x2 y1x3 y3x1), |y|^2 against 1 and
// 1 against |x|^2; the last eight are zero on the target side.  The instruction
// drops what lies below the last place of its running sum, so the products
// stand in rising order.  Error of r^2 in units of 2^-24 (|x|^2 + |y|^2), rms,
// sources around the targets / one / three box widths off: 0.75 / 0.80 / 0.93
// (mean -0.2 to -0.3), axis by axis 0.90 / 0.93 / 1.04, v_mfma_f32_16x16x4 0.84 /
// 0.82 / 0.77, whose 41 cycles do not overlap with the vector ALU (19 cycles here,
// partly hidden).  y2x3 and y3x2 in the free slots change no bit; 32 slots with
// zeros between the orders give 0.72 / 0.76 / 0.86 and a leaf output of 8.0
// instead of 7.8 ms (n = 1e6, 32 columns).  The split of the entries and right
// operands dominates the action's error: 4.1e-6 at n = 5e4, 32 columns, in every
// one of these layouts (4.4e-6 with the FP32 instruction and its order of sums).
struct Split3 {
  __bf16 t[3];
  __device__ __forceinline__ explicit Split3(float v) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      t[i] = (__bf16)v;
      v -= (float)t[i];
    }
  }
};
constexpr int kDistGroups = 3;         // eight k-slots each; the fourth group is zero
constexpr int kSlot[3] = {19, 11, 0};  // first slot of the products of 1, 2^-8, 2^-16

// The k-slots of the source operand (SOURCE: of -2 y' and |y'|^2) or of the
// target operand (of x' and |x'|^2).
template <int D, bool SOURCE>
__device__ __forceinline__ void distance_slots(const float (&v)[D], float s2, __bf16 (&k)[24]) {
  const __bf16 one = (__bf16)1.f;
#pragma unroll
  for (int i = 0; i < 24; ++i) k[i] = (__bf16)0.f;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const Split3 u(v[d]);
    k[kSlot[0] + d] = u.t[0];
    k[kSlot[1] + 2 * d] = u.t[SOURCE ? 0 : 1];
    k[kSlot[1] + 2 * d + 1] = u.t[SOURCE ? 1 : 0];
    k[kSlot[2] + 3 * d] = u.t[1];
    k[kSlot[2] + 3 * d + 1] = u.t[SOURCE ? 0 : 2];
    k[kSlot[2] + 3 * d + 2] = u.t[SOURCE ? 2 : 0];
  }
  const Split3 u(s2);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int at = kSlot[i] + (i == 0 ? 3 : (i == 1 ? 6 : 9));
    k[at + (SOURCE ? 0 : 1)] = u.t[i];
    k[at + (SOURCE ? 1 : 0)] = one;
  }
}

// the source operand of -2 y' and |y'|^2: group g of this source
template <int D>
__device__ __forceinline__ void source_operand(const float (&y)[D], float s2,
                                               bf16x8 (&out)[kDistGroups]) {
  __bf16 a[24];
  distance_slots<D, true>(y, s2, a);
#pragma unroll
  for (int g = 0; g < kDistGroups; ++g)
#pragma unroll
    for (int i = 0; i < 8; ++i) out[g][i] = a[8 * g + i];
}

// the target operand of x' and |x'|^2: the k-slots of lane group lk
template <int D>
__device__ __forceinline__ bf16x8 target_operand(const float (&x)[D], float s2, int lk) {
  __bf16 b[24];
  distance_slots<D, false>(x, s2, b);
  bf16x8 out;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    out[i] = lk == 0 ? b[i] : (lk == 1 ? b[8 + i] : (lk == 2 ? b[16 + i] : (__bf16)0.f));
  return out;
}

// One K-step of 32 sources for the row tiles of a wave, distances from the
// matrix cores: ya, yb are this lane's source operands of the two 16-source
// halves, xb its target operands, Bh, Bl the right operands.
template <int KT, int NT, bool ALL>
__device__ __forceinline__ void gram_step(bf16x8 ya, bf16x8 yb, const u16 *Bh, const u16 *Bl,
                                          const bf16x8 (&xb)[kRT], const bool (&tile_on)[kRT], int ntl,
                                          const KernelParams<float> &kp, f32x4 (&acc)[kRT][NT]) {
  // the entries of every row tile first, then the right operands one column
  // tile at a time: few registers are live at once
  bf16x8 ah[kRT], al[kRT];
#pragma unroll
  for (int rt = 0; rt < kRT; ++rt) {
    if (!ALL && !tile_on[rt]) continue;
    const f32x4 g0 = mma_bf16(ya, xb[rt], splat4(0.f));
    const f32x4 g1 = mma_bf16(yb, xb[rt], splat4(0.f));
    float ev[8];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      ev[v] = gram_kernel<KT>(g0[v], kp);
      ev[4 + v] = gram_kernel<KT>(g1[v], kp);
    }
    split8(ev, ah[rt], al[rt]);
  }
  contract<NT, ALL>(ah, al, Bh, Bl, tile_on, ntl, acc);
}

// ---------------------------------------------------------------------------
// Leaf output: one workgroup per target-leaf task, 8 waves, each wave owns row
// tiles {rg, rg + wrows} of the current 256-row pass and 16 NT rhs columns.
// Far field: A = V_t^T (rows x q) on FP32 MFMA as in the FP32 form (a small
// share of the work); near field on BF16 MFMA.
template <int D, int KT, int NT>
__global__ __launch_bounds__(kThreads, kOcc<NT>) void k_leaf_output_bf16(
    DevTreeView<float> rows, DevTreeView<float> cols, DevPatternView pat,
    InterpParams<float> ip, KernelParams<float> kp, int nrhs, const float *__restrict__ xs,
    const float *__restrict__ tlhs, double *__restrict__ out, int64_t ldo, int natural,
    float *__restrict__ part) {
  constexpr int NC = 16 * NT;
  constexpr int NCP = NC + 16;  // padded stride of the staged far moments
  constexpr bool kGram = kGramNear<KT>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int P1 = ip.P1, q = ip.q;
  const int qpad = (q + 3) & ~3;
  float *F = reinterpret_cast<float *>(smem_raw);               // [D][P1][kRowsP]
  int *aidx = reinterpret_cast<int *>(F + D * P1 * kRowsP);     // [qpad] packed indices
  float *Un = reinterpret_cast<float *>(aidx + ((qpad + 3) & ~3));  // union region
  float *Ms = Un;                                  // far: [kFarChunk][NCP] moments
  // near: [D][kChunk] source points, or with kGram [kDistGroups][kChunk]
  // distance operands of the sources
  float *Ys = Un;
  bf16x8 *Yd = reinterpret_cast<bf16x8 *>(Un);
  u16 *Xh = reinterpret_cast<u16 *>(Yd + kDistGroups * kChunk);  // near: [NC][kChunkP] rhs, hi
  u16 *Xl = Xh + NC * kChunkP;                         // near: [NC][kChunkP] rhs, lo
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int task = pat.near_order[blockIdx.x];
  if (task < 0) return;
  const int li = pat.near_task[4 * task], flags = pat.near_task[4 * task + 3];
  int n0 = pat.near_task[4 * task + 1], n1 = pat.near_task[4 * task + 2];
  const bool split = (flags & kTaskSplit) != 0;
  const bool do_far = (flags & kTaskFar) != 0 && pat.has_far && blockIdx.y == 0;
  list_part(n0, n1);
  const int c = rows.leaves[li];
  const int b0 = rows.begin[c], sz = rows.size[c];
  for (int e = threadIdx.x; e < qpad; e += kThreads)
    aidx[e] = basis_index<float, D>(e < q ? e : 0, ip);
  for (int pbase = 0; pbase < sz; pbase += kRows) {
    __syncthreads();
    if (do_far && threadIdx.x < kRows) {
      const int i = pbase + threadIdx.x;
      if (i < sz) {
#pragma unroll
        for (int d = 0; d < D; ++d)
          basis_1d<float>(rows.unit[(int64_t)d * rows.npts + b0 + i], ip,
                          F + (d * P1) * kRowsP + threadIdx.x, kRowsP);
      } else {
        for (int d = 0; d < D; ++d)
          for (int a = 0; a < P1; ++a) F[(d * P1 + a) * kRowsP + threadIdx.x] = 0.f;
      }
    }
    const int R = (min(kRows, sz - pbase) + 15) / 16;
    const int kspl = k_split(R), wrows = kWaves / kspl, rg = wave % wrows, sg = wave / wrows;
    float x[kRT][D];
    bool tile_on[kRT];
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) {
      const int tile_row0 = pbase + (rg + wrows * rt) * 16;
      tile_on[rt] = tile_row0 < sz;
      const int i = tile_row0 + lr;
#pragma unroll
      for (int d = 0; d < D; ++d)
        x[rt][d] = i < sz ? rows.pts[(int64_t)d * rows.npts + b0 + i] : 0.f;
    }
    // distance operands of the targets, x' = sigma (x - centre of the leaf)
    float ctr[D];
    bf16x8 xb[kRT];
    const float sig = gram_sigma<KT>(kp);
#pragma unroll
    for (int d = 0; d < D; ++d)
      ctr[d] = rows.bbmin[(int64_t)c * D + d] + 0.5f * rows.bbsize[(int64_t)c * D + d];
    if constexpr (kGram) {
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        float s2 = 0.f, v[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          v[d] = (x[rt][d] - ctr[d]) * sig;
          s2 = fmat(v[d], v[d], s2);
        }
        xb[rt] = target_operand<D>(v, s2, lk);
      }
    }
    for (int rc = 0; rc < nrhs; rc += NC) {
      f32x4 acc[kRT][NT];
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = f32x4{0, 0, 0, 0};
      const int ntl = min(NT, (nrhs - rc + 15) >> 4);
      // far field (first task of the leaf): FP32 MFMA, K-steps of 4 moments
      for (int a0 = 0; do_far && a0 < qpad; a0 += kFarChunk) {
        const int na = min(kFarChunk, qpad - a0);
        __syncthreads();
        for (int e = threadIdx.x; e < kFarChunk * NC; e += kThreads) {
          const int al = e / NC, r = e % NC;
          const int alpha = a0 + al;
          Ms[al * NCP + r] = (alpha < q && rc + r < nrhs)
                                 ? tlhs[((int64_t)c * q + alpha) * nrhs + rc + r]
                                 : 0.f;
        }
        __syncthreads();
        for (int ks = 4 * sg; ks < na; ks += 4 * kspl) {
          const int al = ks + lk;
          const int pk = aidx[a0 + al];
          float b[NT];
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) b[nt] = Ms[al * NCP + nt * 16 + lr];
#pragma unroll
          for (int rt = 0; rt < kRT; ++rt) {
            if (!tile_on[rt]) continue;
            const int row = (rg + wrows * rt) * 16 + lr;
            float v = F[(0 * P1 + unpack(pk, 0)) * kRowsP + row];
#pragma unroll
            for (int d = 1; d < D; ++d) v *= F[(d * P1 + unpack(pk, d)) * kRowsP + row];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
              if (nt < ntl) acc[rt][nt] = mma_f32(v, b[nt], acc[rt][nt]);
          }
        }
      }
      // near field: chunks of kChunk sources fetched one chunk ahead into
      // registers, staged as coordinates Ys and the BF16 split of the rhs
      // (a thread takes two neighbouring sources of a column: 32-bit stores)
      constexpr int KX = kChunk * NC / (2 * kThreads);  // rhs pairs per thread
      // coordinates per thread: with kGram thread jj < kChunk loads all D of
      // source jj (its row of the distance operand needs |y'|^2)
      constexpr int KY = kGram ? D : (D * kChunk + kThreads - 1) / kThreads;
      static_assert(kChunk * NC % (2 * kThreads) == 0, "staging layout");
      static_assert(kChunk <= kThreads, "one source per thread in the distance staging");
      float py[KY], px[KX][2];
      int nb = n0, j0 = 0, pnj = 0;
      auto fetch = [&]() {
        const int run = min(pat.near_run[nb], n1 - nb);
        const int s = pat.near_src[nb], sl = pat.near_src[nb + run - 1];
        const int sb = cols.begin[s], ss = cols.begin[sl] + cols.size[sl] - sb;
        pnj = min(kChunk, ss - j0);
        if constexpr (kGram) {
          const int jj = threadIdx.x;
#pragma unroll
          for (int d = 0; d < D; ++d) {  // padding sources sit at the centre
            const float *pt = cols.pts + ((int64_t)d * cols.npts + sb + j0);
            py[d] = (jj < kChunk && jj < pnj) ? pt[(uint32_t)jj] : ctr[d];
          }
        } else {
#pragma unroll
          for (int k = 0; k < KY; ++k) {
            const int e = threadIdx.x + kThreads * k;
            const int d = e / kChunk, jj = e % kChunk;
            py[k] = (e < D * kChunk && jj < pnj)
                        ? cols.pts[(int64_t)d * cols.npts + sb + j0 + jj]
                        : 0.f;
          }
        }
        // a uniform base and 32-bit offsets: no 64-bit address per load
        const float *xt = xs + ((int64_t)(sb + j0) * nrhs + rc);
        const int pr = threadIdx.x % NC, pj = 2 * (threadIdx.x / NC);
#pragma unroll
        for (int k = 0; k < KX; ++k) {
          const int jj = pj + 2 * (kThreads / NC) * k;
#pragma unroll
          for (int u = 0; u < 2; ++u)
            px[k][u] = (jj + u < pnj && rc + pr < nrhs)
                           ? xt[(uint32_t)((jj + u) * nrhs + pr)]
                           : 0.f;
        }
        j0 += kChunk;
        if (j0 >= ss) {
          nb += run;
          j0 = 0;
        }
      };
      bool more = nb < n1;
      if (more) fetch();
      while (more) {
        const int nj = pnj;
        __syncthreads();
        if constexpr (kGram) {
          const int jj = threadIdx.x;
          if (jj < kChunk) {
            float s2 = 0.f, v[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
              v[d] = (py[d] - ctr[d]) * sig;
              s2 = fmat(v[d], v[d], s2);
              v[d] *= -2.f;
            }
            bf16x8 op[kDistGroups];
            source_operand<D>(v, s2, op);
#pragma unroll
            for (int g = 0; g < kDistGroups; ++g) Yd[g * kChunk + jj] = op[g];
          }
        } else {
#pragma unroll
          for (int k = 0; k < KY; ++k) {
            const int e = threadIdx.x + kThreads * k;
            if (e < D * kChunk) Ys[e] = py[k];
          }
        }
#pragma unroll
        for (int k = 0; k < KX; ++k) {
          const int e = threadIdx.x + kThreads * k;
          const int jj = 2 * (e / NC), r = e % NC;
          store_pair(Xh, Xl, r * kChunkP + (kGram ? gram_pos(jj) : jj), px[k][0], px[k][1]);
        }
        __syncthreads();
        more = nb < n1;
        if (more) fetch();
        const int nsteps = (nj + kKB - 1) & ~(kKB - 1);
        // all row tiles valid and all column tiles used (the common case): no
        // branches in a K-step, one basic block for the scheduler
        bool all_on = ntl == NT;
#pragma unroll
        for (int rt = 0; rt < kRT; ++rt) all_on = all_on && tile_on[rt];
        if constexpr (kGram) {
          const int gl = min(lk, kDistGroups - 1);  // group 3: zero in xb
          auto steps = [&](auto all_t) {
            for (int ks = kKB * sg; ks < nsteps; ks += kKB * kspl) {
              const int off = lr * kChunkP + ks + 8 * lk;  // this lane group's eight k-slots
              gram_step<KT, NT, decltype(all_t)::value>(
                  Yd[gl * kChunk + ks + lr], Yd[gl * kChunk + ks + 16 + lr], Xh + off, Xl + off,
                  xb, tile_on, ntl, kp, acc);
            }
          };
          if (all_on)
            steps(std::true_type{});
          else
            steps(std::false_type{});
        } else {
          // kernels with a cusp at r = 0: differences on the VALU
          auto steps = [&](auto all_t) {
            constexpr bool ALL = decltype(all_t)::value;
            for (int ks = kKB * sg; ks < nsteps; ks += kKB * kspl) {
              const int j8 = ks + 8 * lk;  // this lane group's eight sources
              float y[D][8];
#pragma unroll
              for (int d = 0; d < D; ++d)
#pragma unroll
                for (int i = 0; i < 8; ++i) y[d][i] = Ys[d * kChunk + j8 + i];
              bf16x8 ah[kRT], al[kRT];
#pragma unroll
              for (int rt = 0; rt < kRT; ++rt) {
                if (!ALL && !tile_on[rt]) continue;
                float ev[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                  float r2 = 0.f;
#pragma unroll
                  for (int d = 0; d < D; ++d) {
                    const float dd = x[rt][d] - y[d][i];
                    r2 = fmat(dd, dd, r2);
                  }
                  ev[i] = kernel_r2<KT, float>(r2, kp);
                }
                split8(ev, ah[rt], al[rt]);
              }
              const int off = lr * kChunkP + j8;
              contract<NT, ALL>(ah, al, Xh + off, Xl + off, tile_on, ntl, acc);
            }
          };
          if (all_on && KT >= 0)
            steps(std::true_type{});
          else
            steps(std::false_type{});
        }
      }
      if (kspl > 1) add_groups<NT>(acc, Un, kspl, wrows, rg, sg, tile_on, lr, lk);
      // store: C row 4 lk + v of tile (rg + wrows rt), column lr of rhs tile nt
#pragma unroll
      for (int rt = 0; rt < kRT; ++rt) {
        if (!tile_on[rt] || sg != 0) continue;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int col = rc + nt * 16 + lr;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int i = pbase + (rg + wrows * rt) * 16 + 4 * lk + v;
            if (i < sz && col < nrhs) {
              if (gridDim.y > 1) {
                part[((int64_t)blockIdx.y * rows.npts + b0 + i) * nrhs + col] = acc[rt][nt][v];
                continue;
              }
              const int64_t row = natural ? (int64_t)rows.perm[b0 + i] : (int64_t)(b0 + i);
              double *p = out + row + (int64_t)col * ldo;
              if (split)
                atomic_accumulate(p, (double)acc[rt][nt][v]);
              else
                *p = (double)acc[rt][nt][v];
            }
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Coupling: one workgroup per target-cluster task; rows = the q target nodes
// (tiles of 16, kRT per wave, q <= 256), K = the nodes of the far sources in
// K-steps of 32, N = 16 NT rhs columns.  A chunk of kChunk rows holds
// G = kChunk / qpad whole sources when that is 2 or more, else kChunk nodes of
// one source; rows past a source's q nodes or past the list carry zero
// moments.  With fewer than 9 row tiles the waves split the K-steps too.
template <int D, int KT, int NT>
__global__ __launch_bounds__(kThreads, kOcc<NT>) void k_coupling_bf16(
    DevTreeView<float> rows, DevTreeView<float> cols, DevPatternView pat,
    InterpParams<float> ip, KernelParams<float> kp, int nrhs, const float *__restrict__ mom,
    float *__restrict__ tlhs, float *__restrict__ part) {
  constexpr int NC = 16 * NT;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int q = ip.q;
  const int qpad = (q + 3) & ~3;
  float *U = reinterpret_cast<float *>(smem_raw);  // [D][qpad] unit node coordinates
  // [kDistGroups][kChunk] distance operands of the sources, y' = node - centre
  // of the target cluster.  Far blocks are separated (dist >= radius / eta), so
  // the cancellation in |y'|^2 - 2 x'.y' + |x'|^2 stays near the rounding of the
  // direct form.
  bf16x8 *Yd = reinterpret_cast<bf16x8 *>(U + D * qpad);  // qpad floats: 16-byte aligned
  u16 *Mh = reinterpret_cast<u16 *>(Yd + kDistGroups * kChunk);  // [NC][kChunkP] moments, hi
  u16 *Ml = Mh + NC * kChunkP;                         // [NC][kChunkP] moments, lo
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int task = pat.far_order[blockIdx.x];
  if (task < 0) return;
  const int t = pat.far_task[4 * task];
  int f0 = pat.far_task[4 * task + 1], f1 = pat.far_task[4 * task + 2];
  list_part(f0, f1);
  // sums of this part: its slab, or the coupling sums themselves
  float *dst_all = gridDim.y > 1 ? part + (int64_t)blockIdx.y * rows.ncl * ip.q * nrhs : tlhs;
  const bool split = (pat.far_task[4 * task + 3] & kTaskSplit) != 0;
  const int kspl = k_split((q + 15) / 16), wrows = kWaves / kspl, rg = wave % wrows,
            sg = wave / wrows;
  const int G = max(1, kChunk / qpad);
  const float rqpad = 1.0f / (float)qpad;  // bl / qpad = floor((bl + 0.5) / qpad), bl < 256
  for (int e = threadIdx.x; e < D * qpad; e += kThreads) {
    const int d = e / qpad, b = e - d * qpad, bb = b < q ? b : 0;
    U[e] = ip.td ? ip.unodes[d * q + bb] : ip.xi[unpack(basis_index<float, D>(bb, ip), d)];
  }
  float ctr[D];
  bf16x8 xb[kRT];  // distance operands of the target nodes
  const float sig = gram_sigma<KT>(kp);
  const int gl = min(lk, kDistGroups - 1);  // group 3: zero in xb
  bool tile_on[kRT];
#pragma unroll
  for (int d = 0; d < D; ++d) ctr[d] = rows.bbmin[t * D + d] + 0.5f * rows.bbsize[t * D + d];
#pragma unroll
  for (int rt = 0; rt < kRT; ++rt) {
    const int tile_row0 = (rg + wrows * rt) * 16;
    tile_on[rt] = tile_row0 < q;
    const int row = tile_row0 + lr < q ? tile_row0 + lr : 0;
    const int pk = basis_index<float, D>(row, ip);
    float s2 = 0.f, v[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const float u = ip.td ? ip.unodes[d * q + row] : ip.xi[unpack(pk, d)];
      v[d] = (u * rows.bbsize[t * D + d] + rows.bbmin[t * D + d] - ctr[d]) * sig;
      s2 = fmat(v[d], v[d], s2);
    }
    xb[rt] = target_operand<D>(v, s2, lk);
  }
  __syncthreads();  // U
  // source slot and node of row bl of a chunk of nsrc whole sources (G >= 2);
  // node -1: a padding row
  auto chunk_row = [&](int bl, int nsrc, int &slot, int &node) {
    slot = (int)(((float)bl + 0.5f) * rqpad);
    node = bl - slot * qpad;
    if (slot >= nsrc || node >= q) node = -1;
    if (slot >= nsrc) slot = 0;
  };
  for (int rc = 0; rc < nrhs; rc += NC) {
    f32x4 acc[kRT][NT];
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[rt][nt] = f32x4{0, 0, 0, 0};
    const int ntl = min(NT, (nrhs - rc + 15) >> 4);
    bool all_on = ntl == NT;
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) all_on = all_on && tile_on[rt];
    // all row tiles valid and all column tiles used (the common case): no
    // branches in a K-step, one basic block for the scheduler
    auto chunk_steps = [&](int nrows, auto all_t) {
      for (int ks = kKB * sg; ks < nrows; ks += kKB * kspl) {
        const int off = lr * kChunkP + ks + 8 * lk;  // eight k-slots (gram_pos order)
        gram_step<KT, NT, decltype(all_t)::value>(
            Yd[gl * kChunk + ks + lr], Yd[gl * kChunk + ks + 16 + lr], Mh + off, Ml + off, xb,
            tile_on, ntl, kp, acc);
      }
    };
    constexpr int KM = kChunk * NC / (2 * kThreads);  // staged moment pairs per thread
    static_assert(kChunk * NC % (2 * kThreads) == 0, "staging layout");
    static_assert(kChunk <= kThreads, "one node per thread in the distance staging");
    float py[D], pm[KM][2];  // py: the D coordinates of node threadIdx.x of the chunk
    int f = f0, nbe = 0;
    int pn = 0;
    auto fetch = [&]() {
      const int nsrc = G > 1 ? min(G, f1 - f) : 1;
      const int be = nbe;
      pn = G > 1 ? nsrc * qpad : min(kChunk, qpad - be);
      if (G > 1) {
        if (threadIdx.x < kChunk) {
          int slot, node;
          chunk_row(threadIdx.x, nsrc, slot, node);
          const int s = pat.far_src[f + slot];
#pragma unroll
          for (int d = 0; d < D; ++d)
            py[d] = U[d * qpad + (node < 0 ? 0 : node)] * cols.bbsize[s * D + d] +
                    cols.bbmin[s * D + d];
        }
#pragma unroll
        for (int k = 0; k < KM; ++k) {
          const int e = threadIdx.x + kThreads * k;
          const int bl = 2 * (e / NC), r = e % NC;
          int slot, node;  // of both rows of the pair: qpad is even
          chunk_row(bl, nsrc, slot, node);
          // from 32 columns on a wave's rows (4 or 2) lie in one source: qpad
          // is a multiple of 4
          if constexpr (NT >= 2) slot = __builtin_amdgcn_readfirstlane(slot);
          const float *ms = mom + ((int64_t)pat.far_src[f + slot] * q * nrhs + rc);
#pragma unroll
          for (int u = 0; u < 2; ++u)
            pm[k][u] = (node >= 0 && node + u < q && rc + r < nrhs)
                           ? ms[(uint32_t)((node + u) * nrhs + r)]
                           : 0.f;
        }
      } else {
        const int s = pat.far_src[f];
        const float *ms = mom + ((int64_t)s * q * nrhs + rc);
        if (threadIdx.x < kChunk) {
          const int node = be + (int)threadIdx.x < q ? be + (int)threadIdx.x : 0;
#pragma unroll
          for (int d = 0; d < D; ++d)
            py[d] = U[d * qpad + node] * cols.bbsize[s * D + d] + cols.bbmin[s * D + d];
        }
#pragma unroll
        for (int k = 0; k < KM; ++k) {
          const int e = threadIdx.x + kThreads * k;
          const int bl = 2 * (e / NC), r = e % NC;
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int node = be + bl + u;
            pm[k][u] = (bl + u < pn && node < q && rc + r < nrhs)
                           ? ms[(uint32_t)(node * nrhs + r)]
                           : 0.f;
          }
        }
      }
      if (G > 1) {
        f += nsrc;
      } else {
        nbe += kChunk;
        if (nbe >= qpad) {
          ++f;
          nbe = 0;
        }
      }
    };
    auto stage = [&]() {
      if (threadIdx.x < kChunk) {
        const int bl = threadIdx.x;
        float s2 = 0.f, v[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          v[d] = (py[d] - ctr[d]) * sig;
          s2 = fmat(v[d], v[d], s2);
          v[d] *= -2.f;
        }
        bf16x8 op[kDistGroups];
        source_operand<D>(v, s2, op);
#pragma unroll
        for (int g = 0; g < kDistGroups; ++g) Yd[g * kChunk + bl] = op[g];
      }
#pragma unroll
      for (int k = 0; k < KM; ++k) {
        const int e = threadIdx.x + kThreads * k;
        const int bl = 2 * (e / NC), r = e % NC;
        store_pair(Mh, Ml, r * kChunkP + gram_pos(bl), pm[k][0], pm[k][1]);
      }
    };
    bool more = f < f1;
    if (more) fetch();
    while (more) {
      const int nrows = (pn + kKB - 1) & ~(kKB - 1);
      __syncthreads();
      stage();
      __syncthreads();
      more = f < f1;
      if (more) fetch();  // the next chunk's loads overlap this one's K-steps
      if (all_on)
        chunk_steps(nrows, std::true_type{});
      else
        chunk_steps(nrows, std::false_type{});
    }
    if (kspl > 1)
      add_groups<NT>(acc, reinterpret_cast<float *>(Mh), kspl, wrows, rg, sg, tile_on, lr, lk);
#pragma unroll
    for (int rt = 0; rt < kRT; ++rt) {
      if (!tile_on[rt] || sg != 0) continue;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int col = rc + nt * 16 + lr;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int alpha = (rg + wrows * rt) * 16 + 4 * lk + v;
          if (alpha < q && col < nrhs) {
            float *p = dst_all + ((int64_t)t * q + alpha) * nrhs + col;
            if (split)
              atomic_accumulate(p, acc[rt][nt][v]);
            else
              *p = acc[rt][nt][v];
          }
        }
      }
    }
  }
}

template <int NT>
size_t leaf_output_bf16_lds(int D, int P1, int q) {
  constexpr int NC = 16 * NT;
  const int qpad = (q + 3) & ~3;
  const size_t far = (size_t)kFarChunk * (NC + 16) * sizeof(float);
  const size_t near =
      (size_t)kDistGroups * kChunk * 16 + (size_t)2 * NC * kChunkP * sizeof(u16);
  return (size_t)D * P1 * kRowsP * sizeof(float) + (size_t)((qpad + 3) & ~3) * sizeof(int) +
         (far > near ? far : near);
}

template <int NT>
size_t coupling_bf16_lds(int D, int q) {
  constexpr int NC = 16 * NT;
  const int qpad = (q + 3) & ~3;
  return (size_t)D * qpad * sizeof(float) + (size_t)kDistGroups * kChunk * 16 +
         (size_t)2 * NC * kChunkP * sizeof(u16);
}

template <int D, int NT>
hipError_t launch_bf16_nt(bool output, const MfmaLaunch<float> &a) {
  const size_t lds_out = leaf_output_bf16_lds<NT>(D, a.ip.P1, a.ip.q);
  const size_t lds_cpl = coupling_bf16_lds<NT>(D, a.ip.q);
  float *slabs = nullptr;
  const int parts = launch_parts(output, a, kWaves, &slabs);
  const dim3 grid(output ? a.pat.nnear_order : a.pat.nfar_order, (unsigned)parts);
#define FMCA_BF16_LAUNCH(K)                                                                   \
  if (output)                                                                                 \
    hipLaunchKernelGGL((k_leaf_output_bf16<D, K, NT>), grid, dim3(kThreads), lds_out, a.stream,    \
                       a.rows, a.cols, a.pat, a.ip, a.kp, a.nrhs, a.xs, a.tlhs, a.out, a.ldo, \
                       a.natural ? 1 : 0, slabs);                                             \
  else                                                                                        \
    hipLaunchKernelGGL((k_coupling_bf16<D, K, NT>), grid, dim3(kThreads), lds_cpl, a.stream,       \
                       a.rows, a.cols, a.pat, a.ip, a.kp, a.nrhs, a.mom, a.tlhs, slabs)
  switch (a.kp.kt) {
    case KT_EXPONENTIAL:
      FMCA_BF16_LAUNCH(KT_EXPONENTIAL);
      break;
    case KT_MATERN32:
      FMCA_BF16_LAUNCH(KT_MATERN32);
      break;
    case KT_MATERN52:
      FMCA_BF16_LAUNCH(KT_MATERN52);
      break;
    case KT_GAUSSIAN:
      FMCA_BF16_LAUNCH(KT_GAUSSIAN);
      break;
    default:
      FMCA_BF16_LAUNCH(-1);
  }
#undef FMCA_BF16_LAUNCH
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || parts == 1) return e;
  return launch_add_parts<float>(output, a.rows, a.ip.q, a.nrhs, parts, slabs, a.tlhs, a.out,
                                 a.ldo, a.natural, a.stream);
}

// Columns per pass: 16, 32, or 64 for more than 32 columns where the staging
// fits: one evaluation of the entries for 64 columns (n = 1e6: 12.9 ms in the
// leaf output against 2 x 7.7 ms).
inline int bf16_nt(bool output, int D, int P1, int q, int nrhs) {
  if (nrhs <= 16) return 1;
  if (nrhs > 32 && (output ? leaf_output_bf16_lds<4>(D, P1, q) : coupling_bf16_lds<4>(D, q)) <=
                       64 * 1024)
    return 4;
  return 2;
}

template <int D>
hipError_t launch_bf16_d(bool output, const MfmaLaunch<float> &a) {
  switch (bf16_nt(output, D, a.ip.P1, a.ip.q, a.nrhs)) {
    case 1:
      return launch_bf16_nt<D, 1>(output, a);
    case 2:
      return launch_bf16_nt<D, 2>(output, a);
  }
  return launch_bf16_nt<D, 4>(output, a);
}

}  // namespace

// Where the BF16 form is the faster one.  A chunk of 128 sources or nodes is
// staged by eight waves between two barriers; small row counts leave most of a
// K-step's tiles empty and short lists most of a chunk, and the FP32 form, of
// four waves and smaller tiles, is faster there.  FP32 / BF16 (us):
//   leaf output, 16 / 64 columns: 6 rows (2-D degree 1, n = 2e5) 465 / 1087 and
//     1266 / 3487; 24 rows (2-D degree 3, n = 2e5) 218 / 333 and 699 / 983; 49
//     rows with 831 sources (2-D degree 5, n = 2e5) 216 / 266 and 682 / 822, with
//     3429 (3-D degree 2, n = 2e5) 804 / 709 and 2246 / 1945; 62 rows with 869,
//     but only 64 leaves (n = 4000) 30 / 28 and 58 / 39;
//   coupling: q = 16 (2-D degree 3, n = 2e5) 207 / 307 and 647 / 1152; q = 36
//     with 663 nodes (2-D degree 5, n = 2e5) 253 / 306 and 908 / 1147, with 1132
//     (clusters) 242 / 226 and 946 / 907; q = 27 with 2335 (3-D degree 2,
//     n = 2e5) 817 / 702 and 2844 / 2844; few clusters (n = 4000, q = 25) 29 / 23.
bool bf16_pays(bool output, const MfmaLaunch<float> &a) {
  if (output)
    return a.rows.npts > (int64_t)48 * a.rows.nleaves &&
           (a.pat.near_per_task >= 1000 || a.rows.nleaves < 512);
  const int q = a.ip.q;
  return q > 48 || (q > 16 && (a.pat.far_per_task * q >= 700 || a.rows.ncl < 512));
}

bool bf16_supported(bool output, int D, int P1, int q, int nrhs, int kt, int vmask) {
  if (nrhs < kMfmaMinRhs) return false;
  if (vmask != (1 << KV_VALUE) || kt >= KT_COUNT) return false;  // kernel values only
  const size_t limit = 64 * 1024;
  const int nt = nrhs <= 16 ? 1 : 2;
  if (output)
    return (nt == 1 ? leaf_output_bf16_lds<1>(D, P1, q) : leaf_output_bf16_lds<2>(D, P1, q)) <=
           limit;
  if (q > kRows) return false;
  return (nt == 1 ? coupling_bf16_lds<1>(D, q) : coupling_bf16_lds<2>(D, q)) <= limit;
}

hipError_t launch_bf16(bool output, const MfmaLaunch<float> &a, float *xs, float *mom) {
  {
    // the right operand this launch stages, split once here (rewritten by
    // the next action's permutation / upward pass)
    float *x = output ? xs : mom;
    const int64_t n = (output ? a.cols.npts : (int64_t)a.cols.ncl * a.ip.q) * a.nrhs;
    if (n > 0) {
      const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, 8192);
      hipLaunchKernelGGL(k_split_inplace, dim3(grid), dim3(256), 0, a.stream, x, n);
    }
  }
  switch (a.rows.dim) {
    case 1:
      return launch_bf16_d<1>(output, a);
    case 2:
      return launch_bf16_d<2>(output, a);
    case 3:
      return launch_bf16_d<3>(output, a);
  }
  return hipErrorInvalidValue;
}

}  // namespace fmca_amd
