// Channel-mixing linear layers on the matrix cores, fp32 in and out.
//
//   OUT[n, m, :] = scale * X[n, m, :] . W[g(n)][l(m)]      (scale = 1/sqrt(K) in the model)
//
// for features with 16 components per node (l(m) = floor(sqrt(m)), four weight blocks per group) or with a
// single scalar component per node (one weight block per group).
//
// A workgroup of four wavefronts owns a tile of 128 nodes x one component m x all Nout columns, so
// every row of the tile uses the same K x Nout weight block W[g][l(m)].  K is walked in chunks of 32:
// the X rows of the tile (each chunk of a row is one 128-byte line) and the matching columns of the
// TRANSPOSED weights ([Nout, K], which the caller already keeps for the backward) are staged in LDS
// with coalesced 16-byte loads, and each wave feeds the matrix cores with 16-byte LDS reads.  Weights
// therefore cross L2 once per 128 rows instead of once per 32.  All (group, m, tile) combinations go out in
// a single launch; per-element weights are selected through a node permutation that lists the nodes group
// by group, without any host synchronisation.
//
// Arithmetic (the kernel for few rows multiplies fp32 values): every fp32 operand is split into three bf16 pieces when it is staged (a = hi + mid + lo, 24 mantissa bits
// in all), and the product is accumulated in fp32 from the six piece products that matter (hi.hi, hi.mid, mid.hi, hi.lo,
// lo.hi, mid.mid; the dropped ones are below 2^-24 of the product) on v_mfma_f32_32x32x16_bf16, whose rate is 16x that of
// the fp32 matrix instruction.  The result matches an fp32 GEMM to rounding (measured rms error 1.7e-7 against fp64 on
// unit-variance data, plain fp32 accumulation 2.0e-7), and the GEMM phase is a third of what v_mfma_f32_32x32x2_f32 on the
// fp32 values needs (measured 1.2-1.4x faster end to end at every width from 64 to 256), so the kernel runs at what
// its memory traffic allows.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "mfma_f32.hpp"
#include "mfma_rows.hpp"
#include "mfma_split.hpp"

namespace cm {
namespace {

constexpr int kWaves = 4;
constexpr int kTileNodes = 32 * kWaves;  // rows per workgroup (MFMA M = 32 per wave)
constexpr int kKC = 32;                  // K columns staged per step
constexpr int kLdH = kKC + 8;            // padded LDS row stride of a bf16 plane (elements; 80 bytes: conflict-free b128 reads)

// A wave's 32 x (32 NT) block of accumulators to memory, four bytes per lane and store (a store instruction covers two
// rows of 128 bytes): OUT = acc * scale (+ residual).  The residual may be OUT itself, so the compiler cannot move a
// load of it across a store: all of a lane's residual values are read before its first store (every element is read
// and written by the same lane), instead of one dependent load per store.  The product is rounded before the residual is
// added, as in the kernels that stage it in LDS.
template <int NT>
__device__ __forceinline__ void store_block(const v16f (&acc)[NT], const int *sNode, int wave, int half, int mrow, int ncomp, int m,
                                            int row_stride, int col0, float scale, const float *residual, float *OUT) {
  if (residual) {
    float res[16][NT];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int node = sNode[32 * wave + 8 * (r / 4) + 4 * half + (r % 4)];
      const float *rp = residual + (static_cast<int64_t>(node >= 0 ? node : 0) * ncomp + m) * row_stride + col0 + mrow;
#pragma unroll
      for (int t = 0; t < NT; ++t) res[r][t] = node >= 0 ? rp[32 * t] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int node = sNode[32 * wave + 8 * (r / 4) + 4 * half + (r % 4)];
      if (node < 0) continue;
      float *op = OUT + (static_cast<int64_t>(node) * ncomp + m) * row_stride + col0 + mrow;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma clang fp contract(off)
        const float v = acc[t][r] * scale;
        op[32 * t] = v + res[r][t];
      }
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int node = sNode[32 * wave + 8 * (r / 4) + 4 * half + (r % 4)];
    if (node < 0) continue;
    float *op = OUT + (static_cast<int64_t>(node) * ncomp + m) * row_stride + col0 + mrow;
#pragma unroll
    for (int t = 0; t < NT; ++t) op[32 * t] = acc[t][r] * scale;
  }
}

// A workgroup computes 32 * NT output columns, starting at column blockIdx.y * 32 * NT of the nout_total columns of a row
// (one workgroup per tile for all columns where there are many tiles; few tiles are spread over more workgroups, 32
// columns each, which shortens the chain of staging and matrix instructions a tile waits for: every output element sums
// the same products in the same order either way).  SCALED: X is multiplied by row_scale on the way in
// At 160 and 192 columns two workgroups fit a compute unit by their LDS (70 / 77 KB) and, told so, the compiler keeps the
// kernel within the 256 registers that leaves each wave (measured 25-30 % faster on [N,16,C] features there).
template <int NT, bool SCALED>
__global__ __launch_bounds__(kWaves *kWave, ((NT == 5 || NT == 6) ? 2 : 1)) void linear_kernel(const float *__restrict__ X, const float *__restrict__ WT,
                                                               const int32_t *__restrict__ node_perm,
                                                               const int32_t *__restrict__ group_offsets, int nnodes,
                                                               int ngroups, int zero_last_group, int ncomp, int K,
                                                               float scale, const float *__restrict__ row_scale,
                                                               const float *residual, float *OUT, int nout_total) {
  constexpr int NOUT = 32 * NT;
  const int col0 = blockIdx.y * NOUT;
  // three bf16 planes per operand: plane p of X at sAp + p * kTileNodes * kLdH, of the weights at sBp + p * NOUT * kLdH
  // (77 KB at Nout = 192, 92 KB at 256: beyond 64 KB, within the 160 KB of a gfx950 compute unit)
  __shared__ __attribute__((aligned(16))) __bf16 sAp[3 * kTileNodes * kLdH];
  __shared__ __attribute__((aligned(16))) __bf16 sBp[3 * NOUT * kLdH];
  __shared__ int sNode[kTileNodes];

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = tid / kWave;
  // the components of a tile are neighbours in the launch order: they share the tile's row_scale rows and touch
  // adjacent rows of X and OUT while those are hot
  const int m = blockIdx.x % ncomp;  // component 0..ncomp-1
  const int l = ncomp == 1 ? 0 : l_of_m(m);
  const int nblocks = ncomp == 1 ? 1 : 4;  // weight blocks per group

  // locate (group, first position in the grouped node order) of this tile
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x / ncomp, kTileNodes, g, pos0, gend)) return;
  const int nrows = min(kTileNodes, gend - pos0);

  if (tid < kTileNodes) {
    int node = -1;
    if (tid < nrows) {
      node = node_perm ? node_perm[pos0 + tid] : pos0 + tid;
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = -1;
    }
    sNode[tid] = node;
  }
  __syncthreads();

  if (zero_last_group && g == ngroups - 1) {
    // rows that belong to no weight group: the product is defined as zero (a residual still passes through)
    for (int i = tid; i < kTileNodes * NOUT; i += kWaves * kWave) {
      const int node = sNode[i / NOUT];
      if (node >= 0) {
        const int64_t at = (static_cast<int64_t>(node) * ncomp + m) * nout_total + col0 + i % NOUT;
        OUT[at] = residual ? residual[at] : 0.f;
      }
    }
    return;
  }
  const float *Wg = WT + ((static_cast<int64_t>(g) * nblocks + l) * nout_total + col0) * K;  // [NOUT, K] of [nout_total, K]

  v16f acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  // staging map: kKC / 4 threads x 16 bytes cover the staged columns of a row
  constexpr int kTPR = kKC / 4;                    // threads per row
  constexpr int kRPP = kWaves * kWave / kTPR;      // rows per pass
  const int srow = tid / kTPR;
  const int scol = (tid % kTPR) * 4;
  // MFMA operand map: row / column within the 32-wide block and which half of the 8-wide k step
  const int mrow = lane % 32;
  const int half = lane / 32;

  constexpr int A_PASSES = kTileNodes / kRPP;
  constexpr int B_PASSES = NOUT / kRPP;
  f4 pa[A_PASSES], pb[B_PASSES], ps[SCALED ? A_PASSES : 1];
  // global -> register prefetch of one K chunk; the next chunk is in flight while the current one is multiplied
  auto prefetch = [&](int kc) {
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i) {
      const int node = sNode[kRPP * i + srow];
      pa[i] = zero4();
      if (node >= 0) {
        pa[i] = ld4_stream(X + (static_cast<int64_t>(node) * ncomp + m) * K + kc + scol);
        // optional per-node, per-column factor shared by all components (the contraction's upstream gradient); it is
        // applied when the chunk moves to LDS, so that nothing waits for these loads here
        if constexpr (SCALED) ps[i] = ld4(row_scale + static_cast<int64_t>(node) * K + kc + scol);
      }
    }
#pragma unroll
    for (int i = 0; i < B_PASSES; ++i) pb[i] = ld4(Wg + static_cast<int64_t>(kRPP * i + srow) * K + kc + scol);
  };
  prefetch(0);
  for (int kc = 0; kc < K; kc += kKC) {
    __syncthreads();  // previous chunk fully consumed
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i) {
      f4 v = pa[i];
      if constexpr (SCALED) v *= ps[i];
      bf16x4 h, md, lw;
      split3(v, h, md, lw);
      const int at = (kRPP * i + srow) * kLdH + scol;
      *reinterpret_cast<bf16x4 *>(sAp + at) = h;
      *reinterpret_cast<bf16x4 *>(sAp + kTileNodes * kLdH + at) = md;
      *reinterpret_cast<bf16x4 *>(sAp + 2 * kTileNodes * kLdH + at) = lw;
    }
#pragma unroll
    for (int i = 0; i < B_PASSES; ++i) {
      bf16x4 h, md, lw;
      split3(pb[i], h, md, lw);
      const int at = (kRPP * i + srow) * kLdH + scol;
      *reinterpret_cast<bf16x4 *>(sBp + at) = h;
      *reinterpret_cast<bf16x4 *>(sBp + NOUT * kLdH + at) = md;
      *reinterpret_cast<bf16x4 *>(sBp + 2 * NOUT * kLdH + at) = lw;
    }
    __syncthreads();
    if (kc + kKC < K) prefetch(kc + kKC);

#pragma unroll
    for (int ks = 0; ks < kKC; ks += 16) {
      // a lane feeds 8 consecutive k of its row: k = ks + 8 * half .. + 7
      const int aoff = (32 * wave + mrow) * kLdH + ks + 8 * half;
      bf16x8 a[3], b[NT][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p] = *reinterpret_cast<const bf16x8 *>(sAp + p * kTileNodes * kLdH + aoff);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[t][p] = *reinterpret_cast<const bf16x8 *>(sBp + p * NOUT * kLdH + (32 * t + mrow) * kLdH + ks + 8 * half);
      // piece products from small to large; consecutive MFMAs go to different accumulators
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[t][0], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[t][2], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[t][1], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[t][0], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[t][1], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[t][0], acc[t], 0, 0, 0);
    }
  }

  // accumulator r of a lane is row 8*(r/4) + 4*(lane/32) + r%4, column lane%32 of the wave's 32x32 block
  store_block<NT>(acc, sNode, wave, half, mrow, ncomp, m, nout_total, col0, scale, residual, OUT);
}

// -----------------------------------------------------------------------------------------------
// Few rows: 16 nodes x one component x 16 output columns per wave, operands straight to registers (mfma_f32.hpp).  No LDS,
// no barrier: a wave waits for the group offsets, for its node's place in the permutation, and once for everything else.
// In the 21-atom step a launch takes 3.1 us where tiles of 128 rows took 5.7, in the 216-atom, 128-channel step 4.2 and
// 6.3 - 8.5 us where they took 8.7 and 10.7.
template <int KQ, bool SCALED, int CB>
__global__ __launch_bounds__(kWaves *kWave) void linear_few_rows_kernel(const float *__restrict__ X, const float *__restrict__ WT,
                                                                        const int32_t *__restrict__ node_perm,
                                                                        const int32_t *__restrict__ group_offsets, int nnodes,
                                                                        int ngroups, int zero_last_group, int ncomp, float scale,
                                                                        const float *__restrict__ row_scale, const float *residual,
                                                                        float *OUT, int nout) {
  constexpr int K = 16 * KQ;
  const int lane = threadIdx.x % kWave;
  const int row = lane % few::kRows, part = lane / few::kRows;
  const int col0 = few::kRows * CB * (blockIdx.y * (blockDim.x / kWave) + threadIdx.x / kWave);
  const int m = blockIdx.x % ncomp;
  const int l = ncomp == 1 ? 0 : l_of_m(m);
  const int nblocks = ncomp == 1 ? 1 : 4;
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x / ncomp, few::kRows, g, pos0, gend)) return;
  int node = -1;
  if (pos0 + row < gend) node = node_perm ? node_perm[pos0 + row] : pos0 + row;
  const bool here = static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t in = here ? node : 0;  // a row that is not there computes node 0's and drops it
  const int64_t at = (in * ncomp + m) * nout + col0 + 4 * part;
  f4 res[CB], out[CB];
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    res[c] = residual ? ld4(residual + at + few::kRows * c) : zero4();
    out[c] = zero4();
  }
  if (!(zero_last_group && g == ngroups - 1)) {  // (rows of no weight group: the product is defined as zero)
    const float *wp = WT + ((static_cast<int64_t>(g) * nblocks + l) * nout + col0 + row) * K + 4 * part;
    few::Rows<KQ> w[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) w[c] = few::load_rows<KQ>(wp + few::kRows * c * K);
    few::Rows<KQ> x = few::load_rows<KQ>(X + (in * ncomp + m) * K + 4 * part);
    if constexpr (SCALED) {
      const few::Rows<KQ> s = few::load_rows<KQ>(row_scale + in * K + 4 * part);
#pragma unroll
      for (int q = 0; q < KQ; ++q) x.v[q] *= s.v[q];
    }
    few::product<KQ, CB>(x, w, out);
  }
  if (!here) return;
#pragma unroll
  for (int c = 0; c < CB; ++c) {
#pragma clang fp contract(off)  // the product is rounded before the residual is added, as everywhere
    f4 v = out[c] * scale;
    if (residual) v += res[c];
    st4(OUT + at + few::kRows * c, v);
  }
}

// -----------------------------------------------------------------------------------------------
// Few tiles (a system of a few hundred atoms): the launch is over in a few microseconds, most of which a workgroup of the
// kernel above spends waiting for one K chunk after the other, with next to nothing to multiply in between.  Here a
// workgroup (one tile, one component, 32 output columns) requests every K chunk of both operands, the row scales and
// the residual values at once and waits for memory once; K = 32 KCH.  Staging, operand split, piece products and their
// order, and the epilogue's roundings are those of the kernel above: the same bits.
template <int KCH, bool SCALED>
__global__ __launch_bounds__(kWaves *kWave) void linear_few_tiles_kernel(const float *__restrict__ X, const float *__restrict__ WT,
                                                                         const int32_t *__restrict__ node_perm,
                                                                         const int32_t *__restrict__ group_offsets, int nnodes,
                                                                         int ngroups, int zero_last_group, int ncomp, float scale,
                                                                         const float *__restrict__ row_scale, const float *residual,
                                                                         float *OUT, int nout_total) {
  constexpr int K = kKC * KCH;
  constexpr int NOUT = 32;
  const int col0 = blockIdx.y * NOUT;
  __shared__ __attribute__((aligned(16))) __bf16 sAp[3 * kTileNodes * kLdH];
  __shared__ __attribute__((aligned(16))) __bf16 sBp[3 * NOUT * kLdH];
  __shared__ int sNode[kTileNodes];

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = tid / kWave;
  const int m = blockIdx.x % ncomp;
  const int l = ncomp == 1 ? 0 : l_of_m(m);
  const int nblocks = ncomp == 1 ? 1 : 4;

  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x / ncomp, kTileNodes, g, pos0, gend)) return;
  const int nrows = min(kTileNodes, gend - pos0);
  if (tid < kTileNodes) {
    int node = -1;
    if (tid < nrows) {
      node = node_perm ? node_perm[pos0 + tid] : pos0 + tid;
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = -1;
    }
    sNode[tid] = node;
  }
  __syncthreads();

  if (zero_last_group && g == ngroups - 1) {
    for (int i = tid; i < kTileNodes * NOUT; i += kWaves * kWave) {
      const int node = sNode[i / NOUT];
      if (node >= 0) {
        const int64_t at = (static_cast<int64_t>(node) * ncomp + m) * nout_total + col0 + i % NOUT;
        OUT[at] = residual ? residual[at] : 0.f;
      }
    }
    return;
  }
  const float *Wg = WT + ((static_cast<int64_t>(g) * nblocks + l) * nout_total + col0) * K;  // [NOUT, K] of [nout_total, K]

  constexpr int kTPR = kKC / 4;
  constexpr int kRPP = kWaves * kWave / kTPR;
  static_assert(kRPP == NOUT, "one pass of the staging map covers the 32 weight rows");
  constexpr int A_PASSES = kTileNodes / kRPP;
  const int srow = tid / kTPR;
  const int scol = (tid % kTPR) * 4;
  const int mrow = lane % 32;
  const int half = lane / 32;

  // everything this workgroup reads, requested before anything is waited for
  f4 pa[KCH][A_PASSES], pb[KCH], ps[SCALED ? KCH : 1][A_PASSES];
#pragma unroll
  for (int i = 0; i < A_PASSES; ++i) {
    const int node = sNode[kRPP * i + srow];
    const float *xp = X + (static_cast<int64_t>(node >= 0 ? node : 0) * ncomp + m) * K + scol;
    const float *sp = SCALED ? row_scale + static_cast<int64_t>(node >= 0 ? node : 0) * K + scol : nullptr;
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      pa[c][i] = node >= 0 ? ld4_stream(xp + kKC * c) : zero4();
      if constexpr (SCALED) ps[c][i] = node >= 0 ? ld4(sp + kKC * c) : zero4();
    }
  }
#pragma unroll
  for (int c = 0; c < KCH; ++c) pb[c] = ld4(Wg + static_cast<int64_t>(srow) * K + kKC * c + scol);
  float res[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int node = sNode[32 * wave + 8 * (r / 4) + 4 * half + (r % 4)];
    res[r] = (residual && node >= 0) ? residual[(static_cast<int64_t>(node) * ncomp + m) * nout_total + col0 + mrow] : 0.f;
  }

  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int c = 0; c < KCH; ++c) {
    if (c > 0) __syncthreads();  // previous chunk fully consumed
#pragma unroll
    for (int i = 0; i < A_PASSES; ++i) {
      f4 v = pa[c][i];
      if constexpr (SCALED) v *= ps[c][i];
      bf16x4 h, md, lw;
      split3(v, h, md, lw);
      const int at = (kRPP * i + srow) * kLdH + scol;
      *reinterpret_cast<bf16x4 *>(sAp + at) = h;
      *reinterpret_cast<bf16x4 *>(sAp + kTileNodes * kLdH + at) = md;
      *reinterpret_cast<bf16x4 *>(sAp + 2 * kTileNodes * kLdH + at) = lw;
    }
    {
      bf16x4 h, md, lw;
      split3(pb[c], h, md, lw);
      const int at = srow * kLdH + scol;
      *reinterpret_cast<bf16x4 *>(sBp + at) = h;
      *reinterpret_cast<bf16x4 *>(sBp + NOUT * kLdH + at) = md;
      *reinterpret_cast<bf16x4 *>(sBp + 2 * NOUT * kLdH + at) = lw;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < kKC; ks += 16) {
      const int aoff = (32 * wave + mrow) * kLdH + ks + 8 * half;
      bf16x8 a[3], b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        a[p] = *reinterpret_cast<const bf16x8 *>(sAp + p * kTileNodes * kLdH + aoff);
        b[p] = *reinterpret_cast<const bf16x8 *>(sBp + p * NOUT * kLdH + mrow * kLdH + ks + 8 * half);
      }
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
    }
  }

#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int node = sNode[32 * wave + 8 * (r / 4) + 4 * half + (r % 4)];
    if (node < 0) continue;
    float *op = OUT + (static_cast<int64_t>(node) * ncomp + m) * nout_total + col0 + mrow;
    {
#pragma clang fp contract(off)  // the product is rounded before the residual is added, as everywhere
      const float v = acc[r] * scale;
      *op = residual ? v + res[r] : v;
    }
  }
}

// -----------------------------------------------------------------------------------------------
// Variant with the feature rows on a ring of raw fp32 chunks in LDS, filled by direct global -> LDS loads.
//
// What bounds the kernel above is the amount of X that a workgroup has in flight: one 16 KB chunk, and only while it
// multiplies the previous one.  Here the X chunks never pass through registers: each wave fetches the 32 rows it
// multiplies itself, 16 bytes per lane, straight into a three-stage ring (global_load_lds_dwordx4), so one or two chunks
// are in flight at all times; it splits its rows into the bf16 pieces as it feeds the matrix cores (every row is split
// once, by its own wave, so this costs what the staging pass did, and the staged piece planes of X with their LDS
// writes and re-reads go away).  The weights take the old road (registers -> pieces -> LDS planes), one chunk ahead.
//
// Vector-memory operations retire in issue order and one counter covers them all.  The compiler would wait for "all
// of them" wherever it sees a load under a branch or a direct-to-LDS load that may alias a later LDS read, which
// would drain the ring at every chunk.  So every vector-memory operation of the main loop is issued from inline assembly,
// unseen by the compiler, in a fixed order, and waited for explicitly:
//     iteration c:   barrier | wait: all but the 4 loads of X chunk c+1 | weights c -> planes | issue weights c+1
//                    (and scales c+1), then X chunk c+2 | barrier | multiply chunk c
// The assembly statements that wait also carry the loaded registers as read-write operands, which keeps every use
// behind the wait.  M0 (the LDS address of a direct load) is written inside those statements; nothing else in this
// kernel uses it.
//
// LDS layout of a ring stage: row r of the tile at r * 128 bytes, its eight 16-byte pieces at positions
// piece ^ (r & 7), so that the 32 rows a wave reads at the same piece index fall on different banks (a direct load
// writes lane i at base + 16 i: the layout is chosen through which piece each lane fetches).
// -----------------------------------------------------------------------------------------------
constexpr int kStages = 3;
constexpr int kStageBytes = kTileNodes * kKC * 4;

// M0 is written here and named as clobbered; the compiler reserves that register and warns that it does not track it
// across the statement, which is the point of the remark in the comment above: nothing else in this kernel may rely on it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const float *src, unsigned lds_byte_address) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(src), "s"(lds_byte_address) : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ void ldg16(f4 &dst, const float *src) {
  asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(dst) : "v"(src) : "memory");
}
// Marks the point from which a register that a hand-issued load lands in holds the loaded value (the wait that covers the
// load precedes it): no use can move above it, and the build's scan of the generated code, which refuses any instruction
// that touches such a register between the load's issue and this mark, reads the comment it leaves in the assembly.
__device__ __forceinline__ void after_wait(f4 &v) { asm volatile("; landed %0" : "+v"(v)); }

// two workgroups per compute unit (two waves per SIMD) wherever LDS allows it: 256 registers per lane
template <int NT, bool SCALED>
__global__ __launch_bounds__(kWaves *kWave, (NT <= 4 ? 2 : 1)) void linear_ring_kernel(const float *__restrict__ X, const float *__restrict__ WT,
                                                                    const int32_t *__restrict__ node_perm,
                                                                    const int32_t *__restrict__ group_offsets, int nnodes,
                                                                    int ngroups, int zero_last_group, int ncomp, int K,
                                                                    float scale, const float *__restrict__ row_scale,
                                                                    const float *residual, float *OUT) {
  constexpr int NOUT = 32 * NT;
  __shared__ __attribute__((aligned(16))) float sRaw[kStages * kTileNodes * kKC];
  __shared__ __attribute__((aligned(16))) __bf16 sBp[3 * NOUT * kLdH];
  __shared__ int sNode[kTileNodes];

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int m = blockIdx.x % ncomp;
  const int l = ncomp == 1 ? 0 : l_of_m(m);
  const int nblocks = ncomp == 1 ? 1 : 4;

  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x / ncomp, kTileNodes, g, pos0, gend)) return;
  const int nrows = min(kTileNodes, gend - pos0);

  if (tid < kTileNodes) {
    int node = -1;
    if (tid < nrows) {
      node = node_perm ? node_perm[pos0 + tid] : pos0 + tid;
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = -1;
    }
    sNode[tid] = node;
  }
  __syncthreads();

  if (zero_last_group && g == ngroups - 1) {
    for (int i = tid; i < kTileNodes * NOUT; i += kWaves * kWave) {
      const int node = sNode[i / NOUT];
      if (node >= 0) {
        const int64_t at = (static_cast<int64_t>(node) * ncomp + m) * NOUT + i % NOUT;
        OUT[at] = residual ? residual[at] : 0.f;
      }
    }
    return;
  }
  const float *Wg = WT + (static_cast<int64_t>(g) * nblocks + l) * NOUT * K;  // [NOUT, K]

  v16f acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  // weights: staging map as in the kernel above (8 threads x 16 bytes per row of the chunk, 32 rows per pass)
  constexpr int kTPR = kKC / 4;
  constexpr int kRPP = kWaves * kWave / kTPR;
  static_assert(kRPP == 32 && NOUT % kRPP == 0, "staging map");
  const int srow = tid / kTPR;
  const int scol = (tid % kTPR) * 4;
  const float *wsrc = Wg + static_cast<int64_t>(srow) * K + scol;  // + 32 i K for pass i, + kc
  // matrix-core operand map
  const int mrow = lane % 32;
  const int half = lane / 32;

  // X: one direct load covers 8 rows x 128 bytes; a wave issues four per chunk, for its own 32 rows.  Rows beyond the
  // tile fetch row 0 of X (their products are never stored).
  const int drow = lane / 8;
  const int dpiece = (lane & 7) ^ drow;
  const float *xsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int node = sNode[32 * wave + 8 * i + drow];
    xsrc[i] = X + (static_cast<int64_t>(node >= 0 ? node : 0) * ncomp + m) * K + 4 * dpiece;
  }
  const unsigned raw_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(sRaw)) + static_cast<unsigned>(wave) * (32 * kKC * 4);
  auto issue_x = [&](int kc, int stage) {
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16(xsrc[i] + kc, raw_base + static_cast<unsigned>(stage) * kStageBytes + i * (8 * kKC * 4));
  };
  // the wave's own A fragments: 8 consecutive k of row 32 wave + mrow, i.e. pieces ks/4 + 2 half and the next one
  const float *araw = sRaw + (32 * wave + mrow) * kKC;
  const int swz = mrow & 7;

  f4 pb[NT];
  f4 sc[2][4];
  const float *ssrc = nullptr;
  if constexpr (SCALED) {
    const int node = sNode[32 * wave + mrow];
    ssrc = row_scale + static_cast<int64_t>(node >= 0 ? node : 0) * K + 8 * half;
  }
  auto issue_w = [&](int kc, auto par) {
    constexpr int P = decltype(par)::value;
#pragma unroll
    for (int i = 0; i < NT; ++i) ldg16(pb[i], wsrc + static_cast<int64_t>(kRPP * i) * K + kc);
    if constexpr (SCALED) {
#pragma unroll
      for (int q = 0; q < 4; ++q) ldg16(sc[P][q], ssrc + kc + 16 * (q / 2) + 4 * (q % 2));
    }
  };

  // What the next iteration consumes has landed when an iteration (or the prologue) ends: the wait sits at the end of
  // the code that issued the loads, so that every register a load was issued into passes through after_wait before
  // the loop's back edge (a copy the compiler makes there then copies the loaded value).
  auto landed = [&](auto par) {
    constexpr int P = decltype(par)::value;
#pragma unroll
    for (int i = 0; i < NT; ++i) after_wait(pb[i]);
    if constexpr (SCALED) {
#pragma unroll
      for (int q = 0; q < 4; ++q) after_wait(sc[P][q]);
    }
  };
  const int nch = K / kKC;
  issue_w(0, std::integral_constant<int, 0>{});
  issue_x(0, 0);
  if (nch > 1) {
    issue_x(kKC, 1);
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  // all but the four loads of X chunk 1
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  landed(std::integral_constant<int, 0>{});

  auto iteration = [&](int c, int stage, auto par) {
    constexpr int P = decltype(par)::value;
    const int kc = c * kKC;
    // every wave has finished multiplying chunk c - 1: the weight planes and ring stage (c + 2) % 3 are free.  Weights
    // (and scales) of chunk c and X chunk c have landed (waited for where they were issued); the four loads of X chunk
    // c + 1 may still be out
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      bf16x4 h, md, lw;
      split3(pb[i], h, md, lw);
      const int at = (kRPP * i + srow) * kLdH + scol;
      *reinterpret_cast<bf16x4 *>(sBp + at) = h;
      *reinterpret_cast<bf16x4 *>(sBp + NOUT * kLdH + at) = md;
      *reinterpret_cast<bf16x4 *>(sBp + 2 * NOUT * kLdH + at) = lw;
    }
    if (c + 1 < nch) issue_w(kc + kKC, std::integral_constant<int, 1 - P>{});
    if (c + 2 < nch) issue_x(kc + 2 * kKC, stage >= 1 ? stage - 1 : 2);  // (stage + 2) % 3
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // weight planes written

    const float *ast = araw + stage * (kTileNodes * kKC);
#pragma unroll
    for (int ks = 0; ks < kKC; ks += 16) {
      const int piece = ks / 4 + 2 * half;
      f4 r0 = *reinterpret_cast<const f4 *>(ast + 4 * (piece ^ swz));
      f4 r1 = *reinterpret_cast<const f4 *>(ast + 4 * ((piece + 1) ^ swz));
      if constexpr (SCALED) {
        r0 *= sc[P][2 * (ks / 16)];
        r1 *= sc[P][2 * (ks / 16) + 1];
      }
      bf16x4 h0, m0, l0, h1, m1, l1;
      split3(r0, h0, m0, l0);
      split3(r1, h1, m1, l1);
      bf16x8 a[3], b[NT][3];
      a[0] = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
      a[1] = __builtin_shufflevector(m0, m1, 0, 1, 2, 3, 4, 5, 6, 7);
      a[2] = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[t][p] = *reinterpret_cast<const bf16x8 *>(sBp + p * NOUT * kLdH + (32 * t + mrow) * kLdH + ks + 8 * half);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[t][0], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[t][2], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[t][1], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[t][0], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[t][1], acc[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[t][0], acc[t], 0, 0, 0);
    }
    // the next chunk's weights, scales and X rows: everything but the four loads of the X chunk after it, if one was issued
    if (c + 1 < nch) {
      if (c + 2 < nch)
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    landed(std::integral_constant<int, 1 - P>{});
  };
  int stage = 0;
  for (int c = 0; c < nch; c += 2) {
    iteration(c, stage, std::integral_constant<int, 0>{});
    stage = stage == 2 ? 0 : stage + 1;
    if (c + 1 >= nch) break;
    iteration(c + 1, stage, std::integral_constant<int, 1>{});
    stage = stage == 2 ? 0 : stage + 1;
  }
  // Nothing is in flight here (the last chunk waited for everything and issued nothing); said once more in a form that
  // the build's scan of the generated code, which does not know that the loop issues only while it goes on, can read.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  if constexpr (NT <= 4) {
    // Output through LDS, so that rows leave as 16-byte stores (a lane's accumulators are one column of 16 rows: stored
    // directly they are 64 four-byte stores per lane).  Every wave is past its last multiply after the barrier, so the
    // ring and the weight planes are free: each wave lays its 32 x Nout block out row-major in its own piece of them.
    asm volatile("s_barrier" ::: "memory");
    constexpr int TILE = 32 * NOUT;  // floats per wave
    static_assert(4 * TILE <= kStages * kTileNodes * kKC || (3 * TILE <= kStages * kTileNodes * kKC && TILE * 4 <= 3 * NOUT * kLdH * 2),
                  "output staging does not fit the ring and the weight planes");
    float *tile = (4 * TILE <= kStages * kTileNodes * kKC || wave < 3) ? sRaw + wave * TILE : reinterpret_cast<float *>(sBp);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 8 * (r / 4) + 4 * half + (r % 4);
#pragma unroll
      for (int t = 0; t < NT; ++t) tile[row * NOUT + 32 * t + mrow] = acc[t][r] * scale;
    }
    constexpr int PPR = NOUT / 4;  // 16-byte pieces per row
#pragma unroll
    for (int i = 0; i < TILE / 4 / kWave; ++i) {
      const int q = i * kWave + lane;
      const int row = q / PPR, col = 4 * (q % PPR);
      const int node = sNode[32 * wave + row];
      if (node >= 0) {
        const int64_t at = (static_cast<int64_t>(node) * ncomp + m) * NOUT + col;
        f4 v = *reinterpret_cast<const f4 *>(tile + row * NOUT + col);
        if (residual) v += ld4(residual + at);  // may be OUT itself: every element is read and written by the same lane
        st4(OUT + at, v);
      }
    }
  } else {
    store_block<NT>(acc, sNode, wave, half, mrow, ncomp, m, NOUT, 0, scale, residual, OUT);
  }
}

// -----------------------------------------------------------------------------------------------
// Variant with the weights resident in LDS (16 components per node, K = Nout = 64, 96 or 128).
//
// The kernels above stage the K x Nout weight block again for every tile of 128 rows (as many bytes from L2 as the tile
// has from HBM) and walk K in barrier-separated phases.  Here a launch has one workgroup per compute unit, and a
// workgroup takes a contiguous piece of the list of all 16-row tiles, ordered by (weight group, l, node tile, m within
// l), so that it needs one or two weight blocks in its whole life: it splits a block once into three bf16 planes that
// cover all of K (102 KB at 128 x 128) and then its eight waves run independently of each other, one 16-row tile at a
// time, with no barrier until the weight block changes.
//
// Two accumulators: the products of the high pieces have one, the five others, below 2^-8 of them, another (mfma_rows.hpp), so a
// sum of K terms is rounded K / 32 times at its own size.  rms error against fp64 (normal values), one accumulator -> two: 64 columns
// 1.12e-7 -> 5.0e-8, 96 1.41e-7 -> 5.8e-8, 128 1.65e-7 -> 6.5e-8 (with row_scale 7.4e-8).  Two fp16 pieces of rows and columns scaled to their
// largest values and three products are faster at 128 columns (25 000 nodes 90 -> 75 us; equal at 64 and 96) but hold an operand to
// 2^-23 and drop products of 2^-22 (a row of one value: 7.5 2^-24 off), and a value 2^-20 of its row's largest has 19 bits left: not fp32.
//
// Two waves per SIMD on 16-row tiles: a wave alone on its SIMD, on 32-row tiles (32x32x16 instructions, half the weight
// fragments per row), issues an instruction every six cycles.  us, four waves -> eight, shared weights / a weight block per element / row_scale /
// both: 10 752 x 64 21.3 / 25.5 / 23.8 / 27.9 -> 20.1 / 22.2 / 21.7 / 26.2, 25 000 x 96 64 / 70 / 70 / 76 -> 58 / 64 / 64 / 68, 25 000 x 128 91 / 101 / 102 /
// 108 -> 90 / 96 / 92 / 98, where matrix instructions and fragment reads take 31 us each of the 62 that its bytes need.  Twelve waves are
// equal at 64 and 96 columns and spill at 128.
//
// What a wave has in flight lives in registers, not in LDS: the loads of tile i + 1 (8 x 16 bytes per lane at 128
// columns, whole 128-byte lines of 8 rows per instruction) are issued before tile i is multiplied and land in
// accumulator-file registers; 64 KB per compute unit are on their way at any time.  When its turn comes a tile changes
// from that row-major layout to the operand layout of the matrix instruction (a lane holds 8 values of one row per
// 32-wide k step) through the wave's own corner of LDS, up to 96 columns at a time.
// The operands are swapped with respect to the kernels above (weights as the row operand, X rows as the column operand): a lane's
// accumulators are then 4 consecutive output columns of one row; a block of 32 columns goes back through the same corner of LDS
// and leaves as whole lines.
//
// Contract of the hand-issued memory operations of the tile loop (the loads and the stores): a load names its landing
// registers at issue time although the data arrives by the explicit wait that precedes their first use, which is
// sound only while the compiler neither copies nor spills them in between; they are accumulator-file registers,
// which nothing else in the kernel wants, and the build refuses scratch memory in this kernel and any instruction other
// than a load that writes a register its loads land in.  A store is followed by the two idle issue slots that the hardware needs before the
// stored registers may be overwritten (the compiler inserts them for the stores it knows; without them the last lanes of
// the following block were stored instead).
//
// Loads of 32 bytes per lane and row, which is what a lane feeds per k step, request every line four times, and the kernel then
// ran at the rate of the compute unit's queue of outstanding misses (25 000 x 128 118 us; whole lines: 99 us); stores under a
// branch make the compiler wait for everything in flight at the top of the loop (hence no conditional rows, see the row numbers below).
// -----------------------------------------------------------------------------------------------
constexpr int kResWaves = 8;
constexpr int kResRows = 16;   // rows of a tile
constexpr int kResSegRows = 2048;  // rows whose numbers a segment keeps in LDS
using rows::v4f;
constexpr int kResMaxGroups = 128;
constexpr int kResMinNodes = 2048;
constexpr int kOutLd = 36;            // floats per row of a wave's output staging block (32 columns + 16 bytes)

// Row ranges of the weight groups in the grouped node order and their first 16-row tiles in the list of all tiles (ncomp rows per node):
// off[g] and cum[g] for g = 0 .. ngroups, by one wave, 64 groups at a time.  (One thread that walks the groups waits for memory once or
// twice per group: ten groups, 2 500 nodes.)
__device__ __forceinline__ void first_tiles(const int32_t *__restrict__ group_offsets, int ngroups, int nnodes, int ncomp, int lane, int *off, int *cum) {
  int before = 0;
  for (int g0 = 0; g0 < ngroups; g0 += kWave) {
    const int g = g0 + lane;
    const bool has = g < ngroups;
    const int lo = has && group_offsets ? group_offsets[g] : 0, hi = has ? (group_offsets ? group_offsets[g + 1] : nnodes) : 0;
    const int tiles = ncomp * ((max(hi - lo, 0) + kResRows - 1) / kResRows);
    int upto = tiles;  // inclusive prefix sum over the lanes
    for (int d = 1; d < kWave; d <<= 1) {
      const int v = __shfl_up(upto, d);
      if (lane >= d) upto += v;
    }
    if (has) off[g] = lo, cum[g] = before + upto - tiles;
    if (g == ngroups - 1) off[ngroups] = hi, cum[ngroups] = before + upto;
    before += __shfl(upto, kWave - 1);
  }
}

// A workgroup's piece of the list of all tiles, tiles [first, last).  With row_scale (SCALED) the 2 l + 1 tiles of a node tile share its
// row_scale rows: a node tile of l = 0 fetches and multiplies them for one tile, of l = 3 for seven, and with pieces of as many tiles each the
// launch waited for those of l = 0.  A node tile counts 2 l + 1 + 1/2 there (a quarter: the same within 2 %).  us, shared weights / ten
// weight groups, equal pieces -> these: 12 000 x 64 24.5 / 26.4 -> 24.1 / 27.9, 60 000 x 64 101 / 102 -> 94 / 94, 25 000 x 96 68.7 / 70.6 -> 65.1 /
// 68.0, 25 000 x 128 94.8 / 101 -> 91.6 / 98.1 (89 / 96 without row_scale), 60 000 x 128 236 / 252 -> 219 / 228.  With one weight block per l an l
// gets whole workgroups, so that none of them stages two blocks; with more, where pieces cross blocks anyway, the workgroups of
// an XCD take neighbouring pieces, whose rows of row_scale meet in its L2.  (The kernel with weights in registers waits for its matrix
// instructions: equal pieces there, 12 000 x 192 86.7 / 97.8 -> 85.1 / 90.2.)
struct Share {
  int first, last;
};
constexpr int kXcds = 8;
template <bool SCALED>
__device__ __forceinline__ Share own_share(const int *cum, int ngroups) {
  const auto whole = [](int64_t n, int index, int of) { return static_cast<int>(n * index / of); };
  const int of = gridDim.x, index = blockIdx.x, ntiles = cum[ngroups];
  if constexpr (!SCALED) return {whole(ntiles, index, of), whole(ntiles, index + 1, of)};
  const auto cost_before = [](int l) { return 2 * l * l + l; };  // of the l blocks before l, per node tile, in half tiles
  constexpr int kCost = 36;                                      // = cost_before(4)
  if (ngroups == 1 && of >= kCost) {
    int l = 0, first = 0, end = (of * cost_before(1) + kCost / 2) / kCost;  // workgroups [first, end) have l
    while (index >= end) ++l, first = end, end = (of * cost_before(l + 1) + kCost / 2) / kCost;
    const int before = ntiles / 16 * l * l, tiles = ntiles / 16 * (2 * l + 1);
    return {before + whole(tiles, index - first, end - first), before + whole(tiles, index + 1 - first, end - first)};
  }
  const auto tile_at = [&](int piece) {
    int64_t cost = static_cast<int64_t>(ntiles / 16) * kCost * piece / of;
    int g = 0, l = 0;
    while (g < ngroups - 1 && static_cast<int64_t>(cum[g + 1] / 16) * kCost <= cost) ++g;
    cost -= static_cast<int64_t>(cum[g] / 16) * kCost;
    const int64_t tiles = (cum[g + 1] - cum[g]) / 16;
    while (l < 3 && tiles * cost_before(l + 1) <= cost) ++l;
    const int64_t in_l = (cost - tiles * cost_before(l)) * (2 * l + 1) / (cost_before(l + 1) - cost_before(l));
    return static_cast<int>(cum[g] + min(tiles * (l * l) + in_l, tiles * 16));
  };
  const int piece = of % kXcds == 0 ? index % kXcds * (of / kXcds) + index / kXcds : index;
  return {tile_at(piece), tile_at(piece + 1)};
}

template <int K, int NT, bool SCALED>
__global__ __launch_bounds__(kResWaves *kWave, kResWaves / 4) void linear_resident_kernel(
    const float *__restrict__ X, const float *__restrict__ WT, const int32_t *__restrict__ node_perm,
    const int32_t *__restrict__ group_offsets, int nnodes, int ngroups, int zero_last_group, float scale,
    const float *__restrict__ row_scale, float *__restrict__ OUT) {
  constexpr int NOUT = 32 * NT;
  static_assert(K == NOUT, "square weights");
  constexpr int LD = K + 8;      // row stride of a plane in elements: an odd number of 16-byte units
  constexpr int KS = K / 32;
  __shared__ __attribute__((aligned(16))) __bf16 sW[3 * NOUT * LD];
  __shared__ int sId[kResSegRows];
  constexpr int kChunk = K <= 96 ? K : 64;  // columns of X per trip through LDS
  constexpr int kTLd = kChunk + 4;          // floats per row of the transposition block: an odd number of 16-byte units
  constexpr int kStageFloats = kResRows * (kTLd > kOutLd ? kTLd : kOutLd);  // a wave's own corner of LDS
  __shared__ __attribute__((aligned(16))) float sStage[kResWaves * kStageFloats];
  __shared__ int sOff[kResMaxGroups + 1];
  __shared__ int sCum[kResMaxGroups + 1];

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r16 = lane % 16, quarter = lane / 16;

  // groups that have weights, their row ranges in the grouped node order and their first tile in the tile list
  const int ngw = zero_last_group ? ngroups - 1 : ngroups;
  if (wave == 0) first_tiles(group_offsets, ngw, nnodes, 16, lane, sOff, sCum);
  if (zero_last_group) {
    // rows that belong to no weight group: the product is defined as zero (a residual still passes through)
    const int z0 = group_offsets[ngroups - 1], nz = group_offsets[ngroups] - z0;
    constexpr int rowq = 16 * NOUT / 4;
    const int64_t total = static_cast<int64_t>(nz) * rowq;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + tid; i < total; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
      const int node = node_perm[z0 + static_cast<int>(i / rowq)];
      if (static_cast<unsigned>(node) < static_cast<unsigned>(nnodes)) st4(OUT + static_cast<int64_t>(node) * 16 * NOUT + 4 * (i % rowq), zero4());
    }
  }
  __syncthreads();

  const Share share = own_share<SCALED>(sCum, ngw);
  const int i1 = share.last;
  int i = share.first;
  int g = 0, staged_g = -1, staged_l = -1;

  while (i < i1) {
    while (sCum[g + 1] <= i) ++g;
    const int tg = (sCum[g + 1] - sCum[g]) / 16;  // node tiles of the group
    const int l = l_of_m((i - sCum[g]) / tg);
    const int nm = 2 * l + 1;
    const int blk0 = sCum[g] + tg * l * l;        // first tile of (g, l): tile blk0 + t * nm + (m - l * l)
    const int t_first = (i - blk0) / nm;
    const int seg_end = min(min(i1, blk0 + tg * nm), blk0 + (t_first + kResSegRows / kResRows) * nm);
    const int t_count = (seg_end - 1 - blk0) / nm - t_first + 1;
    const int off0 = sOff[g], off1 = sOff[g + 1];
    const bool new_weights = g != staged_g || l != staged_l;

    // W^T[j, :] of block (g, l) -> three planes.  All loads of a thread first, ahead of the row numbers: one trip through L2.
    const float *Wg = WT + (static_cast<int64_t>(g) * 4 + l) * NOUT * K;
    constexpr int kPieces = (NOUT * (K / 4) + kResWaves * kWave - 1) / (kResWaves * kWave);
    const auto piece_of = [&](int it) {  // beyond the block: its last piece once more
      const int q = it * (kResWaves * kWave) + tid;
      return NOUT * (K / 4) % (kResWaves * kWave) == 0 ? q : min(q, NOUT * (K / 4) - 1);
    };
    f4 wv[kPieces];
    if (new_weights) {
#pragma unroll
      for (int it = 0; it < kPieces; ++it) {
        const int q = piece_of(it);
        wv[it] = ld4(Wg + static_cast<int64_t>(q / (K / 4)) * K + 4 * (q % (K / 4)));
      }
    }
    __syncthreads();  // every wave is done with the previous segment
    // Row numbers of the segment's node tiles.  A row beyond the end of the group (or an index outside the node range)
    // stands in for the first row of its tile: it then computes that row's values once more and stores the same bits
    // to the same place, so that no load or store of the tile loop is conditional.
    for (int r = tid; r < kResRows * t_count; r += kResWaves * kWave) {
      const int p0 = off0 + kResRows * (t_first + r / kResRows);
      const int p = p0 + r % kResRows;
      int node = node_perm ? node_perm[p < off1 ? p : p0] : (p < off1 ? p : p0);
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = node_perm ? node_perm[p0] : p0;
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = 0;
      sId[r] = node;
    }
    if (new_weights) {
#pragma unroll
      for (int it = 0; it < kPieces; ++it) {
        const int q = piece_of(it);
        const int at = q / (K / 4) * LD + 4 * (q % (K / 4));
        bf16x4 h, md, lw;
        split3(wv[it], h, md, lw);
        *reinterpret_cast<bf16x4 *>(sW + at) = h;
        *reinterpret_cast<bf16x4 *>(sW + NOUT * LD + at) = md;
        *reinterpret_cast<bf16x4 *>(sW + 2 * NOUT * LD + at) = lw;
      }
      staged_g = g;
      staged_l = l;
    }
    __syncthreads();

    // this wave's contiguous share of the segment
    const int per = (seg_end - i + kResWaves - 1) / kResWaves;
    const int wb = i + wave * per, we = min(seg_end, wb + per);
    i = seg_end;
    if (wb >= we) continue;

    // Tile loop.  Every global access in it is issued from assembly in a fixed order and waited for by an explicit count
    // (the compiler would sink part of a prefetch down to its use and then wait for everything that is in flight, the
    // stores of the previous tile included):
    //     tile i:  wait: all but the stores of tile i - 1 | landing registers (times row_scale) -> LDS -> pieces
    //              | issue the loads of tile i + 1 | multiply | output block by block through LDS, issue the stores
    // Loads are whole lines: one instruction fetches 128 bytes of each of 8 rows (lane = 16-byte piece opiece of row
    // 8 rg + orow; in 32-byte pieces, which is what a lane feeds per k step, every line would be requested four times and
    // the compute unit's queue of outstanding misses would hold a quarter of the bytes).  The landed values change to the
    // operand layout through the wave's own corner of LDS, kChunk columns at a time.
    constexpr int kRg = kResRows / 8;
    constexpr int kLines = kChunk / 32;  // 128-byte lines of a row per chunk
    constexpr int kChunks = K / kChunk;
    static_assert(K % kChunk == 0 && kChunk % 32 == 0, "chunks of whole lines");
    f4 land[kRg * K / 32];                     // index (chunk * kRg + rg) * kLines + line
    f4 sland[SCALED ? kRg * K / 32 : 1];
    float *stg = sStage + wave * kStageFloats;
    const int orow = lane / 8, opiece = lane % 8;
    int t_scales = -1;  // node tile whose row_scale rows are in (or on their way into) sland
    auto issue = [&](int idx, int &m_of, int &tb_of) {
      const int j = idx - blk0;
      const int t = j / nm;
      m_of = l * l + (j - t * nm);
      tb_of = kResRows * (t - t_first);
#pragma unroll
      for (int rg = 0; rg < kRg; ++rg) {
        const int nd = sId[tb_of + 8 * rg + orow];
        const float *xp = X + (static_cast<int64_t>(nd) * 16 + m_of) * K + 4 * opiece;
#pragma unroll
        for (int c = 0; c < kChunks; ++c)
#pragma unroll
          for (int ln = 0; ln < kLines; ++ln)
            asm volatile("global_load_dwordx4 %0, %1, off offset:%2 nt" : "=a"(land[(c * kRg + rg) * kLines + ln]) : "v"(xp), "n"(4 * (c * kChunk + 32 * ln)) : "memory");
      }
      if constexpr (SCALED) {
        // the 2 l + 1 tiles of a node tile follow each other and share their row_scale rows: fetched once (these loads
        // are older than the stores the wait at the top of a tile lets stay out, whether they are issued or not)
        if (t != t_scales) {
          t_scales = t;
#pragma unroll
          for (int rg = 0; rg < kRg; ++rg) {
            const float *sp = row_scale + static_cast<int64_t>(sId[tb_of + 8 * rg + orow]) * K + 4 * opiece;
#pragma unroll
            for (int c = 0; c < kChunks; ++c)
#pragma unroll
              for (int ln = 0; ln < kLines; ++ln)
                asm volatile("global_load_dwordx4 %0, %1, off offset:%2" : "=a"(sland[(c * kRg + rg) * kLines + ln]) : "v"(sp), "n"(4 * (c * kChunk + 32 * ln)) : "memory");
          }
        }
      }
    };
    // a base per plane: the third lies beyond the offset an LDS read can hold, and an address per fragment would take 32 registers
    const __bf16 *wl[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      unsigned at = (q * NOUT + r16) * LD + 8 * quarter;
      asm("" : "+v"(at));
      wl[q] = sW + at;
    }
    int m_next, tb_next;
    issue(wb, m_next, tb_next);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    for (int idx = wb; idx < we; ++idx) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRg * NT) : "memory");
      const int m_cur = m_next, tb_cur = tb_next;
      bf16x8 x[KS][3];
#pragma unroll
      for (int c = 0; c < kChunks; ++c) {
        wave_lds_fence();
#pragma unroll
        for (int rg = 0; rg < kRg; ++rg)
#pragma unroll
          for (int ln = 0; ln < kLines; ++ln) {
            const int j = (c * kRg + rg) * kLines + ln;
            asm volatile("; landed %0" : "+a"(land[j]));
            f4 v = land[j];
            if constexpr (SCALED) {
              asm volatile("; landed %0" : "+a"(sland[j]));
              v *= sland[j];
            }
            *reinterpret_cast<f4 *>(stg + (8 * rg + orow) * kTLd + 32 * ln + 4 * opiece) = v;
          }
        wave_lds_fence();
        // k step s of the chunk: the lane's values are columns 32 s + 8 quarter + {0..7}
        f4 cur[kChunk / 16];
#pragma unroll
        for (int i = 0; i < kChunk / 16; ++i) cur[i] = ld4(stg + r16 * kTLd + 32 * (i / 2) + 8 * quarter + 4 * (i % 2));
        if (c == kChunks - 1 && idx + 1 < we) issue(idx + 1, m_next, tb_next);
#pragma unroll
        for (int sc = 0; sc < kChunk / 32; ++sc) split3(cur[2 * sc], cur[2 * sc + 1], x[c * (kChunk / 32) + sc]);
      }
      __builtin_amdgcn_sched_barrier(0);
      float *orows[kRg];
#pragma unroll
      for (int r = 0; r < kRg; ++r)
        orows[r] = OUT + (static_cast<int64_t>(sId[tb_cur + 8 * r + orow]) * 16 + m_cur) * NOUT + 4 * opiece;

      constexpr int GB = NT % 2 == 0 ? 4 : 2;  // column blocks of 16 at a time
#pragma unroll
      for (int t0 = 0; t0 < 2 * NT; t0 += GB) {
        v4f acc[GB], small[GB];
#pragma unroll
        for (int t = 0; t < GB; ++t) acc[t] = small[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          bf16x8 w[GB][3];
#pragma unroll
          for (int t = 0; t < GB; ++t)
#pragma unroll
            for (int q = 0; q < 3; ++q) w[t][q] = *reinterpret_cast<const bf16x8 *>(wl[q] + 16 * (t0 + t) * LD + 32 * s);
          rows::add_products(w, x[s], acc, small);
          if (K == 128) __builtin_amdgcn_sched_barrier(0);  // fragment reads of later steps hoisted further would not fit the register file
        }
        // accumulator r of a lane: output column 16 t + 4 quarter + r of row r16 of the tile.  A block of 32 columns goes
        // through the wave's own corner of LDS (rows padded to 9 x 16 bytes: conflict-free both ways) and leaves as whole
        // 128-byte lines, 8 rows per store.
#pragma unroll
        for (int t = 0; t < GB; t += 2) {
          wave_lds_fence();
#pragma unroll
          for (int q = 0; q < 2; ++q) st4(stg + r16 * kOutLd + 16 * q + 4 * quarter, f4((acc[t + q] + small[t + q]) * scale));
          wave_lds_fence();
#pragma unroll
          for (int r = 0; r < kRg; ++r) {
            const f4 v = *reinterpret_cast<const f4 *>(stg + (8 * r + orow) * kOutLd + 4 * opiece);
            // the two idle issue slots are what the compiler puts between a 16-byte store and an instruction that
            // overwrites the registers it stores from; it does not see this store
            asm volatile("global_store_dwordx4 %0, %1, off offset:%2\n\ts_nop 1" : : "v"(orows[r]), "v"(v), "n"(64 * (t0 + t)) : "memory");
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // every landing register has been consumed: nothing this wave issued can still write a register
  }
}

// -----------------------------------------------------------------------------------------------
// Variant with the weights resident in registers (160 to 256 columns, K = Nout; COMP = 16 components per node or one).
//
// Three planes of 160 x 160 weights and more do not fit LDS next to anything else, and the tiled kernels stage the block
// again for every 128 rows in barrier-separated phases that one or two waves per SIMD cannot overlap: 192 columns ran at
// 2.8-3.0 TB/s of their bytes, 256 at 2.2.  The register file of a compute unit holds 512 KB: here a workgroup takes a
// contiguous piece of the list of all 16-row tiles (as the kernel above does), wave w keeps the pieces of its 16 CB weight
// columns for all of K in its registers (6 CB K / 16 of them) until the weight block changes, and all waves multiply the
// same tile of X rows, whose piece planes they share through LDS, double-buffered with one barrier per tile.  X goes
// global -> LDS as raw fp32 by direct loads; a wave splits exactly the pieces it fetched itself, so only the planes are
// shared.  The waves of a SIMD take turns in the order of their phases: every other one multiplies the current tile before
// it splits the next.
//
// Operands as in the kernel above (weights as the row operand): a lane's accumulators are four consecutive output columns of
// one row, stored as 16 bytes.  v_mfma_f32_16x16x32_bf16: K steps of 32, pieces, products and accumulators as above.
//
// Vector-memory operations of the tile loop are issued from assembly: the loads of tile k + 2 right after the split of tile
// k + 1, then the stores of a tile; the wait before a split lets exactly those stores stay out.
//
// CB: 16 columns per wave give 10, 12 and 14 waves, three or four per SIMD (32 columns per wave: 5, 6 and 7 waves, two on
// some SIMDs and one on others; 5-8 % slower at 160 and 192); at 256 columns 32 per wave (8 waves) are equal up to 20 000
// nodes and 1 % faster with row_scale.  32-row tiles: 1-3 % slower.  Two or three tiles requested ahead instead of one: no
// faster (656 -> 664 us at 100 000 x 192).
//
// Measured against the tiled kernels (plain / row_scale): 100 000 x 192 810 / 860 -> 655 / 675 us, 50 000 x 160 326 / 345 ->
// 285 / 290, 20 000 x 224 255 / 272 -> 180 / 190, 40 000 x 256 595 / 643 -> 415 / 445, 12 000 x 256 183 / 198 -> 122 / 145,
// equal at 2 048 nodes.  Without its matrix instructions 192 columns take 520 us (4.7 TB/s, the rate of a copy), without
// loads, stores and split 514 us: what is left is their overlap.  All that with one accumulator; with two, us and rms error against fp64:
// 100 000 x 192 672 -> 685, 1.96e-7 -> 7.8e-8, 20 000 x 192 129 -> 133, 10 007 x 224 92 -> 93, 2.14e-7 -> 8.4e-8, 12 000 x 256 130 -> 130, 2.31e-7 -> 8.9e-8,
// 10 007 x 160 57 -> 57, 1.77e-7 -> 7.2e-8.  (Two fp16 pieces of scaled rows and columns and three products, not fp32 any more: 584, -, -, 98 and 53.)
// -----------------------------------------------------------------------------------------------
constexpr int kWideMinScalarNodes = 8192;
constexpr int kWideSegRows = 2048;  // rows whose node numbers a segment keeps in LDS

template <int NT, int CB, int COMP, bool SCALED>
__global__ __launch_bounds__(2 * NT / CB * kWave, (2 * NT / CB + 3) / 4) void linear_wide_kernel(const float *__restrict__ X, const float *__restrict__ WT,
                                                                   const int32_t *__restrict__ node_perm,
                                                                   const int32_t *__restrict__ group_offsets, int nnodes, int ngroups,
                                                                   int zero_last_group, float scale,
                                                                   const float *__restrict__ row_scale, const float *residual, float *OUT) {
  constexpr int K = 32 * NT;                  // = Nout
  constexpr int TR = 16;                      // rows of a tile
  constexpr int WAVES = 2 * NT / CB;          // a wave owns CB blocks of 16 output columns
  constexpr int RB = TR / 16;                 // row blocks
  constexpr int LD = K + 8;                   // row stride of a plane in elements: an odd number of 16-byte units
  constexpr int KS = K / 32;
  constexpr int PIECES = TR * K / 4 / (WAVES * kWave);  // 16-byte pieces of a tile per thread
  constexpr int STORES = CB * RB;             // per wave and tile
  constexpr int kSegTiles = kWideSegRows / TR;
  __shared__ __attribute__((aligned(16))) __bf16 sP[2][3][TR * LD];
  __shared__ __attribute__((aligned(16))) float sRaw[TR * K];
  __shared__ __attribute__((aligned(16))) float sScale[SCALED ? TR * K : 4];
  __shared__ int sId[kWideSegRows];
  __shared__ int sOff[kResMaxGroups + 1];
  __shared__ int sCum[kResMaxGroups + 1];

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r16 = lane % 16, quarter = lane / 16;
  const bool late = (wave / 4 & 1) != 0;  // multiplies before it splits

  const int ngw = zero_last_group ? ngroups - 1 : ngroups;
  if (wave == 0) first_tiles(group_offsets, ngw, nnodes, COMP, lane, sOff, sCum);
  if (zero_last_group) {
    // rows that belong to no weight group: the product is defined as zero (a residual still passes through)
    const int z0 = group_offsets[ngroups - 1], nz = group_offsets[ngroups] - z0;
    constexpr int rowq = COMP * K / 4;
    const int64_t total = static_cast<int64_t>(nz) * rowq;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + tid; i < total; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
      const int node = node_perm[z0 + static_cast<int>(i / rowq)];
      if (static_cast<unsigned>(node) < static_cast<unsigned>(nnodes)) {
        const int64_t at = static_cast<int64_t>(node) * COMP * K + 4 * (i % rowq);
        st4(OUT + at, residual ? ld4(residual + at) : zero4());
      }
    }
  }
  __syncthreads();

  // this thread's pieces of a tile: row and 16-byte column piece
  int prow[PIECES], pcol[PIECES];
#pragma unroll
  for (int j = 0; j < PIECES; ++j) {
    const int p = (j * WAVES + wave) * kWave + lane;
    prow[j] = p / (K / 4);
    pcol[j] = 4 * (p % (K / 4));
  }
  const unsigned raw_lds = static_cast<unsigned>(reinterpret_cast<uintptr_t>(sRaw)) + wave * (kWave * 16);
  const unsigned scale_lds = static_cast<unsigned>(reinterpret_cast<uintptr_t>(sScale)) + wave * (kWave * 16);

  const Share share = own_share<false>(sCum, ngw);
  const int i1 = share.last;
  int i = share.first;
  int g = 0, held_g = -1, held_l = -1;
  bf16x8 w[KS][CB][3];  // weight pieces: k step, column block, piece

  while (i < i1) {
    while (sCum[g + 1] <= i) ++g;
    const int tg = (sCum[g + 1] - sCum[g]) / COMP;  // node tiles of the group
    const int l = COMP == 1 ? 0 : l_of_m((i - sCum[g]) / tg);
    const int nm = 2 * l + 1;
    const int blk0 = sCum[g] + tg * l * l;        // first tile of (g, l): tile blk0 + t * nm + (m - l * l)
    const int t_first = (i - blk0) / nm;
    const int seg_end = min(min(i1, blk0 + tg * nm), blk0 + (t_first + kSegTiles) * nm);
    const int t_count = (seg_end - 1 - blk0) / nm - t_first + 1;
    const int off0 = sOff[g], off1 = sOff[g + 1];

    __syncthreads();  // every wave is done with the previous segment
    // Row numbers of the segment's node tiles; a row beyond the end of the group stands in for the first row of its tile
    // (the same values to the same place once more), so that no load or store of the tile loop is conditional.
    for (int r = tid; r < TR * t_count; r += WAVES * kWave) {
      const int p0 = off0 + TR * (t_first + r / TR);
      const int p = p0 + r % TR;
      int node = node_perm ? node_perm[p < off1 ? p : p0] : (p < off1 ? p : p0);
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = node_perm ? node_perm[p0] : p0;
      if (static_cast<unsigned>(node) >= static_cast<unsigned>(nnodes)) node = 0;
      sId[r] = node;
    }
    if (g != held_g || l != held_l) {
      // a lane feeds 8 consecutive k of one weight column per step
      int at = (16 * CB * wave + r16) * K + 8 * quarter;
      asm volatile("" : "+v"(at));  // computed here: ahead of the loops it would be registers that 224 columns do not have
      const float *Wg = WT + (static_cast<int64_t>(g) * (COMP == 1 ? 1 : 4) + l) * K * K + at;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int s = 0; s < KS; ++s) split3(ld4(Wg + 16 * cb * K + 32 * s), ld4(Wg + 16 * cb * K + 32 * s + 4), w[s][cb]);
      held_g = g;
      held_l = l;
    }
    __syncthreads();

    const int n = seg_end - i;
    int t_scales = -1;  // node tile whose row_scale rows are in (or on their way into) sScale
    auto where = [&](int k, int &m, int &tb) {  // component and first entry of sId of the segment's tile k
      const int j = i + k - blk0;
      const int t = j / nm;
      m = l * l + (j - t * nm);
      tb = TR * (t - t_first);
    };
    auto issue = [&](int k) {
      int m, tb;
      where(k, m, tb);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's reads of the raw rows are done
#pragma unroll
      for (int j = 0; j < PIECES; ++j)
        dma16(X + (static_cast<int64_t>(sId[tb + prow[j]]) * COMP + m) * K + pcol[j], raw_lds + j * (WAVES * kWave * 16));
      if constexpr (SCALED) {
        if (tb != t_scales) {
          t_scales = tb;
#pragma unroll
          for (int j = 0; j < PIECES; ++j)
            dma16(row_scale + static_cast<int64_t>(sId[tb + prow[j]]) * K + pcol[j], scale_lds + j * (WAVES * kWave * 16));
        }
      }
    };
    auto split = [&](int k) {
      __bf16 *plane = &sP[k & 1][0][0];
#pragma unroll
      for (int j = 0; j < PIECES; ++j) {
        const int p = (j * WAVES + wave) * kWave + lane;
        f4 v = *reinterpret_cast<const f4 *>(sRaw + 4 * p);
        if constexpr (SCALED) v *= *reinterpret_cast<const f4 *>(sScale + 4 * p);
        bf16x4 h, md, lw;
        split3(v, h, md, lw);
        const int at = prow[j] * LD + pcol[j];
        *reinterpret_cast<bf16x4 *>(plane + at) = h;
        *reinterpret_cast<bf16x4 *>(plane + TR * LD + at) = md;
        *reinterpret_cast<bf16x4 *>(plane + 2 * TR * LD + at) = lw;
      }
    };
    auto multiply = [&](int k) {
      int m, tb;
      where(k, m, tb);
      const __bf16 *plane = &sP[k & 1][0][0] + r16 * LD + 8 * quarter;
      static_assert(RB == 1, "a lane's sums belong to one row");
      v4f acc[CB], small[CB];
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[cb] = small[cb] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 x[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) x[q] = *reinterpret_cast<const bf16x8 *>(plane + q * (TR * LD) + 32 * s);
        rows::add_products(w[s], x, acc, small);
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int64_t row_at = (static_cast<int64_t>(sId[tb + 16 * rb + r16]) * COMP + m) * K + 16 * CB * wave + 4 * quarter;
        float *op = OUT + row_at;
        f4 res[CB];
        if constexpr (COMP == 1) {
          // May be OUT itself.  A place that stands in for the first row of its tile reads and writes that row from another
          // lane of the same wave: all of them have the residual before any of them stores, as long as a tile is one block
          // of rows (with a single weight group, which is how this form is launched, no row stands in for another tile's).
          static_assert(RB == 1, "stand-in rows of a later block would read what the first block has stored");
#pragma unroll
          for (int cb = 0; cb < CB; ++cb) res[cb] = residual ? ld4(residual + row_at + 16 * cb) : zero4();
        }
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          v4f v;
          {
#pragma clang fp contract(off)  // the product is rounded before the residual is added, as everywhere
            v = (acc[cb] + small[cb]) * scale;
            if (COMP == 1 && residual) v = v + res[cb];
          }
          // (the two idle issue slots: see the stores of the kernel above)
          asm volatile("global_store_dwordx4 %0, %1, off offset:%2\n\ts_nop 1" : : "v"(op), "v"(v), "n"(64 * cb) : "memory");
        }
      }
    };

    issue(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    split(0);
    if (n > 1) issue(1);
    // before the first split of the loop only loads are out; the wait below is exact from the second tile on
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    for (int k = 0; k < n; ++k) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // planes of tile k complete, those of tile k - 1 free
      if (late) multiply(k);
      if (k + 1 < n) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STORES) : "memory");  // the loads of tile k + 1; the stores after them may stay out
        split(k + 1);
        if (k + 2 < n) issue(k + 2);
      }
      if (!late) multiply(k);
    }
    i = seg_end;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// -----------------------------------------------------------------------------------------------
// A workgroup per 128 rows of one weight block (square weights; 16 components per node or one): from some hundred to some thousand nodes.
//
// There a launch is a few microseconds of waiting: the kernels with resident weights walk a list of tiles that crosses weight blocks (a
// new block is a trip through L2, three barriers and the split of all its columns again, with nothing else to do meanwhile), the tiled
// ones walk K in phases.  Here a workgroup has one weight block and each of its eight waves one tile of 16 rows, so everything is asked
// for at once: group offsets, then the weights and the row numbers, then the rows, one barrier, the products, the stores.  Rows of a
// degree are counted node by node (row r of degree l is component l^2 + r % (2l + 1) of the block's node r / (2l + 1)): the rows of a wave lie
// side by side in memory.  Operands and arithmetic: mfma_rows.hpp (a load covers 64 bytes of a row).
// Columns are split over COLS / 16 NB workgroups where the rows alone leave compute units idle, and where the planes of all would not fit LDS.
// -----------------------------------------------------------------------------------------------
constexpr int kBlockWaves = 8;
constexpr int kBlockRows = 16 * kBlockWaves;

__host__ __device__ __forceinline__ int row_blocks(int nodes, int ncomp) {
  const auto of = [&](int nm) { return (nodes * nm + kBlockRows - 1) / kBlockRows; };
  return ncomp == 1 ? of(1) : of(1) + of(3) + of(5) + of(7);
}

template <int KS, int NB, bool SCALED>
__global__ __launch_bounds__(kBlockWaves *kWave, KS <= 3 || (KS == 4 && NB == 4 && !SCALED) || (KS == 5 && NB == 5 && !SCALED) ? 4 : 2) void linear_block_kernel(
    const float *__restrict__ X, const float *__restrict__ WT, const int32_t *__restrict__ node_perm, const int32_t *__restrict__ group_offsets,
    int nnodes, int ngroups, int zero_last_group, int ncomp, float scale, const float *__restrict__ row_scale, const float *residual, float *OUT) {
  constexpr int K = 32 * KS;
  constexpr int NOUT = K;
  constexpr int COLS = 16 * NB;  // columns of this workgroup
  __shared__ __attribute__((aligned(16))) rows::Planes<KS, COLS> planes;

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r16 = lane % 16, quarter = lane / 16;
  const int col0 = blockIdx.y * COLS;

  // weight group, its first place in the node order and its number of nodes; the block among the group's
  int g = 0, off0 = 0, n = nnodes, block = blockIdx.x;
  if (group_offsets) {  // 64 groups at a time, one per lane
    for (int g0 = 0;; g0 += kWave) {
      if (g0 >= ngroups) return;
      const bool has = g0 + lane < ngroups;
      const int lo = has ? group_offsets[g0 + lane] : 0, hi = has ? group_offsets[g0 + lane + 1] : 0;
      const int blocks = row_blocks(max(hi - lo, 0), ncomp);
      int upto = blocks;  // inclusive prefix sum over the lanes
      for (int d = 1; d < min(ngroups - g0, kWave); d <<= 1) {
        const int v = __shfl_up(upto, d);
        if (lane >= d) upto += v;
      }
      const unsigned long long owners = __ballot(has && block < upto);
      if (owners != 0) {
        const int owner = __ffsll(static_cast<long long>(owners)) - 1;
        g = g0 + owner;
        block -= __builtin_amdgcn_readlane(upto - blocks, owner);
        off0 = __builtin_amdgcn_readlane(lo, owner);
        n = __builtin_amdgcn_readlane(hi, owner) - off0;
        break;
      }
      block -= __builtin_amdgcn_readlane(upto, kWave - 1);
    }
  }
  int l = 0, nm = 1;
  if (ncomp != 1) {
    while (block >= (n * nm + kBlockRows - 1) / kBlockRows) {
      block -= (n * nm + kBlockRows - 1) / kBlockRows;
      ++l, nm += 2;
    }
  }
  const bool zero = zero_last_group && g == ngroups - 1;

  // this lane's row: its number first (the rows are waited for longest), then the weights
  const int r = block * kBlockRows + 16 * wave + r16;
  const int t = r / nm;
  int node = off0 + t;
  bool valid = t < n;
  if (node_perm) node = node_perm[valid ? node : off0];
  rows::Fetched<KS, COLS, kBlockWaves * kWave> weights;
  if (!zero) weights.request(WT + ((static_cast<int64_t>(g) * (ncomp == 1 ? 1 : 4) + l) * NOUT + col0) * K);
  valid = valid && static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  if (!valid) node = 0;  // read, never stored
  const int64_t row = static_cast<int64_t>(node) * ncomp + (valid ? l * l + (r - t * nm) : 0);
  float *const op = OUT + row * NOUT + col0 + 4 * quarter;
  const float *const rp = residual ? residual + row * NOUT + col0 + 4 * quarter : nullptr;
  if (zero) {  // the product is defined as zero (a residual still passes through)
    if (!valid) return;
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) st4(op + 16 * cb, rp ? ld4(rp + 16 * cb) : zero4());
    return;
  }
  f4 x[2 * KS], factor[SCALED ? 2 * KS : 1];
  rows::load(X + row * K, x);
  if constexpr (SCALED) rows::load(row_scale + static_cast<int64_t>(node) * K, factor);
  weights.store(planes);
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) x[i] *= factor[i];
  }
  const rows::Operand<KS> operand(x);
  __syncthreads();

  constexpr int GB = rows::blocks_at_a_time(NB);
#pragma unroll
  for (int c0 = 0; c0 < NB; c0 += GB) {
    f4 res[GB], v[GB];
#pragma unroll
    for (int c = 0; c < GB; ++c) res[c] = rp ? ld4(rp + 16 * (c0 + c)) : zero4();
    rows::product(planes, operand, c0, scale, v);
#pragma unroll
    for (int c = 0; c < GB; ++c) {
      {
#pragma clang fp contract(off)  // the product is rounded before the residual is added, as everywhere
        if (rp) v[c] = v[c] + res[c];
      }
      if (valid) st4(op + 16 * (c0 + c), v[c]);
    }
  }
}

// Whether the kernels that keep square weights in LDS (64 to 128 columns) or in registers (160 and more) take a call.
bool resident_weights(int64_t nnodes, int ncomp, int K, int ngroups, bool grouped, bool residual) {
  if (ncomp == 16) return K >= 64 && !residual && ngroups <= kResMaxGroups && nnodes >= kResMinNodes;
  return K >= 160 && !grouped && nnodes >= kWideMinScalarNodes;
}

// Column blocks (of 16) per workgroup of linear_block_kernel, or 0: another kernel.  Each line from both sides, us, shared weights / ten weight
// groups / row_scale / both, the kernel that would run otherwise -> this one:
//  - half of the columns where that leaves no more than one workgroup per compute unit (all -> half: 700 x 128 9.2 / 10.2 / 10.6 / 11.2 ->
//    6.9 / 7.7 / 8.4 / 8.9, 1 000 x 128 with groups, two on some: 10.4 -> 11.0).
//  - up to one round of workgroups always: 2 000 x 64 6.2 / 7.9 / 6.9 / 8.5 -> 5.5 / 7.6 / 6.0 / 8.9, 1 500 x 128 11.9 / 16.8 / 13.0 / 18.5 -> 10.2 /
//    11.3 / 11.8 / 12.9, 1 500 x 160 17.3 / 21.5 / 18.5 / 23.4 -> 14.3 / 15.9 / 16.3 / 17.9, 700 x 192 15.3 / 20.7 / 16.9 / 22.5 -> 11.6 / 12.9 / 14.0 / 15.3,
//    700 x 224 18.1 / 27.7 / 19.4 / 29.5 -> 14.2 / 16.5 / 17.4 / 19.0, 300 x 256 15.3 / 33 / 16.7 / 33 -> 10.6 / 13.1 / 13.6 / 14.8; one component 12 000 x 160
//    10.6 / 14.9 / 11.3 / 21.4 -> 9.3 / 10.0 / 11.9 / 12.4, 12 000 x 192 12.5 / 17.5 / 13.4 / 27.1 -> 11.2 / 11.9 / 14.3 / 15.0, 6 000 x 256 17.7 / 16.9 / 21.6 / 21.4 ->
//    10.8 / 12.5 / 14.8 / 16.7.  (One component, 224 columns, up to 4 096 nodes: the tiled kernel cuts its tiles to 32 columns there, 10.9 -> 12.5.)
//  - beyond it against resident weights at 64 and 96 columns, two workgroups per compute unit: up to four (8 192 nodes; 5 000 x 64 12.2 / 17.2 / 13.3 / 17.6 ->
//    11.0 / 12.3 / 12.5 / 13.4, 8 000 x 96 27.8 / 31.7 / 29.0 / 31.5 -> 22.8 / 24.8 / 25.1 / 27.0).  It stays ahead on its own beyond that, but not in a step, where X and the
//    result share the last-level cache with everything else (12 000 x 96 881 -> 900, 10 752 x 64 in 512 graphs 318 -> 320): the other kernel has the loads
//    of a tile under way while it works on the one before.  At 128 columns one workgroup fits a compute unit, and a second round pays
//    where at least half of it is filled: 2 500 16.7 / 20.1 / 18.0 / 22.5 -> 17.9 / 19.7 / 19.3 / 21.4, 3 500 23.3 / 26.1 / 22.1 / 27.3 -> 20.2 / 23.8 / 21.8 / 25.8,
//    5 000 27.1 / 31.5 / 27.7 / 34.2 -> 27.5 / 30.7 / 29.5 / 33.1.  Beyond 128 columns it does not: 2 500 x 160 21.2 / 26.6 / 22.7 / 29.8 -> 25.4 / 27.3 / 27.1 / 29.5, 2 500 x
//    224 32 / 40 / 34 / 43 -> 40 / 45 / 44 / 50, 16 000 and 24 000 x 192 of one component 14.7 / 20.7 -> 12.3 / 19.9 and 18.2 / 21.6 -> 20.0 / 22.6.
//  - beyond it where resident weights are not to be had, against the tiled kernels.  Up to 128 columns always (16 components with a residual / 130 groups: 9 000 x 32
//    22 / 42 -> 12 / 12, 15 000 x 64 39 / 82 -> 32 / 33, 30 000 x 96 149 / 164 -> 127 / 99, 30 000 x 128 202 / 191 -> 160 / 171; 32 columns, plain, 30 000 28.2 -> 21.2, 100 000
//    80.0 -> 81.9; one component 100 000 x 96 26.7 -> 20.2, 33 000 x 128 16.2 -> 16.8: it has the arithmetic of the chains of such products, node_glue.hip).  With many
//    weight groups, each of which costs the others sixteen part-filled tiles and this one four, always (130: 1 000 x 160 94 -> 42, 20 000 x 160 208 -> 179, 20 000
//    x 192 271 -> 258, 2 500 x 256 288 -> 100).  With a residual on 16 components up to 6 000 nodes (5 000 x 192 66 -> 56, 5 000 x 256 114 -> 103; 9 000 101 -> 102, 188 ->
//    192), at 160 columns always (20 000 160 -> 155).  With few groups below 2 048 nodes at 224 columns (1 500 49 -> 31, 2 000 49 -> 42) and, unless the tiled kernel's
//    workgroups are one round, at 256 (700 32 -> 24, 1 000 34 -> 33, 1 500 in two rounds 59 -> 44, 2 000 60 -> 53), not at 160 and 192 (2 000 22.4 ->
//    27.3, 28.4 -> 33.3); one component at 224 (33 000 50 -> 40; with row_scale 50 000 56 -> 70), at 192 24 000 21.6 -> 22.6.
int block_columns(int64_t nnodes, int ncomp, int K, int ngroups, bool grouped, bool scaled, bool residual) {
  // a workgroup per 128 rows, and on average half of the weight blocks end in one more
  const int64_t rows = ceil_div(nnodes * ncomp, kBlockRows) + (grouped ? static_cast<int64_t>(ngroups) * (ncomp == 1 ? 1 : 4) / 2 : 0);
  const int64_t units = device_compute_units();
  const int all = K / 16, most = K <= 160 ? all : (K == 256 ? all / 4 : all / 2);  // what fits LDS
  const int64_t round = units / (all / most);
  const bool resident = resident_weights(nnodes, ncomp, K, ngroups, grouped, residual);
  if (2 * rows <= round && K != 224 && K != 32) return most / 2;  // (so few rows of 32 columns are the few-rows kernel's)
  if (rows <= round) return K == 224 && ncomp == 1 && !grouped && nnodes <= 4096 ? 0 : most;
  if (resident) return (K < 128 && rows <= 4 * units) || (K == 128 && 2 * rows > 3 * units && rows <= 2 * units) ? most : 0;
  if (K <= 128) return most;
  if (ncomp == 1) return K == 224 && grouped && !scaled ? most : 0;
  if (ngroups > 16) return most;
  if (nnodes >= kResMinNodes) return K == 160 || nnodes <= 6000 ? most : 0;
  if (!grouped || K <= 192) return 0;
  return K == 224 || rows <= 2 * round || 4 * 16 * (ceil_div(nnodes, 128) + ngroups / 2) > 5 * units ? most : 0;
}

template <int KS, int NB>
int launch_block(const float *X, const float *WT, const int32_t *perm, const int32_t *offs, int64_t nnodes, int ngroups,
                 int zero_last_group, int ncomp, float scale, const float *row_scale, const float *residual, float *OUT, hipStream_t st) {
  // every weight block may end in one that is not full
  const int64_t blocks = offs ? nnodes * ncomp / kBlockRows + static_cast<int64_t>(ngroups) * (ncomp == 1 ? 1 : 4)
                              : row_blocks(static_cast<int>(nnodes), ncomp);
  const dim3 grid(static_cast<unsigned>(blocks), 2 * KS / NB), block(kBlockWaves * kWave);
  if (row_scale)
    hipLaunchKernelGGL((linear_block_kernel<KS, NB, true>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, ncomp, scale, row_scale, residual, OUT);
  else
    hipLaunchKernelGGL((linear_block_kernel<KS, NB, false>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, ncomp, scale, row_scale, residual, OUT);
  return check_launch("cm_linear");
}

template <int NT, int CB, int COMP>
int launch_wide(const float *X, const float *WT, const int32_t *perm, const int32_t *offs, int64_t nnodes, int ngroups,
                int zero_last_group, float scale, const float *row_scale, const float *residual, float *OUT, hipStream_t st) {
  const int64_t tiles = COMP * (ceil_div(nnodes, 16) + (offs ? ngroups : 0));  // at most
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>(device_compute_units(), tiles))), block(2 * NT / CB * kWave);
  if (row_scale)
    hipLaunchKernelGGL((linear_wide_kernel<NT, CB, COMP, true>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, scale, row_scale, residual, OUT);
  else
    hipLaunchKernelGGL((linear_wide_kernel<NT, CB, COMP, false>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, scale, row_scale, residual, OUT);
  return check_launch("cm_linear");
}

template <int K, int NT>
int launch_resident(const float *X, const float *WT, const int32_t *perm, const int32_t *offs, int64_t nnodes, int ngroups,
                    int zero_last_group, float scale, const float *row_scale, float *OUT, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(device_compute_units())), block(kResWaves * kWave);
  if (row_scale)
    hipLaunchKernelGGL((linear_resident_kernel<K, NT, true>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, scale, row_scale, OUT);
  else
    hipLaunchKernelGGL((linear_resident_kernel<K, NT, false>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, scale, row_scale, OUT);
  return check_launch("cm_linear");
}

template <int KQ, int CB>
int launch_few_rows(const float *X, const float *WT, const int32_t *perm, const int32_t *offs, int64_t nnodes, int ngroups,
                    int zero_last_group, int ncomp, int Nout, float scale, const float *row_scale, const float *residual, float *OUT,
                    hipStream_t st) {
  const int64_t tiles = ceil_div(nnodes, few::kRows) + (offs ? ngroups : 0);
  const int cols = Nout / (few::kRows * CB), waves = cols % 4 == 0 ? 4 : (cols % 3 == 0 ? 3 : (cols % 2 == 0 ? 2 : 1));
  const dim3 grid(static_cast<unsigned>(tiles * ncomp), static_cast<unsigned>(cols / waves)), block(waves * kWave);
  if (row_scale)
    hipLaunchKernelGGL((linear_few_rows_kernel<KQ, true, CB>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, ncomp, scale, row_scale, residual, OUT, Nout);
  else
    hipLaunchKernelGGL((linear_few_rows_kernel<KQ, false, CB>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, ncomp, scale, row_scale, residual, OUT, Nout);
  return check_launch("cm_linear");
}

template <int NT>
int launch(const float *X, const float *WT, const int32_t *perm, const int32_t *offs, int64_t nnodes, int ngroups,
           int zero_last_group, int ncomp, int K, float scale, const float *row_scale, const float *residual, float *OUT,
           hipStream_t st) {
  const int64_t tiles = ceil_div(nnodes, kTileNodes) + (offs ? ngroups : 0);
  const dim3 grid(static_cast<unsigned>(tiles * ncomp)), block(kWaves * kWave);
  constexpr int NOUT = 32 * NT;
  // few tiles (less than half a workgroup per compute unit): 32 columns per workgroup
  if (NT > 1 && tiles * ncomp * 2 <= device_compute_units()) {
    const dim3 split(grid.x, NT);
    if (K <= 4 * kKC) {  // every chunk requested at once (registers for four of them)
#define CM_FEW(KCH_, SCALED_)                                                                                                       \
  hipLaunchKernelGGL((linear_few_tiles_kernel<KCH_, SCALED_>), split, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups, \
                     zero_last_group, ncomp, scale, row_scale, residual, OUT, NOUT)
      switch (K / kKC) {
        case 1: if (row_scale) CM_FEW(1, true); else CM_FEW(1, false); break;
        case 2: if (row_scale) CM_FEW(2, true); else CM_FEW(2, false); break;
        case 3: if (row_scale) CM_FEW(3, true); else CM_FEW(3, false); break;
        default: if (row_scale) CM_FEW(4, true); else CM_FEW(4, false); break;
      }
#undef CM_FEW
      return check_launch("cm_linear");
    }
    if (row_scale)
      hipLaunchKernelGGL((linear_kernel<1, true>), split, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                         zero_last_group, ncomp, K, scale, row_scale, residual, OUT, NOUT);
    else
      hipLaunchKernelGGL((linear_kernel<1, false>), split, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                         zero_last_group, ncomp, K, scale, row_scale, residual, OUT, NOUT);
    return check_launch("cm_linear");
  }
  // The ring variant wherever it runs two workgroups per compute unit or the plain one does not either (Nout up to 128,
  // and 224 / 256), and K has more than one chunk to overlap; measured at 25 000 nodes: 108 vs 119-127 us at 128
  // columns, 76 vs 80-83 at 96, equal at 64, 224 and 256, slower at 32 (one chunk), 160 and 192 (one workgroup per CU).
  // The row_scale variant at 256 columns does not fit the register file and would spill, which the hand-issued loads
  // of the ring kernel do not tolerate (the build checks that no instantiated ring kernel uses scratch memory): it
  // runs on the plain kernel.
  constexpr bool kRing = NT == 2 || NT == 3 || NT == 4 || NT >= 7;
  constexpr bool kRingScaled = kRing && NT < 8;
  if constexpr (kRing) {
    if (K > kKC && (!row_scale || kRingScaled)) {
      if constexpr (kRingScaled) {
        if (row_scale) {
          hipLaunchKernelGGL((linear_ring_kernel<NT, true>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes),
                             ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT);
          return check_launch("cm_linear");
        }
      }
      hipLaunchKernelGGL((linear_ring_kernel<NT, false>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                         zero_last_group, ncomp, K, scale, row_scale, residual, OUT);
      return check_launch("cm_linear");
    }
  }
  if (row_scale)
    hipLaunchKernelGGL((linear_kernel<NT, true>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, ncomp, K, scale, row_scale, residual, OUT, NOUT);
  else
    hipLaunchKernelGGL((linear_kernel<NT, false>), grid, block, 0, st, X, WT, perm, offs, static_cast<int>(nnodes), ngroups,
                       zero_last_group, ncomp, K, scale, row_scale, residual, OUT, NOUT);
  return check_launch("cm_linear");
}

}  // namespace
}  // namespace cm

extern "C" int cm_linear(const float *X, const float *W_T, const int32_t *node_perm, const int32_t *group_offsets,
                         int64_t nnodes, int ngroups, int zero_last_group, int ncomp, int K, int Nout, float scale,
                         const float *row_scale, const float *residual, float *OUT, cm_stream_t stream) {
  CM_REQUIRE(ncomp == 1 || ncomp == 16, "cm_linear: ncomp=%d must be 1 or 16", ncomp);
  CM_REQUIRE(!zero_last_group || (group_offsets != nullptr && ngroups >= 2),
             "cm_linear: a zero group needs node_perm / group_offsets and at least one weight group before it");
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 16, "cm_linear: nnodes out of range");
  CM_REQUIRE(K >= 32 && K <= 256 && K % 32 == 0, "cm_linear: K=%d must be a multiple of 32 in [32, 256]", K);
  CM_REQUIRE(Nout >= 32 && Nout <= 256 && Nout % 32 == 0, "cm_linear: Nout=%d must be a multiple of 32 in [32, 256]", Nout);
  CM_REQUIRE(ngroups >= 1, "cm_linear: ngroups must be at least 1");
  CM_REQUIRE((node_perm == nullptr) == (group_offsets == nullptr), "cm_linear: node_perm and group_offsets go together");
  CM_REQUIRE(group_offsets != nullptr || ngroups == 1, "cm_linear: ngroups > 1 needs node_perm / group_offsets");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && W_T && OUT, "cm_linear: NULL pointer");
  hipStream_t st = cm::as_stream(stream);
  // few rows, any width: the kernel without tiles (the line: mfma_f32.hpp)
  if (cm::few::applies(nnodes, ncomp, Nout)) {
    const bool one = cm::few::blocks(nnodes, ncomp, Nout) <= cm::few::kOneColumnBlock;
    switch (K / 32) {
#define CM_CASE(KC_) \
      case KC_: return (one ? cm::launch_few_rows<2 * KC_, 1> : cm::launch_few_rows<2 * KC_, 2>)(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, Nout, scale, row_scale, residual, OUT, st);
      CM_CASE(1) CM_CASE(2) CM_CASE(3) CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8)
#undef CM_CASE
    }
  }
  // up to some thousand nodes (cm::block_columns): a workgroup per 128 rows of one weight block
  if (K == Nout) {
    switch (32 * K + cm::block_columns(nnodes, ncomp, K, ngroups, group_offsets != nullptr, row_scale != nullptr, residual != nullptr)) {
#define CM_CASE(KS_, NB_) \
      case 32 * 32 * KS_ + NB_: return cm::launch_block<KS_, NB_>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, scale, row_scale, residual, OUT, st);
      CM_CASE(1, 2) CM_CASE(2, 4) CM_CASE(2, 2) CM_CASE(3, 6) CM_CASE(3, 3) CM_CASE(4, 8) CM_CASE(4, 4) CM_CASE(5, 10) CM_CASE(5, 5)
      CM_CASE(6, 6) CM_CASE(6, 3) CM_CASE(7, 7) CM_CASE(8, 4) CM_CASE(8, 2)
#undef CM_CASE
    }
  }
  // 16 components per node, square weights, beyond: up to 128 columns the kernel that keeps the weights in LDS (measured against the ring kernel at 25 000 nodes: 87 vs 102-112 us at 128 channels, 58 vs 67-71 at 96, 42 vs
  // 47 at 64; 360 vs 430 us at 100 000 x 128); at 160 to 256 columns the one that keeps them in registers
  const bool resident = K == Nout && cm::resident_weights(nnodes, ncomp, K, ngroups, group_offsets != nullptr, residual != nullptr);
  if (resident && ncomp == 16) {
    switch (K) {
#define CM_CASE(K_, NT_) \
      case K_: return cm::launch_resident<K_, NT_>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, scale, row_scale, OUT, st);
      CM_CASE(64, 2) CM_CASE(96, 3) CM_CASE(128, 4)
#undef CM_CASE
#define CM_CASE(NT_, CB_) \
      case 32 * NT_: return cm::launch_wide<NT_, CB_, 16>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, scale, row_scale, nullptr, OUT, st);
      CM_CASE(5, 1) CM_CASE(6, 1) CM_CASE(7, 1) CM_CASE(8, 2)
#undef CM_CASE
    }
  }
  // One component per node, one weight group, 160 columns and more, beyond one round of the kernel above: the same kernel (100 000 x
  // 192 65.7 -> 51.3 us against the tiled one)
  if (resident && ncomp == 1) {
    switch (K) {
#define CM_CASE(NT_, CB_) \
      case 32 * NT_: return cm::launch_wide<NT_, CB_, 1>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, scale, row_scale, residual, OUT, st);
      CM_CASE(5, 1) CM_CASE(6, 1) CM_CASE(7, 1) CM_CASE(8, 2)
#undef CM_CASE
    }
  }
  switch (Nout / 32) {
    case 1: return cm::launch<1>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 2: return cm::launch<2>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 3: return cm::launch<3>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 4: return cm::launch<4>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 5: return cm::launch<5>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 6: return cm::launch<6>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 7: return cm::launch<7>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
    case 8: return cm::launch<8>(X, W_T, node_perm, group_offsets, nnodes, ngroups, zero_last_group, ncomp, K, scale, row_scale, residual, OUT, st);
  }
  return CM_EINVAL;
}
