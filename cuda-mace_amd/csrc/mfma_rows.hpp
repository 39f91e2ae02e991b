// Products of 16 rows per wave with a square weight block whose fp16 planes the workgroup keeps in LDS, fp32 in and out: shared by
// linear.hip and node_glue.hip, which return the same bits.
//
// Arithmetic: two fp16 pieces per operand and three products on v_mfma_f32_16x16x32_f16 (mfma_split.hpp), the products with a low piece
// in an accumulator of their own; weights are the row operand.  Row lane % 16 of the wave's 16 belongs to the lanes r, r + 16, r + 32, r +
// 48; lane group q = lane / 16 holds columns 16 i + 4 q + {0..3} of it for every i.  For k step s a lane feeds its columns of i = 2 s and 2 s
// + 1 (the order of k within a step does not matter as long as the weight planes are written in the same one), and the sums it gets for
// block c of 16 output columns are columns 16 c + 4 q + {0..3}: the result lies as the operand did, and a chain of products needs no exchange.
#pragma once

#include "common.hpp"
#include "mfma_split.hpp"

namespace cm {
namespace rows {

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float largest4(f4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); }

// Weight planes of COLS columns of a block with K = 32 KS rows, [piece][column][k], and what takes the columns' scales back.
template <int KS, int COLS>
struct Planes {
  static constexpr int K = 32 * KS;
  static constexpr int LD = K + 8;  // row stride of a plane in elements: an odd number of 16-byte units
  _Float16 w[2 * COLS * LD];
  float column[COLS];
};

// A thread's part of such a block on its way from memory (W^T, rows of K): four threads per column.
constexpr int kThreadsPerColumn = 4;
template <int KS, int COLS, int THREADS>
struct Fetched {
  static constexpr int kPasses = (COLS * kThreadsPerColumn + THREADS - 1) / THREADS;
  f4 v[kPasses][2 * KS];

  __device__ __forceinline__ static int column(int pass) { return pass * (THREADS / kThreadsPerColumn) + static_cast<int>(threadIdx.x) / kThreadsPerColumn; }

  __device__ __forceinline__ void request(const float *__restrict__ WT) {
    const float *at = WT + 4 * (threadIdx.x % kThreadsPerColumn);
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int col = min(column(p), COLS - 1);  // beyond the last: that one again
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) v[p][i] = ld4(at + static_cast<int64_t>(col) * (32 * KS) + 16 * i);
    }
  }

  // scaled by powers of two, split and written; column[] = scale times what takes the column's scale back
  __device__ __forceinline__ void store(Planes<KS, COLS> &to, float scale) const {
    constexpr int LD = Planes<KS, COLS>::LD;
    const int part = threadIdx.x % kThreadsPerColumn;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int col = column(p);
      float big = 0.f;
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) big = fmaxf(big, largest4(v[p][i]));
      big = fmaxf(big, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, big), 0xB1, 0xf, 0xf, false)));
      big = fmaxf(big, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, big), 0x4E, 0xf, 0xf, false)));
      const PieceScale of = piece_scale(big, kLeastColumnExponent);
      if (col < COLS) {
        _Float16 *at = to.w + col * LD + 8 * part;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          f16x4 h0, l0, h1, l1;
          split2(v[p][2 * s], of.s, h0, l0);
          split2(v[p][2 * s + 1], of.s, h1, l1);
          *reinterpret_cast<f16x8 *>(at + 32 * s) = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
          *reinterpret_cast<f16x8 *>(at + COLS * LD + 32 * s) = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        if (part == 0) to.column[col] = ldexpf(scale, of.exponent);
      }
    }
  }
};

// The pieces of a lane's part of a row (columns 16 i + 4 q + {0..3} in v[i]), scaled by the row's largest value.
template <int KS>
struct Operand {
  f16x8 x[KS][2];
  int exponent;

  __device__ __forceinline__ explicit Operand(const f4 (&v)[2 * KS]) {
    float big = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) big = fmaxf(big, largest4(v[i]));
    big = fmaxf(big, __shfl_xor(big, 16));
    big = fmaxf(big, __shfl_xor(big, 32));  // the four lanes of a row
    const PieceScale of = piece_scale(big, kLeastRowExponent);
    exponent = of.exponent;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      f16x4 h0, l0, h1, l1;
      split2(v[2 * s], of.s, h0, l0);
      split2(v[2 * s + 1], of.s, h1, l1);
      x[s][0] = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
      x[s][1] = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
};

// GB blocks of 16 output columns from block c0 on: columns 16 (c0 + c) + 4 q + {0..3} of the lane's row in out[c]
template <int GB, int KS, int COLS>
__device__ __forceinline__ void product(const Planes<KS, COLS> &p, const Operand<KS> &a, int c0, f4 (&out)[GB]) {
  constexpr int LD = Planes<KS, COLS>::LD;
  const int lane = threadIdx.x % kWave;
  const int r16 = lane % 16, quarter = lane / 16;
  const _Float16 *wl = p.w + r16 * LD + 8 * quarter;
  v4f acc[GB], small[GB];  // products of high pieces, and those with a low one
#pragma unroll
  for (int c = 0; c < GB; ++c) acc[c] = small[c] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    f16x8 wh[GB], wo[GB];
#pragma unroll
    for (int c = 0; c < GB; ++c) {
      wh[c] = *reinterpret_cast<const f16x8 *>(wl + 16 * (c0 + c) * LD + 32 * s);
      wo[c] = *reinterpret_cast<const f16x8 *>(wl + COLS * LD + 16 * (c0 + c) * LD + 32 * s);
    }
#pragma unroll
    for (int c = 0; c < GB; ++c) small[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[c], a.x[s][1], small[c], 0, 0, 0);
#pragma unroll
    for (int c = 0; c < GB; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[c], a.x[s][0], acc[c], 0, 0, 0);
#pragma unroll
    for (int c = 0; c < GB; ++c) small[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wo[c], a.x[s][0], small[c], 0, 0, 0);
  }
#pragma unroll
  for (int c = 0; c < GB; ++c) {
    out[c] = (acc[c] + small[c]) * ld4(p.column + 16 * (c0 + c) + 4 * quarter);
#pragma unroll
    for (int k = 0; k < 4; ++k) out[c][k] = __builtin_ldexpf(out[c][k], a.exponent);
  }
}
// column blocks at a time: independent chains for the matrix instructions, registers for their accumulators and fragments
constexpr int blocks_at_a_time(int blocks) { return blocks % 4 == 0 ? 4 : (blocks % 3 == 0 ? 3 : (blocks % 2 == 0 ? 2 : 1)); }

// all 2 KS blocks of a square product
template <int KS>
__device__ __forceinline__ void product_all(const Planes<KS, 32 * KS> &p, const Operand<KS> &a, f4 (&out)[2 * KS]) {
  constexpr int GB = blocks_at_a_time(2 * KS);
#pragma unroll
  for (int c0 = 0; c0 < 2 * KS; c0 += GB) {
    f4 part[GB];
    product(p, a, c0, part);
#pragma unroll
    for (int c = 0; c < GB; ++c) out[c0 + c] = part[c];
  }
}

// the lane's part of a row of K = 16 NB columns
template <int NB>
__device__ __forceinline__ void load(const float *row, f4 (&v)[NB]) {
  const float *at = row + 4 * (threadIdx.x % kWave / 16);
#pragma unroll
  for (int i = 0; i < NB; ++i) v[i] = ld4(at + 16 * i);
}
template <int NB>
__device__ __forceinline__ void store(float *row, const f4 (&v)[NB]) {
  float *at = row + 4 * (threadIdx.x % kWave / 16);
#pragma unroll
  for (int i = 0; i < NB; ++i) st4(at + 16 * i, v[i]);
}

}  // namespace rows
}  // namespace cm
