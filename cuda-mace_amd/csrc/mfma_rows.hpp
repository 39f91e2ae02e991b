// Products of 16 rows per wave with a square weight block whose bf16 planes the workgroup keeps in LDS, fp32 in and out: shared by
// linear.hip and node_glue.hip, which return the same bits.
//
// Arithmetic: three bf16 pieces per operand and six products on v_mfma_f32_16x16x32_bf16 (mfma_split.hpp), those of the two high pieces
// in one accumulator and the others in a second; weights are the row operand.  Row lane % 16 of the wave's 16 belongs to the lanes r, r + 16, r + 32, r +
// 48; lane group q = lane / 16 holds columns 16 i + 4 q + {0..3} of it for every i.  For k step s a lane feeds its columns of i = 2 s and 2 s
// + 1 (the order of k within a step does not matter as long as the weight planes are written in the same one), and the sums it gets for
// block c of 16 output columns are columns 16 c + 4 q + {0..3}: the result lies as the operand did, and a chain of products needs no exchange.
#pragma once

#include "common.hpp"
#include "mfma_split.hpp"

namespace cm {
namespace rows {

typedef float v4f __attribute__((ext_vector_type(4)));

// Weight planes of COLS columns of a block with K = 32 KS rows, [piece][column][k].
template <int KS, int COLS>
struct Planes {
  static constexpr int K = 32 * KS;
  static constexpr int LD = K + 8;  // row stride of a plane in elements: an odd number of 16-byte units
  __bf16 w[3 * COLS * LD];
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

  __device__ __forceinline__ void store(Planes<KS, COLS> &to) const {
    constexpr int LD = Planes<KS, COLS>::LD;
    const int part = threadIdx.x % kThreadsPerColumn;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
      const int col = column(p);
      if (col < COLS) {
        __bf16 *at = to.w + col * LD + 8 * part;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          bf16x8 piece[3];
          split3(v[p][2 * s], v[p][2 * s + 1], piece);
#pragma unroll
          for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8 *>(at + q * (COLS * LD) + 32 * s) = piece[q];
        }
      }
    }
  }
};

// The pieces of a lane's part of a row (columns 16 i + 4 q + {0..3} in v[i]).
template <int KS>
struct Operand {
  bf16x8 x[KS][3];

  __device__ __forceinline__ explicit Operand(const f4 (&v)[2 * KS]) {
#pragma unroll
    for (int s = 0; s < KS; ++s) split3(v[2 * s], v[2 * s + 1], x[s]);
  }
};

// The six piece products of a k step that matter, into the accumulators of GB blocks: those of the high pieces in acc, the others, below 2^-8 of
// them, from the smallest on in small, so that a sum of K terms is rounded K / 32 times at its own size (in one accumulator: six times as
// often).  Consecutive instructions go to different accumulators.
template <int GB>
__device__ __forceinline__ void add_products(const bf16x8 (&w)[GB][3], const bf16x8 (&x)[3], v4f (&acc)[GB], v4f (&small)[GB]) {
  constexpr int kW[5] = {0, 2, 1, 0, 1}, kX[5] = {2, 0, 1, 1, 0};
#pragma unroll
  for (int q = 0; q < 5; ++q) {
#pragma unroll
    for (int c = 0; c < GB; ++c) small[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c][kW[q]], x[kX[q]], small[c], 0, 0, 0);
    if (q == 2) {
#pragma unroll
      for (int c = 0; c < GB; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c][0], x[0], acc[c], 0, 0, 0);
    }
  }
}

// GB blocks of 16 output columns from block c0 on: scale times columns 16 (c0 + c) + 4 q + {0..3} of the lane's row in out[c]
template <int GB, int KS, int COLS>
__device__ __forceinline__ void product(const Planes<KS, COLS> &p, const Operand<KS> &a, int c0, float scale, f4 (&out)[GB]) {
  constexpr int LD = Planes<KS, COLS>::LD;
  const int lane = threadIdx.x % kWave;
  const int r16 = lane % 16, quarter = lane / 16;
  const __bf16 *wl = p.w + r16 * LD + 8 * quarter;
  v4f acc[GB], small[GB];
#pragma unroll
  for (int c = 0; c < GB; ++c) acc[c] = small[c] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    bf16x8 w[GB][3];
#pragma unroll
    for (int c = 0; c < GB; ++c)
#pragma unroll
      for (int q = 0; q < 3; ++q) w[c][q] = *reinterpret_cast<const bf16x8 *>(wl + (q * COLS + 16 * (c0 + c)) * LD + 32 * s);
    add_products(w, a.x[s], acc, small);
  }
#pragma unroll
  for (int c = 0; c < GB; ++c) out[c] = (acc[c] + small[c]) * scale;
}
// column blocks at a time: independent chains for the matrix instructions, registers for their accumulators and fragments
constexpr int blocks_at_a_time(int blocks) { return blocks % 4 == 0 ? 4 : (blocks % 3 == 0 ? 3 : (blocks % 2 == 0 ? 2 : 1)); }

// all 2 KS blocks of a square product
template <int KS>
__device__ __forceinline__ void product_all(const Planes<KS, 32 * KS> &p, const Operand<KS> &a, float scale, f4 (&out)[2 * KS]) {
  constexpr int GB = blocks_at_a_time(2 * KS);
#pragma unroll
  for (int c0 = 0; c0 < 2 * KS; c0 += GB) {
    f4 part[GB];
    product(p, a, c0, scale, part);
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
