// Products of a few rows, fp32 in and out, on v_mfma_f32_16x16x4_f32 with both operands straight from memory (or an fp32
// tile in LDS) in registers: shared by linear.hip and node_glue.hip for systems of some hundred to a few thousand nodes.
//
// A wave computes 16 rows x 16 output columns.  Such a launch is over in a few microseconds, and what it spends them on
// is the chain of waits of one wave: with the operand split of mfma_split.hpp that chain holds the staging, two barriers
// and ~90 vector instructions per 32 columns of K, here it is the loads of both operands, all in flight at once, and
// K / 4 matrix instructions of 32 cycles (0.43 us at K = 128).  The split is worth its instructions where a launch is
// bound by the matrix rate (the bf16 form has 16 times the rate of this one, for six products), not here.
#pragma once

#include "common.hpp"

namespace cm {
namespace few {

constexpr int kRows = 16;

// A lane's share of 16 operand rows of K = 16 KQ columns: of row lane % 16 the columns 16 q + 4 (lane / 16) .. + 3.  The
// matrix instruction that takes element i of piece q sums over the columns 16 q + 4 g + i of the four lane groups g.
template <int KQ>
struct Rows {
  f4 v[KQ];
};

// `at`: the lane's row (lane % 16), already advanced by 4 (lane / 16) columns
template <int KQ>
__device__ __forceinline__ Rows<KQ> load_rows(const float *at) {
  Rows<KQ> r;
#pragma unroll
  for (int q = 0; q < KQ; ++q) r.v[q] = ld4(at + 16 * q);
  return r;
}

// X . W for 16 rows of X and 16 CB columns of W (rows of the transposed weights): the lane receives columns
// 4 (lane / 16) .. + 3 of row lane % 16 of each block, 16 consecutive bytes of the output row.  Four chains of sums, added
// up at the end: the whole sum in one chain has up to twice the rms error of the split form (2e-7 against 1e-7 at K = 64),
// in four a little less than it (8e-8; node energies of a 400-atom model 4.7e-7 against 4.9e-7).
template <int KQ, int CB>
__device__ __forceinline__ void product(const Rows<KQ> &x, const Rows<KQ> (&wt)[CB], f4 (&out)[CB]) {
  f4 sum[CB][4];
#pragma unroll
  for (int c = 0; c < CB; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[c][i] = zero4();
#pragma unroll
  for (int q = 0; q < KQ; ++q)
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f4 &chain = sum[c][(q + i) % 4];
        chain = __builtin_amdgcn_mfma_f32_16x16x4f32(wt[c].v[q][i], x.v[q][i], chain, 0, 0, 0);
      }
#pragma unroll
  for (int c = 0; c < CB; ++c) out[c] = (sum[c][0] + sum[c][1]) + (sum[c][2] + sum[c][3]);
}

// Where it is taken, in 16 x 16 blocks of output per launch.  Every block reads its 16 rows of both operands itself, so
// the traffic between L2 and the compute units grows with the blocks where a tile of 128 rows shares it, and one block
// after the other waits for the fp32 matrix rate.  Measured (us, the tiled kernels -> this one):
//   [N, C]      216 x 64 5.0 -> 2.7, 216 x 128 6.7 -> 3.6, 2 000 x 128 6.9 -> 3.7, 2 000 x 256 10.8 -> 7.7, 10 000 x 64 5.5 -> 4.7;
//               even at 5 000 x 128 and 192 (2 500 and 3 750 blocks).  At 96 and 128 columns the line is one tile of 16 rows
//               per compute unit (1 536 and 2 048 blocks), where the chains of these products (node_glue.hip) change with it: steps of
//               3 500 x 128 421 -> 412 us, 4 000 454 -> 444, 4 500 513 -> 523 (chains forward / backward 17.1 / 17.1 -> 16.9 / 12.6, 17.6 / 17.0 -> 23.6 /
//               23.2 at 5 000).  At 256 columns the kernel with a workgroup per 128 rows is faster from 2 048 on (2 500 x 256 13.6 -> 8.3, 2 500 x
//               224 equal)
//   [N, 16, C]  216 x 64 5.3 -> 2.9, 216 x 128 7.2 -> 5.0, 500 x 96 6.9 -> 5.5, 216 x 192 9.9 -> 8.6 (2 688 blocks); even at 500 x 128
//               and 1 000 x 64 (4 000 blocks), slower beyond
// From 1 024 blocks (a wave on every SIMD) a wave takes two neighbouring blocks of columns and reads its rows once for
// both (2 000 x 192 7.2 -> 5.1, 216 x 16 x 128 5.7 -> 5.0).
inline int64_t blocks(int64_t nnodes, int ncomp, int columns) { return ceil_div(nnodes, kRows) * ncomp * (columns / kRows); }
constexpr int64_t kOneColumnBlock = 1024;
inline bool applies(int64_t nnodes, int ncomp, int columns) {
  const int64_t limit = ncomp > 1 ? 3072 : (columns == 96 ? 1536 : (columns == 128 || columns == 256 ? 2048 : 2560));
  return blocks(nnodes, ncomp, columns) <= limit;
}

}  // namespace few
}  // namespace cm
