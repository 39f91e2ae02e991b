// The chains of [N, C] x [C, C] products between the two interaction layers, one launch per direction.
//
// Between the first layer's contraction and the second layer's message passing the model applies three small linears to
// the same rows (reference: models/InvariantMACE.py:41-53 linear_matmul for the product's linear and linear_up, :56-74
// the per-element skip connection):
//
//   forward    h1 = B1 . Wprod1          sc = skip_e(h1)   (weights of the node's element)      X2 = h1 . Wup
//   backward   gh1 = gX2 . Wup^T + g1 + skip_e^T(g2)       gB1 = gh1 . Wprod1^T
//
// As separate launches of the linear kernel each of them keeps the device busy for a few microseconds and costs a launch; here a wave takes
// 16 nodes of one element through the whole chain, the rows in its registers (Chain below), or, for few nodes, a workgroup does.
// Arithmetic, operand split and accumulation order are those of the linear kernels (mfma_rows.hpp, mfma_f32.hpp), and every
// intermediate is rounded to fp32 where the separate launches store it, so the chain returns the bits of the separate launches.
//
// A third launch has the product linear of the second layer, the readouts and the product of their derivative (node_head below).
//
// g1 and g2 are the gradients of minus the (weighted) sum of node energies with respect to the two layers' features:
// g1[n, c] = -weight[n] scale w1[c] is formed here from the linear readout's weights; g2 = -dE/dh2 arrives as dE/dh2 and
// its sign goes into the scale of the skip product.
#include <type_traits>

#include "common.hpp"
#include "mfma_f32.hpp"
#include "mfma_rows.hpp"
#include "node_glue.hpp"
#include "node_glue_device.hpp"
#include "readout_device.hpp"

// Products and the additions that follow them stay separate roundings, as they are where separate launches store the
// product before the next one adds to it.
#pragma clang fp contract(off)

namespace cm {
namespace {

// A workgroup of WAVES waves: a wave takes 16 nodes of one element through the whole chain.  The result of a product lies in the lanes
// as the operand of the next one does (mfma_rows.hpp), so the rows never leave the registers, and the waves meet only where the
// workgroup's weight planes change: all three blocks fit LDS together up to 64 columns, two at 96, one at 128.  Before, tiles of 32 or
// 128 nodes exchanged the rows through LDS and staged operands for each 32 columns of K between two barriers (us, forward / backward):
// 10 752 x 64 12.5 / 11.1 -> 7.4 / 7.3, 60 000 x 64 21.5 / 18.4 -> 19.5 / 19.8, 5 000 x 96 13.7 / 12.9 -> 12.0 / 12.2, 25 000 x 96 19.7 / 17.0 -> 16.8 / 16.8,
// 5 000 x 128 15.3 / 14.0 -> 17.4 / 17.1, 14 000 x 128 21.1 / 19.0 -> 19.5 / 18.2, 25 000 x 128 26.9 / 23.4 -> 25.3 / 25.0 (its 51 MB take 10), 60 000 x 128 52.6 / 48.4 ->
// 48.1 / 49.2.  What is left at 128 columns: matrix instructions and fragment reads of 128 rows, and the split of three weight
// blocks, each between two barriers.
template <int NT, int WAVES>
struct Chain {
  static constexpr int C = 32 * NT, NB = 2 * NT;
  static constexpr int kThreads = WAVES * kWave, kRows = 16 * WAVES;
  static constexpr int kSlots = NT <= 2 ? 3 : (NT == 3 ? 2 : 1);  // weight blocks whose planes fit LDS together
  using Planes = rows::Planes<NT, C>;
  using Weights = rows::Fetched<NT, C, kThreads>;
  using Operand = rows::Operand<NT>;
  // another block in the place of one that every wave has multiplied
  __device__ static void replace(Planes &planes, const Weights &w) {
    __syncthreads();
    w.store(planes);
    __syncthreads();
  }
};

// ---- forward: h1 = B1 . Wprod, sc = skip_scale h1 . Wskip[element], X2 = h1 . Wup ---------------------------------
template <int NT, int WAVES>
__global__ __launch_bounds__(WAVES *kWave) void node_glue_forward_kernel(
    const float *__restrict__ B1, const float *__restrict__ prod_WT, const float *__restrict__ skip_WT,
    const float *__restrict__ up_WT, const int32_t *__restrict__ node_perm, const int32_t *__restrict__ group_offsets, int nnodes,
    int ngroups, float skip_scale, float *__restrict__ h1, float *__restrict__ sc, float *__restrict__ X2) {
  using S = Chain<NT, WAVES>;
  constexpr int C = S::C;
  __shared__ __attribute__((aligned(16))) typename S::Planes planes[S::kSlots];
  typename S::Weights w_prod, w_up, w_skip;
  w_prod.request(prod_WT);
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x, S::kRows, g, pos0, gend)) return;
  const int pos = pos0 + threadIdx.x / kWave * 16 + threadIdx.x % 16;
  const int node = node_perm[pos < gend ? pos : pos0];
  const bool here = pos < gend && static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t at = static_cast<int64_t>(here ? node : 0) * C;
  const bool no_element = g == ngroups - 1;  // nodes of no element: the skip connection is defined as zero there
  f4 v[S::NB], h[S::NB];
  rows::load(B1 + at, v);
  w_up.request(up_WT);
  if (!no_element) w_skip.request(skip_WT + static_cast<int64_t>(g) * C * C);
  __builtin_amdgcn_sched_barrier(0);  // all on their way before the first is waited for
  w_prod.store(planes[0]);
  if constexpr (S::kSlots >= 2) w_up.store(planes[1 % S::kSlots]);
  if (S::kSlots == 3 && !no_element) w_skip.store(planes[2 % S::kSlots]);
  __syncthreads();
  rows::product_all(planes[0], typename S::Operand(v), 1.0f, h);
  if (here) rows::store(h1 + at, h);
  const typename S::Operand operand(h);
  if constexpr (S::kSlots == 1) S::replace(planes[0], w_up);
  rows::product_all(planes[1 % S::kSlots], operand, 1.0f, v);
  if (here) rows::store(X2 + at, v);
  if (no_element) {
#pragma unroll
    for (int i = 0; i < S::NB; ++i) v[i] = zero4();
  } else {
    if constexpr (S::kSlots < 3) S::replace(planes[2 % S::kSlots], w_skip);
    rows::product_all(planes[2 % S::kSlots], operand, skip_scale, v);
  }
  if (here) rows::store(sc + at, v);
}

// ---- few nodes (few::applies): tiles of 16, one wave per 16 output columns, products of mfma_f32.hpp ------------------
// All weights of the chain and the tile's rows are requested before anything is waited for; between two products stands one
// trip of the 16 rows through LDS.  Same products and roundings as the few-rows linear kernel, so again the bits of the
// separate launches.  Measured at 216 nodes and 64 channels against 32-row tiles of the kernels above: forward 9.3 ->
// 4.4 us, backward 8.7 -> 5.4.
template <int NT>
struct FewShared {
  static constexpr int C = 32 * NT;
  static constexpr int kThreads = 2 * NT * kWave;
  static constexpr int kLd = C + 4;  // padded row stride (floats)
  float tile[few::kRows * kLd];
};

// The wave's 16 columns of the tile's rows to LDS, and all columns of the lane's row back as an operand.
template <class S>
__device__ __forceinline__ void put(S &s, f4 v) {
  const int lane = threadIdx.x % kWave;
  *reinterpret_cast<f4 *>(s.tile + (lane % few::kRows) * S::kLd + few::kRows * (threadIdx.x / kWave) + 4 * (lane / few::kRows)) = v;
}
template <class S>
__device__ __forceinline__ few::Rows<S::C / 16> get(const S &s) {
  const int lane = threadIdx.x % kWave;
  return few::load_rows<S::C / 16>(s.tile + (lane % few::kRows) * S::kLd + 4 * (lane / few::kRows));
}

template <int NT>
__global__ __launch_bounds__(2 * NT *kWave) void node_glue_forward_few_kernel(
    const float *__restrict__ B1, const float *__restrict__ prod_WT, const float *__restrict__ skip_WT,
    const float *__restrict__ up_WT, const int32_t *__restrict__ node_perm, const int32_t *__restrict__ group_offsets, int nnodes,
    int ngroups, float skip_scale, float *__restrict__ h1, float *__restrict__ sc, float *__restrict__ X2) {
  constexpr int C = 32 * NT, KQ = C / 16;
  using S = FewShared<NT>;
  __shared__ __attribute__((aligned(16))) S s;
  const int lane = threadIdx.x % kWave;
  const int row = lane % few::kRows, part = lane / few::kRows, col0 = few::kRows * (threadIdx.x / kWave);
  const int64_t wat = static_cast<int64_t>(col0 + row) * C + 4 * part;
  few::Rows<KQ> wp[1] = {few::load_rows<KQ>(prod_WT + wat)}, wu[1], ws[1];
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x, few::kRows, g, pos0, gend)) return;
  const int node = pos0 + row < gend ? node_perm[pos0 + row] : -1;
  const bool here = static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t in = here ? node : 0;
  const bool no_element = g == ngroups - 1;  // nodes of no element: the skip connection is defined as zero there
  const few::Rows<KQ> x = few::load_rows<KQ>(B1 + in * C + 4 * part);
  ws[0] = few::load_rows<KQ>(skip_WT + static_cast<int64_t>(no_element ? 0 : g) * C * C + wat);
  wu[0] = few::load_rows<KQ>(up_WT + wat);
  __builtin_amdgcn_sched_barrier(0);  // the weights of all three products on their way before the first one waits
  const int64_t at = in * C + col0 + 4 * part;
  f4 v[1];
  few::product<KQ, 1>(x, wp, v);
  put(s, v[0]);
  if (here) st4(h1 + at, v[0]);
  __syncthreads();
  const few::Rows<KQ> h = get(s);
  few::product<KQ, 1>(h, wu, v);
  if (here) st4(X2 + at, v[0]);
  few::product<KQ, 1>(h, ws, v);
  if (here) st4(sc + at, no_element ? zero4() : v[0] * skip_scale);
}

// ---- backward: gh1 = gX2 . Wup^T + g1 - skip_scale dE/dh2 . Wskip[element]^T, gB1 = gh1 . Wprod^T ------------------
// four columns of it
__device__ __forceinline__ f4 gh1_of(f4 up, f4 skip, const double *w1, double scale, double node_weight, float factor, bool no_element) {
  f4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = cm::gh1_of(up[i], skip[i], w1[i], scale, node_weight, factor, no_element);
  return r;
}

template <int NT, int WAVES>
__global__ __launch_bounds__(WAVES *kWave) void node_glue_backward_kernel(
    const float *__restrict__ gX2, const float *__restrict__ d_h2, const float *__restrict__ up_W, const float *__restrict__ skip_W,
    const float *__restrict__ prod_W, const double *__restrict__ w1, double scale, const double *__restrict__ node_weights,
    const int32_t *__restrict__ node_perm, const int32_t *__restrict__ group_offsets, int nnodes, int ngroups, float skip_scale,
    float *__restrict__ gB1, EnergySums sums, int first_tile) {
  using S = Chain<NT, WAVES>;
  constexpr int C = S::C;
  __shared__ __attribute__((aligned(16))) typename S::Planes planes[S::kSlots];
  if (static_cast<int>(blockIdx.x) < first_tile) {
    // workgroups ahead of the tiles: the energy of one graph each, from node energies an earlier launch wrote
    static_assert(sizeof(planes) >= S::kThreads * sizeof(double), "the planes' place holds the partial sums");
    graph_energy<S::kThreads>(sums, blockIdx.x, reinterpret_cast<double *>(planes));
    return;
  }
  typename S::Weights w_up, w_skip, w_prod;
  w_up.request(up_W);
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x - first_tile, S::kRows, g, pos0, gend)) return;
  const int pos = pos0 + threadIdx.x / kWave * 16 + threadIdx.x % 16;
  const int node = node_perm[pos < gend ? pos : pos0];
  const bool here = pos < gend && static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t in = here ? node : 0, at = in * C;
  const bool no_element = g == ngroups - 1;
  f4 v[S::NB], d[S::NB], up[S::NB], skip[S::NB];
  rows::load(gX2 + at, v);
  if (!no_element) w_skip.request(skip_W + static_cast<int64_t>(g) * C * C);
  rows::load(d_h2 + at, d);
  w_prod.request(prod_W);
  const double nw = node_weights ? node_weights[in] : 1.0;
  __builtin_amdgcn_sched_barrier(0);  // all on their way before the first is waited for
  w_up.store(planes[0]);
  if (S::kSlots >= 2 && !no_element) w_skip.store(planes[1 % S::kSlots]);
  if constexpr (S::kSlots == 3) w_prod.store(planes[2 % S::kSlots]);
  __syncthreads();
  rows::product_all(planes[0], typename S::Operand(v), 1.0f, up);
  if (!no_element) {
    if constexpr (S::kSlots == 1) S::replace(planes[0], w_skip);
    rows::product_all(planes[1 % S::kSlots], typename S::Operand(d), -skip_scale, skip);
  } else {
#pragma unroll
    for (int i = 0; i < S::NB; ++i) skip[i] = zero4();
  }
#pragma unroll
  for (int i = 0; i < S::NB; ++i) v[i] = gh1_of(up[i], skip[i], w1 + 16 * i + 4 * (threadIdx.x % kWave / 16), scale, nw, 1.0f, no_element);
  if constexpr (S::kSlots < 3) S::replace(planes[2 % S::kSlots], w_prod);
  rows::product_all(planes[2 % S::kSlots], typename S::Operand(v), 1.0f, d);
  if (here) rows::store(gB1 + at, d);
}

template <int NT>
__global__ __launch_bounds__(2 * NT *kWave) void node_glue_backward_few_kernel(
    const float *__restrict__ gX2, const float *__restrict__ d_h2, const float *__restrict__ up_W, const float *__restrict__ skip_W,
    const float *__restrict__ prod_W, const double *__restrict__ w1, double scale, const double *__restrict__ node_weights,
    const int32_t *__restrict__ node_perm, const int32_t *__restrict__ group_offsets, int nnodes, int ngroups, float skip_scale,
    float *__restrict__ gB1, EnergySums sums, int first_tile) {
  constexpr int C = 32 * NT, KQ = C / 16;
  using S = FewShared<NT>;
  __shared__ __attribute__((aligned(16))) S s;
  if (static_cast<int>(blockIdx.x) < first_tile) {
    constexpr int kSum = S::kThreads >= 512 ? 512 : (S::kThreads >= 256 ? 256 : 128);
    static_assert(sizeof(s.tile) >= kSum * sizeof(double), "the tile holds the partial sums");
    graph_energy<kSum, 8>(sums, blockIdx.x, reinterpret_cast<double *>(s.tile));
    return;
  }
  const int lane = threadIdx.x % kWave;
  const int row = lane % few::kRows, part = lane / few::kRows, col0 = few::kRows * (threadIdx.x / kWave);
  const int64_t wat = static_cast<int64_t>(col0 + row) * C + 4 * part;
  few::Rows<KQ> wu[1] = {few::load_rows<KQ>(up_W + wat)}, ws[1], wp[1];
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x - first_tile, few::kRows, g, pos0, gend)) return;
  const int node = pos0 + row < gend ? node_perm[pos0 + row] : -1;
  const bool here = static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t in = here ? node : 0;
  const bool no_element = g == ngroups - 1;
  const few::Rows<KQ> x = few::load_rows<KQ>(gX2 + in * C + 4 * part), d = few::load_rows<KQ>(d_h2 + in * C + 4 * part);
  ws[0] = few::load_rows<KQ>(skip_W + static_cast<int64_t>(no_element ? 0 : g) * C * C + wat);
  wp[0] = few::load_rows<KQ>(prod_W + wat);
  const double nw = node_weights ? node_weights[in] : 1.0;
  __builtin_amdgcn_sched_barrier(0);
  f4 v[1], u[1];
  few::product<KQ, 1>(x, wu, v);
  few::product<KQ, 1>(d, ws, u);
  put(s, gh1_of(v[0], u[0], w1 + col0 + 4 * part, scale, nw, -skip_scale, no_element));
  __syncthreads();
  few::product<KQ, 1>(get(s), wp, v);
  if (here) st4(gB1 + in * C + col0 + 4 * part, v[0]);
}

// From 96 channels on the three products of a tile are too much for one compute unit (its eight waves share four matrix
// pipes: 3 x 0.9 us at 128 channels, and 3 x 64 KB of weights on their way to it), so the chain is cut at h1 / gh1 and each
// part spreads its 16-column blocks over the device like any linear.  Measured in the step of 216 nodes and 128 channels
// (32-row tiles -> both launches): forward 15.4 -> 9.3 us, backward 16.3 -> 11.4 (one launch of the chain above: 10.8, 13.1).
// Beyond 128 channels the same two cuts serve the step of few nodes (node_chains_cut), three launches fewer: 216 x 192 181 -> 172 us per
// step, 500 x 224 255 -> 248, 216 x 256 209 -> 202, 60 x 192 160 -> 154, 1 000 x 256 349 -> 343.
template <int KQ>
__global__ __launch_bounds__(4 * kWave) void node_glue_skip_up_kernel(const float *__restrict__ h1, const float *__restrict__ skip_WT,
                                                                      const float *__restrict__ up_WT, const int32_t *__restrict__ node_perm,
                                                                      const int32_t *__restrict__ group_offsets, int nnodes, int ngroups,
                                                                      float skip_scale, float *__restrict__ sc, float *__restrict__ X2) {
  constexpr int C = 16 * KQ;
  const int lane = threadIdx.x % kWave;
  const int row = lane % few::kRows, part = lane / few::kRows;
  const int block = blockIdx.y * (blockDim.x / kWave) + threadIdx.x / kWave;  // the first KQ: X2, the others: sc
  const bool skip = block >= KQ;
  const int col0 = few::kRows * (skip ? block - KQ : block);
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x, few::kRows, g, pos0, gend)) return;
  const int node = pos0 + row < gend ? node_perm[pos0 + row] : -1;
  const bool here = static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t in = here ? node : 0;
  f4 v[1] = {zero4()};
  if (!(skip && g == ngroups - 1)) {
    const float *W = skip ? skip_WT + static_cast<int64_t>(g) * C * C : up_WT;
    const few::Rows<KQ> w[1] = {few::load_rows<KQ>(W + static_cast<int64_t>(col0 + row) * C + 4 * part)};
    few::product<KQ, 1>(few::load_rows<KQ>(h1 + in * C + 4 * part), w, v);
  }
  if (here) st4((skip ? sc : X2) + in * C + col0 + 4 * part, skip ? v[0] * skip_scale : v[0]);
}

template <int KQ>
__global__ __launch_bounds__(4 * kWave) void node_glue_gh1_kernel(const float *__restrict__ gX2, const float *__restrict__ d_h2,
                                                                  const float *__restrict__ up_W, const float *__restrict__ skip_W,
                                                                  const double *__restrict__ w1, double scale,
                                                                  const double *__restrict__ node_weights, const int32_t *__restrict__ node_perm,
                                                                  const int32_t *__restrict__ group_offsets, int nnodes, int ngroups,
                                                                  float skip_scale, float *__restrict__ gh1, EnergySums sums, int first_tile) {
  constexpr int C = 16 * KQ;
  constexpr int kSum = 128;
  if (static_cast<int>(blockIdx.x) < first_tile) {
    __shared__ double partial[kSum];
    if (blockIdx.y == 0) graph_energy<kSum, 16>(sums, blockIdx.x, partial);
    return;
  }
  const int lane = threadIdx.x % kWave;
  const int row = lane % few::kRows, part = lane / few::kRows;
  const int col0 = few::kRows * (blockIdx.y * (blockDim.x / kWave) + threadIdx.x / kWave);
  int g, pos0, gend;
  if (!locate_group_tile(group_offsets, ngroups, nnodes, blockIdx.x - first_tile, few::kRows, g, pos0, gend)) return;
  const int node = pos0 + row < gend ? node_perm[pos0 + row] : -1;
  const bool here = static_cast<unsigned>(node) < static_cast<unsigned>(nnodes);
  const int64_t in = here ? node : 0;
  const bool no_element = g == ngroups - 1;
  const int64_t wat = static_cast<int64_t>(col0 + row) * C + 4 * part;
  const few::Rows<KQ> wu[1] = {few::load_rows<KQ>(up_W + wat)};
  const few::Rows<KQ> ws[1] = {few::load_rows<KQ>(skip_W + static_cast<int64_t>(no_element ? 0 : g) * C * C + wat)};
  f4 v[1], u[1];
  few::product<KQ, 1>(few::load_rows<KQ>(gX2 + in * C + 4 * part), wu, v);
  few::product<KQ, 1>(few::load_rows<KQ>(d_h2 + in * C + 4 * part), ws, u);
  if (!here) return;
  st4(gh1 + in * C + col0 + 4 * part, gh1_of(v[0], u[0], w1 + col0 + 4 * part, scale, node_weights ? node_weights[in] : 1.0, -skip_scale, no_element));
}

// ---- head: h2 = B2 . Wprod + sc, readouts of h1 and h2, gB2 = -w dE/dh2 . Wprod^T (w: the node's weight) --------------
// Between the second layer's contraction and the backward chain every step is per node: a product with a residual, the
// readouts (readout.hip has their arithmetic and the meaning of the operands), and the product of their derivative.  h2 stays on
// chip: of the [N, C] rows only dE/dh2 is written besides gB2, for the skip connection's gradient.  The readouts are
// bound by nothing but the fp64 matrix rate and the chain of a tile, 0.9 us each way at 128 x 128 on four matrix pipes.
// Measured inside the step, three launches -> one (us): 21 x 64 9.0 -> 5.2, 216 x 128 14.8 -> 12.4, 2 000 x 128 15.4 -> 12.5 (tiles
// of 16 nodes), 5 000 x 96 24.0 -> 15.6, 10 752 x 64 23.9 -> 13.5, 25 000 x 128 66.6 -> 40 (its 112 MB, half of them the fp64 feature
// rows, take 21); with the rows of 16 nodes in a wave's registers, as in the chains above, 5 000 x 96 16.1 -> 15.4, 10 752 x 64 14.3 -> 11.5,
// 25 000 x 128 41.7 -> 39.4, and 5 000 x 128 16.8 -> 21.5, whose weight blocks take turns in LDS.
// Without d_h2 (energies alone) the kernel ends with the energies.  Bits of the separate launches, as above.
// A wave has all classes of pieces of its 16 nodes (in the separate kernel four waves share them); the weights of the readouts
// wait in LDS.
template <int NT, int WAVES>
__global__ __launch_bounds__(WAVES *kWave) void node_head_kernel(
    const float *__restrict__ B2, const float *__restrict__ sc, const float *__restrict__ h1, const float *__restrict__ prod_WT,
    const float *__restrict__ prod_W, readout::Weights w, readout::Outputs out, const double *__restrict__ node_weights, int nnodes,
    float *__restrict__ d_h2, float *__restrict__ gB2) {
  using S = Chain<NT, WAVES>;
  constexpr int C = S::C, kHidden = readout::kHidden, kClasses = readout::kClasses;
  constexpr int kLdW = kHidden + 2;  // row stride of W2a in LDS (doubles): the four lane groups of a read start 64 bytes apart in bank space
  constexpr int kSlots = NT <= 3 ? 2 : 1;
  __shared__ __attribute__((aligned(16))) typename S::Planes planes[kSlots];
  __shared__ __attribute__((aligned(16))) double sW[C * kLdW], sw1[C];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int col = lane % 16, part = lane / 16;
  const int node = blockIdx.x * S::kRows + tid / kWave * 16 + col;
  const bool here = node < nnodes;
  const int64_t at = static_cast<int64_t>(here ? node : 0) * C;

  typename S::Weights w_prod, w_back;
  w_prod.request(prod_WT);
  f4 x[S::NB], h2[S::NB], a[S::NB];
  rows::load(B2 + at, x);
  constexpr int kWPer = (C * kHidden + S::kThreads - 1) / S::kThreads;
  double w2a[kWPer];
#pragma unroll
  for (int i = 0; i < kWPer; ++i) {
    const int q = tid + i * S::kThreads, c = q / kHidden, j = q % kHidden;
    w2a[i] = c < C && j < w.hidden ? w.W2a[c * w.hidden + j] : 0.0;
  }
  const double w1v = tid < C ? w.w1[tid] : 0.0;
  const int row = here && out.rows ? out.rows[node] : node;
  const bool row_ok = here && static_cast<unsigned>(row) < static_cast<unsigned>(nnodes);
  if (d_h2) w_back.request(prod_W);
  __builtin_amdgcn_sched_barrier(0);  // all on their way before the first is waited for
  w_prod.store(planes[0]);
#pragma unroll
  for (int i = 0; i < kWPer; ++i) {
    const int q = tid + i * S::kThreads;
    if (q < C * kHidden) sW[q / kHidden * kLdW + q % kHidden] = w2a[i];
  }
  if (tid < C) sw1[tid] = w1v;
  static_assert(S::kThreads >= C, "a thread per channel");
  if (kSlots == 2 && d_h2) w_back.store(planes[1 % kSlots]);
  rows::load(sc + at, a);  // the residual
  const typename S::Operand operand(x);
  __syncthreads();
  rows::product_all(planes[0], operand, 1.0f, h2);
#pragma unroll
  for (int p = 0; p < S::NB; ++p) h2[p] = h2[p] + a[p];
  rows::load(h1 + at, a);

  readout::d4v z[kClasses];
  double e1[kClasses];
#pragma unroll
  for (int k = 0; k < kClasses; ++k) z[k] = readout::d4v{0.0, 0.0, 0.0, 0.0}, e1[k] = 0.0;
#pragma unroll
  for (int p = 0; p < S::NB; ++p) {
    const int c = 16 * p + 4 * part;
    double wz[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wz[i] = sW[(c + i) * kLdW + readout::operand_row(col)];
    readout::add_z(z[p % kClasses], wz, h2[p]);
    readout::add_linear(e1[p % kClasses], *reinterpret_cast<const readout::d2v *>(sw1 + c), *reinterpret_cast<const readout::d2v *>(sw1 + c + 2), a[p]);
    if (out.feats64 && row_ok) readout::store_feats(out.feats64 + static_cast<int64_t>(row) * (2 * C) + c, C, a[p], h2[p]);
  }
  // sums in pairs, (0 + 1) + (2 + 3), of classes and of hidden units
  const readout::d4v zsum = (z[0] + z[1]) + (z[2] + z[3]);
  double esum = (e1[0] + e1[1]) + (e1[2] + e1[3]), e2[4], d[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const double gate = 4 * part + i < w.hidden ? w.w2b[4 * part + i] * w.act_cst : 0.0;
    readout::activate(gate, zsum[i], e2[i], d[i]);
  }
  esum = esum + ((e2[0] + e2[1]) + (e2[2] + e2[3]));
  const double en = readout::node_energy(esum, w.scale, w.shift);
  if (here && part == 0) readout::store_energy(out, node, row, row_ok, en);
  if (!d_h2) return;
  const double nw = node_weights && here ? node_weights[node] : 1.0;
#pragma unroll
  for (int p = 0; p < S::NB; ++p) {
    const double *wp = sW + (16 * p + readout::operand_row(col)) * kLdW + 4 * part;
    const double wd[4] = {wp[0], wp[1], wp[2], wp[3]};
    f4 g = readout::derivative(wd, d, w.scale);
    if (node_weights) {
#pragma unroll
      for (int i = 0; i < 4; ++i) g[i] = static_cast<float>(static_cast<double>(g[i]) * nw);
    }
    x[p] = g;
  }
  if (here) rows::store(d_h2 + at, x);
  if constexpr (kSlots == 1) S::replace(planes[0], w_back);
  rows::product_all(planes[1 % kSlots], typename S::Operand(x), -1.0f, h2);
  if (here) rows::store(gB2 + at, h2);
}

// Few nodes: tiles of 16, a wave per 16 columns, the readouts' sums shared by the waves as in the separate kernel.
template <int NT>
__global__ __launch_bounds__(2 * NT *kWave) void node_head_few_kernel(
    const float *__restrict__ B2, const float *__restrict__ sc, const float *__restrict__ h1, const float *__restrict__ prod_WT,
    const float *__restrict__ prod_W, readout::Weights w, readout::Outputs out, const double *__restrict__ node_weights, int nnodes,
    float *__restrict__ d_h2, float *__restrict__ gB2) {
  constexpr int C = 32 * NT, KQ = C / 16, kWaves = 2 * NT;
  constexpr int kClasses = readout::kClasses, kUsed = KQ < kClasses ? KQ : kClasses;  // classes that have a piece
  constexpr int kPer = (KQ + kClasses - 1) / kClasses;                                // pieces of a class
  using S = FewShared<NT>;
  __shared__ __attribute__((aligned(16))) S s;
  __shared__ double sZ[kUsed][4][kWave], sE[kUsed][kWave], sE2[4][kWave], sD[4][kWave];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int row = lane % few::kRows, part = lane / few::kRows, col0 = few::kRows * wave;
  const int64_t wat = static_cast<int64_t>(col0 + row) * C + 4 * part;
  const int node = blockIdx.x * few::kRows + row;
  const bool here = node < nnodes;
  const int64_t in = here ? node : 0;
  few::Rows<KQ> wp[1] = {few::load_rows<KQ>(prod_WT + wat)}, wq[1];
  const few::Rows<KQ> x = few::load_rows<KQ>(B2 + in * C + 4 * part);
  __builtin_amdgcn_sched_barrier(0);  // the first product's operands first: the loads of a compute unit return one after the other
  const int64_t at = in * C + col0 + 4 * part;
  const f4 residual = ld4(sc + at);
  // what this wave needs for the readouts: class `wave` of the pieces, element `wave` of z, piece `wave` of the derivative
  f4 a[kPer];
  double wz[kPer][4], wd[4];
  readout::d2v wl[kPer][2];
  if (wave < kUsed) {
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int c = 16 * (wave + kClasses * u) + 4 * part;
      if (c >= C) break;  // the same for the whole wave
      a[u] = ld4(h1 + in * C + c);
      wl[u][0] = *reinterpret_cast<const readout::d2v *>(w.w1 + c), wl[u][1] = *reinterpret_cast<const readout::d2v *>(w.w1 + c + 2);
#pragma unroll
      for (int i = 0; i < 4; ++i) wz[u][i] = readout::operand_row(row) < w.hidden ? w.W2a[(c + i) * w.hidden + readout::operand_row(row)] : 0.0;
    }
  }
  const double *wd_at = w.W2a + static_cast<int64_t>(16 * wave + readout::operand_row(row)) * w.hidden + 4 * part;
  if (w.hidden == readout::kHidden) {
    const readout::d2v lo = reinterpret_cast<const readout::d2v *>(wd_at)[0], hi = reinterpret_cast<const readout::d2v *>(wd_at)[1];
    wd[0] = lo.x, wd[1] = lo.y, wd[2] = hi.x, wd[3] = hi.y;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) wd[i] = 4 * part + i < w.hidden ? wd_at[i] : 0.0;
  }
  auto gate_of = [&](int i) { return 4 * part + i < w.hidden ? w.w2b[4 * part + i] * w.act_cst : 0.0; };
  const double gate = gate_of(wave % 4);
  const int to = here && out.rows ? out.rows[in] : node;
  const bool to_ok = here && static_cast<unsigned>(to) < static_cast<unsigned>(nnodes);
  const double nw = node_weights ? node_weights[in] : 1.0;
  if (d_h2) wq[0] = few::load_rows<KQ>(prod_W + wat);
  __builtin_amdgcn_sched_barrier(0);  // all operands on their way before the first product waits

  f4 v[1];
  few::product<KQ, 1>(x, wp, v);
  put(s, v[0] + residual);
  __syncthreads();
  if (wave < kUsed) {
    readout::d4v z{0.0, 0.0, 0.0, 0.0};
    double e1 = 0.0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int c = 16 * (wave + kClasses * u) + 4 * part;
      if (c >= C) break;
      const f4 b = *reinterpret_cast<const f4 *>(s.tile + row * S::kLd + c);
      readout::add_z(z, wz[u], b);
      readout::add_linear(e1, wl[u][0], wl[u][1], a[u]);
      if (out.feats64 && to_ok) readout::store_feats(out.feats64 + static_cast<int64_t>(to) * (2 * C) + c, C, a[u], b);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) sZ[wave][i][lane] = z[i];
    sE[wave][lane] = e1;
  }
  __syncthreads();
  auto total = [&](const auto &get_class) {
    double q[kClasses];
#pragma unroll
    for (int k = 0; k < kClasses; ++k) q[k] = k < kUsed ? get_class(k < kUsed ? k : 0) : 0.0;
    return (q[0] + q[1]) + (q[2] + q[3]);
  };
  for (int i = wave; i < 4; i += kWaves) {
    const double z_i = total([&](int k) { return sZ[k][i][lane]; });
    readout::activate(i == wave ? gate : gate_of(i), z_i, sE2[i][lane], sD[i][lane]);
  }
  __syncthreads();
  if (wave == 0) {
    const double e = total([&](int k) { return sE[k][lane]; }) + ((sE2[0][lane] + sE2[1][lane]) + (sE2[2][lane] + sE2[3][lane]));
    const double en = readout::node_energy(e, w.scale, w.shift);
    if (here && part == 0) readout::store_energy(out, node, to, to_ok, en);
  }
  if (!d_h2) return;
  const double d[4] = {sD[0][lane], sD[1][lane], sD[2][lane], sD[3][lane]};
  f4 g = readout::derivative(wd, d, w.scale);
  if (node_weights) {
#pragma unroll
    for (int i = 0; i < 4; ++i) g[i] = static_cast<float>(static_cast<double>(g[i]) * nw);
  }
  if (here) st4(d_h2 + at, g);
  put(s, g);  // the rows of h2 have been read
  __syncthreads();
  few::product<KQ, 1>(get(s), wq, v);
  if (here) st4(gB2 + at, v[0] * -1.0f);
}

// Four waves per workgroup (64 nodes) while that is one round of workgroups, eight beyond.  us, four / eight waves, forward and backward:
// 5 000 x 128 17.5 + 17.0 / 21.7 + 22.1, 10 752 x 64 7.4 + 7.3 / 8.8 + 9.5, 16 000 x 96 14.4 + 13.6 / 15.9 + 15.9; 18 000 x 64 12.6 + 12.8 /
// 9.8 + 9.9, 18 000 x 128 33.1 + 32.8 / 23.9 + 23.3, 25 000 x 96 23.5 + 23.6 / 16.8 + 17.0.
inline bool four_waves(int64_t nnodes) { return ceil_div(nnodes, 128) * 2 < device_compute_units(); }

// The chains cut at h1 / gh1 (few nodes): product and skip + up, or gh1 and product.
template <int NT>
int launch_forward_cut(const float *B1, const float *prod_WT, const float *skip_WT, const float *up_WT, const int32_t *perm, const int32_t *offs,
                       int64_t nnodes, int ngroups, float skip_scale, float *h1, float *sc, float *X2, hipStream_t st) {
  constexpr int kBlocks = 4 * NT, kPerGroup = NT == 3 ? 3 : 4;
  static_assert(kBlocks % kPerGroup == 0, "the blocks divide evenly among the workgroups");
  const unsigned tiles = static_cast<unsigned>(ceil_div(nnodes, few::kRows) + ngroups);
  const int rc = cm_linear(B1, prod_WT, nullptr, nullptr, nnodes, 1, 0, 1, 32 * NT, 32 * NT, 1.0f, nullptr, nullptr, h1, st);
  if (rc != CM_OK) return rc;
  hipLaunchKernelGGL((node_glue_skip_up_kernel<2 * NT>), dim3(tiles, kBlocks / kPerGroup), dim3(kPerGroup * kWave), 0, st, h1, skip_WT, up_WT, perm,
                     offs, static_cast<int>(nnodes), ngroups, skip_scale, sc, X2);
  return check_launch("cm_node_glue_forward");
}
template <int NT>
int launch_backward_cut(const float *gX2, const float *d_h2, const float *up_W, const float *skip_W, const float *prod_W, const double *w1,
                        double scale, const double *node_weights, const int32_t *perm, const int32_t *offs, int64_t nnodes, int ngroups,
                        float skip_scale, float *gh1, float *gB1, const EnergySums &sums, hipStream_t st) {
  constexpr int kBlocks = 2 * NT, kPerGroup = NT % 2 == 0 ? 4 : (NT % 3 == 0 ? 3 : 2);
  static_assert(kBlocks % kPerGroup == 0, "the blocks divide evenly among the workgroups");
  const unsigned extra = sums.out ? static_cast<unsigned>(sums.ngraphs) : 0u;
  const unsigned tiles = static_cast<unsigned>(ceil_div(nnodes, few::kRows) + ngroups);
  hipLaunchKernelGGL((node_glue_gh1_kernel<2 * NT>), dim3(tiles + extra, kBlocks / kPerGroup), dim3(kPerGroup * kWave), 0, st, gX2, d_h2, up_W, skip_W,
                     w1, scale, node_weights, perm, offs, static_cast<int>(nnodes), ngroups, skip_scale, gh1, sums, static_cast<int>(extra));
  const int rc = check_launch("cm_node_glue_backward");
  if (rc != CM_OK) return rc;
  return cm_linear(gh1, prod_W, nullptr, nullptr, nnodes, 1, 0, 1, 32 * NT, 32 * NT, 1.0f, nullptr, nullptr, gB1, st);
}

template <int NT>
int launch_forward(const float *B1, const float *prod_WT, const float *skip_WT, const float *up_WT, const int32_t *perm,
                   const int32_t *offs, int64_t nnodes, int ngroups, float skip_scale, float *h1, float *sc, float *X2,
                   hipStream_t st) {
  if (few::applies(nnodes, 1, 32 * NT)) {
    const unsigned tiles = static_cast<unsigned>(ceil_div(nnodes, few::kRows) + ngroups);
    if constexpr (NT >= 3) {
      return launch_forward_cut<NT>(B1, prod_WT, skip_WT, up_WT, perm, offs, nnodes, ngroups, skip_scale, h1, sc, X2, st);
    } else {
      hipLaunchKernelGGL((node_glue_forward_few_kernel<NT>), dim3(tiles), dim3(2 * NT * kWave), 0, st, B1, prod_WT, skip_WT, up_WT, perm,
                         offs, static_cast<int>(nnodes), ngroups, skip_scale, h1, sc, X2);
    }
    return check_launch("cm_node_glue_forward");
  }
  const auto launch = [&](auto waves) {
    constexpr int kW = decltype(waves)::value;
    const unsigned tiles = static_cast<unsigned>(ceil_div(nnodes, 16 * kW) + ngroups);
    hipLaunchKernelGGL((node_glue_forward_kernel<NT, kW>), dim3(tiles), dim3(kW * kWave), 0, st, B1, prod_WT, skip_WT, up_WT, perm, offs,
                       static_cast<int>(nnodes), ngroups, skip_scale, h1, sc, X2);
  };
  if (four_waves(nnodes)) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 8>{});
  return check_launch("cm_node_glue_forward");
}

template <int NT>
int launch_backward(const float *gX2, const float *d_h2, const float *up_W, const float *skip_W, const float *prod_W,
                    const double *w1, double scale, const double *node_weights, const int32_t *perm, const int32_t *offs,
                    int64_t nnodes, int ngroups, float skip_scale, float *gh1, float *gB1, const EnergySums &sums, hipStream_t st) {
  const unsigned extra = sums.out ? static_cast<unsigned>(sums.ngraphs) : 0u;
  if (few::applies(nnodes, 1, 32 * NT)) {
    const unsigned tiles = static_cast<unsigned>(ceil_div(nnodes, few::kRows) + ngroups);
    if (NT >= 3 && gh1)
      return launch_backward_cut<NT>(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, perm, offs, nnodes, ngroups, skip_scale, gh1, gB1, sums, st);
    hipLaunchKernelGGL((node_glue_backward_few_kernel<NT>), dim3(tiles + extra), dim3(2 * NT * kWave), 0, st, gX2, d_h2, up_W, skip_W,
                       prod_W, w1, scale, node_weights, perm, offs, static_cast<int>(nnodes), ngroups, skip_scale, gB1, sums,
                       static_cast<int>(extra));
    return check_launch("cm_node_glue_backward");
  }
  const auto launch = [&](auto waves) {
    constexpr int kW = decltype(waves)::value;
    const unsigned tiles = static_cast<unsigned>(ceil_div(nnodes, 16 * kW) + ngroups);
    hipLaunchKernelGGL((node_glue_backward_kernel<NT, kW>), dim3(tiles + extra), dim3(kW * kWave), 0, st, gX2, d_h2, up_W, skip_W, prod_W, w1, scale,
                       node_weights, perm, offs, static_cast<int>(nnodes), ngroups, skip_scale, gB1, sums, static_cast<int>(extra));
  };
  if (four_waves(nnodes)) launch(std::integral_constant<int, 4>{});
  else launch(std::integral_constant<int, 8>{});
  return check_launch("cm_node_glue_backward");
}

template <int NT>
int launch_head(const float *B2, const float *sc, const float *h1, const float *prod_WT, const float *prod_W, const readout::Weights &w,
                const readout::Outputs &out, const double *node_weights, int64_t nnodes, float *d_h2, float *gB2, hipStream_t st) {
  const int n = static_cast<int>(nnodes);
  if (few::applies(nnodes, 1, 32 * NT))
    hipLaunchKernelGGL((node_head_few_kernel<NT>), dim3(static_cast<unsigned>(ceil_div(nnodes, few::kRows))), dim3(2 * NT * kWave), 0, st, B2, sc, h1,
                       prod_WT, prod_W, w, out, node_weights, n, d_h2, gB2);
  else if (four_waves(nnodes))
    hipLaunchKernelGGL((node_head_kernel<NT, 4>), dim3(static_cast<unsigned>(ceil_div(nnodes, 64))), dim3(4 * kWave), 0, st, B2, sc, h1, prod_WT,
                       prod_W, w, out, node_weights, n, d_h2, gB2);
  else
    hipLaunchKernelGGL((node_head_kernel<NT, 8>), dim3(static_cast<unsigned>(ceil_div(nnodes, 128))), dim3(8 * kWave), 0, st, B2, sc, h1, prod_WT,
                       prod_W, w, out, node_weights, n, d_h2, gB2);
  return check_launch("cm_mace_step");
}

}  // namespace
}  // namespace cm

extern "C" int cm_node_glue_supported(int channels) { return channels >= 32 && channels <= 128 && channels % 32 == 0; }

extern "C" int cm_node_glue_forward(const float *B1, const float *prod_WT, const float *skip_WT, const float *up_WT,
                                    const int32_t *node_perm, const int32_t *group_offsets, int64_t nnodes, int ngroups,
                                    int channels, float skip_scale, float *h1, float *sc, float *X2, cm_stream_t stream) {
  CM_REQUIRE(cm_node_glue_supported(channels), "cm_node_glue_forward: channels=%d must be 32, 64, 96 or 128", channels);
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 256, "cm_node_glue_forward: nnodes out of range");
  CM_REQUIRE(ngroups >= 2, "cm_node_glue_forward: ngroups counts the elements plus the group of nodes without one");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(B1 && prod_WT && skip_WT && up_WT && node_perm && group_offsets && h1 && sc && X2, "cm_node_glue_forward: NULL pointer");
  hipStream_t st = cm::as_stream(stream);
  switch (channels / 32) {
    case 1: return cm::launch_forward<1>(B1, prod_WT, skip_WT, up_WT, node_perm, group_offsets, nnodes, ngroups, skip_scale, h1, sc, X2, st);
    case 2: return cm::launch_forward<2>(B1, prod_WT, skip_WT, up_WT, node_perm, group_offsets, nnodes, ngroups, skip_scale, h1, sc, X2, st);
    case 3: return cm::launch_forward<3>(B1, prod_WT, skip_WT, up_WT, node_perm, group_offsets, nnodes, ngroups, skip_scale, h1, sc, X2, st);
    case 4: return cm::launch_forward<4>(B1, prod_WT, skip_WT, up_WT, node_perm, group_offsets, nnodes, ngroups, skip_scale, h1, sc, X2, st);
  }
  return CM_EINVAL;
}

namespace cm {

// Up to 1 536 blocks: beyond, a product is faster on tiles of 128 rows that share its operands (2 500 x 256 as three launches 28 us, cut 33).
bool node_chains_cut(int64_t nnodes, int channels) {
  return channels > 128 && few::blocks(nnodes, 1, channels) <= 1536 && few::applies(nnodes, 1, channels);
}

int node_glue_forward_cut(const float *B1, const float *prod_WT, const float *skip_WT, const float *up_WT, const int32_t *node_perm,
                          const int32_t *group_offsets, int64_t nnodes, int ngroups, int channels, float skip_scale, float *h1, float *sc, float *X2,
                          hipStream_t st) {
  switch (channels / 32) {
#define CM_CASE(NT_) \
    case NT_: return launch_forward_cut<NT_>(B1, prod_WT, skip_WT, up_WT, node_perm, group_offsets, nnodes, ngroups, skip_scale, h1, sc, X2, st);
    CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8)
#undef CM_CASE
    default: set_error("node glue: channels=%d not supported", channels); return CM_EINVAL;
  }
}

// cm_node_glue_backward whose launch also sums the node energies per graph (operands checked by the caller, cm_mace_step)
int node_glue_backward_with_energy_sums(const float *gX2, const float *d_h2, const float *up_W, const float *skip_W, const float *prod_W,
                                        const double *w1, double scale, const double *node_weights, const int32_t *node_perm,
                                        const int32_t *group_offsets, int64_t nnodes, int ngroups, int channels, float skip_scale, float *gh1,
                                        float *gB1, const double *node_es, const int32_t *graph_ptr, int ngraphs, double *energies,
                                        const double *graph_e0, double *total_energies, hipStream_t st) {
  const EnergySums sums{node_es, node_weights, graph_ptr, energies, ngraphs, graph_e0, total_energies};
  switch (channels / 32) {
    case 1: return launch_backward<1>(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, node_perm, group_offsets, nnodes, ngroups, skip_scale, gh1, gB1, sums, st);
    case 2: return launch_backward<2>(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, node_perm, group_offsets, nnodes, ngroups, skip_scale, gh1, gB1, sums, st);
    case 3: return launch_backward<3>(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, node_perm, group_offsets, nnodes, ngroups, skip_scale, gh1, gB1, sums, st);
    case 4: return launch_backward<4>(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, node_perm, group_offsets, nnodes, ngroups, skip_scale, gh1, gB1, sums, st);
#define CM_CASE(NT_) \
    case NT_: return launch_backward_cut<NT_>(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, node_perm, group_offsets, nnodes, ngroups, skip_scale, gh1, gB1, sums, st);
    CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8)
#undef CM_CASE
    default: set_error("node glue: channels=%d not supported", channels); return CM_EINVAL;
  }
}

int node_head(const float *B2, const float *sc, const float *h1, const float *prod_WT, const float *prod_W, const readout::Weights &w,
              const readout::Outputs &out, const double *node_weights, int64_t nnodes, int channels, float *d_h2, float *gB2, hipStream_t st) {
  CM_REQUIRE(w.hidden >= 1 && w.hidden <= readout::kHidden, "cm_mace_step: hidden=%d must be in [1, %d]", w.hidden, readout::kHidden);
  switch (channels / 32) {
    case 1: return launch_head<1>(B2, sc, h1, prod_WT, prod_W, w, out, node_weights, nnodes, d_h2, gB2, st);
    case 2: return launch_head<2>(B2, sc, h1, prod_WT, prod_W, w, out, node_weights, nnodes, d_h2, gB2, st);
    case 3: return launch_head<3>(B2, sc, h1, prod_WT, prod_W, w, out, node_weights, nnodes, d_h2, gB2, st);
    case 4: return launch_head<4>(B2, sc, h1, prod_WT, prod_W, w, out, node_weights, nnodes, d_h2, gB2, st);
    default: set_error("node head: channels=%d not supported", channels); return CM_EINVAL;
  }
}

}  // namespace cm

extern "C" int cm_node_glue_backward(const float *gX2, const float *d_h2, const float *up_W, const float *skip_W,
                                     const float *prod_W, const double *w1, double scale, const double *node_weights,
                                     const int32_t *node_perm, const int32_t *group_offsets, int64_t nnodes, int ngroups,
                                     int channels, float skip_scale, float *gB1, cm_stream_t stream) {
  CM_REQUIRE(cm_node_glue_supported(channels), "cm_node_glue_backward: channels=%d must be 32, 64, 96 or 128", channels);
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 256, "cm_node_glue_backward: nnodes out of range");
  CM_REQUIRE(ngroups >= 2, "cm_node_glue_backward: ngroups counts the elements plus the group of nodes without one");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(gX2 && d_h2 && up_W && skip_W && prod_W && w1 && node_perm && group_offsets && gB1, "cm_node_glue_backward: NULL pointer");
  return cm::node_glue_backward_with_energy_sums(gX2, d_h2, up_W, skip_W, prod_W, w1, scale, node_weights, node_perm, group_offsets,
                                                 nnodes, ngroups, channels, skip_scale, nullptr, gB1, nullptr, nullptr, 0, nullptr, nullptr,
                                                 nullptr, cm::as_stream(stream));
}
