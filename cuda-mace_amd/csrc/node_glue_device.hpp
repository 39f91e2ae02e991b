// Pieces of the step between the layers that node_glue.hip and few_nodes.hip share.
#pragma once

#include "common.hpp"

namespace cm {

// Energies per graph, riding in the backward launch (its tiles do not depend on them): out[g] = sum over the graph's nodes
// of weight[n] * node_es[n], strided partial sums of the workgroup's threads (the largest power of two of them) and a tree
// over them: a fixed order.
struct EnergySums {
  const double *node_es, *node_weights;
  const int32_t *graph_ptr;
  double *out;
  int ngraphs;
  const double *graph_e0;  // a constant per graph added into `total` (NULL: zero)
  double *total;           // NULL: not asked for
};
template <int THREADS, int PARTS = 4>  // THREADS: a power of two, at most the workgroup's size
__device__ __forceinline__ void graph_energy(const EnergySums &q, int graph, double *part) {
#pragma clang fp contract(off)
  const int tid = threadIdx.x;
  if (tid < THREADS) {
    const int lo = q.graph_ptr[graph], hi = q.graph_ptr[graph + 1];
    auto term = [&](int i) { return q.node_weights ? q.node_weights[i] * q.node_es[i] : q.node_es[i]; };
    // PARTS strided partial sums per thread, their loads requested together: one sum after the other waits for memory
    // once per node, and this workgroup would outlast the tiles of the launch
    double sum[PARTS];
#pragma unroll
    for (int k = 0; k < PARTS; ++k) sum[k] = 0.0;
    for (int i = lo + tid; i < hi; i += PARTS * THREADS) {
      double t[PARTS];
#pragma unroll
      for (int k = 0; k < PARTS; ++k) t[k] = i + k * THREADS < hi ? term(i + k * THREADS) : 0.0;
#pragma unroll
      for (int k = 0; k < PARTS; ++k) sum[k] += t[k];
    }
#pragma unroll
    for (int d = PARTS / 2; d > 0; d /= 2)
#pragma unroll
      for (int k = 0; k < d; ++k) sum[k] += sum[k + d];
    part[tid] = sum[0];
  }
  __syncthreads();
  for (int d = THREADS / 2; d > 0; d >>= 1) {
    if (tid < d) part[tid] += part[tid + d];
    __syncthreads();
  }
  if (tid == 0) {
    q.out[graph] = part[0];
    if (q.total) q.total[graph] = part[0] + (q.graph_e0 ? q.graph_e0[graph] : 0.0);
  }
}

// gh1 = gX2 . Wup^T + g1 - skip_scale dE/dh2 . Wskip^T of one column of a node from the two products (factor: what takes the
// second one to -skip_scale dE/dh2 . Wskip^T); every addition a rounding of its own, as where separate launches store what they add to.
__device__ __forceinline__ float gh1_of(float up, float skip, double w1, double scale, double node_weight, float factor, bool no_element) {
#pragma clang fp contract(off)
  const float g1 = static_cast<float>(-1.0 * scale * w1 * node_weight);
  const float sum = up + g1;
  return no_element ? sum : sum + skip * factor;
}

}  // namespace cm
