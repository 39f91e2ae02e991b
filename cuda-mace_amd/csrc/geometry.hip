// Edge geometry: vectors and lengths from positions, and the scatter of their gradients back to
// the atoms (what makes forces out of per-edge gradients).
//
// Forward: vec[e] = pos[b[e]] - pos[a[e]] + shift[e] in fp64, rounded once to fp32 for the
// kernels downstream, plus its length.  Backward: the gradient of an atom is the signed sum of the
// edge-vector gradients over the edges that start (a) or end (b) at it; both sums run over
// contiguous index ranges (CSR of the sorted row a, sender-sorted view of row b), a wave or a
// quarter of one per atom, accumulated in fp64 with a fixed reduction order -- no atomics, bit-reproducible.
//
// Optional row map: with `rows` given, atom n of the edge lists is row rows[n] of `pos` and of the position gradient.
// A caller that works on a relabelled copy of the graph then keeps positions and forces in its own order and needs no
// gather on the way in or out.
#include "common.hpp"

namespace cm {
namespace {

__device__ __forceinline__ int row_of(const int32_t *__restrict__ rows, int n) { return rows ? rows[n] : n; }

__global__ void edge_geometry_forward_kernel(const double *__restrict__ pos, const int32_t *__restrict__ a,
                                             const int32_t *__restrict__ b, const double *__restrict__ shifts,
                                             const int32_t *__restrict__ rows, int64_t nedges, int nnodes,
                                             float *__restrict__ vec, float *__restrict__ len) {
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (e >= nedges) return;
  double v[3];
  edge_vector_f64(pos, a, b, shifts, rows, e, nnodes, v);
  vec[3 * e + 0] = static_cast<float>(v[0]);
  vec[3 * e + 1] = static_cast<float>(v[1]);
  vec[3 * e + 2] = static_cast<float>(v[2]);
  len[e] = static_cast<float>(sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]));
}

// total gradient with respect to the edge vector: g_vec + g_len * vec / |vec| (vec recomputed in fp64).  Without a
// length gradient nothing but g_vec is touched.
template <bool HAS_GLEN>
__device__ __forceinline__ void edge_grad(const double *__restrict__ pos, const double *__restrict__ shifts,
                                          const int32_t *__restrict__ a, const int32_t *__restrict__ b,
                                          const int32_t *__restrict__ rows, const float *__restrict__ gvec,
                                          const float *__restrict__ glen, int64_t e, int nnodes, double (&g)[3]) {
  if constexpr (!HAS_GLEN) {
#pragma unroll
    for (int k = 0; k < 3; ++k) g[k] = gvec ? static_cast<double>(gvec[3 * e + k]) : 0.0;
    return;
  }
  const int ia = a[e], ib = b[e];
  g[0] = g[1] = g[2] = 0.0;
  if (static_cast<unsigned>(ia) >= static_cast<unsigned>(nnodes) || static_cast<unsigned>(ib) >= static_cast<unsigned>(nnodes)) return;
  double v[3];
  const int ra = row_of(rows, ia), rb = row_of(rows, ib);
#pragma unroll
  for (int k = 0; k < 3; ++k) v[k] = pos[3 * rb + k] - pos[3 * ra + k] + shifts[3 * e + k];
  const double r = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  const double s = r > 0.0 ? static_cast<double>(glen[e]) / r : 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) g[k] = (gvec ? static_cast<double>(gvec[3 * e + k]) : 0.0) + s * v[k];
}

template <bool HAS_GLEN>
__global__ void edge_grad_kernel(const double *__restrict__ pos, const double *__restrict__ shifts,
                                 const int32_t *__restrict__ a, const int32_t *__restrict__ b,
                                 const int32_t *__restrict__ rows, const float *__restrict__ gvec,
                                 const float *__restrict__ glen, int64_t nedges, int nnodes, double *__restrict__ gshift) {
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (e >= nedges) return;
  double g[3];
  edge_grad<HAS_GLEN>(pos, shifts, a, b, rows, gvec, glen, e, nnodes, g);
  gshift[3 * e + 0] = g[0];
  gshift[3 * e + 1] = g[1];
  gshift[3 * e + 2] = g[2];
}

// LANES per atom.  A wave's time is its chain of dependent loads (offsets, edge number, gradient) and the reduction.  Up to
// kFewAtoms atoms a wave takes one, and its edges in one or two trips; beyond, where every SIMD has several waves, four
// atoms share a wave's chain and reduction, with four edges per lane and trip whose loads are requested together.  In the step
// (us; forces alone, a wave per atom -> 16 lanes): 10 752 x 10 8.8 -> 4.9, 25 000 x 52 22.6 -> 20.0, 100 000 x 52 77 -> 65.
// VIRIAL: the atom's share of the virial from the edges that start at it, as the comment on virials in step.hip has it, instead of
// in a launch of its own: 216 x 90 edges 5.7 + 5.5 -> 6.0 (16 lanes 11.0), 1 000 x 52 5.3 (16 lanes 7.7), 5 000 x 52 9.1 + 5.0 -> 12.1,
// 12 000 x 24 14.1 + 5.8 -> 13.5; alone, 5 000 x 52 with 64 lanes 9.6 and with 16 lanes 6.4.
// Runs of 128 neighbouring atoms on an XCD: gradients of edges that end at neighbours share lines (25 000 x 52 20.0 -> 17.2, 100 000 x 52 65.7 -> 62.3).
constexpr int64_t kFewAtoms = 2048;
template <int LANES, bool HAS_GLEN, bool VIRIAL>
__global__ __launch_bounds__(256) void edge_geometry_backward_kernel(
    const double *__restrict__ pos, const double *__restrict__ shifts, const int32_t *__restrict__ a,
    const int32_t *__restrict__ b, const int32_t *__restrict__ rows, const int32_t *__restrict__ a_first_occ,
    const int32_t *__restrict__ b_perm, const int32_t *__restrict__ b_offsets, const float *__restrict__ gvec,
    const float *__restrict__ glen, int64_t nedges, int nnodes, double *__restrict__ gpos, const float *__restrict__ vec,
    double *__restrict__ node_virial) {
  constexpr int kEdgesAhead = kWave / LANES;
  const int lane = threadIdx.x % LANES;
  const int node = place_on_xcd<LANES / 2>(blockIdx.x, gridDim.x) * (blockDim.x / LANES) + threadIdx.x / LANES;
  const bool here = node < nnodes;
  double acc[3] = {0.0, 0.0, 0.0}, vir[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int kb0 = 0, kb1 = 0, ea0 = 0, ea1 = 0, row = 0;
  if (here) {
    kb0 = b_offsets[node], kb1 = b_offsets[node + 1];
    ea0 = a_first_occ[node], ea1 = a_first_occ[nnodes + node];
    clamp_edge_range(ea0, ea1, nedges);
    row = row_of(rows, node);
  }
  // every load of a trip is issued whatever its edge (one beyond the list reads the list's last and is dropped): loads under a
  // branch of their own are waited for one after the other
  auto take = [&](int e, bool counts, double (&g)[3]) {
    if constexpr (HAS_GLEN) {
      g[0] = g[1] = g[2] = 0.0;
      if (counts) edge_grad<true>(pos, shifts, a, b, rows, gvec, glen, e, nnodes, g);
    } else {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const float v = gvec ? gvec[3 * static_cast<int64_t>(e) + i] : 0.f;
        g[i] = counts ? static_cast<double>(v) : 0.0;
      }
    }
  };
  // edges that end at this atom (row b): + gradient
  for (int k0 = kb0 + lane; k0 < kb1; k0 += LANES * kEdgesAhead) {
    int e[kEdgesAhead];
    double g[kEdgesAhead][3];
#pragma unroll
    for (int u = 0; u < kEdgesAhead; ++u) e[u] = b_perm[min(k0 + u * LANES, kb1 - 1)];
#pragma unroll
    for (int u = 0; u < kEdgesAhead; ++u) {
      const bool known = static_cast<unsigned>(e[u]) < static_cast<uint64_t>(nedges);
      take(known ? e[u] : 0, known && k0 + u * LANES < kb1, g[u]);
    }
#pragma unroll
    for (int u = 0; u < kEdgesAhead; ++u)
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i] += g[u][i];
  }
  // edges that start at this atom (row a, contiguous): - gradient
  for (int e0 = ea0 + lane; e0 < ea1; e0 += LANES * kEdgesAhead) {
    double g[kEdgesAhead][3];
    float v[kEdgesAhead][3];
#pragma unroll
    for (int u = 0; u < kEdgesAhead; ++u) {
      const int e = min(e0 + u * LANES, ea1 - 1);
      take(e, e0 + u * LANES < ea1, g[u]);
      if constexpr (VIRIAL) {
#pragma unroll
        for (int i = 0; i < 3; ++i) v[u][i] = vec[3 * static_cast<int64_t>(e) + i];
      }
    }
#pragma unroll
    for (int u = 0; u < kEdgesAhead; ++u) {
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i] -= g[u][i];
      if constexpr (VIRIAL) {
        const bool counts = e0 + u * LANES < ea1;
        const double v0 = counts ? v[u][0] : 0.f, v1 = counts ? v[u][1] : 0.f, v2 = counts ? v[u][2] : 0.f;
        vir[0] += v0 * g[u][0], vir[1] += v1 * g[u][1], vir[2] += v2 * g[u][2];
        vir[3] += 0.5 * (v1 * g[u][2] + v2 * g[u][1]), vir[4] += 0.5 * (v0 * g[u][2] + v2 * g[u][0]);
        vir[5] += 0.5 * (v0 * g[u][1] + v1 * g[u][0]);
      }
    }
  }
#pragma unroll
  for (int off = LANES / 2; off > 0; off >>= 1) {
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i] += __shfl_xor(acc[i], off);
    if constexpr (VIRIAL) {
#pragma unroll
      for (int i = 0; i < 6; ++i) vir[i] += __shfl_xor(vir[i], off);
    }
  }
  if (here && lane == 0) {
#pragma unroll
    for (int i = 0; i < 3; ++i) gpos[3 * static_cast<int64_t>(row) + i] = acc[i];
    if constexpr (VIRIAL) {
#pragma unroll
      for (int i = 0; i < 6; ++i) node_virial[6 * static_cast<int64_t>(node) + i] = vir[i];
    }
  }
}

template <bool HAS_GLEN, bool VIRIAL>
void launch_backward(const double *pos, const double *shifts, const int32_t *a, const int32_t *b, const int32_t *rows, const int32_t *a_first_occ,
                     const int32_t *b_perm, const int32_t *b_offsets, const float *gvec, const float *glen, int64_t nedges, int64_t nnodes,
                     double *gpos, const float *vec, double *node_virial, hipStream_t st) {
  const int lanes = nnodes <= kFewAtoms ? kWave : 16;
  const dim3 grid(static_cast<unsigned>(ceil_div(nnodes, 256 / lanes))), block(256);
  if (nnodes <= kFewAtoms)
    hipLaunchKernelGGL((edge_geometry_backward_kernel<kWave, HAS_GLEN, VIRIAL>), grid, block, 0, st, pos, shifts, a, b, rows, a_first_occ, b_perm, b_offsets,
                       gvec, glen, nedges, static_cast<int>(nnodes), gpos, vec, node_virial);
  else
    hipLaunchKernelGGL((edge_geometry_backward_kernel<16, HAS_GLEN, VIRIAL>), grid, block, 0, st, pos, shifts, a, b, rows, a_first_occ, b_perm, b_offsets,
                       gvec, glen, nedges, static_cast<int>(nnodes), gpos, vec, node_virial);
}

}  // namespace
}  // namespace cm

namespace cm {

int forces_and_node_virials(const float *grad_vectors, const float *vec, const int32_t *node_rows, const int32_t *a_first_occ,
                            const int32_t *b_perm, const int32_t *b_offsets, int64_t nnodes, int64_t nedges, double *forces,
                            double *node_virial, hipStream_t st) {
  launch_backward<false, true>(nullptr, nullptr, nullptr, nullptr, node_rows, a_first_occ, b_perm, b_offsets, grad_vectors, nullptr, nedges, nnodes, forces,
                               vec, node_virial, st);
  return check_launch("cm_mace_step (forces)");
}

}  // namespace cm

extern "C" int cm_edge_geometry_forward(const double *positions, const int32_t *row_a, const int32_t *row_b,
                                        const double *shifts, const int32_t *node_rows, int64_t nnodes, int64_t nedges,
                                        float *vectors, float *lengths, cm_stream_t stream) {
  CM_REQUIRE(nedges >= 0 && nnodes >= 0 && nnodes < INT32_MAX / 4, "cm_edge_geometry_forward: sizes out of range");
  if (nedges == 0) return CM_OK;
  CM_REQUIRE(positions && row_a && row_b && shifts && vectors && lengths, "cm_edge_geometry_forward: NULL pointer");
  const int block = 256;
  hipLaunchKernelGGL(cm::edge_geometry_forward_kernel, dim3(static_cast<unsigned>(cm::ceil_div(nedges, block))), dim3(block),
                     0, cm::as_stream(stream), positions, row_a, row_b, shifts, node_rows, nedges, static_cast<int>(nnodes), vectors,
                     lengths);
  return cm::check_launch("cm_edge_geometry_forward");
}

extern "C" int cm_edge_geometry_backward(const double *positions, const int32_t *row_a, const int32_t *row_b,
                                         const double *shifts, const int32_t *node_rows, const int32_t *a_first_occ,
                                         const int32_t *b_perm, const int32_t *b_offsets, const float *grad_vectors,
                                         const float *grad_lengths,
                                         int64_t nnodes, int64_t nedges, double *grad_positions, double *grad_shifts,
                                         cm_stream_t stream) {
  CM_REQUIRE(nedges >= 0 && nnodes >= 0 && nnodes < INT32_MAX / 4, "cm_edge_geometry_backward: sizes out of range");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(a_first_occ && b_offsets, "cm_edge_geometry_backward: NULL index structure");
  CM_REQUIRE(nedges == 0 || (positions && row_a && row_b && shifts && b_perm), "cm_edge_geometry_backward: NULL pointer");
  hipStream_t st = cm::as_stream(stream);
  if (grad_positions) {
    if (grad_lengths)
      cm::launch_backward<true, false>(positions, shifts, row_a, row_b, node_rows, a_first_occ, b_perm, b_offsets, grad_vectors, grad_lengths, nedges,
                                       nnodes, grad_positions, nullptr, nullptr, st);
    else
      cm::launch_backward<false, false>(positions, shifts, row_a, row_b, node_rows, a_first_occ, b_perm, b_offsets, grad_vectors, nullptr, nedges, nnodes,
                                        grad_positions, nullptr, nullptr, st);
  }
  if (grad_shifts && nedges > 0) {
    const int block = 256;
    const dim3 grid(static_cast<unsigned>(cm::ceil_div(nedges, block)));
    if (grad_lengths)
      hipLaunchKernelGGL(cm::edge_grad_kernel<true>, grid, dim3(block), 0, st, positions, shifts, row_a, row_b, node_rows,
                         grad_vectors, grad_lengths, nedges, static_cast<int>(nnodes), grad_shifts);
    else
      hipLaunchKernelGGL(cm::edge_grad_kernel<false>, grid, dim3(block), 0, st, positions, shifts, row_a, row_b, node_rows,
                         grad_vectors, grad_lengths, nedges, static_cast<int>(nnodes), grad_shifts);
  }
  return cm::check_launch("cm_edge_geometry_backward");
}
