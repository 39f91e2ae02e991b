// The readouts' arithmetic per node, shared by readout.hip and node_glue.hip (which computes them between two products): both
// return the same bits.
#pragma once

#include "common.hpp"

namespace cm {
namespace readout {

typedef double d2v __attribute__((ext_vector_type(2)));
typedef double d4v __attribute__((ext_vector_type(4)));

constexpr int kHidden = 16;   // largest hidden width
constexpr int kClasses = 4;   // the 16-channel pieces of a node are summed in classes, piece p in class p % 4, added up at the end

struct Weights {
  const double *w1, *W2a, *w2b;  // [C], [C, hidden], [hidden]
  double act_cst, scale, shift;
  int hidden;
};
struct Outputs {
  double *node_es;          // [N]
  double *feats64;          // [N, 2 C] or NULL, in the rows below
  const int32_t *rows;      // row of feats64 and node_total that a node is written to (NULL: its own)
  const double *node_e0;    // [N] or NULL
  double *node_total;       // [N] or NULL
};

// Operand row `col` of the first product is hidden unit 4 (col % 4) + col / 4, so that element i of z in lane group g is
// unit 4 g + i, which is where the second product wants it; row `col` of the second is channel 4 (col % 4) + col / 4 of its
// piece, so that a lane's four results are neighbours in memory.
__device__ __forceinline__ int operand_row(int col) { return 4 * (col % 4) + col / 4; }

// four channels of one piece into the sums of its class: z (16 hidden units x 16 nodes) and the first readout
__device__ __forceinline__ void add_z(d4v &z, const double (&wz)[4], f4 h2) {
#pragma unroll
  for (int i = 0; i < 4; ++i) z = __builtin_amdgcn_mfma_f64_16x16x4f64(wz[i], static_cast<double>(h2[i]), z, 0, 0, 0);
}
__device__ __forceinline__ void add_linear(double &e1, d2v w01, d2v w23, f4 h1) {
  e1 += static_cast<double>(h1.x) * w01.x;
  e1 += static_cast<double>(h1.y) * w01.y;
  e1 += static_cast<double>(h1.z) * w23.x;
  e1 += static_cast<double>(h1.w) * w23.y;
}
// energy and derivative of a hidden unit; gate: its w2b times the normalisation of the gate
__device__ __forceinline__ void activate(double gate, double z, double &e, double &d) {
  const double sig = 1.0 / (1.0 + exp(-z));
  e = gate * z * sig;
  d = gate * (sig + z * sig * (1.0 - sig));
}
// node energy from the lanes' sums (lanes 16 g + node: channels and hidden units of group g)
__device__ __forceinline__ double node_energy(double e, double scale, double shift) {
  e += __shfl_xor(e, 16);
  e += __shfl_xor(e, 32);
  return scale * e + shift;
}
// four channels of dE/dh2 of a node, the lane's share of the 16 channels x 16 nodes of a piece
__device__ __forceinline__ f4 derivative(const double (&wd)[4], const double (&d)[4], double scale) {
  d4v g{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < 4; ++i) g = __builtin_amdgcn_mfma_f64_16x16x4f64(wd[i], d[i], g, 0, 0, 0);
  return f4{static_cast<float>(scale * g[0]), static_cast<float>(scale * g[1]), static_cast<float>(scale * g[2]), static_cast<float>(scale * g[3])};
}
// four channels of both feature rows in double precision
__device__ __forceinline__ void store_feats(double *f, int C, f4 h1, f4 h2) {
  reinterpret_cast<d2v *>(f)[0] = d2v{h1.x, h1.y};
  reinterpret_cast<d2v *>(f)[1] = d2v{h1.z, h1.w};
  reinterpret_cast<d2v *>(f + C)[0] = d2v{h2.x, h2.y};
  reinterpret_cast<d2v *>(f + C)[1] = d2v{h2.z, h2.w};
}
__device__ __forceinline__ void store_energy(const Outputs &o, int node, int row, bool row_ok, double en) {
  o.node_es[node] = en;
  if (o.node_total && row_ok) o.node_total[row] = en + (o.node_e0 ? o.node_e0[node] : 0.0);
}

}  // namespace readout
}  // namespace cm
