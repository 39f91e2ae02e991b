// Internal entry of geometry.hip for the one-call step.
#pragma once

#include "common.hpp"

namespace cm {

// cm_edge_geometry_backward of vector gradients alone that also writes node_virial [nnodes, 6] (xx, yy, zz, yz, xz, xy): the sum
// over the edges that start at an atom of 1/2 (vec (x) g + g (x) vec), vec [nedges, 3] the edge vectors.  Operands as checked by
// the caller; nnodes > 0.
int forces_and_node_virials(const float *grad_vectors, const float *vec, const int32_t *node_rows, const int32_t *a_first_occ,
                            const int32_t *b_perm, const int32_t *b_offsets, int64_t nnodes, int64_t nedges, double *forces,
                            double *node_virial, hipStream_t st);

}  // namespace cm
