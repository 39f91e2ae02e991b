// Internal entry of node_glue.hip for the one-call step.
#pragma once

#include "common.hpp"
#include "readout_device.hpp"

namespace cm {

// cm_node_glue_backward whose launch also sums the node energies per graph in extra workgroups (energies[g] = sum over
// graph g's nodes of node_weights[n] * node_es[n]; fixed order; total_energies[g] = energies[g] + graph_e0[g] when asked
// for, a missing graph_e0 counting as zero).  node_es must have been written by an earlier launch on the same stream.
// gh1: [nnodes, channels] of scratch memory.  Operands as checked by the caller.
int node_glue_backward_with_energy_sums(const float *gX2, const float *d_h2, const float *up_W, const float *skip_W, const float *prod_W,
                                        const double *w1, double scale, const double *node_weights, const int32_t *node_perm,
                                        const int32_t *group_offsets, int64_t nnodes, int ngroups, int channels, float skip_scale, float *gh1,
                                        float *gB1, const double *node_es, const int32_t *graph_ptr, int ngraphs, double *energies,
                                        const double *graph_e0, double *total_energies, hipStream_t st);

// Beyond 128 channels, few nodes: whether node_glue_forward_cut and node_glue_backward_with_energy_sums take the step's products between
// the layers, two launches per direction (the same products as three or four launches of the linear kernel).
bool node_chains_cut(int64_t nnodes, int channels);
int node_glue_forward_cut(const float *B1, const float *prod_WT, const float *skip_WT, const float *up_WT, const int32_t *node_perm,
                          const int32_t *group_offsets, int64_t nnodes, int ngroups, int channels, float skip_scale, float *h1, float *sc, float *X2,
                          hipStream_t st);

// h2 = B2 . Wprod + sc (kept on chip), the readouts of h1 and h2 with everything cm_readout_forward writes, and, with d_h2
// given, d_h2 = weight dE/dh2 (node_weights NULL: one) and gB2 = -d_h2 . Wprod^T.  32 to 128 channels (cm_node_glue_supported).
int node_head(const float *B2, const float *sc, const float *h1, const float *prod_WT, const float *prod_W, const readout::Weights &w,
              const readout::Outputs &out, const double *node_weights, int64_t nnodes, int channels, float *d_h2, float *gB2, hipStream_t st);

}  // namespace cm
