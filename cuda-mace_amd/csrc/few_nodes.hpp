// Internal entry of few_nodes.hip for the one-call step.
#pragma once

#include "common.hpp"
#include "node_glue_device.hpp"
#include "readout_device.hpp"

namespace cm {
namespace fewnodes {

// Whether the step of this size (forces, or energies alone) takes a node through a whole layer per launch.
bool applies(const cm_mace_weights &w, int64_t nnodes, int64_t nedges, bool forces);

// Where the step keeps what one launch leaves for the next (rows of the workspace; energies alone: the second line NULL).
struct Scratch {
  float *vec, *X2, *h1, *sc;
  int32_t *live, *groups;  // [2 N] edge ranges up to the last edge inside the cutoff; [2 N] weight group and element of every node
  float *grad1, *d_h2, *gXe, *gv1, *gv2;
};

// First layer, edge vectors and live ranges included: vec, live, groups, h1, sc, X2 and, for forces, grad1.
int first_layer(const cm_mace_weights &w, const cm_mace_graph &g, const double *positions, const double *shifts, const Scratch &s, hipStream_t st);
// Second layer up to the node energies and, for forces, back to the gradients of its edges: d_h2, gXe, gv2.
int second_layer(const cm_mace_weights &w, const cm_mace_graph &g, const readout::Outputs &out, const Scratch &s, hipStream_t st);
// The rest of the backward chain down to the edge gradients of both layers, gv1, and the graph energies.
int back_to_edges(const cm_mace_weights &w, const cm_mace_graph &g, const EnergySums &sums, const Scratch &s, hipStream_t st);

}  // namespace fewnodes
}  // namespace cm
