// One energy + forces evaluation of the two-layer invariant model: the library enqueues every kernel of the step
// itself, forward and then the hand-written backward chain, through the same entry points a caller could use one by
// one.  Nothing here computes; this file is the order of the launches and the layout of the workspace.
//
// Forward                                         Backward (seed -1 on every node energy: the chain delivers forces)
//   vec        = pos[snd] - pos[rcv] + shift        g1 = -scale w1 (every node), g2 = -dE/dh2 (never stored: the sign
//                                                             goes into the scale of the linears that read dE/dh2)
//   live       = edge ranges up to the last pair
//                inside the cutoff (forward MP only)
//   M1         = MP(X1, vec, spline 0)              gB2       = g2 . Wprod2^T
//   A          = mix0(M1)        (per element)      gA        = (gB2 * grad2) . Wmix1^T      (contraction backward folded)
//   B1, grad1  = contraction 0 (A)                  gX2, gv2  = MP backward(X2, vec, spline 1, gA)
//   h1         = B1 . Wprod1                        gh1       = gX2 . Wup^T + g1 ;  gh1 += skip^T(g2)
//   sc         = skip(h1)        (per element)      gB1       = gh1 . Wprod1^T
//   X2         = h1 . Wup                           gA        = (gB1 * grad1) . Wmix0^T      (per element)
//   M2         = MP(X2, vec, spline 1)              gv1       = MP backward(X1, vec, spline 0, gA)   (no gX: X1 is constant)
//   A          = mix1(M2)                           forces    = geometry backward(gv1 + gv2)
//   B2, grad2  = contraction 1 (A)                  virials   = 1/2 sum_e (vec (x) gv + gv (x) vec), per node, then per graph
//   h2         = B2 . Wprod2 + sc                               (on request)
//   E_n, dE/dh2, feats = readouts(h1, h2);  E_graph = sum over the graph's nodes
// With node weights (cm_mace_graph.node_weights) E_graph = sum_n weight[n] E_n and the seed of node n is -weight[n]: g1's
// rows and the rows of dE/dh2 are multiplied by the node's weight before the chain starts.
#include <cstdlib>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "few_nodes.hpp"
#include "geometry.hpp"
#include "mp_common.hpp"
#include "node_glue.hpp"
#include "readout.hpp"

namespace cm {
namespace {

// ---- optional per-stage timing: events on the launch stream around chosen stages of the step --------------------
constexpr int kStages = 25;
struct Pending {
  int stage;
  hipEvent_t start, stop;
};
std::mutex g_timing_mutex;
unsigned g_timing_mask = 0;  // bit s set: stage s is bracketed by events
std::vector<Pending> g_pending;
std::vector<hipEvent_t> g_event_pool;
double g_stage_ms[kStages] = {};
int64_t g_stage_launches[kStages] = {};

hipEvent_t take_event() {
  if (!g_event_pool.empty()) {
    hipEvent_t e = g_event_pool.back();
    g_event_pool.pop_back();
    return e;
  }
  hipEvent_t e = nullptr;
  (void)hipEventCreate(&e);
  return e;
}

// Brackets one stage with events when its bit is set; used only through CM_STAGE below.
struct StageTimer {
  hipStream_t st;
  int stage;
  hipEvent_t start = nullptr;
  StageTimer(hipStream_t s, int stage_, unsigned mask) : st(s), stage(stage_) {
    if (mask >> stage & 1u) {
      std::lock_guard<std::mutex> lock(g_timing_mutex);
      start = take_event();
      if (start) (void)hipEventRecord(start, st);
    }
  }
  ~StageTimer() {
    if (!start) return;
    std::lock_guard<std::mutex> lock(g_timing_mutex);
    hipEvent_t stop = take_event();
    if (stop) {
      (void)hipEventRecord(stop, st);
      g_pending.push_back({stage, start, stop});
    } else {
      g_event_pool.push_back(start);
    }
  }
};

__global__ void fill_f64_kernel(double *p, int64_t n, double value) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    p[i] = value;
}

// p[i] = src[i], or zero without a source
__global__ void copy_or_zero_f64_kernel(double *p, const double *src, int64_t n) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    p[i] = src ? src[i] : 0.0;
}

// Edge vectors and the edge range of every receiver node cut back to its last edge inside the cutoff, one launch.
// Thread i forms the vector of edge i (fp64 difference of the positions plus the shift, rounded once to fp32: the
// arithmetic of cm_edge_geometry_forward), writes it as the row of `vec` the backward chain reads and, for the forward kernel with
// the table in LDS, as a record of 16 bytes with the sender (either may be NULL), and, where a backward chain follows (gv1 and gv2 given), clears the vector
// gradients of an edge beyond the cutoff (the backward edge passes skip the edges behind a node's mark, and write the same
// zeros for those before it), and leaves a bit per edge inside the cutoff for the sender pass (live_bits, may be NULL).  The thread of a receiver's
// last edge closes the receiver's range: live[n] = first_occ[n], live[nnodes + n] = one past the last edge e of the node
// with |vec[e]| <= r_max (the node's first edge if there is none).  The message-passing kernels, forward and backward,
// skip the edges behind that mark, which contribute exact zeros.  A Verlet list holds a third more pairs than the cutoff
// takes in; the model orders each node's pairs with those of the skin shell last, nearest first, so that most of them
// fall behind the mark.  The closing thread reads the mark off the workgroup's ballots of "inside the cutoff" where the
// node's edges up to the mark lie among the workgroup's 256; otherwise it walks back from the workgroup's first edge,
// forming those vectors again (a walk over all of a node's tail, one line of memory per lane and access, cost a list
// with a skin 60 us per step).  The length is the one the message-passing kernels compute from the same fp32 vector.
__device__ __forceinline__ int walk_back_to_live_edge(const double *__restrict__ pos, const int32_t *__restrict__ a,
                                                      const int32_t *__restrict__ b, const double *__restrict__ shifts,
                                                      const int32_t *__restrict__ rows, int nnodes, float r_max, int e0, int e) {
  // by the whole wave, 64 edges per trip, with the same arguments in every lane: one past the last live edge of e0 .. e - 1, or e0
  while (e > e0) {
    const int q = e - 1 - static_cast<int>(threadIdx.x % kWave);
    double w[3];
    edge_vector_f64(pos, a, b, shifts, rows, max(q, e0), nnodes, w);
    const bool live = q >= e0 && mp::edge_length(static_cast<float>(w[0]), static_cast<float>(w[1]), static_cast<float>(w[2])) <= r_max;
    const unsigned long long lives = __ballot(live);
    if (lives != 0) return e - (__ffsll(static_cast<long long>(lives)) - 1);
    e = max(e - kWave, e0);
  }
  return e;
}

__global__ __launch_bounds__(256) void geometry_live_range_kernel(const double *__restrict__ pos, const int32_t *__restrict__ a,
                                                                  const int32_t *__restrict__ b, const double *__restrict__ shifts,
                                                                  const int32_t *__restrict__ rows, const int32_t *__restrict__ first_occ,
                                                                  float r_max, int nnodes, int64_t nedges, float *__restrict__ vec,
                                                                  float4 *__restrict__ records, int32_t *__restrict__ live,
                                                                  float *__restrict__ gv1, float *__restrict__ gv2,
                                                                  unsigned long long *__restrict__ live_bits) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  const int lane = threadIdx.x % kWave;
  bool inside = false;
  int recv = -1, next_recv = -2;
  if (i < nedges) {
    double v[3];
    edge_vector_f64(pos, a, b, shifts, rows, i, nnodes, v);
    const float v0 = static_cast<float>(v[0]), v1 = static_cast<float>(v[1]), v2 = static_cast<float>(v[2]);
    if (vec) {
      vec[3 * i + 0] = v0;
      vec[3 * i + 1] = v1;
      vec[3 * i + 2] = v2;
    }
    if (records) records[i] = make_float4(v0, v1, v2, __int_as_float(b[i]));
    inside = mp::edge_length(v0, v1, v2) <= r_max;
    if (!inside && gv1) {
      gv1[3 * i + 0] = gv1[3 * i + 1] = gv1[3 * i + 2] = 0.f;
      gv2[3 * i + 0] = gv2[3 * i + 1] = gv2[3 * i + 2] = 0.f;
    }
    recv = a[i];
    next_recv = i + 1 < nedges ? a[i + 1] : -2;
  }
  // "inside the cutoff" of the workgroup's 256 consecutive edges, one word per wave (every thread arrives here)
  __shared__ unsigned long long s_inside[4];
  const int wave = threadIdx.x / kWave;
  const unsigned long long inside_mask = __ballot(inside);
  if (lane == 0) {
    s_inside[wave] = inside_mask;
    if (live_bits && i < nedges) live_bits[i / kWave] = inside_mask;
  }
  __syncthreads();
  const bool closes = i < nedges && recv != next_recv && static_cast<unsigned>(recv) < static_cast<unsigned>(nnodes);
  int e0 = 0, e = -1, from = 0;  // from: where the walk begins if the ballots do not settle it
  if (closes) {
    int e1 = first_occ[nnodes + recv];
    e0 = first_occ[recv];
    clamp_edge_range(e0, e1, nedges);
    from = e1;
    if (e1 == i + 1) {  // this is the last edge of the receiver's range, as in every sorted list
      const int64_t group_first = i - threadIdx.x;  // first edge of the workgroup
      // the node's edges in this workgroup, from this wave down: the highest one inside the cutoff
      for (int w = wave; w >= 0 && e < 0; --w) {
        const int64_t wave_first = group_first + w * kWave;
        if (wave_first + kWave <= e0) break;  // the node's range begins above this wave
        const int hi = w == wave ? lane : kWave - 1;
        const int lo = e0 > wave_first ? static_cast<int>(e0 - wave_first) : 0;
        const unsigned long long upto = hi == kWave - 1 ? ~0ull : (1ull << (hi + 1)) - 1ull;
        const unsigned long long mine = s_inside[w] & upto & ~((1ull << lo) - 1ull);
        if (mine != 0) e = static_cast<int>(wave_first) + (63 - __clzll(static_cast<long long>(mine))) + 1;
      }
      if (e < 0 && e0 >= group_first) e = e0;
      from = static_cast<int>(group_first);
    }
  }
  // what is left, a node at a time, by all lanes (every lane of the wave arrives here)
  for (unsigned long long left = __ballot(closes && e < 0); left != 0; left &= left - 1) {
    const int of = __ffsll(static_cast<long long>(left)) - 1;
    const int found = walk_back_to_live_edge(pos, a, b, shifts, rows, nnodes, r_max, __builtin_amdgcn_readlane(e0, of), __builtin_amdgcn_readlane(from, of));
    if (lane == of) e = found;
  }
  if (closes) {
    live[recv] = e0;
    live[nnodes + recv] = e;
  }
  if (i < nnodes) {  // a node without edges: an empty range
    const int n = static_cast<int>(i);
    int e0 = first_occ[n], e1 = first_occ[nnodes + n];
    clamp_edge_range(e0, e1, nedges);
    if (e0 >= e1) {
      live[n] = e0;
      live[nnodes + n] = e0;
    }
  }
}

// out[g] = sum of x over the nodes ptr[g] .. ptr[g + 1]: one workgroup per graph, every thread a strided partial sum, a
// tree over the partials: the same order on every run.
constexpr int kSumThreads = 1024;
__device__ __forceinline__ void segment_sum(const double *__restrict__ x, const double *__restrict__ weights, const int32_t *__restrict__ ptr,
                                            double *__restrict__ out, const double *__restrict__ graph_e0, double *__restrict__ total, int graph) {
  __shared__ double part[kSumThreads];
  const int lo = ptr[graph], hi = ptr[graph + 1];
  auto term = [&](int i) { return weights ? weights[i] * x[i] : x[i]; };
  // four strided partial sums per thread, their loads requested together (one sum waits for memory once per element)
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  int i = lo + threadIdx.x;
  for (; i + 3 * kSumThreads < hi; i += 4 * kSumThreads) {
    const double t0 = term(i), t1 = term(i + kSumThreads), t2 = term(i + 2 * kSumThreads), t3 = term(i + 3 * kSumThreads);
    s0 += t0, s1 += t1, s2 += t2, s3 += t3;
  }
  for (; i < hi; i += kSumThreads) s0 += term(i);
  part[threadIdx.x] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  for (int d = kSumThreads / 2; d > 0; d >>= 1) {
    if (threadIdx.x < d) part[threadIdx.x] += part[threadIdx.x + d];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[graph] = part[0];
    if (total) total[graph] = part[0] + (graph_e0 ? graph_e0[graph] : 0.0);
  }
}

__global__ __launch_bounds__(kSumThreads) void segment_sum_f64_kernel(const double *__restrict__ x, const double *__restrict__ weights,
                                                                     const int32_t *__restrict__ ptr, double *__restrict__ out,
                                                                     const double *__restrict__ graph_e0, double *__restrict__ total) {
  segment_sum(x, weights, ptr, out, graph_e0, total, blockIdx.x);
}

// Between the readouts and the backward chain of the separate launches (beyond 128 channels): the graph energies, a workgroup each,
// and in the others the seeds of the chain, a wave per node: g1[n, c] = -weight[n] * scale * w1[c], the gradient of
// -sum(weight * node energies) with respect to the first layer's features (the linear readout), without weights the same row
// for every node; with weights d_h2's rows (the second readout's derivative) times the node's weight.  One launch instead of two or,
// with weights, three, each of them a latency for a small system, with the sum of a large graph alongside the rows.  In the step (us):
// 60 x 192 7 -> 3.2, 12 000 x 256 with weights 23.5 -> 11.6, 100 000 x 192 41 -> 32 (the rows, 16 bytes per lane, and the sum alike).
__global__ __launch_bounds__(kSumThreads) void energies_and_seeds_kernel(const double *__restrict__ node_es, const double *__restrict__ node_weights,
                                                                        const int32_t *__restrict__ ptr, double *__restrict__ energies,
                                                                        const double *__restrict__ graph_e0, double *__restrict__ total, int ngraphs,
                                                                        float *__restrict__ g1, float *__restrict__ d_h2,
                                                                        const double *__restrict__ w1, double scale, int nnodes, int C) {
  if (static_cast<int>(blockIdx.x) < ngraphs) {
    segment_sum(node_es, node_weights, ptr, energies, graph_e0, total, blockIdx.x);
    return;
  }
  constexpr int kWaves = kSumThreads / kWave;
  const int c = 4 * (threadIdx.x % kWave);
  if (c >= C) return;
  double w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) w[k] = w1[c + k];
  for (int n = (blockIdx.x - ngraphs) * kWaves + threadIdx.x / kWave; n < nnodes; n += (gridDim.x - ngraphs) * kWaves) {
    const int64_t at = static_cast<int64_t>(n) * C + c;
    const double nw = node_weights ? node_weights[n] : 1.0;
    f4 g;
#pragma unroll
    for (int k = 0; k < 4; ++k) g[k] = static_cast<float>(-1.0 * scale * w[k] * nw);
    st4(g1 + at, g);
    if (node_weights) {
      f4 d = ld4(d_h2 + at);
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = static_cast<float>(static_cast<double>(d[k]) * nw);
      st4(d_h2 + at, d);
    }
  }
}

// Virials from the per-edge gradients the backward chain ends with: under a symmetric strain every edge vector becomes
// vec + vec . strain, so -dE/d strain = 1/2 sum_e (vec_e (x) gv_e + gv_e (x) vec_e) with gv_e = -dE/d vec_e, which is what
// the chain delivers.  Two levels, both in a fixed order: per receiver node (with the forces, geometry.hip), then per graph.
// node_virial [nnodes, 6]: xx, yy, zz, yz, xz, xy.
// virials[g] (3 x 3, symmetric) = sum of node_virial over the graph's nodes; one workgroup per graph, strided partial sums
// and a tree over them.  stress[g] = -virials[g] / volume (cell and stress may be NULL), the volume as the triple product of
// the cell vectors: in a launch of its own it was 4 to 5 us at any size.
__device__ __forceinline__ double cell_volume(const double *c) {
  return fabs(c[0] * (c[4] * c[8] - c[5] * c[7]) + c[1] * (c[5] * c[6] - c[3] * c[8]) + c[2] * (c[3] * c[7] - c[4] * c[6]));
}

__global__ __launch_bounds__(kSumThreads) void graph_virial_kernel(const double *__restrict__ node_virial,
                                                                   const int32_t *__restrict__ ptr, double *__restrict__ virials,
                                                                   const double *__restrict__ cell, double *__restrict__ stress) {
  __shared__ double part[6][kSumThreads];
  const int lo = ptr[blockIdx.x], hi = ptr[blockIdx.x + 1];
  double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int i = lo + threadIdx.x; i < hi; i += kSumThreads) {
#pragma unroll
    for (int k = 0; k < 6; ++k) s[k] += node_virial[6 * static_cast<int64_t>(i) + k];
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) part[k][threadIdx.x] = s[k];
  __syncthreads();
  for (int d = kSumThreads / 2; d > 0; d >>= 1) {
    if (threadIdx.x < d) {
#pragma unroll
      for (int k = 0; k < 6; ++k) part[k][threadIdx.x] += part[k][threadIdx.x + d];
    }
    __syncthreads();
  }
  if (threadIdx.x < 9) {
    const int a = threadIdx.x / 3, b = threadIdx.x % 3;
    const double v = part[a == b ? a : 6 - a - b][0];  // xx, yy, zz, yz, xz, xy
    const int64_t at = 9 * static_cast<int64_t>(blockIdx.x);
    virials[at + threadIdx.x] = v;
    if (stress) stress[at + threadIdx.x] = -v / cell_volume(cell + at);
  }
}

__global__ void stress_kernel(const double *__restrict__ virials, const double *__restrict__ cell, int64_t ngraphs,
                              double *__restrict__ stress) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i < 9 * ngraphs) stress[i] = -virials[i] / cell_volume(cell + i / 9 * 9);
}

// Results of a step to a caller on the host: the values straight into its memory, every word its own flag (see cm_report).
constexpr int kMaxReports = 4;
constexpr unsigned long long kNotYet = 0x7ff4c0dec0dec0deull;  // a NaN that no arithmetic returns

struct Reports {
  const unsigned long long *src[kMaxReports];
  int64_t end[kMaxReports];  // where the array's values end in the host's memory
};

__global__ __launch_bounds__(256) void report_kernel(Reports r, int64_t n, unsigned long long *__restrict__ host) {
  for (int64_t k = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; k < n; k += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    int a = 0;
    while (k >= r.end[a]) ++a;
    __hip_atomic_store(host + k, r.src[a][k - (a ? r.end[a - 1] : 0)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// A fixed amount of dependent-free fp32 multiply-adds per lane, nothing else: what a box's vector ALUs deliver, for
// telling boxes apart when the step's VALU-bound kernels differ between runs.
__global__ __launch_bounds__(256) void probe_fma_kernel(float *out, int iters) {
  float a[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) a[k] = 1.0f + 0.001f * static_cast<float>(threadIdx.x + k);
  const float m = 0.999f, c = 0.0005f;
  for (int i = 0; i < iters; ++i) {
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = fmaf(a[k], m, c);
  }
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < 8; ++k) sum += a[k];
  if (sum == 123.456f) out[0] = sum;  // never true: keeps the loop
}

inline size_t align256(size_t n) { return (n + 255) & ~static_cast<size_t>(255); }

// Carves the workspace; the same walk sizes it (base == nullptr) and lays it out.  Energies alone keep nothing for a backward
// chain: no gradient rows, no E x C of per-edge gradients, one message for both layers (the first layer's is read before the
// second's is written, and so is what its contraction leaves).
struct Layout {
  float *vec, *records, *gv1, *gv2, *bufM1, *bufM2, *bufA, *edge_scratch;
  float *B1, *h1, *sc, *X2, *B2, *h2, *d_h2, *g1, *gB, *gX2, *gh1a, *gh1;
  int32_t *live;         // [2 N] edge ranges cut back to the last edge inside the cutoff
  double *node_virial;   // [N, 6]
  uint32_t *live_bits;   // a bit per edge inside the cutoff, until the virials are written to the same place; NULL where they do not fit it
  size_t bytes;

  Layout(void *base, int64_t N, int64_t E, int C, bool forces) {
    size_t at = 0;
    auto take = [&](size_t n) {
      char *p = base ? static_cast<char *>(base) + at : nullptr;
      at += align256(n);
      return p;
    };
    auto f = [&](int64_t n) { return reinterpret_cast<float *>(take(static_cast<size_t>(n) * sizeof(float))); };
    auto backward = [&](int64_t n) { return forces ? f(n) : nullptr; };
    const int64_t NC = N * C;
    vec = f(3 * E), h2 = f(NC);
    // Energies alone read no vectors but the records', and write h2 when the last record has been read: there the records lie
    // across both, where they fit (with more neighbours than channels they do not, and the forward reads vectors and senders)
    // With forces they lie where the backward pass, which begins after the last forward has read them, puts its per-edge
    // gradients: E C floats, of which C >= 32 are an edge's, and they take four.
    records = forces ? nullptr : (E <= NC ? vec : nullptr);
    gv1 = backward(3 * E), gv2 = backward(3 * E);
    bufM1 = f(16 * NC), bufM2 = forces ? f(16 * NC) : bufM1, bufA = f(16 * NC);
    edge_scratch = backward(E * C);
    if (forces) records = edge_scratch;
    B1 = f(NC), h1 = f(NC), sc = f(NC), X2 = f(NC), B2 = forces ? f(NC) : B1, d_h2 = backward(NC);
    g1 = backward(NC), gB = backward(NC), gX2 = backward(NC), gh1a = backward(NC), gh1 = backward(NC);
    live = reinterpret_cast<int32_t *>(take(static_cast<size_t>(2 * N) * sizeof(int32_t)));
    node_virial = forces ? reinterpret_cast<double *>(take(static_cast<size_t>(6 * N) * sizeof(double))) : nullptr;
    live_bits = forces && E > 0 && (E + kWave - 1) / kWave <= 6 * N ? reinterpret_cast<uint32_t *>(node_virial) : nullptr;
    bytes = at;
  }
};

}  // namespace
}  // namespace cm

extern "C" int cm_probe_fma(float *out, int workgroups, int iters, cm_stream_t stream) {
  CM_REQUIRE(out && workgroups > 0 && iters > 0, "cm_probe_fma: NULL output or empty launch");
  hipLaunchKernelGGL(cm::probe_fma_kernel, dim3(static_cast<unsigned>(workgroups)), dim3(256), 0, cm::as_stream(stream), out, iters);
  return cm::check_launch("cm_probe_fma");
}

// A driver on the host waits for a few thousand numbers after each step.  As one concatenation, one copy and a wait for the
// stream they came 12 us after the step's last kernel had ended at 216 atoms; here a kernel writes them into the host's memory and the
// host polls the words, which it has set to a value that no result has (and that is no error if one has it: after two
// milliseconds the host waits for the stream instead, as it does where the step itself takes longer).  From the call of the step to
// its results in hand 120 -> 113 us, and the host has 30 us less to do in between (the stress' launch, concatenation, copy).
extern "C" int cm_report(int narrays, const double *const *src, const int64_t *counts, double *host, cm_stream_t stream) {
  static const char *what = "cm_report";
  CM_REQUIRE(narrays >= 0 && narrays <= cm::kMaxReports && (narrays == 0 || (src && counts)), "%s: 0 to %d arrays", what, cm::kMaxReports);
  cm::Reports r{};
  int64_t n = 0;
  int used = 0;
  for (int k = 0; k < narrays; ++k) {
    CM_REQUIRE(counts[k] >= 0 && counts[k] < INT32_MAX, "%s: count out of range", what);
    if (counts[k] == 0) continue;
    CM_REQUIRE(src[k] && host, "%s: NULL array", what);
    n += counts[k];
    r.src[used] = reinterpret_cast<const unsigned long long *>(src[k]), r.end[used++] = n;
  }
  if (n == 0) return CM_OK;
  hipStream_t st = cm::as_stream(stream);
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  CM_REQUIRE(hipStreamIsCapturing(st, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone,
             "%s: a stream under capture delivers nothing to the host", what);
  unsigned long long *words = reinterpret_cast<unsigned long long *>(host);
  for (int64_t k = 0; k < n; ++k) __atomic_store_n(words + k, cm::kNotYet, __ATOMIC_RELAXED);
  hipLaunchKernelGGL(cm::report_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(cm::ceil_div(n, 256), 64))), dim3(256), 0, st, r, n, words);
  const int rc = cm::check_launch(what);
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
  int64_t landed = 0;
  while (rc == CM_OK && landed < n && std::chrono::steady_clock::now() < until)
    while (landed < n && __atomic_load_n(words + landed, __ATOMIC_RELAXED) != cm::kNotYet) ++landed;
  if (landed == n) return CM_OK;
  const hipError_t err = hipStreamSynchronize(st);
  if (rc == CM_OK && err != hipSuccess) {
    cm::set_error("%s: %s", what, hipGetErrorString(err));
    return CM_ELAUNCH;
  }
  return rc;
}

// The largest squared distance between the rows of two arrays in host memory; a NaN coordinate gives infinity.
extern "C" double cm_host_max_displacement(const double *positions, const double *reference, int64_t nnodes) {
#pragma clang fp contract(off)
  double worst = 0.0;
  for (int64_t n = 0; n < nnodes; ++n) {
    const double d0 = positions[3 * n] - reference[3 * n], d1 = positions[3 * n + 1] - reference[3 * n + 1], d2 = positions[3 * n + 2] - reference[3 * n + 2];
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    if (!(r2 <= worst)) worst = r2 == r2 ? r2 : __builtin_inf();
  }
  return worst;
}

extern "C" int cm_stress(const double *virials, const double *cell, int64_t ngraphs, double *stress, cm_stream_t stream) {
  CM_REQUIRE(ngraphs >= 0 && ngraphs < INT32_MAX / 16, "cm_stress: number of graphs out of range");
  if (ngraphs == 0) return CM_OK;
  CM_REQUIRE(virials && cell && stress, "cm_stress: NULL pointer");
  hipLaunchKernelGGL(cm::stress_kernel, dim3(static_cast<unsigned>(cm::ceil_div(9 * ngraphs, 256))), dim3(256), 0, cm::as_stream(stream),
                     virials, cell, ngraphs, stress);
  return cm::check_launch("cm_stress");
}

extern "C" size_t cm_mace_step_workspace(int64_t nnodes, int64_t nedges, int channels) {
  if (nnodes < 0 || nedges < 0 || channels <= 0) return 0;
  return cm::Layout(nullptr, nnodes, nedges, channels, true).bytes;
}

extern "C" size_t cm_mace_energy_workspace(int64_t nnodes, int64_t nedges, int channels) {
  if (nnodes < 0 || nedges < 0 || channels <= 0) return 0;
  return cm::Layout(nullptr, nnodes, nedges, channels, false).bytes;
}

// Runs one stage; with the stage's timing bit set, between two events recorded on the stream.
#define CM_STAGE(id, call)                          \
  do {                                              \
    cm::StageTimer timer_(st, (id), timing_mask);   \
    const int rc_ = (call);                         \
    if (rc_ != CM_OK) return rc_;                   \
  } while (0)

extern "C" int cm_mace_step_timing(unsigned stage_mask) {
  std::lock_guard<std::mutex> lock(cm::g_timing_mutex);
  cm::g_timing_mask = stage_mask & ((1u << cm::kStages) - 1u);
  for (cm::Pending &p : cm::g_pending) {
    cm::g_event_pool.push_back(p.start);
    cm::g_event_pool.push_back(p.stop);
  }
  cm::g_pending.clear();
  for (int s = 0; s < cm::kStages; ++s) cm::g_stage_ms[s] = 0.0, cm::g_stage_launches[s] = 0;
  return CM_OK;
}

extern "C" int cm_mace_step_timing_read(double *total_ms, int64_t *launches, int capacity) {
  CM_REQUIRE(total_ms && launches && capacity >= cm::kStages, "cm_mace_step_timing_read: need room for %d stages", cm::kStages);
  std::lock_guard<std::mutex> lock(cm::g_timing_mutex);
  for (cm::Pending &p : cm::g_pending) {
    float ms = 0.f;
    if (hipEventSynchronize(p.stop) == hipSuccess && hipEventElapsedTime(&ms, p.start, p.stop) == hipSuccess) {
      cm::g_stage_ms[p.stage] += ms;
      cm::g_stage_launches[p.stage] += 1;
    }
    cm::g_event_pool.push_back(p.start);
    cm::g_event_pool.push_back(p.stop);
  }
  cm::g_pending.clear();
  for (int s = 0; s < cm::kStages; ++s) total_ms[s] = cm::g_stage_ms[s], launches[s] = cm::g_stage_launches[s];
  return cm::kStages;
}

namespace {

// The end of the step: forces, and virials on request, from the edge gradients of both layers.
int forces_of_step(const cm::Layout &L, const cm_mace_graph *g, const double *positions, const double *shifts, double *forces, double *virials,
                   const double *cell, double *stress, unsigned timing_mask, cm_stream_t stream) {
  const int64_t N = g->nnodes, E = g->nedges;
  hipStream_t st = cm::as_stream(stream);
  if (virials) {
    CM_STAGE(23, cm::forces_and_node_virials(L.gv1, L.vec, g->node_rows, g->first_occ, g->sender_perm, g->sender_offsets, N, E, forces, L.node_virial, st));
    cm::StageTimer timer_(st, 24, timing_mask);
    hipLaunchKernelGGL(cm::graph_virial_kernel, dim3(g->ngraphs), dim3(cm::kSumThreads), 0, st, L.node_virial, g->graph_ptr, virials,
                       cell, stress);
  } else {
    CM_STAGE(23, cm_edge_geometry_backward(positions, g->receiver, g->sender, shifts, g->node_rows, g->first_occ, g->sender_perm,
                                           g->sender_offsets, L.gv1, nullptr, N, E, forces, nullptr, stream));
  }
  return cm::check_launch("cm_mace_step");
}

// The step of cm_mace_step, or, with want_forces false, its forward half alone: no backward chain, and none of what only
// that chain reads (the contractions' gradient tables, the readouts' derivative, cleared edge gradients) is formed, written or
// given room.
int run_step(const cm_mace_weights *w, const cm_mace_graph *g, const double *positions, const double *shifts, void *workspace,
             size_t workspace_bytes, double *interaction_energy, double *node_energy, bool want_forces, double *forces,
             double *node_feats, double *virials, const double *cell, double *stress, double *total_energy, double *total_node_energy,
             cm_stream_t stream) {
  CM_REQUIRE(w && g, "cm_mace_step: NULL weights or graph");
  CM_REQUIRE(!stress || (virials && cell), "cm_mace_step_stress: stress needs virials and the cell");
  const int64_t N = g->nnodes, E = g->nedges;
  const int C = w->channels, ne = w->nelements;
  CM_REQUIRE(N >= 0 && E >= 0 && g->ngraphs >= 1, "cm_mace_step: negative size or no graph");
  CM_REQUIRE(cm_channels_supported(C), "cm_mace_step: channels=%d must be a multiple of 32 in [32, 256]", C);
  CM_REQUIRE(ne >= 1, "cm_mace_step: nelements must be at least 1");
  CM_REQUIRE(interaction_energy && g->graph_ptr, "cm_mace_step: NULL energy output or graph_ptr");
  hipStream_t st = cm::as_stream(stream);
  unsigned timing_mask;
  {
    std::lock_guard<std::mutex> lock(cm::g_timing_mutex);
    timing_mask = cm::g_timing_mask;
  }
  if (timing_mask != 0) {
    // events recorded into a capture cannot be read back: a captured step is not timed
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) timing_mask = 0;
  }
  if (N == 0) {
    hipLaunchKernelGGL(cm::fill_f64_kernel, dim3(1), dim3(64), 0, st, interaction_energy, static_cast<int64_t>(g->ngraphs), 0.0);
    if (virials)
      hipLaunchKernelGGL(cm::fill_f64_kernel, dim3(1), dim3(64), 0, st, virials, static_cast<int64_t>(9) * g->ngraphs, 0.0);
    if (stress)
      if (const int rc = cm_stress(virials, cell, g->ngraphs, stress, stream); rc != CM_OK) return rc;
    if (total_energy)
      hipLaunchKernelGGL(cm::copy_or_zero_f64_kernel, dim3(1), dim3(64), 0, st, total_energy, g->graph_e0, static_cast<int64_t>(g->ngraphs));
    return cm::check_launch("cm_mace_step");
  }
  CM_REQUIRE(positions && node_energy && (forces || !want_forces), "cm_mace_step: NULL positions or output");
  CM_REQUIRE(N < INT32_MAX / 4 && E < INT32_MAX, "cm_mace_step: sizes out of range");
  CM_REQUIRE(E == 0 || shifts, "cm_mace_step: NULL shifts");
  CM_REQUIRE(g->first_occ && g->sender_offsets && g->elem_perm && g->elem_offsets && g->onehot_perm && g->onehot_offsets && g->X1,
             "cm_mace_step: NULL graph structure");
  CM_REQUIRE(E == 0 || (g->receiver && g->sender && g->sender_perm), "cm_mace_step: NULL edge list");
  for (int t = 0; t < 2; ++t)
    CM_REQUIRE(w->spline[t] && w->mix_WT[t] && w->mix_W[t] && w->T3[t] && w->T2[t] && w->T1[t] && w->prod_WT[t] && w->prod_W[t] &&
                   (w->mono3[t] == nullptr) == (w->mono2[t] == nullptr),
               "cm_mace_step: NULL weight of layer %d", t);
  CM_REQUIRE(w->r_knots && w->up_WT && w->up_W && w->skip_WT && w->skip_W && w->w1 && w->W2a && w->w2b, "cm_mace_step: NULL weight");
  const cm::Layout L(workspace, N, E, C, want_forces);
  if (workspace == nullptr || workspace_bytes < L.bytes) {
    cm::set_error("cm_mace_step / cm_mace_energy: workspace of %zu bytes, need %zu", workspace_bytes, L.bytes);
    return CM_ENOSPC;
  }
  CM_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "cm_mace_step: workspace must be 256-byte aligned");
  const int32_t *oh_perm = g->onehot_perm, *oh_off = g->onehot_offsets;
  const int32_t *el_perm = g->elem_perm, *el_off = g->elem_offsets;
  const float *none = nullptr;

  const char *glue_env = getenv("CM_STEP_GLUE");  // development switch: smallest node count that takes the chained kernels; -1: none
  const int glue_min = glue_env ? atoi(glue_env) : 0;
  // Few nodes: a workgroup takes a node through a whole layer (few_nodes.hip), three launches and the forces.
  if (glue_min >= 0 && N >= glue_min && cm::fewnodes::applies(*w, N, E, want_forces)) {
    const cm::fewnodes::Scratch s{L.vec, L.X2, L.h1, L.sc, L.live, reinterpret_cast<int32_t *>(L.bufA), want_forces ? L.bufM1 : nullptr, L.d_h2,
                                  L.edge_scratch, L.gv1, L.gv2};
    CM_REQUIRE(w->hidden >= 1 && w->hidden <= cm::readout::kHidden, "cm_mace_step: hidden=%d must be in [1, %d]", w->hidden, cm::readout::kHidden);
    CM_REQUIRE(E < INT32_MAX / 3, "cm_mace_step: number of edges out of range");
    CM_STAGE(1, cm::fewnodes::first_layer(*w, *g, positions, shifts, s, st));
    CM_STAGE(7, cm::fewnodes::second_layer(*w, *g, cm::readout::Outputs{node_energy, node_feats, g->node_rows, g->node_e0, total_node_energy}, s, st));
    if (!want_forces) {
      cm::StageTimer timer_(st, 12, timing_mask);
      hipLaunchKernelGGL(cm::segment_sum_f64_kernel, dim3(g->ngraphs), dim3(cm::kSumThreads), 0, st, node_energy, g->node_weights,
                         g->graph_ptr, interaction_energy, g->graph_e0, total_energy);
      return cm::check_launch("cm_mace_energy");
    }
    CM_STAGE(21, cm::fewnodes::back_to_edges(*w, *g, cm::EnergySums{node_energy, g->node_weights, g->graph_ptr, interaction_energy, g->ngraphs,
                                                                    g->graph_e0, total_energy}, s, st));
    return forces_of_step(L, g, positions, shifts, forces, virials, cell, stress, timing_mask, stream);
  }

  // ---- forward ----
  // The forward kernel with the table in LDS reads an edge's vector and sender once per pair of degrees and 16 channels: one load
  // of 16 bytes from one place instead of two loads from two arrays (forward pass alone, 25 000 x 128 238 -> 229 us, 12 000 x 256
  // 235 -> 218, 40 000 x 192 600 -> 573, 10 007 x 160 128 -> 124; writing the records 3 us at 25 000 x 52).
  const bool records = E > 0 && L.records && E <= cm::mp::kMaxRecords && cm::mp::sliced_forward_applies(N, E, C, w->nknots);
  if (E > 0) {
    cm::StageTimer timer_(st, 0, timing_mask);
    hipLaunchKernelGGL(cm::geometry_live_range_kernel, dim3(static_cast<unsigned>(cm::ceil_div(std::max(N, E), 256))), dim3(256), 0, st,
                       positions, g->receiver, g->sender, shifts, g->node_rows, g->first_occ, w->r_max, static_cast<int>(N), E,
                       want_forces || !records ? L.vec : nullptr, records ? reinterpret_cast<float4 *>(L.records) : nullptr, L.live, L.gv1,
                       L.gv2, reinterpret_cast<unsigned long long *>(L.live_bits));
  }
  const int32_t *fo_live = E > 0 ? L.live : g->first_occ;
  const float *X[2] = {g->X1, L.X2};
  float *bufM[2] = {L.bufM1, L.bufM2};
  float *B[2] = {L.B1, L.B2};
  float *h[2] = {L.h1, L.h2};
  // the three [N, C] products between the layers (and their three transposes in the backward) as one launch each
  const bool glue = cm_node_glue_supported(C) != 0 && glue_min >= 0 && N >= glue_min;
  // beyond 128 channels and for few nodes the same in two launches; the head stays three, and weights of the nodes need their pass over dE/dh2
  const bool cut = !glue && glue_min >= 0 && cm::node_chains_cut(N, C);
  const bool cut_backward = cut && !g->node_weights;
  for (int t = 0; t < 2; ++t) {
    if (t == 1 && !glue && !cut) {
      // residual skip connection per element and linear_up, both of the first layer's output
      CM_STAGE(5, cm_linear(L.h1, w->skip_WT, oh_perm, oh_off, N, ne + 1, 1, 1, C, C, w->skip_scale, none, none, L.sc, stream));
      CM_STAGE(6, cm_linear(L.h1, w->up_WT, nullptr, nullptr, N, 1, 0, 1, C, C, 1.0f, none, none, L.X2, stream));
    }
    if (records)
      CM_STAGE(t == 0 ? 1 : 7, cm::mp::edge_forward_from_records(X[t], L.records, w->r_knots, w->spline[t], w->nknots, w->r_width, w->r_max, fo_live, N,
                                                                 E, C, bufM[t], st));
    else
      CM_STAGE(t == 0 ? 1 : 7, cm_mp_edge_forward(X[t], L.vec, w->r_knots, w->spline[t], w->nknots, w->r_width, w->r_max, g->sender, fo_live, N,
                               E, C, bufM[t], stream));
    if (t == 0)
      CM_STAGE(2, cm_linear(bufM[t], w->mix_WT[t], oh_perm, oh_off, N, ne + 1, 1, 16, C, C, w->mix_scale[t], none, none, L.bufA, stream));
    else
      CM_STAGE(8, cm_linear(bufM[t], w->mix_WT[t], nullptr, nullptr, N, 1, 0, 16, C, C, w->mix_scale[t], none, none, L.bufA, stream));
    // the contraction's gradient table takes the place of the message, which is no longer needed
    float *table = want_forces ? bufM[t] : nullptr;
    CM_STAGE(t == 0 ? 3 : 9, cm_symcon_forward(L.bufA, el_perm, el_off, w->mono3[t], w->n3[t], w->mono2[t], w->n2[t], w->T3[t], w->T2[t], w->T1[t], N,
                              ne, C, B[t], table, stream));
    if (t == 0 && glue)
      CM_STAGE(4, cm_node_glue_forward(L.B1, w->prod_WT[0], w->skip_WT, w->up_WT, oh_perm, oh_off, N, ne + 1, C, w->skip_scale, L.h1, L.sc,
                                       L.X2, stream));
    else if (t == 0 && cut)
      CM_STAGE(4, cm::node_glue_forward_cut(L.B1, w->prod_WT[0], w->skip_WT, w->up_WT, oh_perm, oh_off, N, ne + 1, C, w->skip_scale, L.h1, L.sc, L.X2,
                                            st));
    else if (t == 0 || !glue)
      CM_STAGE(t == 0 ? 4 : 10, cm_linear(B[t], w->prod_WT[t], nullptr, nullptr, N, 1, 0, 1, C, C, 1.0f, none, t == 1 ? L.sc : none, h[t], stream));
  }
  if (glue)  // with the product linear before the readouts and, for forces, the one behind their derivative
    CM_STAGE(11, cm::node_head(L.B2, L.sc, L.h1, w->prod_WT[1], w->prod_W[1],
                               cm::readout::Weights{w->w1, w->W2a, w->w2b, w->act_cst, w->scale, w->shift, w->hidden},
                               cm::readout::Outputs{node_energy, node_feats, g->node_rows, g->node_e0, total_node_energy}, g->node_weights, N, C,
                               want_forces ? L.d_h2 : nullptr, L.gB, st));
  else
    CM_STAGE(11, cm::readout_forward_with_totals(L.h1, L.h2, w->w1, w->W2a, w->w2b, w->act_cst, w->scale, w->shift, N, C, w->hidden,
                                                 node_energy, want_forces ? L.d_h2 : nullptr, node_feats, g->node_rows, g->node_e0, total_node_energy, st));
  if (!want_forces) {
    cm::StageTimer timer_(st, 12, timing_mask);
    hipLaunchKernelGGL(cm::segment_sum_f64_kernel, dim3(g->ngraphs), dim3(cm::kSumThreads), 0, st, node_energy, g->node_weights,
                       g->graph_ptr, interaction_energy, g->graph_e0, total_energy);
  }

  if (!want_forces) return cm::check_launch("cm_mace_energy");

  // ---- backward: d(-sum of node energies) / d positions ----
  // The seed is -1 on every node energy (-weight[n] with node weights), so the readouts' backward needs no pass of its
  // own: the gradient with respect to the second layer's features is -d_h2 (the sign goes into the scale of the two
  // linears that consume it, which is exact; node weights scale its rows first), the one with respect to the first
  // layer's is a constant row (times the node's weight).
  if (!glue && !cut_backward) {  // the chained kernels form the constant rows themselves, weight the others, and take the energy sums along
    cm::StageTimer timer_(st, 13, timing_mask);
    const unsigned rows = static_cast<unsigned>(std::min<int64_t>(cm::ceil_div(N, cm::kSumThreads / cm::kWave), 1024));
    hipLaunchKernelGGL(cm::energies_and_seeds_kernel, dim3(g->ngraphs + rows), dim3(cm::kSumThreads), 0, st, node_energy, g->node_weights, g->graph_ptr,
                       interaction_energy, g->graph_e0, total_energy, g->ngraphs, L.g1, L.d_h2, w->w1, w->scale, static_cast<int>(N), C);
  }
  // layer 1 (second interaction)
  if (!glue)
    CM_STAGE(14, cm_linear(L.d_h2, w->prod_W[1], nullptr, nullptr, N, 1, 0, 1, C, C, -1.0f, none, none, L.gB, stream));
  CM_STAGE(15, cm_linear(L.bufM2, w->mix_W[1], nullptr, nullptr, N, 1, 0, 16, C, C, w->mix_scale[1], L.gB, none, L.bufA, stream));
  CM_REQUIRE(E < INT32_MAX / 3, "cm_mace_step: number of edges out of range");
  CM_STAGE(16, cm::mp::edge_backward_with_live_bits(L.X2, L.vec, w->r_knots, w->spline[1], w->nknots, w->r_width, w->r_max, L.bufA, g->sender, fo_live,
                                                    g->sender_perm, g->sender_offsets, N, E, C, L.gX2, L.gv2, L.edge_scratch, L.live_bits, st));
  // layer 0 (first interaction): its input features depend on the species alone, so no gradient with respect to them
  if (glue || cut_backward) {
    CM_STAGE(17, cm::node_glue_backward_with_energy_sums(L.gX2, L.d_h2, w->up_W, w->skip_W, w->prod_W[0], w->w1, w->scale, g->node_weights,
                                                         oh_perm, oh_off, N, ne + 1, C, w->skip_scale, L.gh1, L.gB, node_energy, g->graph_ptr,
                                                         g->ngraphs, interaction_energy, g->graph_e0, total_energy, st));
  } else {
    CM_STAGE(17, cm_linear(L.gX2, w->up_W, nullptr, nullptr, N, 1, 0, 1, C, C, 1.0f, none, L.g1, L.gh1a, stream));
    CM_STAGE(18, cm_linear(L.d_h2, w->skip_W, oh_perm, oh_off, N, ne + 1, 1, 1, C, C, -w->skip_scale, none, L.gh1a, L.gh1, stream));
    CM_STAGE(19, cm_linear(L.gh1, w->prod_W[0], nullptr, nullptr, N, 1, 0, 1, C, C, 1.0f, none, none, L.gB, stream));
  }
  CM_STAGE(20, cm_linear(L.bufM1, w->mix_W[0], oh_perm, oh_off, N, ne + 1, 1, 16, C, C, w->mix_scale[0], L.gB, none, L.bufA, stream));
  // its vector gradient is written onto the second layer's: gv1 = (this layer's) + gv2
  CM_STAGE(21, cm::mp::edge_backward_onto(g->X1, L.vec, w->r_knots, w->spline[0], w->nknots, w->r_width, w->r_max, L.bufA, g->sender,
                                         fo_live, N, E, C, L.gv1, L.gv2, st));
  return forces_of_step(L, g, positions, shifts, forces, virials, cell, stress, timing_mask, stream);
}

}  // namespace

extern "C" int cm_mace_step(const cm_mace_weights *weights, const cm_mace_graph *graph, const double *positions, const double *shifts,
                            void *workspace, size_t workspace_bytes, double *interaction_energy, double *node_energy,
                            double *forces, double *node_feats, double *virials, double *total_energy, double *total_node_energy,
                            cm_stream_t stream) {
  return run_step(weights, graph, positions, shifts, workspace, workspace_bytes, interaction_energy, node_energy, true, forces,
                  node_feats, virials, nullptr, nullptr, total_energy, total_node_energy, stream);
}

extern "C" int cm_mace_step_stress(const cm_mace_weights *weights, const cm_mace_graph *graph, const double *positions,
                                   const double *shifts, const double *cell, void *workspace, size_t workspace_bytes,
                                   double *interaction_energy, double *node_energy, double *forces, double *node_feats,
                                   double *virials, double *stress, double *total_energy, double *total_node_energy,
                                   cm_stream_t stream) {
  return run_step(weights, graph, positions, shifts, workspace, workspace_bytes, interaction_energy, node_energy, true, forces,
                  node_feats, virials, cell, stress, total_energy, total_node_energy, stream);
}

extern "C" int cm_mace_energy(const cm_mace_weights *weights, const cm_mace_graph *graph, const double *positions,
                              const double *shifts, void *workspace, size_t workspace_bytes, double *interaction_energy,
                              double *node_energy, double *node_feats, double *total_energy, double *total_node_energy,
                              cm_stream_t stream) {
  return run_step(weights, graph, positions, shifts, workspace, workspace_bytes, interaction_energy, node_energy, false, nullptr,
                  node_feats, nullptr, nullptr, nullptr, total_energy, total_node_energy, stream);
}
