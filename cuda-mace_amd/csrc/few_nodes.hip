// The step of few nodes: a workgroup takes one node through everything between two exchanges with its neighbours, so that a step is
// three launches and the forces instead of fifteen.
//
// A step of some ten to some hundred atoms spends its time on the chain of its launches: each is over in 3 to 6 us, next to nothing of
// which is arithmetic or traffic, and waits for what the one before has written (21 atoms x 64 channels: 16 launches, 71 us).  All that
// crosses from one node to another is the gather of the sender rows in the two message passes and of the per-edge gradients on the way
// back; between those a node's rows [16, C] fit a workgroup's LDS, the weights (4 C^2 per mixing, C^2 per product) come from L2 in as many
// bytes as the node's table rows do, and every product of one row is K multiply-adds per column, which the vector ALU does in less time
// than 16 rows of a matrix instruction, fifteen of them empty, would take.
//
//   first_layer    vectors, live edge range, M1, A, B1 and grad1, h1, sc, X2                    (stages of step.hip in its notation)
//   second_layer   M2, A, B2, h2, the readouts, gB2, gA, gv2 and the per-edge rows of gX2
//   back_to_edges  gX2 (sender pass), gh1, gB1, gA, gv1; extra workgroups: the graph energies
//
// Every sum is formed in the order of the launch it stands for: v_mfma_f32_16x16x4_f32 and v_mfma_f64_16x16x4_f64 add their four products one
// after the other, fused, k ascending (checked bit for bit against fma chains), so the chains of mfma_f32.hpp and readout_device.hpp are
// chains of fmaf and fma here, and the step returns the bits of the separate launches.
#include "common.hpp"
#include "few_nodes.hpp"
#include "mfma_f32.hpp"
#include "mp_spline_device.hpp"
#include "node_glue.hpp"
#include "symcon_device.hpp"

namespace cm {
namespace fewnodes {
namespace {

using namespace mp;

// Threads of a workgroup: 512 while every node has a compute unit to itself, 256 and two nodes to a unit beyond.
constexpr int kAlone = 512, kShared = 256;
template <int T>
constexpr int kMostParts = T == kAlone ? 6 : 4;  // of the forward (forward_parts; with more than a node per unit it gives no more than four)

// Workgroup barrier that orders LDS alone: loads of weights that a thread has requested stay in flight across it.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// the wave's number in a scalar register: a branch on it is the wave's, and what one side holds takes no registers of the other
__device__ __forceinline__ int wave_number() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

// ---- products of one row ------------------------------------------------------------------------------------------------
// The chain of channel k in mfma_f32.hpp's product is (k / 16 + k % 4) % 4, its place there 4 (k / 16) + k % 16 / 4.  A row that is about to be
// multiplied lies in LDS chain by chain, so that a thread reads its chain's values 16 bytes at a time.
template <int C>
__device__ __forceinline__ int place(int k) {
  return ((k / 16 + k % 4) & 3) * (C / 4) + 4 * (k / 16) + k % 16 / 4;
}
// channel at place j of chain ch
__device__ __forceinline__ int channel_at(int ch, int j) { return 16 * (j / 4) + 4 * (j % 4) + ((ch - j / 4) & 3); }

// A thread's share of NMAT products of a row and a [C, C] matrix W[k][column]: one chain of four neighbouring columns, 16 bytes per load (a
// load costs the path from L1 about as much with 4 bytes per lane).
template <int C, int NMAT>
struct Products {
  f4 w[C / 4];
  // whole waves: a lane beyond the last unit repeats that one
  __device__ __forceinline__ static bool here() { return wave_number() * kWave < C * NMAT; }
  __device__ __forceinline__ static int thread() { return min(static_cast<int>(threadIdx.x), C * NMAT - 1); }
  __device__ __forceinline__ void request(const float *W0, const float *W1 = nullptr) {
    if (!here()) return;
    const int unit = thread() % C, ch = unit / (C / 4);
    const float *W = (thread() < C ? W0 : W1) + 4 * (unit % (C / 4));
#pragma unroll
    for (int j = 0; j < C / 4; ++j) w[j] = ld4(W + channel_at(ch, j) * C);
  }
  // x0, x1: the rows, by place; partial sums to part[matrix][chain][column]
  __device__ __forceinline__ void run(const float *x0, const float *x1, float *part) const {
    if (!here()) return;
    const int unit = thread() % C, ch = unit / (C / 4);
    const float *x = (thread() < C ? x0 : x1) + ch * (C / 4);
    f4 sum = zero4();
#pragma unroll
    for (int j = 0; j < C / 4; j += 4) {
      const f4 v = ld4(x + j);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) sum[q] = fmaf(w[j + i][q], v[i], sum[q]);
    }
    st4(part + 4 * thread(), sum);
  }
};
// the four chains of a column
template <int C>
__device__ __forceinline__ float column(const float *part, int c) {
  return (part[c] + part[C + c]) + (part[2 * C + c] + part[3 * C + c]);
}

// The channel mixing of a node's 16 rows, a [C, C] block per degree: a thread has one chain of four neighbouring columns for the rows of
// its set, all of one degree.  Sets are as many as the threads allow, in an order that gives the four SIMDs equal work (wave w is SIMD w % 4's).
template <int C, int T>
struct Mixing {
  static constexpr int kSpan = C <= 64 ? C : 128;  // threads of a set: whole waves from 64 columns on, the last one partly idle at 96
  static constexpr int kSets = T / kSpan;
  static_assert(kSets == 2 || kSets == 4 || kSets == 8 || kSets == 16, "sets");
  f4 w[C / 4];
  __device__ __forceinline__ static int set() {
    const int s = threadIdx.x / kSpan;
    return kSpan >= kWave ? __builtin_amdgcn_readfirstlane(s) : s;
  }
  __device__ __forceinline__ static int unit() { return threadIdx.x % kSpan; }
  // degree of a set (4: none)
  __device__ __forceinline__ static int degree_of(int set) {
    if constexpr (kSets == 16) return l_of_m(set & 15);
    if constexpr (kSets == 8) return (0x14102233 >> (4 * set)) & 7;  // as in run
    return set == 0 ? 3 : (set == 1 ? 2 : (set == 2 ? 0 : 1));  // (of two sets the first degree)
  }
  __device__ __forceinline__ static bool here() { return degree_of(set()) < 4 && unit() < C; }
  __device__ __forceinline__ void request(const float *W) { request_degree(W, degree_of(set())); }
  __device__ __forceinline__ void request_degree(const float *W, int l) {
    if (!here()) return;
    const int ch = unit() / (C / 4);
    const float *at = W + static_cast<int64_t>(l) * (C * C) + 4 * (unit() % (C / 4));
#pragma unroll
    for (int j = 0; j < C / 4; ++j) w[j] = ld4(at + channel_at(ch, j) * C);
  }
  template <int M0, int N>
  __device__ __forceinline__ void rows(const float *x, float *part) const {
    if (unit() >= C) return;
    const int ch = unit() / (C / 4);
    const float *xc = x + M0 * C + ch * (C / 4);
    f4 sum[N];
#pragma unroll
    for (int m = 0; m < N; ++m) sum[m] = zero4();
#pragma unroll
    for (int j = 0; j < C / 4; j += 4)
#pragma unroll
      for (int m = 0; m < N; ++m) {
        const f4 v = ld4(xc + m * C + j);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) sum[m][q] = fmaf(w[j + i][q], v[i], sum[m][q]);
      }
    float *to = part + ch * (16 * C) + M0 * C + 4 * (unit() % (C / 4));
#pragma unroll
    for (int m = 0; m < N; ++m) st4(to + m * C, sum[m]);
  }
  // x: [16][C] by place; partial sums to part[chain][16][C].  W: the weights once more, for sets of two degrees.
  __device__ __forceinline__ void run(const float *x, float *part, const float *W) {
    const int s = set();
    if constexpr (kSets == 16) {
      rows<0, 1>(x + s * C, part + s * C);
    } else if constexpr (kSets == 8) {
      switch (s) {
        case 0: rows<9, 4>(x, part); break;
        case 1: rows<13, 3>(x, part); break;
        case 2: rows<4, 3>(x, part); break;
        case 3: rows<7, 2>(x, part); break;
        case 4: rows<0, 1>(x, part); break;
        case 5: rows<1, 1>(x, part); break;
        case 7: rows<2, 2>(x, part); break;
      }
    } else if constexpr (kSets == 2) {
      if (s == 0) rows<9, 7>(x, part);
      else rows<4, 5>(x, part);
      request_degree(W, s);
      if (s == 0) rows<0, 1>(x, part);
      else rows<1, 3>(x, part);
    } else {
      switch (s) {
        case 0: rows<9, 7>(x, part); break;
        case 1: rows<4, 5>(x, part); break;
        case 2: rows<0, 1>(x, part); break;
        case 3: rows<1, 3>(x, part); break;
      }
    }
  }
};
template <int C>
__device__ __forceinline__ float mixed(const float *part, int at, float scale) {  // at: m C + column
#pragma clang fp contract(off)
  const float v = (part[at] + part[16 * C + at]) + (part[32 * C + at] + part[48 * C + at]);
  return v * scale;
}

// ---- LDS of a workgroup -----------------------------------------------------------------------------------------------
template <int C, int T, bool FORWARD, bool BACKWARD>
struct Shared {
  static constexpr int kWaves = T / kWave, kStaged = kMostParts<T> * kStageBytes;
  static constexpr int kForward = FORWARD ? kStaged + kMostParts<T> * 16 * C * 4 : 0;
  static constexpr int kMixing = 64 * C * 4, kEdgeSums = BACKWARD ? kWaves * 16 * kChunk * 4 : 0;
  static constexpr int kEdges = kMixing > kEdgeSums ? kMixing : kEdgeSums;  // where the edges staged for the backward pass lie
  static constexpr int kBackward = kEdges + (BACKWARD ? kWaves * kStageBytes : 0);
  // edges staged for the forward and the parts' sums; then partial sums of products or the edges' sums, and behind them, some time before they are
  // needed, the edges staged for the backward pass
  __attribute__((aligned(16))) unsigned char work[kForward > kBackward ? kForward : kBackward];
  __attribute__((aligned(16))) float rows[16 * C];  // operand rows, by place
  __attribute__((aligned(16))) float grad[16 * C];  // gradient rows, by channel
  __attribute__((aligned(16))) float row[3][C];     // operand rows of the products, by place
  float h2[C];
  double z[4][16], e1[4][4], e2[16], d[16];
  float knots[kKnotsInLds];
  int mark, group, element;
  __device__ float *part() { return reinterpret_cast<float *>(work); }
  __device__ float *sums(int p) { return reinterpret_cast<float *>(work + kStaged) + p * (16 * C); }
  __device__ Staged edges() { return Staged(work + kEdges + wave_number() * kStageBytes); }
};

// the waves that contract: the last ones, which come last for parts of the forward too
template <int C, int T>
struct Contraction {
  static constexpr int kFirst = T / kWave - (C + kWave - 1) / kWave;
  static_assert(C <= kFirst * kWave, "the next product's threads are others");
  float t3[CM_SYMCON_N3], t2[CM_SYMCON_N2], t1;
  __device__ __forceinline__ static int channel() { return static_cast<int>(threadIdx.x) - kFirst * kWave; }
  __device__ __forceinline__ static bool here() { return channel() >= 0 && channel() < C; }
  // by whole waves (a lane beyond the last channel reads the last one's)
  __device__ __forceinline__ void request(const float *T3, const float *T2, const float *T1, int element) {
    const int c = min(channel(), C - 1);
#pragma unroll
    for (int t = 0; t < CM_SYMCON_N3; ++t) t3[t] = T3[(static_cast<int64_t>(element) * CM_SYMCON_N3 + t) * C + c];
#pragma unroll
    for (int t = 0; t < CM_SYMCON_N2; ++t) t2[t] = T2[(static_cast<int64_t>(element) * CM_SYMCON_N2 + t) * C + c];
    t1 = T1[static_cast<int64_t>(element) * C + c];
  }
  template <bool GRAD>
  __device__ __forceinline__ float run(const float *part, float scale, float (&g)[16]) const {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = mixed<C>(part, i * C + channel(), scale);
    return symcon::contract<float, GRAD>(x, t3, t2, t1, g);
  }
};

// Message of the node over its edges e0 .. e1 - 1 into s.rows, the parts by waves as in mp_spline_forward_kernel.  `others` is called by the
// waves that contract later, `meanwhile` by every thread between its part and the barrier behind which the parts are added.
template <int C, int T, class S, class Fn0, class Fn>
__device__ __forceinline__ void message(S &s, const float *__restrict__ X, const Spline &sp, const int32_t *__restrict__ sender, int nnodes, int64_t nedges,
                                        int e0, int e1, int parts, Fn0 others, Fn meanwhile) {
  using K = Cfg<C, true>;
  const int wave = wave_number(), lane = threadIdx.x % kWave;
  if (wave < parts) {
    const int64_t len = e1 - e0;
    const int lo = e0 + static_cast<int>(len * wave / parts), hi = e0 + static_cast<int>(len * (wave + 1) / parts);
    typename K::vec acc[16];
    forward_wave<C>(X, sp, sender, nnodes, nedges, lo, hi, Staged(s.work + wave * kStageBytes), acc,
                                      KnotCopy<>::applies(sp) ? s.knots : nullptr);
    using Sums = SlotSums<K>;
    Sums::total(acc);
    if (Sums::holds(lane)) {
      float *to = s.sums(wave) + Sums::first_row(lane) * C + K::off(lane % K::SW);
#pragma unroll
      for (int m = 0; m < Sums::kRows; ++m) K::st(to + m * C, acc[m]);
    }
  }
  if (wave >= Contraction<C, T>::kFirst) others();
  meanwhile();
  lds_barrier();
  for (int i = threadIdx.x; i < 16 * C; i += T) {
    float v = s.sums(0)[i];
    for (int p = 1; p < parts; ++p) v += s.sums(p)[i];
    s.rows[i / C * C + place<C>(i % C)] = v;
  }
  lds_barrier();
}

struct Graph {
  int nnodes, ngroups, nelements;
  int64_t nedges;
  const int32_t *receiver, *sender, *first_occ, *sender_perm, *sender_offsets, *elem_perm, *elem_offsets, *onehot_perm, *onehot_offsets, *rows;
};

// Gradients of the edges e0 .. e1 - 1 of a node from its gradient rows s.grad, as mp_spline_backward_edge_kernel forms them: every edge on its
// own, so the split over the waves is free; a wave takes as many edges as it has slots before another is given some.  The wave's first
// chunk is staged (stage) some time before the gradient rows are there, behind other waits.
template <int C, int T, bool WANT_GX, class S>
struct EdgeGradients {
  using K = Cfg<C>;
  using vec = typename K::vec;
  S &s;
  const Spline &sp;
  const int32_t *sender;
  int nnodes;
  int64_t nedges;
  float *gvec;
  const float *addend;
  int cursor, hi, nlive, base;

  __device__ __forceinline__ Staged staged() const { return s.edges(); }
  __device__ __forceinline__ EdgeGradients(S &s_, const Spline &sp_, const Graph &q, float *gvec_, const float *addend_, int e0, int e1)
      : s(s_), sp(sp_), sender(q.sender), nnodes(q.nnodes), nedges(q.nedges), gvec(gvec_), addend(addend_) {
    const int64_t len = e1 - e0, wave = wave_number();
    const int parts = static_cast<int>(min(static_cast<int64_t>(T / kWave), (len + K::EPW - 1) / K::EPW));
    cursor = wave < parts ? e0 + static_cast<int>(len * wave / parts) : e1;
    hi = wave < parts ? e0 + static_cast<int>(len * (wave + 1) / parts) : e1;
    nlive = 0, base = cursor;
  }
  // the raw edges of the first chunk, and their staging; the knots are in LDS
  __device__ __forceinline__ RawEdge request() const {
    RawEdge r{-1, 0.f, 0.f, 0.f};
    if (cursor >= hi) return r;
    const int64_t e = min(cursor + static_cast<int>(threadIdx.x % kWave), hi - 1);
    r.s = sender[e];
    r.v0 = sp.vec[3 * e + 0], r.v1 = sp.vec[3 * e + 1], r.v2 = sp.vec[3 * e + 2];
    return r;
  }
  template <bool AHEAD>
  __device__ __forceinline__ void stage(RawEdge ahead) {
    if (cursor >= hi) return;
    const int lane = threadIdx.x % kWave;
    base = cursor;
    auto dead = [&](int pass_base, int, unsigned long long, bool lane_is_dead) {
      if (lane_is_dead) {
        const int64_t e = pass_base + lane;
#pragma unroll
        for (int k = 0; k < 3; ++k) gvec[3 * e + k] = addend ? addend[3 * e + k] : 0.f;
      }
    };
    const Staged st = staged();
    wave_lds_fence();
    nlive = stage_edges<true, AHEAD>(nullptr, sender, sp, nnodes, nedges, cursor, hi, lane, st.sY, st.sS, st.sIdx, st.sXr, st.sOrig, dead, ahead, s.knots,
                                     KnotCopy<>::applies(sp));
    wave_lds_fence();
  }
  // the operands of the slots' first edges
  __device__ __forceinline__ void fetch(Operands<K> &o, const float *__restrict__ X, int j) const {
    const int cl = threadIdx.x % K::SW;
    const Staged st = staged();
    fetch_operands<C>(o, X, sp.coeffs, st.sS[j], st.sIdx[j], st.sXr[j], cl < K::LPE ? cl : 0);
  }
  __device__ __forceinline__ void run(const float *__restrict__ X, float *__restrict__ gXe) {
    const int lane = threadIdx.x % kWave, slot = lane / K::SW, cl = lane % K::SW;
    const bool active = cl < K::LPE;
    if (base >= hi) return;
    const Staged st = staged();
    float *const sGY = s.part() + wave_number() * (16 * kChunk);
    vec g[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) g[m] = active ? K::ld(s.grad + m * C + K::off(cl)) : zerov<vec>();
    for (;;) {
      Operands<K> o;
      if (slot < nlive) fetch(o, X, slot);
#pragma unroll 1
      for (int j = slot; j < nlive; j += K::EPW) {
        float y[16], p[16];
        staged_harmonics(st.sY, j, y);
        vec gxe = zerov<vec>(), grq = zerov<vec>();
        edge_products<K, true, true, true, WANT_GX>(o, y, g, p, gxe, grq);
        p[0] = dotv(o.x, grq);
        if constexpr (WANT_GX) {
          if (active) K::st(gXe + static_cast<int64_t>(base + st.sOrig[j]) * C + K::off(cl), gxe);
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(o, X, j + K::EPW < nlive ? j + K::EPW : j);
        slot_reduce16<K::SW>(p, cl);
        store_reduced16<K::SW>(p, cl, j, sGY);
      }
      wave_lds_fence();
      if (lane < nlive) {
        float sums[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) sums[m] = sGY[m * kChunk + lane];
        finish_vector_gradient(sp.vec, base + st.sOrig[lane], sums, addend, gvec);
      }
      if (cursor >= hi) break;
      stage<false>(RawEdge{-1, 0.f, 0.f, 0.f});
    }
  }
};

// copy of the knots; a barrier follows before they are read
template <int T>
__device__ __forceinline__ void copy_knots(const Spline &sp, float *to) {
  if (KnotCopy<>::applies(sp))
    for (int i = threadIdx.x; i < sp.nknots; i += T) to[i] = sp.knots[i];
}

// The group of a node in a grouped order of the nodes (-1: the order does not name it), by the calling wave.
__device__ __forceinline__ int group_of(const int32_t *__restrict__ perm, const int32_t *__restrict__ offsets, int nnodes, int ngroups, int node) {
  const int lane = threadIdx.x % kWave;
  int pos = -1;
  for (int base = 0; base < nnodes && pos < 0; base += 4 * kWave) {
    int at[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) at[k] = perm[min(base + k * kWave + lane, nnodes - 1)];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const unsigned long long found = __ballot(base + k * kWave + lane < nnodes && at[k] == node);
      if (found != 0 && pos < 0) pos = base + k * kWave + __ffsll(static_cast<long long>(found)) - 1;
    }
  }
  if (pos < 0) return -1;
  for (int base = 0; base < ngroups; base += kWave) {
    const int i = min(base + lane, ngroups - 1);
    const unsigned long long found = __ballot(base + lane < ngroups && offsets[i] <= pos && pos < offsets[i + 1]);
    if (found != 0) return base + __ffsll(static_cast<long long>(found)) - 1;
  }
  return -1;
}

// ---- first layer ----------------------------------------------------------------------------------------------------------
struct FirstLayer {
  const double *positions, *shifts;
  const float *X1, *mix, *T3, *T2, *T1, *prod, *up, *skip;  // matrices as [k][column]
  float mix_scale, skip_scale;
  int parts;
  float *vec;
  Scratch s;
};

template <int C, int T, bool FORCES>
__global__ __launch_bounds__(T, 2) void first_layer_kernel(Graph q, Spline sp, FirstLayer a) {
  using S = Shared<C, T, true, false>;
  __shared__ S s;
  const int tid = threadIdx.x;
  const int node = blockIdx.x, wave = wave_number();
  // edge vectors, and the end of the range of edges inside the cutoff; the last two waves look the node's groups up meanwhile
  int e0 = q.first_occ[node], e1 = q.first_occ[q.nnodes + node];
  clamp_edge_range(e0, e1, q.nedges);
  copy_knots<T>(sp, s.knots);
  if (tid == 0) s.mark = e0;
  lds_barrier();
  if (wave == S::kWaves - 1) {
    const int element = group_of(q.elem_perm, q.elem_offsets, q.nnodes, q.nelements, node);
    if (tid % kWave == 0) s.element = element;
  } else if (wave == S::kWaves - 2) {
    const int g = group_of(q.onehot_perm, q.onehot_offsets, q.nnodes, q.ngroups, node);
    if (tid % kWave == 0) s.group = g < 0 ? q.ngroups - 1 : g;
  }
  for (int e = e0 + tid; e < e1; e += T) {
    double v[3];
    edge_vector_f64(a.positions, q.receiver, q.sender, a.shifts, q.rows, e, q.nnodes, v);
    const float v0 = static_cast<float>(v[0]), v1 = static_cast<float>(v[1]), v2 = static_cast<float>(v[2]);
    a.vec[3 * static_cast<int64_t>(e) + 0] = v0;
    a.vec[3 * static_cast<int64_t>(e) + 1] = v1;
    a.vec[3 * static_cast<int64_t>(e) + 2] = v2;
    if (edge_length(v0, v1, v2) <= sp.r_max) {
      atomicMax(&s.mark, e + 1);
    } else if (FORCES) {
#pragma unroll
      for (int k = 0; k < 3; ++k) a.s.gv1[3 * static_cast<int64_t>(e) + k] = a.s.gv2[3 * static_cast<int64_t>(e) + k] = 0.f;
    }
  }
  __syncthreads();  // the vectors are in memory
  e1 = s.mark;
  const int g = s.group, element = s.element;
  const bool no_element = g == q.ngroups - 1;
  if (tid == T - 1) {
    a.s.live[node] = e0;
    a.s.live[q.nnodes + node] = e1;
    a.s.groups[node] = g;
    a.s.groups[q.nnodes + node] = element;
  }

  const float *mix = a.mix + static_cast<int64_t>(no_element ? 0 : g) * (4 * C * C);
  Contraction<C, T> contraction;
  Mixing<C, T> mixing;
  message<C, T>(
      s, a.X1, sp, q.sender, q.nnodes, q.nedges, e0, e1, a.parts, [&]() { contraction.request(a.T3, a.T2, a.T1, max(element, 0)); },
      [&]() {
        if (!no_element) mixing.request(mix);
      });
  if (no_element) {
    for (int i = tid; i < 64 * C; i += T) s.part()[i] = 0.f;
  } else {
    mixing.run(s.rows, s.part(), mix);
  }
  Products<C, 1> prod;
  lds_barrier();
  if (wave < Contraction<C, T>::kFirst) {
    prod.request(a.prod);
  } else if (Contraction<C, T>::here()) {
    const int c = Contraction<C, T>::channel();
    float grad[16];
    float b = contraction.template run<FORCES>(s.part(), a.mix_scale, grad);
    s.row[0][place<C>(c)] = b;
    if constexpr (FORCES) {
#pragma unroll
      for (int i = 0; i < 16; ++i) a.s.grad1[(static_cast<int64_t>(node) * 16 + i) * C + c] = grad[i];
    }
  }
  lds_barrier();
  prod.run(s.row[0], nullptr, s.part());
  Products<C, 2> both;
  both.request(a.up, a.skip + static_cast<int64_t>(no_element ? 0 : g) * C * C);
  lds_barrier();
  const int64_t at = static_cast<int64_t>(node) * C;
  if (tid < C) {
    const float h1 = column<C>(s.part(), tid);
    a.s.h1[at + tid] = h1;
    s.row[1][place<C>(tid)] = h1;
  }
  lds_barrier();
  both.run(s.row[1], s.row[1], s.part());
  lds_barrier();
  if (tid < C) {
    a.s.X2[at + tid] = column<C>(s.part(), tid);
  } else if (tid < 2 * C) {
#pragma clang fp contract(off)
    const float v = column<C>(s.part() + 4 * C, tid - C) * a.skip_scale;
    a.s.sc[at + tid - C] = no_element ? 0.f : v;
  }
}

// ---- second layer, forward and back to its edges ----------------------------------------------------------------------------
struct SecondLayer {
  const float *mix, *mix_T, *T3, *T2, *T1, *prod, *prod_T;
  float mix_scale;
  int parts;
  readout::Weights w;
  readout::Outputs out;
  const double *node_weights;
  Scratch s;
};

template <int C, int T, bool FORCES>
__global__ __launch_bounds__(T, 2) void second_layer_kernel(Graph q, Spline sp, SecondLayer a) {
  using S = Shared<C, T, true, FORCES>;
  constexpr int kHidden = readout::kHidden, kClasses = readout::kClasses, kPieces = C / 16, kPer = (kPieces + kClasses - 1) / kClasses;
  __shared__ S s;
  const int tid = threadIdx.x, lane = tid % kWave, wave = wave_number();
  const int node = blockIdx.x;
  const int e0 = a.s.live[node], e1 = a.s.live[q.nnodes + node];
  const int element = a.s.groups[q.nnodes + node];
  const int64_t at = static_cast<int64_t>(node) * C;
  copy_knots<T>(sp, s.knots);
  EdgeGradients<C, T, true, S> gradients(s, sp, q, a.s.gv2, nullptr, e0, e1);
  lds_barrier();

  Contraction<C, T> contraction;
  Mixing<C, T> mixing;
  message<C, T>(
      s, a.s.X2, sp, q.sender, q.nnodes, q.nedges, e0, e1, a.parts,
      [&]() { contraction.request(a.T3, a.T2, a.T1, max(element, 0)); },
      [&]() { mixing.request(a.mix); });
  mixing.run(s.rows, s.part(), a.mix);
  Products<C, 1> prod;
  // the readouts' weights: the first wave has the hidden units (unit by lane % 16, class by lane / 16), the second the linear readout
  double wz[kPer][16];
  f4 h1v[kPer];
  readout::d2v wl[kPer][2];
  const int unit = lane % 16, cls = lane / 16, lin_cls = lane % 4, lin_part = lane / 16;
  const float residual = tid < C ? a.s.sc[at + tid] : 0.f;
  const int to = a.out.rows ? a.out.rows[node] : node;
  const bool to_ok = static_cast<unsigned>(to) < static_cast<unsigned>(q.nnodes);
  lds_barrier();
  if (wave < Contraction<C, T>::kFirst) {
    prod.request(a.prod);
    if (wave == 0) {
#pragma unroll
      for (int u = 0; u < kPer; ++u)
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const int c = 16 * (cls + kClasses * u) + k;
          wz[u][k] = c < C && unit < a.w.hidden ? a.w.W2a[c * a.w.hidden + unit] : 0.0;
        }
    } else if (wave == 1) {
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int c = 16 * (lin_cls + kClasses * u) + 4 * lin_part;
        const bool in = c < C;
        h1v[u] = in ? ld4(a.s.h1 + at + c) : zero4();
        wl[u][0] = in ? readout::d2v{a.w.w1[c], a.w.w1[c + 1]} : readout::d2v{0.0, 0.0};
        wl[u][1] = in ? readout::d2v{a.w.w1[c + 2], a.w.w1[c + 3]} : readout::d2v{0.0, 0.0};
      }
    }
    if (FORCES) gradients.template stage<false>(RawEdge{-1, 0.f, 0.f, 0.f});
  } else if (Contraction<C, T>::here()) {
    const int c = Contraction<C, T>::channel();
    float grad[16];
    s.row[0][place<C>(c)] = contraction.template run<FORCES>(s.part(), a.mix_scale, grad);
    if constexpr (FORCES) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s.grad[i * C + c] = grad[i];
    }
  }
  lds_barrier();
  prod.run(s.row[0], nullptr, s.part());
  lds_barrier();
  if (FORCES && wave >= Contraction<C, T>::kFirst) gradients.template stage<false>(RawEdge{-1, 0.f, 0.f, 0.f});
  if (tid < C) {
    const float h2 = column<C>(s.part(), tid) + residual;
    s.h2[tid] = h2;
    if (a.out.feats64 && to_ok) {
      double *f = a.out.feats64 + static_cast<int64_t>(to) * (2 * C) + tid;
      f[0] = a.s.h1[at + tid];
      f[C] = h2;
    }
  }
  Products<C, 1> back;
  if (FORCES) back.request(a.prod_T);
  lds_barrier();
  // hidden units and linear readout in the classes and orders of readout_device.hpp
  if (wave == 0) {
    double z = 0.0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int c0 = 16 * (cls + kClasses * u);
      if (c0 >= C) break;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p) z = fma(wz[u][4 * p + i], static_cast<double>(s.h2[c0 + 4 * p + i]), z);
    }
    s.z[cls][unit] = z;
  } else if (wave == 1 && unit < 4) {
    double e1sum = 0.0;
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      if (lin_cls + kClasses * u < kPieces) readout::add_linear(e1sum, wl[u][0], wl[u][1], h1v[u]);
    s.e1[lin_cls][lin_part] = e1sum;
  }
  double wd[kHidden];
  if (FORCES && tid < C) {
#pragma unroll
    for (int k = 0; k < kHidden; ++k) wd[k] = k < a.w.hidden ? a.w.W2a[tid * a.w.hidden + k] : 0.0;
  }
  lds_barrier();
  if (wave == 0) {
    const double gate = unit < a.w.hidden ? a.w.w2b[unit] * a.w.act_cst : 0.0;
    double e2, d;
    readout::activate(gate, (s.z[0][unit] + s.z[1][unit]) + (s.z[2][unit] + s.z[3][unit]), e2, d);
    if (lane < 16) s.e2[unit] = e2, s.d[unit] = d;
    wave_lds_fence();
    const int p = lane / 16;
    const double e = ((s.e1[0][p] + s.e1[1][p]) + (s.e1[2][p] + s.e1[3][p])) + ((s.e2[4 * p] + s.e2[4 * p + 1]) + (s.e2[4 * p + 2] + s.e2[4 * p + 3]));
    const double en = readout::node_energy(e, a.w.scale, a.w.shift);
    if (lane == 0) readout::store_energy(a.out, node, to, to_ok, en);
  }
  if constexpr (FORCES) {
    lds_barrier();
    if (tid < C) {
      double g = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 4; ++p) g = fma(wd[4 * p + i], s.d[4 * p + i], g);
      float d_h2 = static_cast<float>(a.w.scale * g);
      if (a.node_weights) d_h2 = static_cast<float>(static_cast<double>(d_h2) * a.node_weights[node]);
      a.s.d_h2[at + tid] = d_h2;
      s.row[1][place<C>(tid)] = d_h2;
    }
    lds_barrier();
    back.run(s.row[1], nullptr, s.part());
    Mixing<C, T> mixing_back;
    mixing_back.request(a.mix_T);
    lds_barrier();
    if (tid < C) s.h2[tid] = column<C>(s.part(), tid) * -1.0f;
    lds_barrier();
    for (int i = tid; i < 16 * C; i += T) s.rows[i / C * C + place<C>(i % C)] = s.grad[i] * s.h2[i % C];
    lds_barrier();
    mixing_back.run(s.rows, s.part(), a.mix_T);
    lds_barrier();
    for (int i = tid; i < 16 * C; i += T) s.grad[i] = mixed<C>(s.part(), i, a.mix_scale);
    lds_barrier();
    gradients.run(a.s.X2, a.s.gXe);
  }
}

// ---- backward between the layers and through the first one ----------------------------------------------------------------
struct BackToEdges {
  const float *X1, *mix_T, *up_T, *skip_T, *prod_T;
  float mix_scale, skip_scale;
  const double *w1, *node_weights;
  double scale;
  int sender_parts, first_node;
  EnergySums sums;
  Scratch s;
};

// A wave's part of a sender's row sum, in the lanes of its first slot: mp_backward_sender_kernel's batches of four rows per slot.
template <int C>
__device__ __forceinline__ f4 sender_rows(const Spline &sp, const float *__restrict__ gXe, const int32_t *__restrict__ perm, int64_t nedges, int k0, int k1) {
  using K = Cfg<C, false, true>;
  const int lane = threadIdx.x % kWave, slot = lane / K::SW, cl = lane % K::SW;
  f4 acc = zero4();
  if (cl < K::LPE) {
    for (int k = k0 + slot; k < k1; k += 4 * K::EPW) {
      int e[4];
      f4 row[4];
      bool take[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) e[j] = perm[min(k + j * K::EPW, k1 - 1)];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        take[j] = k + j * K::EPW < k1 && static_cast<unsigned>(e[j]) < static_cast<uint64_t>(nedges);
        const int64_t ec = take[j] ? e[j] : 0;
        row[j] = ld4(gXe + ec * C + 4 * cl);
        take[j] = take[j] & (edge_length(sp.vec[3 * ec], sp.vec[3 * ec + 1], sp.vec[3 * ec + 2]) <= sp.r_max);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) row[j] = take[j] ? row[j] : zero4();
      acc += (row[0] + row[1]) + (row[2] + row[3]);
    }
  }
#pragma unroll
  for (int off = kWave / 2; off >= K::SW; off >>= 1) acc += shfl_down4(acc, off);
  return acc;
}

template <int C, int T>
__global__ __launch_bounds__(T, 2) void back_to_edges_kernel(Graph q, Spline sp, BackToEdges a) {
  using S = Shared<C, T, false, true>;
  __shared__ S s;
  const int tid = threadIdx.x, lane = tid % kWave, wave = wave_number();
  if (static_cast<int>(blockIdx.x) < a.first_node) {
    static_assert(sizeof(s.work) >= T * sizeof(double), "the sums' place");
    graph_energy<T>(a.sums, blockIdx.x, reinterpret_cast<double *>(s.work));
    return;
  }
  const int node = blockIdx.x - a.first_node;
  const int g = a.s.groups[node];
  const bool no_element = g == q.ngroups - 1;
  const int e0 = a.s.live[node], e1 = a.s.live[q.nnodes + node];
  const int64_t at = static_cast<int64_t>(node) * C;
  copy_knots<T>(sp, s.knots);
  EdgeGradients<C, T, false, S> gradients(s, sp, q, a.s.gv1, a.s.gv2, e0, e1);
  const RawEdge raw = gradients.request();
  lds_barrier();
  const float *skip_T = a.skip_T + static_cast<int64_t>(no_element ? 0 : g) * C * C;
  Products<C, 2> both;
  if constexpr (C <= 96) both.request(a.up_T, skip_T);  // (no registers for them here beyond)
  {
    using K = Cfg<C, false, true>;
    const int k0 = q.sender_offsets[node], k1 = q.sender_offsets[node + 1];
    const int64_t len = k1 - k0;
    for (int p = wave; p < a.sender_parts; p += S::kWaves) {
      const int lo = k0 + static_cast<int>(len * p / a.sender_parts), hi = k0 + static_cast<int>(len * (p + 1) / a.sender_parts);
      const f4 acc = sender_rows<C>(sp, a.s.gXe, q.sender_perm, q.nedges, lo, hi);
      if (lane < K::LPE) st4(s.part() + p * C + 4 * lane, acc);
    }
  }
  gradients.template stage<true>(raw);
  if constexpr (C > 96) both.request(a.up_T, skip_T);
  const float d_h2 = tid < C ? a.s.d_h2[at + tid] : 0.f;
  lds_barrier();
  if (tid < C) {
    float v = s.part()[tid];
    for (int p = 1; p < a.sender_parts; ++p) v += s.part()[p * C + tid];
    s.row[0][place<C>(tid)] = v;
    s.row[1][place<C>(tid)] = d_h2;
  }
  lds_barrier();
  both.run(s.row[0], s.row[1], s.part());
  Products<C, 1> prod;
  prod.request(a.prod_T);
  lds_barrier();
  if (tid < C)
    s.row[2][place<C>(tid)] = gh1_of(column<C>(s.part(), tid), column<C>(s.part() + 4 * C, tid), a.w1[tid], a.scale,
                                     a.node_weights ? a.node_weights[node] : 1.0, -a.skip_scale, no_element);
  lds_barrier();
  float grad1[(16 * C + T - 1) / T];
#pragma unroll
  for (int i = 0; i < 16 * C / T; ++i) grad1[i] = a.s.grad1[16 * at + tid + i * T];
  prod.run(s.row[2], nullptr, s.part());
  Mixing<C, T> mixing;
  const float *mix_T = a.mix_T + static_cast<int64_t>(no_element ? 0 : g) * (4 * C * C);
  if (!no_element) mixing.request(mix_T);
  lds_barrier();
  if (tid < C) s.h2[tid] = column<C>(s.part(), tid);
  lds_barrier();
#pragma unroll
  for (int p = 0; p < 16 * C / T; ++p) {
    const int i = tid + p * T;
    s.rows[i / C * C + place<C>(i % C)] = grad1[p] * s.h2[i % C];
  }
  lds_barrier();
  if (no_element) {
    for (int i = tid; i < 64 * C; i += T) s.part()[i] = 0.f;
  } else {
    mixing.run(s.rows, s.part(), mix_T);
  }
  lds_barrier();
  for (int i = tid; i < 16 * C; i += T) s.grad[i] = mixed<C>(s.part(), i, a.mix_scale);
  lds_barrier();
  gradients.run(a.X1, nullptr);
}

Graph graph_of(const cm_mace_weights &w, const cm_mace_graph &g) {
  return Graph{static_cast<int>(g.nnodes), w.nelements + 1, w.nelements, g.nedges, g.receiver, g.sender, g.first_occ, g.sender_perm, g.sender_offsets,
               g.elem_perm, g.elem_offsets, g.onehot_perm, g.onehot_offsets, g.node_rows};
}
Spline spline_of(const cm_mace_weights &w, int layer, const Scratch &s) {
  return Spline{s.vec, nullptr, w.r_knots, w.spline[layer], w.nknots, w.r_width, w.r_max};
}

// call(std::integral_constant channels, std::integral_constant threads)
template <class Call>
int dispatch(int channels, int64_t nnodes, Call call) {
  const auto threads = [&](auto c) {
    if (nnodes <= device_compute_units()) call(c, std::integral_constant<int, kAlone>{});
    else call(c, std::integral_constant<int, kShared>{});
    return CM_OK;
  };
  switch (channels) {
    case 32: return threads(std::integral_constant<int, 32>{});
    case 64: return threads(std::integral_constant<int, 64>{});
    case 96: return threads(std::integral_constant<int, 96>{});
    case 128: return threads(std::integral_constant<int, 128>{});
    default: set_error("cm_mace_step: channels=%d not supported", channels); return CM_EINVAL;
  }
}

}  // namespace

// Edges per node up to which the step of few nodes is no slower than the separate launches.  A node has eight waves, or four, whatever its edges;
// the separate launches cut them into as many parts as the chip has room for, and the fewer nodes share a round the more of it they leave
// idle here.  Step in us, the separate launches -> these, edges per node:
//   up to a node per unit   64   20 x 1 571 325 -> 305; 96 20 x 262 174 -> 169, x 524 197 -> 197, x 785 250 -> 269, 60 x 785 262 -> 272, 100 x 785 276 -> 273, x 1 152 362 -> 376,
//                           150 x 1 571 490 -> 494, 256 x 1 571 543 -> 503; 128 20 x 524 228 -> 226, x 785 291 -> 303, 60 x 785 304 -> 303, 100 x 1 152 419 -> 416
//   up to two               32   300 x 1 152 257 -> 253, x 1 571 321 -> 330; 64 300 x 785 305 -> 299, x 1 152 401 -> 410, 384 x 1 152 444 -> 415; 96 257 x 262 202 -> 199, x 367 238 -> 245,
//                           320 x 367 262 -> 257, x 524 330 -> 338, 384 x 524 351 -> 342, x 785 472 -> 479; 128 257 x 262 240 -> 234, x 367 285 -> 292, 384 x 785 554 -> 551
//   a second round          32   513 x 157 111 -> 110, x 209 127 -> 130, x 524 205 -> 243, 768 x 209 141 -> 138, x 262 161 -> 169, 1 024 x 262 175 -> 177; 64 513 x 79 123 -> 120, x 157
//                           153 -> 164, x 524 317 -> 383, 640 x 105 140 -> 138, x 131 155 -> 158, 768 x 157 183 -> 181, x 209 207 -> 209; energies alone 32 768 x 209 67.0 ->
//                           70.0, 1 024 x 209 75.0 -> 74.0, x 262 83.8 -> 85.5; 64 513 x 79 65.7 -> 56.0, 768 x 157 88.1 -> 88.2, x 209 98.3 -> 103.5
static double most_edges_per_node(int channels, int64_t nnodes, bool forces) {
  const double u = static_cast<double>(nnodes) / device_compute_units();
  if (u <= 1.0) return channels <= 64 ? 2000.0 : 430.0 + 1100.0 * u;
  if (u <= 2.0) return channels == 32 ? 1000.0 + 1400.0 * (u - 1.0) : (channels == 64 ? 700.0 + 1600.0 * (u - 1.0) : 290.0 + 600.0 * (u - 1.0));
  const double v = u - 2.0;
  return channels == 32 ? 155.0 + (forces ? 53.0 : 30.0) * v : 85.0 + (forces ? (40.0 + 70.0 * v) * v : 70.0 * v);
}

// Up to a node per compute unit a workgroup of eight waves has a unit to itself, up to two it has four waves and half of one; a second round of
// those pays at 32 and 64 channels, whose weights are small.  Beyond, the launches that share weights between nodes are faster (and round
// otherwise beyond few::applies: 384 nodes at 128 channels, 512 at 96, 768 at 64).  Step in us, the separate launches -> these:
//   32   21 x 9 71 -> 36, 256 x 52 75 -> 42, 512 x 52 85 -> 51, 756 x 9 77 -> 65, 1 000 x 52 99 -> 90, 1 500 x 52 113 -> 131
//   64   21 x 9 71 -> 39, 100 x 52 85 -> 49, 256 x 52 91 -> 53, 500 x 52 111 -> 70, 504 x 9 95 -> 48, 600 x 52 117 -> 113, 756 x 9 102 -> 82
//   96   21 x 9 82 -> 53, 256 x 52 116 -> 72, 500 x 52 138 -> 95, 504 x 9 115 -> 71
//   128  21 x 9 92 -> 62, 216 x 92 141 -> 99, 256 x 52 136 -> 86, 384 x 52 155 -> 115, 378 x 9 132 -> 85
// (eight waves to half of the nodes: 64 channels, 216 x 52, 51 against 55 with four.)
bool applies(const cm_mace_weights &w, int64_t nnodes, int64_t nedges, bool forces) {
  const int C = w.channels;
  return C <= 128 && nnodes <= (C == 32 ? 4 : 3) * device_compute_units() && static_cast<double>(nedges) <= most_edges_per_node(C, nnodes, forces) * static_cast<double>(nnodes) &&
         !w.mono3[0] && !w.mono2[0] && !w.mono3[1] && !w.mono2[1] && w.n3[0] == CM_SYMCON_N3 && w.n2[0] == CM_SYMCON_N2 &&
         w.n3[1] == CM_SYMCON_N3 && w.n2[1] == CM_SYMCON_N2 && few::applies(nnodes, 16, C) && few::applies(nnodes, 1, C) &&
         !sliced_forward_applies(nnodes, nedges, C, w.nknots);
}

int first_layer(const cm_mace_weights &w, const cm_mace_graph &g, const double *positions, const double *shifts, const Scratch &s, hipStream_t st) {
  const FirstLayer a{positions, shifts, g.X1, w.mix_W[0], w.T3[0], w.T2[0], w.T1[0], w.prod_W[0], w.up_W, w.skip_W,
                     w.mix_scale[0], w.skip_scale, edge_forward_parts(w.channels, g.nnodes, g.nedges), s.vec, s};
  const Spline sp = spline_of(w, 0, s);
  const dim3 grid(static_cast<unsigned>(g.nnodes));
  const int rc = dispatch(w.channels, g.nnodes, [&](auto c, auto t) {
    constexpr int kC = decltype(c)::value, kT = decltype(t)::value;
    if (s.grad1) hipLaunchKernelGGL((first_layer_kernel<kC, kT, true>), grid, dim3(kT), 0, st, graph_of(w, g), sp, a);
    else hipLaunchKernelGGL((first_layer_kernel<kC, kT, false>), grid, dim3(kT), 0, st, graph_of(w, g), sp, a);
  });
  if (rc != CM_OK) return rc;
  return check_launch("cm_mace_step (first layer)");
}

int second_layer(const cm_mace_weights &w, const cm_mace_graph &g, const readout::Outputs &out, const Scratch &s, hipStream_t st) {
  const SecondLayer a{w.mix_W[1], w.mix_WT[1], w.T3[1], w.T2[1], w.T1[1], w.prod_W[1], w.prod_WT[1], w.mix_scale[1],
                      edge_forward_parts(w.channels, g.nnodes, g.nedges),
                      readout::Weights{w.w1, w.W2a, w.w2b, w.act_cst, w.scale, w.shift, w.hidden}, out, g.node_weights, s};
  const Spline sp = spline_of(w, 1, s);
  const dim3 grid(static_cast<unsigned>(g.nnodes));
  const int rc = dispatch(w.channels, g.nnodes, [&](auto c, auto t) {
    constexpr int kC = decltype(c)::value, kT = decltype(t)::value;
    if (s.grad1) hipLaunchKernelGGL((second_layer_kernel<kC, kT, true>), grid, dim3(kT), 0, st, graph_of(w, g), sp, a);
    else hipLaunchKernelGGL((second_layer_kernel<kC, kT, false>), grid, dim3(kT), 0, st, graph_of(w, g), sp, a);
  });
  if (rc != CM_OK) return rc;
  return check_launch("cm_mace_step (second layer)");
}

int back_to_edges(const cm_mace_weights &w, const cm_mace_graph &g, const EnergySums &sums, const Scratch &s, hipStream_t st) {
  const BackToEdges a{g.X1, w.mix_WT[0], w.up_WT, w.skip_WT, w.prod_WT[0], w.mix_scale[0], w.skip_scale, w.w1, g.node_weights, w.scale,
                      sender_parts_of(w.channels, g.nnodes, g.nedges), g.ngraphs, sums, s};
  const Spline sp = spline_of(w, 0, s);
  const dim3 grid(static_cast<unsigned>(g.nnodes + g.ngraphs));
  const int rc = dispatch(w.channels, g.nnodes, [&](auto c, auto t) {
    constexpr int kC = decltype(c)::value, kT = decltype(t)::value;
    hipLaunchKernelGGL((back_to_edges_kernel<kC, kT>), grid, dim3(kT), 0, st, graph_of(w, g), sp, a);
  });
  if (rc != CM_OK) return rc;
  return check_launch("cm_mace_step (back to the edges)");
}

}  // namespace fewnodes
}  // namespace cm
