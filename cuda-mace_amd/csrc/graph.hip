// Index structures of one neighbour list, derived on the device in one call and without a host synchronisation.
//
// The model works on a relabelled copy of the graph in which atoms that are close in space have close indices, so that
// the gathers of sender rows hit in cache, and on lists in which every receiver's pairs beyond the cutoff (the skin shell
// of a Verlet list) come last, nearest first, so that the message-passing kernels can stop at the last pair inside the
// cutoff.  The reference has no counterpart: it takes the list as upstream's host-side search returns it
// (tests/test_utils.py:62-105) and rebuilds its own index table inside every forward call
// (jit_wrappers/src/invariant_message_passing_wrapper.cpp:91-93).
//
//   atoms    sorted by (graph, bin of a 3-D grid, original index); grid of at most `bins` cells per axis, cells at least
//            half a cutoff wide, over the bounding box of the positions
//   edges    of the incoming list (sorted by row i) move with their atom i as whole segments; inside a segment the pairs
//            within the cutoff come first, by the new label of atom j (ties in the list's order), then the others by
//            length (ties in the list's order).  No global sort of the edges: a wave ranks the pairs of one atom.
//   derived  CSR offsets of the new row i, the view of the new list sorted by row j.
#include <algorithm>
#include <cfloat>

#include "common.hpp"

// Products and sums as written (no fused multiply-adds): a host restatement then computes the same grid cells and orders
// pairs of equal length identically.
#pragma clang fp contract(off)

namespace cm {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kMaxBoxes = 64;  // partial bounding boxes; a wave reduces them
constexpr int kScanThreads = 1024;
constexpr int kScanStage = 32 * 1024;  // values staged in LDS at a time (128 KB)
constexpr int kSegLds = 512;   // keys of a segment that a wave keeps in LDS
constexpr int kSegKeys = 4;    // keys of a longer one that a lane ranks at a time
constexpr int kBucketLds = 256;  // pairs of one sender that a wave keeps in LDS

// What bounds the whole call is the launches: each holds microseconds of work that waits for the one before.  There are eight
// of them (nine where few bins hold many atoms), where one kernel per step (box, keys, clear, histogram, scan, fill, rank, ...) took seventeen: every counter is
// cleared by the first, the old CSR and the pairs per sender are taken while the atoms are binned, and the offsets of the view
// by sender are known before the pairs are placed, so the pairs drop into their buckets there.
// A list that holds the reverse of each of its pairs and comes with its CSR (what the neighbour search of this library
// delivers) needs neither: an atom sends as many pairs as it receives, and 470 000 atomic additions in the old labels, which lie
// anywhere in space, are 23 of the 100 us that the eight launches take at 12 000 atoms (153 as seventeen).

struct Box {
  double lo[3], hi[3];
};

__device__ __forceinline__ void include(Box &box, const Box &other) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    box.lo[k] = other.lo[k] < box.lo[k] ? other.lo[k] : box.lo[k];
    box.hi[k] = other.hi[k] > box.hi[k] ? other.hi[k] : box.hi[k];
  }
}

// The box of a wave's boxes, in every lane (smallest and largest values: the order does not matter; a NaN is never taken).
__device__ __forceinline__ Box box_of_wave(Box box) {
  for (int d = kWave / 2; d > 0; d >>= 1) {
    Box other;
#pragma unroll
    for (int k = 0; k < 3; ++k) other.lo[k] = __shfl_xor(box.lo[k], d), other.hi[k] = __shfl_xor(box.hi[k], d);
    include(box, other);
  }
  return box;
}

__device__ __forceinline__ Box empty_box() { return Box{{DBL_MAX, DBL_MAX, DBL_MAX}, {-DBL_MAX, -DBL_MAX, -DBL_MAX}}; }

// Workgroups [0, nboxes): the bounding box of a share of the positions each; the others clear `counters`.
__global__ __launch_bounds__(kThreads) void box_and_clear_kernel(const double *__restrict__ pos, int64_t n, int nboxes, Box *__restrict__ boxes,
                                                                 int32_t *__restrict__ counters, int64_t ncounters) {
  __shared__ Box part[kWaves];
  const int t = threadIdx.x;
  if (static_cast<int>(blockIdx.x) >= nboxes) {
    const int64_t step = static_cast<int64_t>(gridDim.x - nboxes) * kThreads;
    for (int64_t k = static_cast<int64_t>(blockIdx.x - nboxes) * kThreads + t; k < ncounters; k += step) counters[k] = 0;
    return;
  }
  Box box = empty_box();
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + t; i < n; i += static_cast<int64_t>(nboxes) * kThreads) {
    Box at;
#pragma unroll
    for (int k = 0; k < 3; ++k) at.lo[k] = at.hi[k] = pos[3 * i + k];
    include(box, at);
  }
  box = box_of_wave(box);
  if (t % kWave == 0) part[t / kWave] = box;
  __syncthreads();
  if (t == 0) {
    for (int w = 1; w < kWaves; ++w) include(box, part[w]);
    boxes[blockIdx.x] = box;
  }
}

// Workgroups [0, node_blocks), a thread per atom: key = ((graph * bins + bx) * bins + by) * bins + bz, and the atoms per key
// (atoms_of_key NULL: not asked for).
// The others, a thread per pair: the old CSR (a change of the value of row_i closes every atom before it and opens every
// atom up to it, values out of range counting as the nearest atom) and the pairs per atom j.
__global__ __launch_bounds__(kThreads) void count_kernel(const double *__restrict__ pos, const int32_t *__restrict__ graph_of_node, int nnodes,
                                                         int node_blocks, const Box *__restrict__ boxes, int nboxes, double min_width, int bins,
                                                         int ngraphs, int32_t *__restrict__ keys, int32_t *__restrict__ atoms_of_key,
                                                         const int32_t *__restrict__ row_i, const int32_t *__restrict__ row_j, int64_t nedges,
                                                         int32_t *__restrict__ first_occ, int32_t *__restrict__ pairs_of_sender) {
  __shared__ double s_box[4];
  const int t = threadIdx.x;
  if (static_cast<int>(blockIdx.x) >= node_blocks) {
    const int64_t e = static_cast<int64_t>(blockIdx.x - node_blocks) * kThreads + t;
    if (e >= nedges) return;
    const auto clamped = [&](int i) { return i < 0 ? 0 : (i >= nnodes ? nnodes - 1 : i); };
    const int cur = clamped(row_i[e]), prev = e > 0 ? clamped(row_i[e - 1]) : -1, j = row_j[e];
    for (int i = prev + 1; i <= cur; ++i) first_occ[i] = static_cast<int32_t>(e);
    for (int i = prev < 0 ? 0 : prev; i < cur; ++i) first_occ[nnodes + i] = static_cast<int32_t>(e);
    if (e == nedges - 1) {
      first_occ[nnodes + cur] = static_cast<int32_t>(nedges);
      for (int i = cur + 1; i < nnodes; ++i) first_occ[i] = first_occ[nnodes + i] = static_cast<int32_t>(nedges);
    }
    if (static_cast<unsigned>(j) < static_cast<unsigned>(nnodes)) atomicAdd(&pairs_of_sender[j], 1);
    return;
  }
  if (t < kWave) {
    const Box box = box_of_wave(t < nboxes ? boxes[t] : empty_box());
    if (t == 0) {
      double extent = 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        s_box[k] = box.lo[k];
        const double e = box.hi[k] - box.lo[k];
        extent = e > extent ? e : extent;
      }
      s_box[3] = extent;
    }
  }
  __syncthreads();
  const int i = blockIdx.x * kThreads + t;
  if (i >= nnodes) return;
  double width = s_box[3] / bins * (1.0 + 1e-12);
  width = width > min_width ? width : min_width;
  int b[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double f = floor((pos[3 * static_cast<int64_t>(i) + k] - s_box[k]) / width);
    b[k] = f < 0.0 ? 0 : (f >= bins ? bins - 1 : static_cast<int>(f));  // NaN positions land in bin 0
  }
  int g = graph_of_node ? graph_of_node[i] : 0;
  g = g < 0 ? 0 : (g >= ngraphs ? ngraphs - 1 : g);
  const int key = ((g * bins + b[0]) * bins + b[1]) * bins + b[2];
  keys[i] = key;
  if (atoms_of_key) atomicAdd(&atoms_of_key[key], 1);
}

// One workgroup: offsets of the bins, and a copy of them that counts up while the bins are filled.
__global__ __launch_bounds__(kScanThreads) void bin_offsets_kernel(const int32_t *__restrict__ atoms_of_key, int nkeys,
                                                                   int32_t *__restrict__ offsets, int32_t *__restrict__ cursor) {
  __shared__ int part[kScanThreads];
  __shared__ int stage[kScanStage];
  const int total = workgroup_exclusive_scan<kScanThreads, kScanStage, int>(
      nkeys, stage, part, [&](int k) { return atoms_of_key[k]; },
      [&](int k, int before, int) { offsets[k] = cursor[k] = before; });
  if (threadIdx.x == 0) offsets[nkeys] = total;
}

__global__ void bin_atoms_kernel(const int32_t *__restrict__ keys, int nnodes, int32_t *__restrict__ cursor, int32_t *__restrict__ binned) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nnodes) binned[atomicAdd(&cursor[keys[i]], 1)] = i;
}

// The atoms of a bin in the order of their indices: perm and its inverse; under the new label, the length of the atom's
// segment and the pairs it sends (pairs_of_sender NULL: as many as it receives).  binned NULL: perm is there.
__global__ void relabel_nodes_kernel(const int32_t *__restrict__ keys, const int32_t *__restrict__ binned, const int32_t *__restrict__ offsets,
                                     const int32_t *__restrict__ old_first_occ, const int32_t *__restrict__ pairs_of_sender, int nnodes,
                                     int64_t nedges, int32_t *__restrict__ perm, int32_t *__restrict__ inverse, int32_t *__restrict__ degree,
                                     int32_t *__restrict__ sent) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nnodes) return;
  int a = p, o;
  if (binned) {
    o = binned[p];
    const int key = keys[o], lo = offsets[key], hi = offsets[key + 1];
    a = lo;
    for (int q = lo; q < hi; ++q) a += binned[q] < o ? 1 : 0;
  } else {
    o = perm[p];
  }
  perm[a] = o;
  inverse[o] = a;
  int e0 = old_first_occ[o], e1 = old_first_occ[nnodes + o];
  clamp_edge_range(e0, e1, nedges);
  degree[a] = e1 - e0;
  sent[a] = pairs_of_sender ? pairs_of_sender[o] : e1 - e0;
}

// Two workgroups.  The first: first_occ[a] = exclusive scan of degree, first_occ[n + a] = inclusive scan (the CSR layout the
// message-passing kernels take: starts, then ends).  The second: the offsets of the view by sender, and a copy to fill by.
// Ranges of the old CSR overlap where the list is not sorted by row i, and then add up to more than nedges, or more than 32 bits hold:
// the sums have 64, and no offset lies beyond the list.
__global__ __launch_bounds__(kScanThreads) void edge_offsets_kernel(const int32_t *__restrict__ degree, const int32_t *__restrict__ sent, int n,
                                                                    int64_t nedges, int32_t *__restrict__ first_occ,
                                                                    int32_t *__restrict__ sender_offsets, int32_t *__restrict__ cursor,
                                                                    int32_t *__restrict__ long_bucket) {
  __shared__ int64_t part[kScanThreads];
  __shared__ int64_t stage[kScanStage / 2];
  const bool by_sender = blockIdx.x == 1;
  const int32_t *__restrict__ counts = by_sender ? sent : degree;
  const auto within = [&](int64_t offset) { return static_cast<int32_t>(offset < nedges ? offset : nedges); };
  const int64_t total = workgroup_exclusive_scan<kScanThreads, kScanStage / 2, int64_t>(
      n, stage, part, [&](int k) { return counts[k]; },
      [&](int k, int64_t before, int64_t value) {
        if (by_sender) {
          sender_offsets[k] = cursor[k] = within(before);
          if (value > kBucketLds) *long_bucket = 1;
        } else {
          first_occ[k] = within(before);
          first_occ[n + k] = within(before + value);
        }
      });
  if (by_sender && threadIdx.x == 0) sender_offsets[n] = within(total);
}

// One wave per new atom: keys of the pairs of its segment (pairs within the cutoff by the new label of atom j, the others
// behind them by length: the bit pattern of a non-negative double orders like its value), their ranks by (key, position in
// the list), the pairs at their places, and each into its sender's bucket in any order.  Of a list that is not sorted by row i, an atom
// has the pairs that find a place, and others stay without: none is written out of range.
// Keys of more pairs than LDS holds go through `key`, and from there through LDS piece by piece, each read by a lane for several of its
// keys.  The whole call, us, every key read from memory for every pair -> that: 200 atoms x 600 pairs 718 -> 423, 1 000 x 900 1 852 -> 990, 5 000 x
// 900 4 359 -> 2 055.  (1 024 keys in LDS are faster up to that number, 342, 862 and 2 050, and make every other list slower: half as many waves to a
// unit, 12 000 x 40 105 -> 106.4, 100 000 x 4 413 -> 438.)
__global__ __launch_bounds__(kWave) void place_edges_kernel(const double *__restrict__ pos, const int32_t *__restrict__ perm,
                                                            const int32_t *__restrict__ inverse, const int32_t *__restrict__ old_first_occ,
                                                            const int32_t *__restrict__ new_first_occ, const int32_t *__restrict__ row_i,
                                                            const int32_t *__restrict__ row_j, const double *__restrict__ shifts, double r_max,
                                                            unsigned long long *__restrict__ key, int nnodes, int64_t nedges,
                                                            int32_t *__restrict__ receiver, int32_t *__restrict__ sender,
                                                            int32_t *__restrict__ edge_perm, double *__restrict__ shifts_out,
                                                            const int32_t *__restrict__ sender_offsets, int32_t *__restrict__ cursor,
                                                            int32_t *__restrict__ bucketed) {
  __shared__ unsigned long long sk[kSegLds];
  const int a = blockIdx.x, lane = threadIdx.x;
  const int o = perm[a];
  int s0 = old_first_occ[o], s1 = old_first_occ[nnodes + o];
  clamp_edge_range(s0, s1, nedges);
  const int base = new_first_occ[a], d = min(s1 - s0, new_first_occ[nnodes + a] - base);
  const bool in_lds = d <= kSegLds;
  for (int t = lane; t < d; t += kWave) {
    const int64_t e = s0 + t;
    const int i = row_i[e], j = row_j[e];
    unsigned long long k = 0x7fffffffull;  // a pair that names no atom: behind the pairs within the cutoff
    if (static_cast<unsigned>(i) < static_cast<unsigned>(nnodes) && static_cast<unsigned>(j) < static_cast<unsigned>(nnodes)) {
      double v[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = (pos[3 * static_cast<int64_t>(j) + c] - pos[3 * static_cast<int64_t>(i) + c]) + shifts[3 * e + c];
      const double len = sqrt((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
      k = len > r_max ? (1ull << 63) | static_cast<unsigned long long>(__double_as_longlong(len))
                      : static_cast<unsigned long long>(static_cast<unsigned>(inverse[j]));
    }
    if (in_lds)
      sk[t] = k;
    else
      key[e] = k;
  }
  __syncthreads();
  struct Pair {
    int j;
    double shift[3];
  };
  const auto pair_of = [&](int k) {
    const int64_t e = s0 + k;
    return Pair{row_j[e], {shifts[3 * e + 0], shifts[3 * e + 1], shifts[3 * e + 2]}};
  };
  const auto place = [&](int k, int rank, const Pair &pair) {
    const int64_t at = base + rank;
    const int j = pair.j;
    const bool named = static_cast<unsigned>(j) < static_cast<unsigned>(nnodes);
    const int s_new = named ? inverse[j] : j;
    receiver[at] = a;
    sender[at] = s_new;
    edge_perm[at] = s0 + k;
#pragma unroll
    for (int c = 0; c < 3; ++c) shifts_out[3 * at + c] = pair.shift[c];
    if (named) {
      const int to = atomicAdd(&cursor[s_new], 1);
      if (to < sender_offsets[s_new + 1]) bucketed[to] = static_cast<int32_t>(at);
    }
  };
  if (in_lds) {
    for (int k = lane; k < d; k += kWave) {
      const unsigned long long mine = sk[k];
      const Pair pair = pair_of(k);  // on its way meanwhile
      int rank = 0;
#pragma unroll 4
      for (int t = 0; t < d; ++t) rank += (sk[t] < mine || (sk[t] == mine && t < k)) ? 1 : 0;
      place(k, rank, pair);
    }
    return;
  }
  for (int first = 0; first < d; first += kSegKeys * kWave) {
    unsigned long long mine[kSegKeys];
    int rank[kSegKeys];
#pragma unroll
    for (int u = 0; u < kSegKeys; ++u) mine[u] = key[s0 + min(first + u * kWave + lane, d - 1)], rank[u] = 0;
    for (int from = 0; from < d; from += kSegLds) {
      const int cnt = min(kSegLds, d - from);
      __syncthreads();  // the piece before has been read
      for (int t = lane; t < cnt; t += kWave) sk[t] = key[s0 + from + t];
      __syncthreads();
      for (int t = 0; t < cnt; ++t) {
        const unsigned long long other = sk[t];
#pragma unroll
        for (int u = 0; u < kSegKeys; ++u) rank[u] += (other < mine[u] || (other == mine[u] && from + t < first + u * kWave + lane)) ? 1 : 0;
      }
    }
#pragma unroll
    for (int u = 0; u < kSegKeys; ++u)
      if (const int k = first + u * kWave + lane; k < d) place(k, rank[u], pair_of(k));
  }
}

// Workgroups [0, sender_blocks), a wave per sender: its pairs in the order of the new list.  Slots that no pair took (a list that
// is not sorted by row i) name pair 0.  A bucket that does not fit a wave's LDS is left to the other workgroups, a thread per slot, which
// leave at once where there is none (long_bucket): one wave would take the square of its pairs, in a row.  The whole call, us, a list of 160 000
// pairs in which one of 20 000 atoms sends 1 000 / 5 000 / 20 000 of them: by waves alone 1 201 / 27 400 / 438 000, so 111 / 282 / 946; every atom
// sends about 400, 200 atoms 413 -> 207; none that many, 12 000 atoms x 40 105.0 -> 105.2, 25 000 x 85 301.3 -> 300.8.
__global__ __launch_bounds__(kThreads) void rank_senders_kernel(const int32_t *__restrict__ sender_offsets, const int32_t *__restrict__ cursor,
                                                                const int32_t *__restrict__ bucketed, const int32_t *__restrict__ sender,
                                                                const int32_t *__restrict__ long_bucket, int sender_blocks, int nnodes,
                                                                int64_t nedges, int32_t *__restrict__ perm) {
  if (static_cast<int>(blockIdx.x) >= sender_blocks) {
    if (*long_bucket == 0) return;
    const int64_t step = static_cast<int64_t>(gridDim.x - sender_blocks) * kThreads;
    for (int64_t p = static_cast<int64_t>(blockIdx.x - sender_blocks) * kThreads + threadIdx.x; p < nedges; p += step) {
      const int mine = bucketed[p];  // anything where no pair took the slot, which then lies in no sender's range
      if (static_cast<uint64_t>(static_cast<int64_t>(mine)) >= static_cast<uint64_t>(nedges)) continue;
      const int a = sender[mine];
      if (static_cast<unsigned>(a) >= static_cast<unsigned>(nnodes)) continue;
      const int lo = sender_offsets[a], end = sender_offsets[a + 1], hi = min(cursor[a], end);
      if (p < lo || p >= hi || end - lo <= kBucketLds) continue;
      int rank = 0;
#pragma unroll 8
      for (int q = lo; q < hi; ++q) rank += bucketed[q] < mine ? 1 : 0;
      perm[lo + rank] = mine;
    }
    return;
  }
  __shared__ int stage[kWaves][kBucketLds];
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
  const int a = blockIdx.x * kWaves + w;
  const int lo = a < nnodes ? sender_offsets[a] : 0, end = a < nnodes ? sender_offsets[a + 1] : 0;
  const int hi = a < nnodes ? min(cursor[a], end) : 0;
  const bool here = end - lo <= kBucketLds;
  if (here)
    for (int p = lo + lane; p < hi; p += kWave) stage[w][p - lo] = bucketed[p];
  __syncthreads();
  if (here)
    for (int p = lo + lane; p < hi; p += kWave) {
      const int mine = stage[w][p - lo];
      int rank = 0;
#pragma unroll 4
      for (int q = 0; q < hi - lo; ++q) rank += stage[w][q] < mine ? 1 : 0;
      perm[lo + rank] = mine;
    }
  for (int p = hi + lane; p < end; p += kWave) perm[p] = 0;
}

// Rows `perm` of several arrays in one launch.  A workgroup copies a few rows of one array, in the widest units that the
// length of its rows and both addresses allow.
constexpr int kMaxRowArrays = 8;

struct RowArrays {
  const char *src[kMaxRowArrays];
  char *dst[kMaxRowArrays];
  int units[kMaxRowArrays], width[kMaxRowArrays], rows[kMaxRowArrays];  // units per row, bytes per unit, rows per workgroup
  unsigned first[kMaxRowArrays + 1];                                    // first workgroup
  int count;
};

template <typename Unit>
__device__ __forceinline__ void copy_rows(const char *src, char *dst, const int32_t *__restrict__ perm, int units, int64_t r0, int rows, int64_t n) {
  const Unit *from = reinterpret_cast<const Unit *>(src);
  Unit *to = reinterpret_cast<Unit *>(dst);
  const unsigned total = static_cast<unsigned>(rows) * static_cast<unsigned>(units);
  for (unsigned k = threadIdx.x; k < total; k += kThreads) {
    const unsigned r = k / static_cast<unsigned>(units);
    const int o = perm[r0 + r];
    if (static_cast<uint64_t>(static_cast<int64_t>(o)) < static_cast<uint64_t>(n))
      to[r0 * units + k] = from[static_cast<int64_t>(o) * units + (k - r * units)];
  }
}

__global__ __launch_bounds__(kThreads) void gather_rows_kernel(RowArrays a, const int32_t *__restrict__ perm, int64_t n) {
  int k = 0;
  while (k + 1 < a.count && blockIdx.x >= a.first[k + 1]) ++k;
  const int64_t r0 = static_cast<int64_t>(blockIdx.x - a.first[k]) * a.rows[k];
  const int rows = static_cast<int>(n - r0 < a.rows[k] ? n - r0 : a.rows[k]);
  switch (a.width[k]) {
    case 16: return copy_rows<int4>(a.src[k], a.dst[k], perm, a.units[k], r0, rows, n);
    case 8: return copy_rows<int2>(a.src[k], a.dst[k], perm, a.units[k], r0, rows, n);
    case 4: return copy_rows<int>(a.src[k], a.dst[k], perm, a.units[k], r0, rows, n);
    default: return copy_rows<char>(a.src[k], a.dst[k], perm, a.units[k], r0, rows, n);
  }
}

inline size_t align256(size_t n) { return (n + 255) & ~static_cast<size_t>(255); }

// Few bins of many atoms: an atom's rank in its bin takes as many reads as the bin has atoms, and all atoms count in a few places.  The sort
// for few keys (sort.hip), which it takes where this holds, ranks within 256 atoms instead.  The whole call, us, that -> this: 4 096 atoms in one bin 436 -> 49,
// in 27 65 -> 47, in 64 53 -> 49; 8 191 in 64 78 -> 49, 20 000 in one 2 005 -> 64, in 64 148 -> 67, 100 000 in one 9 940 -> 181, in 64 620 -> 192.
inline bool many_atoms_per_key(int64_t nnodes, int64_t nkeys) { return nkeys <= 64 && nnodes >= 4096; }

struct PrepareLayout {
  Box *boxes;
  int32_t *counters, *long_bucket, *atoms_of_key, *old_first_occ, *pairs_of_sender;  // the last four are cleared together
  int64_t ncounters;
  int32_t *atom_keys, *bin_offsets, *bin_cursor, *binned, *degree, *sent, *sender_cursor, *bucketed;
  unsigned long long *edge_key;
  bool many_per_key;
  void *sort;  // many_per_key alone
  size_t sort_bytes, bytes;
  PrepareLayout(void *base, int64_t N, int64_t E, int64_t nkeys) {
    size_t at = 0;
    auto take = [&](size_t n) {
      char *p = base ? static_cast<char *>(base) + at : nullptr;
      at += align256(n);
      return p;
    };
    auto ints = [&](int64_t n) { return reinterpret_cast<int32_t *>(take(static_cast<size_t>(n) * 4)); };
    boxes = reinterpret_cast<Box *>(take(kMaxBoxes * sizeof(Box)));
    ncounters = 1 + nkeys + 3 * N;
    counters = ints(ncounters);
    long_bucket = counters;
    atoms_of_key = long_bucket + 1;
    old_first_occ = atoms_of_key + nkeys;
    pairs_of_sender = old_first_occ + 2 * N;
    atom_keys = ints(N);
    bin_offsets = ints(nkeys + 1);
    bin_cursor = ints(nkeys);
    binned = ints(N);
    degree = ints(N);
    sent = ints(N);
    sender_cursor = ints(N);
    bucketed = ints(E);
    edge_key = reinterpret_cast<unsigned long long *>(take(static_cast<size_t>(E) * 8));
    many_per_key = many_atoms_per_key(N, nkeys);
    sort_bytes = many_per_key ? cm_stable_key_sort_workspace(N, nkeys) : 0;
    sort = take(sort_bytes);
    bytes = at;
  }
};

}  // namespace
}  // namespace cm

extern "C" size_t cm_graph_prepare_workspace(int64_t nnodes, int64_t nedges, int ngraphs, int bins) {
  if (nnodes < 0 || nedges < 0 || ngraphs < 1 || bins < 1) return 0;
  return cm::PrepareLayout(nullptr, nnodes, nedges, static_cast<int64_t>(ngraphs) * bins * bins * bins).bytes;
}

namespace cm {
namespace {

int prepare(const double *positions, const int32_t *row_i, const int32_t *row_j, const double *shifts,
                                const int32_t *known_first_occ, const int32_t *graph_of_node, int64_t nnodes, int64_t nedges, int ngraphs, double r_max, int bins,
                                int32_t *node_perm, int32_t *node_inverse, int32_t *receiver, int32_t *sender, int32_t *edge_perm,
                                double *shifts_out, int32_t *first_occ, int32_t *sender_perm, int32_t *sender_offsets,
                                void *workspace, size_t workspace_bytes, cm_stream_t stream, const char *what) {
  CM_REQUIRE(nnodes >= 0 && nedges >= 0 && nnodes < INT32_MAX / 4 && nedges < INT32_MAX / 3, "%s: sizes out of range", what);
  CM_REQUIRE(ngraphs >= 1 && bins >= 1 && bins <= 64, "%s: need at least one graph and 1 to 64 bins per axis", what);
  const int64_t nkeys = static_cast<int64_t>(ngraphs) * bins * bins * bins;
  CM_REQUIRE(nkeys < (int64_t{1} << 24), "%s: ngraphs * bins^3 = %lld keys, at most 2^24 - 1", what, static_cast<long long>(nkeys));
  CM_REQUIRE(r_max > 0.0, "%s: r_max must be positive", what);
  CM_REQUIRE(sender_offsets && (nnodes == 0 || first_occ), "%s: NULL output", what);
  CM_REQUIRE(nnodes == 0 || (positions && node_perm && node_inverse), "%s: NULL node operand", what);
  CM_REQUIRE(nedges == 0 || (row_i && row_j && shifts && receiver && sender && edge_perm && shifts_out && sender_perm),
             "%s: NULL edge operand", what);
  const PrepareLayout L(workspace, nnodes, nedges, nkeys);
  if (workspace == nullptr || workspace_bytes < L.bytes) {
    set_error("%s: workspace of %zu bytes, need %zu", what, workspace_bytes, L.bytes);
    return CM_ENOSPC;
  }
  CM_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "%s: workspace must be 256-byte aligned", what);
  CM_REQUIRE(nnodes > 0 || nedges == 0, "%s: pairs without atoms", what);
  hipStream_t st = as_stream(stream);
  const int N = static_cast<int>(nnodes);
  const int32_t *old_first_occ = known_first_occ ? known_first_occ : L.old_first_occ;
  const dim3 block(kThreads);
  const unsigned gn = static_cast<unsigned>(ceil_div(nnodes, kThreads)), ge = static_cast<unsigned>(ceil_div(nedges, kThreads));
  if (nnodes > 0) {
    // atoms by bin; old CSR and pairs per sender
    const int64_t ncounters = known_first_occ ? 1 + nkeys : L.ncounters;
    const int nboxes = static_cast<int>(std::min<int64_t>(ceil_div(nnodes, 4 * kThreads), kMaxBoxes));
    const unsigned clears = static_cast<unsigned>(std::min<int64_t>(ceil_div(ncounters, 4 * kThreads), 1024));
    hipLaunchKernelGGL(box_and_clear_kernel, dim3(nboxes + clears), block, 0, st, positions, nnodes, nboxes, L.boxes, L.counters, ncounters);
    hipLaunchKernelGGL(count_kernel, dim3(gn + (known_first_occ ? 0 : ge)), block, 0, st, positions, graph_of_node, N, static_cast<int>(gn), L.boxes, nboxes,
                       0.5 * r_max, bins, ngraphs, L.atom_keys, L.many_per_key ? static_cast<int32_t *>(nullptr) : L.atoms_of_key, row_i, row_j, nedges,
                       L.old_first_occ, L.pairs_of_sender);
    if (L.many_per_key) {
      if (const int rc = cm_stable_key_sort(L.atom_keys, nnodes, nkeys, node_perm, L.bin_offsets, L.sort, L.sort_bytes, stream); rc != CM_OK) return rc;
    } else {
      hipLaunchKernelGGL(bin_offsets_kernel, dim3(1), dim3(kScanThreads), 0, st, L.atoms_of_key, static_cast<int>(nkeys), L.bin_offsets,
                         L.bin_cursor);
      hipLaunchKernelGGL(bin_atoms_kernel, dim3(gn), block, 0, st, L.atom_keys, N, L.bin_cursor, L.binned);
    }
    hipLaunchKernelGGL(relabel_nodes_kernel, dim3(gn), block, 0, st, L.atom_keys, L.many_per_key ? static_cast<const int32_t *>(nullptr) : L.binned,
                       L.bin_offsets, old_first_occ,
                       known_first_occ ? static_cast<const int32_t *>(nullptr) : L.pairs_of_sender, N, nedges, node_perm, node_inverse, L.degree, L.sent);
  }
  hipLaunchKernelGGL(edge_offsets_kernel, dim3(2), dim3(kScanThreads), 0, st, L.degree, L.sent, N, nedges, first_occ, sender_offsets,
                     L.sender_cursor, L.long_bucket);
  if (nedges > 0) {
    hipLaunchKernelGGL(place_edges_kernel, dim3(static_cast<unsigned>(nnodes)), dim3(kWave), 0, st, positions, node_perm, node_inverse,
                       old_first_occ, first_occ, row_i, row_j, shifts, r_max, L.edge_key, N, nedges, receiver, sender, edge_perm, shifts_out,
                       sender_offsets, L.sender_cursor, L.bucketed);
    const unsigned sender_blocks = static_cast<unsigned>(ceil_div(nnodes, kWaves));
    hipLaunchKernelGGL(rank_senders_kernel, dim3(sender_blocks + std::min(ge, 1024u)), block, 0, st, sender_offsets, L.sender_cursor, L.bucketed, sender,
                       L.long_bucket, static_cast<int>(sender_blocks), N, nedges, sender_perm);
  }
  return check_launch(what);
}

}  // namespace
}  // namespace cm

extern "C" int cm_graph_prepare(const double *positions, const int32_t *row_i, const int32_t *row_j, const double *shifts,
                                const int32_t *graph_of_node, int64_t nnodes, int64_t nedges, int ngraphs, double r_max, int bins,
                                int32_t *node_perm, int32_t *node_inverse, int32_t *receiver, int32_t *sender, int32_t *edge_perm,
                                double *shifts_out, int32_t *first_occ, int32_t *sender_perm, int32_t *sender_offsets,
                                void *workspace, size_t workspace_bytes, cm_stream_t stream) {
  return cm::prepare(positions, row_i, row_j, shifts, nullptr, graph_of_node, nnodes, nedges, ngraphs, r_max, bins, node_perm, node_inverse, receiver, sender,
                     edge_perm, shifts_out, first_occ, sender_perm, sender_offsets, workspace, workspace_bytes, stream, "cm_graph_prepare");
}

extern "C" int cm_graph_prepare_symmetric(const double *positions, const int32_t *row_i, const int32_t *row_j, const double *shifts,
                                const int32_t *old_first_occ, const int32_t *graph_of_node, int64_t nnodes, int64_t nedges, int ngraphs, double r_max, int bins,
                                int32_t *node_perm, int32_t *node_inverse, int32_t *receiver, int32_t *sender, int32_t *edge_perm,
                                double *shifts_out, int32_t *first_occ, int32_t *sender_perm, int32_t *sender_offsets,
                                void *workspace, size_t workspace_bytes, cm_stream_t stream) {
  CM_REQUIRE(nnodes == 0 || old_first_occ != nullptr, "cm_graph_prepare_symmetric: old_first_occ is NULL");
  return cm::prepare(positions, row_i, row_j, shifts, old_first_occ, graph_of_node, nnodes, nedges, ngraphs, r_max, bins, node_perm, node_inverse, receiver, sender,
                     edge_perm, shifts_out, first_occ, sender_perm, sender_offsets, workspace, workspace_bytes, stream, "cm_graph_prepare_symmetric");
}

extern "C" int cm_gather_rows(const int32_t *perm, int64_t nrows, int narrays, const void *const *src, void *const *dst, const int64_t *row_bytes,
                              cm_stream_t stream) {
  static const char *what = "cm_gather_rows";
  CM_REQUIRE(nrows >= 0 && nrows < INT32_MAX, "%s: nrows out of range", what);
  CM_REQUIRE(narrays >= 0 && narrays <= cm::kMaxRowArrays, "%s: %d arrays, at most %d", what, narrays, cm::kMaxRowArrays);
  CM_REQUIRE(narrays == 0 || (src && dst && row_bytes), "%s: NULL pointer", what);
  CM_REQUIRE(nrows == 0 || narrays == 0 || perm, "%s: perm is NULL", what);
  cm::RowArrays a{};
  uint64_t blocks = 0;
  for (int k = 0; k < narrays; ++k) {
    CM_REQUIRE(row_bytes[k] >= 0 && row_bytes[k] <= (1 << 20), "%s: rows of 0 to 2^20 bytes", what);
    if (row_bytes[k] == 0 || nrows == 0) continue;
    CM_REQUIRE(src[k] && dst[k], "%s: NULL array", what);
    const uintptr_t bits = reinterpret_cast<uintptr_t>(src[k]) | reinterpret_cast<uintptr_t>(dst[k]) | static_cast<uintptr_t>(row_bytes[k]);
    const int at = a.count++, width = bits % 16 == 0 ? 16 : bits % 8 == 0 ? 8 : bits % 4 == 0 ? 4 : 1;
    a.src[at] = static_cast<const char *>(src[k]), a.dst[at] = static_cast<char *>(dst[k]);
    a.width[at] = width, a.units[at] = static_cast<int>(row_bytes[k] / width);
    a.rows[at] = std::max(1, 4 * cm::kThreads / a.units[at]);
    a.first[at] = static_cast<unsigned>(blocks);
    blocks += static_cast<uint64_t>(cm::ceil_div(nrows, a.rows[at]));
  }
  CM_REQUIRE(blocks < (1ull << 31), "%s: too many rows", what);
  if (blocks == 0) return CM_OK;
  hipLaunchKernelGGL(cm::gather_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(cm::kThreads), 0, cm::as_stream(stream), a, perm, nrows);
  return cm::check_launch(what);
}
