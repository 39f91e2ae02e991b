// Neighbour list on the device: all ordered pairs (i, j, S) with |r_j - r_i + S . cell| < cutoff, sorted
// lexicographically by (i, j, Sx, Sy, Sz) -- the edge list the message-passing kernels consume (row i sorted).
//
// Cell list in fractional coordinates of the (possibly triclinic) cell: bins at least half a cutoff wide along every
// axis (measured perpendicular to the other two cell vectors; bins of a whole cutoff hold 1.7 times the candidates, and in a
// cell barely wider than the cutoff six times: a 216-atom crystal with a skin was then one bin and its 27 images), atoms copied bin by bin (in any order inside a bin), one
// wavefront per atom scanning the neighbouring bins with the lanes spread over the bins' atoms taken together.  Two
// passes over the candidates (count, then fill after an exclusive scan) give every atom a contiguous segment; inside a
// segment the hits are placed at their rank under the (j, S) order, so the result is the unique sorted list and
// is reproducible bit for bit.
//
// What bounds it is the chain of dependent memory accesses and the number of launches: a few thousand atoms are a few
// microseconds of work.  Bin by bin (27 bins of a dozen atoms: offsets, then indices, then positions, each waiting for the
// one before) a scan took 25 us at 2 000 atoms and 44 us for a 216-atom crystal with 89 neighbours each; now the bins'
// ranges are looked up side by side and their atoms addressed as one sequence of records.
//
// The accept test uses the ORIGINAL fp64 positions and the integer image S only:
//     v = (r_j - r_i) + (Sx c0 + Sy c1 + Sz c2),   v0 v0 + v1 v1 + v2 v2 < cutoff^2,   (j, S) != (i, 0)
// evaluated left to right without fused multiply-adds, so that a host restatement of the same expression decides
// every borderline pair identically.  Bins only choose the candidates; they are 1e-9 wider than the cutoff so that
// rounding in the fractional coordinates cannot lose a pair.  Atoms may lie outside the cell (unwrapped
// trajectories): the wrap count of each atom enters S.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <type_traits>

#include "common.hpp"

namespace cm {
namespace {

constexpr int kGridThreads = 1024;
constexpr int kOffsetsStage = 16 * 1024;  // values staged in LDS at a time by the offsets scan (128 KB)
constexpr double kBinSlack = 1.0 + 1e-9;
constexpr double kBinsPerCutoff = 2.0;
constexpr int kMaxScan = 32;  // most images of the cell scanned on each side of an atom

struct Grid {
  double inv[9];    // inverse of the effective cell (row-vector convention: frac = r . inv)
  double cellv[9];  // the cell as given (used for S . cell)
  double fmin[3];   // lower bound of the binned range per axis (0 for periodic axes)
  double fscale[3]; // bins per unit of fractional coordinate
  int nb[3];        // bins per axis
  int nscan[3];     // bins to scan on each side
  int periodic[3];
  int status;       // 0 ok, 1 periodic axis with a singular cell, 2 cell thinner than cutoff / 32
};

struct Workspace {
  Grid *grid;
  int32_t *wrap;          // [N, 3]  images the atom was wrapped by along periodic axes
  int32_t *keys;          // [N]     its bin
  int32_t *slot;          // [N]     its place inside the bin
  int32_t *cell_count;    // [max_cells]
  int32_t *cell_offsets;  // [max_cells + 1]
  int32_t *degree;        // [N]
  int32_t *skey;          // [N]     bin, in bin order like the next two
  double *spos;           // [N, 3]  positions as given
  int4 *smeta;            // [N]     index of the atom, its wrap
  size_t total;
};

size_t align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }

Workspace carve(void *base, int64_t n, int64_t max_cells) {
  Workspace w;
  char *p = static_cast<char *>(base);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char *q = p ? p + off : nullptr;
    off += align256(bytes);
    return q;
  };
  auto ints = [&](int64_t count) { return reinterpret_cast<int32_t *>(take(sizeof(int32_t) * static_cast<size_t>(count))); };
  w.grid = reinterpret_cast<Grid *>(take(sizeof(Grid)));
  w.wrap = ints(3 * n);
  w.keys = ints(n);
  w.slot = ints(n);
  w.cell_count = ints(max_cells);
  w.cell_offsets = ints(max_cells + 1);
  w.degree = ints(n);
  w.skey = ints(n);
  w.spos = reinterpret_cast<double *>(take(sizeof(double) * 3 * static_cast<size_t>(n)));
  w.smeta = reinterpret_cast<int4 *>(take(sizeof(int4) * static_cast<size_t>(n)));
  w.total = off;
  return w;
}

__device__ __forceinline__ int floor_div(int a, int b) {
  int q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
  return q;
}

// One workgroup: effective cell and its inverse, extent of the atoms along non-periodic axes, bin counts.  Written to
// *grid (global memory) and *out (LDS; valid for every thread on return).
__device__ __forceinline__ void make_grid(const double *__restrict__ pos, const double *__restrict__ cell, int px, int py, int pz,
                                          double cutoff, int nnodes, int max_cells, Grid *__restrict__ grid, Grid *out) {
  __shared__ double inv[9];
  __shared__ double lo[3][kGridThreads / kWave], hi[3][kGridThreads / kWave];
  __shared__ int singular;
  const int t = threadIdx.x;
  if (t == 0) {
    double c[9];
    for (int k = 0; k < 9; ++k) c[k] = cell ? cell[k] : 0.0;
    const double cx[3] = {c[4] * c[8] - c[5] * c[7], c[5] * c[6] - c[3] * c[8], c[3] * c[7] - c[4] * c[6]};  // c1 x c2
    const double det = c[0] * cx[0] + c[1] * cx[1] + c[2] * cx[2];
    const double n0 = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]), n1 = sqrt(c[3] * c[3] + c[4] * c[4] + c[5] * c[5]),
                 n2 = sqrt(c[6] * c[6] + c[7] * c[7] + c[8] * c[8]);
    const bool bad = !(fabs(det) > 1e-12 * n0 * n1 * n2) || !isfinite(det);
    singular = bad;
    if (bad) {
      for (int k = 0; k < 9; ++k) inv[k] = (k % 4 == 0) ? 1.0 : 0.0;
    } else {
      // inverse of the 3x3 matrix with rows c0, c1, c2: columns are the cross products / det
      const double r = 1.0 / det;
      inv[0] = cx[0] * r;
      inv[3] = cx[1] * r;
      inv[6] = cx[2] * r;
      inv[1] = (c[7] * c[2] - c[8] * c[1]) * r;  // (c2 x c0)
      inv[4] = (c[8] * c[0] - c[6] * c[2]) * r;
      inv[7] = (c[6] * c[1] - c[7] * c[0]) * r;
      inv[2] = (c[1] * c[5] - c[2] * c[4]) * r;  // (c0 x c1)
      inv[5] = (c[2] * c[3] - c[0] * c[5]) * r;
      inv[8] = (c[0] * c[4] - c[1] * c[3]) * r;
    }
  }
  __syncthreads();
  double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  // (the range of a fully periodic cell is the cell: the atoms are not looked at)
  for (int i = t; i < (px && py && pz ? 0 : nnodes); i += kGridThreads) {
    const double x = pos[3 * i], y = pos[3 * i + 1], z = pos[3 * i + 2];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double f = x * inv[k] + y * inv[3 + k] + z * inv[6 + k];
      mn[k] = fmin(mn[k], f);
      mx[k] = fmax(mx[k], f);
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    for (int off = kWave / 2; off > 0; off >>= 1) {
      mn[k] = fmin(mn[k], __shfl_xor(mn[k], off));
      mx[k] = fmax(mx[k], __shfl_xor(mx[k], off));
    }
    if (t % kWave == 0) {
      lo[k][t / kWave] = mn[k];
      hi[k][t / kWave] = mx[k];
    }
  }
  __syncthreads();
  if (t < kWave) {  // an axis per lane (square roots and divisions one after the other by one thread took 3 us)
    Grid &g = *out;
    const int k = min(t, 2);
    const bool mine = t < 3, per = (k == 0 ? px : (k == 1 ? py : pz)) != 0;
    const double height = 1.0 / sqrt(inv[k] * inv[k] + inv[3 + k] * inv[3 + k] + inv[6 + k] * inv[6 + k]);
    double width, low = 0.0;  // distance covered by the binned range of the axis, perpendicular to the other two axes
    if (per) {
      width = height;
    } else {
      double a = INFINITY, b = -INFINITY;
      for (int w = 0; w < kGridThreads / kWave; ++w) {
        a = fmin(a, lo[k][w]);
        b = fmax(b, hi[k][w]);
      }
      const double ext = (nnodes > 0 && b > a) ? (b - a) : 0.0;
      low = nnodes > 0 ? a : 0.0;
      width = ext * height;
    }
    const double bins = floor(kBinsPerCutoff * width / (cutoff * kBinSlack));
    int nb = bins >= 1.0 ? static_cast<int>(fmin(bins, 1.0e6)) : 1;
    if (t < 9) {
      g.inv[t] = inv[t];
      g.cellv[t] = cell ? cell[t] : 0.0;
    }
    // keep the number of bins within what the caller's workspace holds: halve the finest axis until it fits
    int n0 = __shfl(nb, 0), n1 = __shfl(nb, 1), n2 = __shfl(nb, 2);
    while (static_cast<int64_t>(n0) * n1 * n2 > max_cells) {
      int finest = 0;
      if (n1 > n0) finest = 1;
      if (n2 > (finest == 1 ? n1 : n0)) finest = 2;
      if (finest == 0) n0 = (n0 + 1) / 2;
      else if (finest == 1) n1 = (n1 + 1) / 2;
      else n2 = (n2 + 1) / 2;
    }
    nb = k == 0 ? n0 : (k == 1 ? n1 : n2);
    double fscale;
    int nscan;
    if (per) {
      fscale = nb;
      const double binw = width / nb;
      nscan = static_cast<int>(ceil(cutoff * kBinSlack / binw));
    } else {
      // fscale maps (f - fmin) to a bin number; a zero extent puts every atom in bin 0
      const double ext = width > 0.0 ? width : 0.0;
      fscale = ext > 0.0 ? nb * height / ext : 0.0;
      nscan = nb > 1 ? static_cast<int>(ceil(cutoff * kBinSlack / (ext / nb))) : 0;
    }
    if (nscan < 0) nscan = 0;
    const bool thin = nscan > kMaxScan;  // a cell far thinner than the cutoff: refuse rather than scan thousands of images
    if (mine) {
      g.fmin[k] = low;
      g.fscale[k] = fscale;
      g.nb[k] = nb;
      g.nscan[k] = thin ? 0 : nscan;
      g.periodic[k] = per ? 1 : 0;
    }
    const bool any_thin = __ballot(mine && thin) != 0;
    if (t == 0) g.status = any_thin ? 2 : ((singular && (px || py || pz)) ? 1 : 0);
    wave_lds_fence();
    static_assert(sizeof(Grid) % 4 == 0, "copied word by word");
    for (int q = t; q < static_cast<int>(sizeof(Grid) / 4); q += kWave) reinterpret_cast<int *>(grid)[q] = reinterpret_cast<const int *>(out)[q];
  }
  __syncthreads();
}

// Bin of an atom and the images it is wrapped by.
__device__ __forceinline__ int bin_of(const Grid &g, double x, double y, double z, int (&wrap)[3]) {
  int b[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double f = x * g.inv[k] + y * g.inv[3 + k] + z * g.inv[6 + k];
    int w = 0;
    if (g.periodic[k]) {
      const double fl = floor(f);
      f -= fl;
      w = static_cast<int>(fl);
      if (f >= 1.0) {
        f -= 1.0;
        w += 1;
      }
    } else {
      f -= g.fmin[k];
    }
    const int bk = static_cast<int>(f * g.fscale[k]);
    b[k] = bk < 0 ? 0 : (bk > g.nb[k] - 1 ? g.nb[k] - 1 : bk);
    wrap[k] = w;
  }
  return (b[0] * g.nb[1] + b[1]) * g.nb[2] + b[2];
}

// Up to kSmallAtoms atoms and bins: the whole cell list by one workgroup, with the bins counted and scanned in LDS, in place
// of the five launches below.  Beyond that a thread's passes over its atoms cost more than the launches (12 000 atoms: 90
// against 35 us; 2 000: 17 against 28; with a thread's atoms in registers and the grid's axes side by side 2 000 17.5 -> 12.7, 216 10.2 -> 8.6).
constexpr int kSmallAtoms = 4 * 1024;
__global__ __launch_bounds__(kGridThreads) void nl_cells_small_kernel(const double *__restrict__ pos, const double *__restrict__ cell,
                                                                      int px, int py, int pz, double cutoff, int nnodes, int max_cells,
                                                                      Workspace w) {
  extern __shared__ int s_count[];  // [max_cells]
  __shared__ Grid g;
  __shared__ int s_wave[kGridThreads / kWave];
  const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
  for (int c = t; c < max_cells; c += kGridThreads) s_count[c] = 0;
  // a thread's atoms, t, t + 1024, ..., stay in its registers from here on
  constexpr int kMine = kSmallAtoms / kGridThreads;
  double r[kMine][3];
  int key[kMine], slot[kMine], wrap[kMine][3];
#pragma unroll
  for (int u = 0; u < kMine; ++u) {
    const int i = t + u * kGridThreads;
#pragma unroll
    for (int k = 0; k < 3; ++k) r[u][k] = i < nnodes ? pos[3 * i + k] : 0.0;
  }
  make_grid(pos, cell, px, py, pz, cutoff, nnodes, max_cells, w.grid, &g);  // ends with a barrier
  const int ncells = min(g.nb[0] * g.nb[1] * g.nb[2], max_cells);
#pragma unroll
  for (int u = 0; u < kMine; ++u) {
    if (t + u * kGridThreads >= nnodes) break;
    key[u] = bin_of(g, r[u][0], r[u][1], r[u][2], wrap[u]);
    slot[u] = atomicAdd(&s_count[key[u]], 1);
  }
  __syncthreads();
  // exclusive scan in place: a contiguous run of odd length per thread, then over the threads
  const int per = ((ncells + kGridThreads - 1) / kGridThreads) | 1;
  const int lo = min(t * per, ncells), hi = min(lo + per, ncells);
  int sum = 0;
  for (int c = lo; c < hi; ++c) sum += s_count[c];
  int upto = sum;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int v = __shfl_up(upto, d);
    if (lane >= d) upto += v;
  }
  if (lane == kWave - 1) s_wave[wave] = upto;
  __syncthreads();
  int run = upto - sum;
  for (int q = 0; q < wave; ++q) run += s_wave[q];
  for (int c = lo; c < hi; ++c) {
    const int v = s_count[c];
    s_count[c] = run;
    run += v;
  }
  __syncthreads();
  for (int c = t; c < ncells; c += kGridThreads) w.cell_offsets[c] = s_count[c];
  if (t == 0) w.cell_offsets[ncells] = nnodes;
#pragma unroll
  for (int u = 0; u < kMine; ++u) {
    const int i = t + u * kGridThreads;
    if (i >= nnodes) break;
    const int at = s_count[key[u]] + slot[u];
    w.skey[at] = key[u];
    w.smeta[at] = make_int4(i, wrap[u][0], wrap[u][1], wrap[u][2]);
#pragma unroll
    for (int k = 0; k < 3; ++k) w.spos[3 * at + k] = r[u][k];
  }
}

// The same for more atoms: grid, bins (a counter per bin), a scan, the copy into bin order.
__global__ __launch_bounds__(kGridThreads) void nl_grid_kernel(const double *__restrict__ pos, const double *__restrict__ cell,
                                                               int px, int py, int pz, double cutoff, int nnodes,
                                                               int max_cells, Grid *__restrict__ grid) {
  __shared__ Grid g;
  make_grid(pos, cell, px, py, pz, cutoff, nnodes, max_cells, grid, &g);
}

__global__ void nl_clear_kernel(int32_t *__restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ void nl_bin_kernel(const double *__restrict__ pos, int nnodes, Workspace w) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nnodes) return;
  int wr[3];
  const int key = bin_of(*w.grid, pos[3 * static_cast<int64_t>(i)], pos[3 * static_cast<int64_t>(i) + 1], pos[3 * static_cast<int64_t>(i) + 2], wr);
  w.keys[i] = key;
  w.slot[i] = atomicAdd(&w.cell_count[key], 1);
#pragma unroll
  for (int k = 0; k < 3; ++k) w.wrap[3 * static_cast<int64_t>(i) + k] = wr[k];
}

constexpr int kCellStage = 32 * 1024;  // values staged in LDS at a time (128 KB)
__global__ __launch_bounds__(kGridThreads) void nl_cell_scan_kernel(int max_cells, Workspace w) {
  __shared__ int part[kGridThreads];
  __shared__ int stage[kCellStage];
  const int ncells = min(w.grid->nb[0] * w.grid->nb[1] * w.grid->nb[2], max_cells);
  const int total = workgroup_exclusive_scan<kGridThreads, kCellStage, int>(
      ncells, stage, part, [&](int k) { return w.cell_count[k]; }, [&](int k, int before, int) { w.cell_offsets[k] = before; });
  if (threadIdx.x == 0) w.cell_offsets[ncells] = total;
}

__global__ void nl_place_kernel(const double *__restrict__ pos, int nnodes, Workspace w) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i >= nnodes) return;
  const int key = w.keys[i];
  const int64_t at = w.cell_offsets[key] + w.slot[i];
  w.skey[at] = key;
  w.smeta[at] = make_int4(static_cast<int>(i), w.wrap[3 * i], w.wrap[3 * i + 1], w.wrap[3 * i + 2]);
#pragma unroll
  for (int k = 0; k < 3; ++k) w.spos[3 * at + k] = pos[3 * i + k];
}

// Component k of S . cell, term by term from the left.  No contraction into fused multiply-adds.
__device__ __forceinline__ double image_shift(const int (&S)[3], const double *c, int k) {
#pragma clang fp contract(off)
  return (S[0] * c[k] + S[1] * c[3 + k]) + S[2] * c[6 + k];
}

// The accept test; see the head of this file.
__device__ __forceinline__ bool within(const double *pi, const double *pj, const int (&S)[3], const double *c, double rc2) {
#pragma clang fp contract(off)
  double d2 = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double v = (pj[k] - pi[k]) + image_shift(S, c, k);
    d2 = k == 0 ? v * v : d2 + v * v;
  }
  return d2 < rc2;
}

// What the last pass writes when it has a segment's hits in LDS: the list in every form its consumers take.
struct GraphOut {
  int32_t *row_i, *row_j;   // [E]
  int64_t *edge_index;      // [2, E]
  double *unit_shifts;      // [E, 3]
  double *shifts;           // [E, 3]
  int32_t *first_occ;       // [2 N]
  int64_t *batch, *ptr;     // [N] zeros, {0, N}; may be NULL
  int32_t *ptr32;           // {0, N}; may be NULL
};

// A neighbour's place in the order of a segment: its index, then the image S.  The neighbours of one index j are scanned in images B of
// the cell with S = B + (wrap of i) - (wrap of j), so B orders them as S does; |B| <= kMaxScan.
__device__ __forceinline__ unsigned long long order_key(int j, int image) {
  return static_cast<unsigned long long>(static_cast<unsigned>(j)) << 24 | static_cast<unsigned>(image);
}
__device__ __forceinline__ int pack_image(int b0, int b1, int b2) { return (b0 + 128) << 16 | (b1 + 128) << 8 | (b2 + 128); }
__device__ __forceinline__ void unpack_image(int image, int (&b)[3]) {
  b[0] = (image >> 16 & 255) - 128, b[1] = (image >> 8 & 255) - 128, b[2] = (image & 255) - 128;
}

__device__ __forceinline__ bool key_less(int ja, const int32_t *Sa, int jb, const int32_t *Sb) {
  if (ja != jb) return ja < jb;
  if (Sa[0] != Sb[0]) return Sa[0] < Sb[0];
  if (Sa[1] != Sb[1]) return Sa[1] < Sb[1];
  return Sa[2] < Sb[2];
}

// One wavefront per atom, atoms in bin order (the waves of a workgroup share their candidates).
//   COUNT     degree[i] = number of neighbours
//   SCRATCH   the neighbours (j, S) in scan order to scratch[offsets[i] ...] (j in scratch[0:E], S in scratch[E:4E])
//   GRAPH     the neighbours collected in LDS (`cap` of them per wave), each written to its rank under the (j, S) order
// Two times 64 candidates per trip, their look-ups and loads side by side: a trip is a chain of seven LDS reads and a load.  With that and
// the rank from one 64-bit key per neighbour (the compare of index and image took 25 of 41 us at 123 neighbours, many of them images of one
// atom) us, count / graph: 2 000 atoms with 52 neighbours 9.2 / 14.4 -> 7.7 / 10.8, 216 with 123 13.8 / 41 -> 12.9 / 16.7, 12 000
// with 42 17.8 / 36.4 -> 18.3 / 32.6.  64 bins where no more are in reach (large cells, whose bins are halved to fit the workspace) and 64 candidates where no
// more are left: 40 000 with 10, 45 bins and 58 candidates, 29.8 / 49.2 -> 35.8 / 58.7 with 128 of each always, 28.7 / 52.2 with this.
enum class Scan { kCount, kScratch, kGraph };
constexpr int kScanWaves = 4;
template <Scan MODE>
__global__ __launch_bounds__(kScanWaves * kWave) void nl_scan_kernel(Workspace w, double cutoff, int nnodes,
                                                                     const int32_t *__restrict__ offsets, int64_t nedges,
                                                                     int32_t *__restrict__ scratch, GraphOut out, int cap) {
  constexpr int kBins = 2 * kWave;  // bins looked up at a time, two neighbouring ones per lane
  __shared__ int s_before[kScanWaves][kBins], s_first[kScanWaves][kBins], s_image[kScanWaves][kBins];
  extern __shared__ __attribute__((aligned(16))) unsigned char s_hits[];  // GRAPH: per wave cap keys, then cap places in bin order
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int at = blockIdx.x * (blockDim.x / kWave) + wave;
  if (at >= nnodes) return;
  const Grid *grid = w.grid;
  const int nb0 = grid->nb[0], nb1 = grid->nb[1], nb2 = grid->nb[2];
  const int per0 = grid->periodic[0], per1 = grid->periodic[1], per2 = grid->periodic[2];
  const int r0 = grid->nscan[0], r1 = grid->nscan[1], r2 = grid->nscan[2];
  const int key = w.skey[at];
  const int4 me = w.smeta[at];
  const int i = me.x;
  const int wi[3] = {me.y, me.z, me.w};
  const double pi[3] = {w.spos[3 * static_cast<int64_t>(at)], w.spos[3 * static_cast<int64_t>(at) + 1], w.spos[3 * static_cast<int64_t>(at) + 2]};
  const int bi0 = key / (nb1 * nb2), bi1 = (key / nb2) % nb1, bi2 = key % nb2;
  const double rc2 = cutoff * cutoff;
  double c[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) c[k] = grid->cellv[k];
  const int64_t seg = MODE == Scan::kCount ? 0 : offsets[i];
  unsigned long long *hkey = reinterpret_cast<unsigned long long *>(s_hits) + wave * cap;
  int *hk = reinterpret_cast<int *>(s_hits + sizeof(*hkey) * (blockDim.x / kWave) * cap) + wave * cap;
  int count = 0;
  const int m1 = 2 * r1 + 1, m2 = 2 * r2 + 1;
  const int nscan = grid->status == 0 ? (2 * r0 + 1) * m1 * m2 : 0;
  const float per_plane = 1.0f / static_cast<float>(m1 * m2), per_row = 1.0f / static_cast<float>(m2);
  // Exact: q + 1/2 over the divisor is half of its inverse away from an integer, and q < 65^3.
  const auto quotient = [](int q, float inverse) { return static_cast<int>((static_cast<float>(q) + 0.5f) * inverse); };
  // image of the cell that bin number b of an axis lies in, b then being its number in the cell
  const auto wrap = [](int &b, int nb, int reach) {
    const int B = reach <= nb ? (b < 0 ? -1 : (b >= nb ? 1 : 0)) : floor_div(b, nb);
    b -= B * nb;
    return B;
  };
  const auto look_at = [&](int first_bin, auto per_lane) {
    // 64 or 128 bins side by side: where their atoms begin, how many there are, which image of the cell they belong to
    constexpr int U = decltype(per_lane)::value;
    int first[U], cnt[U], image[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      first[u] = cnt[u] = image[u] = 0;
      const int q = first_bin + U * lane + u;
      if (q < nscan) {
        const int q0 = quotient(q, per_plane), in_plane = q - q0 * (m1 * m2), q1 = quotient(in_plane, per_row);
        int b0 = bi0 + q0 - r0, b1 = bi1 + q1 - r1, b2 = bi2 + (in_plane - q1 * m2) - r2;
        int B0 = 0, B1 = 0, B2 = 0;
        if (per0) B0 = wrap(b0, nb0, r0);
        if (per1) B1 = wrap(b1, nb1, r1);
        if (per2) B2 = wrap(b2, nb2, r2);
        if (b0 >= 0 && b0 < nb0 && b1 >= 0 && b1 < nb1 && b2 >= 0 && b2 < nb2) {
          const int id = (b0 * nb1 + b1) * nb2 + b2;
          first[u] = w.cell_offsets[id];
          cnt[u] = w.cell_offsets[id + 1] - first[u];
          image[u] = pack_image(B0, B1, B2);
        }
      }
    }
    int upto = cnt[0] + (U == 2 ? cnt[U - 1] : 0);
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int v = __shfl_up(upto, d);
      if (lane >= d) upto += v;
    }
    const int total = __shfl(upto, kWave - 1);
    wave_lds_fence();  // the previous bins' tables have been read
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s_before[wave][U * lane + u] = upto - cnt[U - 1] - (u == U - 2 ? cnt[0] : 0);
      s_first[wave][U * lane + u] = first[u];
      s_image[wave][U * lane + u] = image[u];
    }
    wave_lds_fence();
    const auto trip = [&](int base, auto sets) {
      constexpr int kSets = decltype(sets)::value;
      int b[kSets], cand[kSets], image_of[kSets], S[kSets][3];
      int64_t k_of[kSets];
      int4 meta[kSets];
      double pj[kSets][3];
#pragma unroll
      for (int u = 0; u < kSets; ++u) b[u] = 0, cand[u] = min(base + u * kWave + lane, total - 1);
      // the last bin whose atoms begin at or before cand: it is not empty, since cand < total
#pragma unroll
      for (int step = U * kWave / 2; step > 0; step >>= 1) {
        int before[kSets];
#pragma unroll
        for (int u = 0; u < kSets; ++u) before[u] = s_before[wave][b[u] + step];
#pragma unroll
        for (int u = 0; u < kSets; ++u) b[u] += before[u] <= cand[u] ? step : 0;
      }
#pragma unroll
      for (int u = 0; u < kSets; ++u) {
        k_of[u] = s_first[wave][b[u]] + (cand[u] - s_before[wave][b[u]]);
        image_of[u] = s_image[wave][b[u]];
      }
#pragma unroll
      for (int u = 0; u < kSets; ++u) {
        meta[u] = w.smeta[k_of[u]];
#pragma unroll
        for (int k = 0; k < 3; ++k) pj[u][k] = w.spos[3 * k_of[u] + k];
      }
#pragma unroll
      for (int u = 0; u < kSets; ++u) {
        unpack_image(image_of[u], S[u]);
        S[u][0] += wi[0] - meta[u].y, S[u][1] += wi[1] - meta[u].z, S[u][2] += wi[2] - meta[u].w;
        const int j = meta[u].x;
        const bool hit = base + u * kWave + lane < total && within(pi, pj[u], S[u], c, rc2) &&
                         !(j == i && S[u][0] == 0 && S[u][1] == 0 && S[u][2] == 0);
        const unsigned long long mask = __ballot(hit);
        const int mine = count + __popcll(mask & ((1ull << lane) - 1ull));
        if constexpr (MODE == Scan::kScratch) {
          if (hit && seg + mine < nedges) {
            scratch[seg + mine] = j;
#pragma unroll
            for (int k = 0; k < 3; ++k) scratch[nedges + 3 * (seg + mine) + k] = S[u][k];
          }
        }
        if constexpr (MODE == Scan::kGraph) {
          if (hit && mine < cap) {
            hkey[mine] = order_key(j, image_of[u]);
            hk[mine] = static_cast<int>(k_of[u]);
          }
        }
        count += __popcll(mask);
      }
    };
    // the last 64 or fewer by themselves: with few candidates in all of the bins the second set would be all of the work again
    for (int base = 0; base < total; base += 2 * kWave) {
      if (total - base > kWave) trip(base, std::integral_constant<int, 2>{});
      else trip(base, std::integral_constant<int, 1>{});
    }
  };
  // a reach of one or two bins (large cells, whose bins are halved to fit the workspace): 64 at a time
  if (nscan <= kWave) look_at(0, std::integral_constant<int, 1>{});
  else
    for (int first_bin = 0; first_bin < nscan; first_bin += kBins) look_at(first_bin, std::integral_constant<int, 2>{});
  if constexpr (MODE == Scan::kCount) {
    if (lane == 0) w.degree[i] = count;
  }
  if constexpr (MODE == Scan::kGraph) {
    wave_lds_fence();
    // never below zero: where the caller's `nedges` ends before the segment begins, nothing of it is written, here neither
    const int d = max(0, min(min(count, cap), static_cast<int>(min(static_cast<int64_t>(offsets[i + 1]), nedges) - seg)));
    // up to the next multiple of four (cap is one): keys above all others
    if (lane < (-d & 3)) hkey[d + lane] = ~0ull;
    wave_lds_fence();
    auto emit = [&](int64_t to, unsigned long long key, int k) {
      const int j = static_cast<int>(key >> 24);
      const int4 meta = w.smeta[k];
      int S[3];
      unpack_image(static_cast<int>(key & 0xffffffu), S);
      S[0] += wi[0] - meta.y, S[1] += wi[1] - meta.z, S[2] += wi[2] - meta.w;
      out.row_i[to] = i;
      out.row_j[to] = j;
      out.edge_index[to] = i;
      out.edge_index[nedges + to] = j;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        out.unit_shifts[3 * to + q] = S[q];
        out.shifts[3 * to + q] = image_shift(S, c, q);
      }
    };
    // two neighbours per lane and pass over the keys
    for (int e0 = 0; e0 < d; e0 += 2 * kWave) {
      unsigned long long key[2];
      int k[2], rank[2] = {0, 0};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int e = min(e0 + u * kWave + lane, d - 1);
        key[u] = hkey[e], k[u] = hk[e];
      }
#pragma unroll 2
      for (int q = 0; q < d; q += 4) {
        unsigned long long other[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) other[v] = hkey[q + v];
#pragma unroll
        for (int v = 0; v < 4; ++v) rank[0] += other[v] < key[0] ? 1 : 0, rank[1] += other[v] < key[1] ? 1 : 0;
      }
      if (d <= 2 * kWave) {  // all of them are in registers: into their order in LDS first, then out in that order, lane by lane
        wave_lds_fence();
#pragma unroll
        for (int u = 0; u < 2; ++u)
          if (u * kWave + lane < d) hkey[rank[u]] = key[u], hk[rank[u]] = k[u];
        wave_lds_fence();
        for (int e = lane; e < d; e += kWave) emit(seg + e, hkey[e], hk[e]);
      } else {
#pragma unroll
        for (int u = 0; u < 2; ++u)
          if (e0 + u * kWave + lane < d) emit(seg + rank[u], key[u], k[u]);
      }
    }
    if (lane == 0) {
      out.first_occ[i] = offsets[i];
      out.first_occ[nnodes + i] = offsets[i + 1];
      if (out.batch) out.batch[i] = 0;
      if (at == 0) {
        if (out.ptr) out.ptr[0] = 0, out.ptr[1] = nnodes;
        if (out.ptr32) out.ptr32[0] = 0, out.ptr32[1] = nnodes;
      }
    }
  }
}

// offsets[0 .. n] = exclusive scan of degree[0 .. n-1] and, next to it, the grid's status and the largest degree; one
// workgroup, every thread a contiguous run.  `counts` (two words of host memory, may be NULL): offsets[n] in the upper half
// of the first, the largest degree and the status above bit 0 in the second, and bit 0 of each set, so that a host that
// polls them needs no order between the two stores (a release to the host would write back the whole L2 first).
__global__ __launch_bounds__(kGridThreads) void nl_offsets_kernel(Workspace w, int n, int32_t *__restrict__ offsets,
                                                                  int32_t *__restrict__ status, int32_t *__restrict__ max_degree,
                                                                  unsigned long long *__restrict__ counts) {
  __shared__ long long part[kGridThreads];
  __shared__ long long stage[kOffsetsStage];
  __shared__ int s_most[kGridThreads / kWave];
  int most = 0;
  const long long total = workgroup_exclusive_scan<kGridThreads, kOffsetsStage, long long>(
      n, stage, part, [&](int k) { return w.degree[k]; },
      [&](int k, long long before, long long value) {
        offsets[k] = static_cast<int32_t>(before > INT32_MAX ? INT32_MAX : before);
        most = max(most, static_cast<int>(value));
      });
  for (int d = kWave / 2; d > 0; d >>= 1) most = max(most, __shfl_xor(most, d));
  if (threadIdx.x % kWave == 0) s_most[threadIdx.x / kWave] = most;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int32_t pairs = static_cast<int32_t>(total > INT32_MAX ? INT32_MAX : total), state = w.grid->status;
    offsets[n] = pairs;
    if (status) *status = state;
    for (int q = 1; q < kGridThreads / kWave; ++q) most = max(most, s_most[q]);
    if (max_degree) *max_degree = most;
    if (counts) {
      const auto word = [](int32_t high, int32_t low) {
        return static_cast<unsigned long long>(static_cast<uint32_t>(high)) << 32 | static_cast<unsigned long long>(low) << 1 | 1ull;
      };
      __hip_atomic_store(counts, word(pairs, 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(counts + 1, word(most, state), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// One wavefront per atom: every hit of its segment goes to its rank under the (j, S) order.
__global__ __launch_bounds__(256) void nl_rank_kernel(const int32_t *__restrict__ offsets, int nnodes, int64_t nedges,
                                                      const int32_t *__restrict__ scratch, int32_t *__restrict__ row_i,
                                                      int32_t *__restrict__ row_j, int32_t *__restrict__ unit_shifts) {
  const int lane = threadIdx.x % kWave;
  const int i = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (i >= nnodes) return;
  const int64_t e0 = offsets[i];
  const int64_t e1 = min(static_cast<int64_t>(offsets[i + 1]), nedges);
  const int32_t *sj = scratch;
  const int32_t *sS = scratch + nedges;
  for (int64_t e = e0 + lane; e < e1; e += kWave) {
    const int j = sj[e];
    const int32_t S[3] = {sS[3 * e], sS[3 * e + 1], sS[3 * e + 2]};
    int rank = 0;
    for (int64_t q = e0; q < e1; ++q) rank += key_less(sj[q], sS + 3 * q, j, S) ? 1 : 0;
    const int64_t at = e0 + rank;
    row_i[at] = i;
    row_j[at] = j;
    unit_shifts[3 * at + 0] = S[0];
    unit_shifts[3 * at + 1] = S[1];
    unit_shifts[3 * at + 2] = S[2];
  }
}

// The view of a list sorted by row j, for a list that holds the reverse (j, i, -S) of each of its pairs (i, j, S), as every
// list of this file does: the pairs sent by s are then the reverses of the pairs of s, in the order of (j, -S), so the view's
// offsets are the list's own and an entry is found by a binary search in the segment of j.  One launch in place of a
// counting sort's five.
__device__ __forceinline__ int compare_pair(int ja, double a0, double a1, double a2, int jb, const double *Sb) {
  if (ja != jb) return ja < jb ? -1 : 1;
  if (a0 != Sb[0]) return a0 < Sb[0] ? -1 : 1;
  if (a1 != Sb[1]) return a1 < Sb[1] ? -1 : 1;
  if (a2 != Sb[2]) return a2 < Sb[2] ? -1 : 1;
  return 0;
}
__global__ __launch_bounds__(256) void nl_sender_view_kernel(const int32_t *__restrict__ row_i, const int32_t *__restrict__ row_j,
                                                             const double *__restrict__ unit_shifts,
                                                             const int32_t *__restrict__ first_occ, int nnodes, int64_t nedges,
                                                             int32_t *__restrict__ perm) {
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (e >= nedges) return;
  const int i = row_i[e], j = row_j[e];
  const bool good = static_cast<unsigned>(i) < static_cast<unsigned>(nnodes) && static_cast<unsigned>(j) < static_cast<unsigned>(nnodes);
  if (!good) {  // not a list of this file: some place, inside the view
    perm[e] = static_cast<int32_t>(e);
    return;
  }
  const double s0 = -unit_shifts[3 * e], s1 = -unit_shifts[3 * e + 1], s2 = -unit_shifts[3 * e + 2];
  int lo = first_occ[j], hi = first_occ[nnodes + j];
  clamp_edge_range(lo, hi, nedges);
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (compare_pair(i, s0, s1, s2, row_j[mid], unit_shifts + 3 * static_cast<int64_t>(mid)) > 0)
      lo = mid + 1;
    else
      hi = mid;
  }
  // images of one neighbour come in the opposite order
  int a0 = first_occ[i], b0 = first_occ[nnodes + i];
  clamp_edge_range(a0, b0, nedges);
  int64_t a = e, b = e;
  while (a > a0 && row_j[a - 1] == j) --a;
  while (b + 1 < b0 && row_j[b + 1] == j) ++b;
  perm[a + (b - e)] = static_cast<int32_t>(min(static_cast<int64_t>(lo), nedges - 1));
}

// ---- the test a Verlet list needs before it is reused: how far has any atom moved since the list was built ----
__global__ void clear_u64_kernel(unsigned long long *out) { *out = 0ull; }

// Non-negative doubles order like their bit patterns, so the maximum over the grid is an integer atomic.
__global__ __launch_bounds__(256) void max_displacement_kernel(const double *__restrict__ positions,
                                                               const double *__restrict__ reference, int64_t nnodes,
                                                               unsigned long long *__restrict__ out) {
#pragma clang fp contract(off)  // squares and sums as written, like the accept test of the list itself
  double worst = 0.0;
  for (int64_t n = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; n < nnodes;
       n += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const double d0 = positions[3 * n + 0] - reference[3 * n + 0];
    const double d1 = positions[3 * n + 1] - reference[3 * n + 1];
    const double d2 = positions[3 * n + 2] - reference[3 * n + 2];
    const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
    worst = r2 > worst ? r2 : worst;  // a NaN coordinate is caught below
    if (!(r2 == r2)) worst = __builtin_inf();
  }
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const double other = __shfl_down(worst, off);
    worst = other > worst ? other : worst;
  }
  if (threadIdx.x % kWave == 0) atomicMax(out, static_cast<unsigned long long>(__double_as_longlong(worst)));
}

}  // namespace
}  // namespace cm

extern "C" int cm_max_displacement(const double *positions, const double *reference, int64_t nnodes, double *out_sq,
                                   cm_stream_t stream) {
  CM_REQUIRE(nnodes >= 0, "cm_max_displacement: negative size");
  CM_REQUIRE(out_sq && (nnodes == 0 || (positions && reference)), "cm_max_displacement: NULL pointer");
  hipStream_t st = cm::as_stream(stream);
  unsigned long long *out = reinterpret_cast<unsigned long long *>(out_sq);
  hipLaunchKernelGGL(cm::clear_u64_kernel, dim3(1), dim3(1), 0, st, out);
  if (nnodes > 0) {
    const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(cm::ceil_div(nnodes, 256), 1024));
    hipLaunchKernelGGL(cm::max_displacement_kernel, dim3(blocks), dim3(256), 0, st, positions, reference, nnodes, out);
  }
  return cm::check_launch("cm_max_displacement");
}

extern "C" size_t cm_neighbour_list_workspace(int64_t nnodes, int64_t max_cells) {
  if (nnodes < 0 || max_cells < 1) return 0;
  return cm::carve(nullptr, nnodes, max_cells).total;
}

namespace cm {
namespace {

// Everything up to the offsets of the segments: the cell list and the count of every atom's neighbours.
int search(const double *positions, const double *cell, int pbc_x, int pbc_y, int pbc_z, double cutoff, int64_t nnodes, int64_t max_cells,
           void *workspace, size_t workspace_bytes, int32_t *offsets, int32_t *status, int32_t *max_degree,
           unsigned long long *counts, hipStream_t st, const char *what) {
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 4, "%s: nnodes out of range", what);
  CM_REQUIRE(max_cells >= 1 && max_cells < INT32_MAX / 2, "%s: max_cells out of range", what);
  CM_REQUIRE(cutoff > 0.0 && std::isfinite(cutoff), "%s: cutoff must be positive and finite", what);
  CM_REQUIRE(offsets != nullptr && (status != nullptr || counts != nullptr), "%s: offsets / status is NULL", what);
  CM_REQUIRE(nnodes == 0 || positions != nullptr, "%s: positions is NULL", what);
  CM_REQUIRE(cell != nullptr || !(pbc_x || pbc_y || pbc_z), "%s: a periodic axis needs a cell", what);
  const Workspace w = carve(workspace, nnodes, max_cells);
  if (workspace == nullptr || workspace_bytes < w.total) {
    set_error("%s: workspace of %zu bytes, need %zu", what, workspace_bytes, w.total);
    return CM_ENOSPC;
  }
  const int n = static_cast<int>(nnodes), cells = static_cast<int>(max_cells);
  if (n <= kSmallAtoms && cells <= kSmallAtoms) {
    hipLaunchKernelGGL(nl_cells_small_kernel, dim3(1), dim3(kGridThreads), static_cast<unsigned>(cells * sizeof(int)), st, positions, cell,
                       pbc_x, pbc_y, pbc_z, cutoff, n, cells, w);
  } else {
    const dim3 per_atom(static_cast<unsigned>(ceil_div(std::max(n, 1), 256))), block(256);
    hipLaunchKernelGGL(nl_grid_kernel, dim3(1), dim3(kGridThreads), 0, st, positions, cell, pbc_x, pbc_y, pbc_z, cutoff, n, cells, w.grid);
    hipLaunchKernelGGL(nl_clear_kernel, dim3(static_cast<unsigned>(ceil_div(cells, 256))), block, 0, st, w.cell_count, cells);
    hipLaunchKernelGGL(nl_bin_kernel, per_atom, block, 0, st, positions, n, w);
    hipLaunchKernelGGL(nl_cell_scan_kernel, dim3(1), dim3(kGridThreads), 0, st, cells, w);
    hipLaunchKernelGGL(nl_place_kernel, per_atom, block, 0, st, positions, n, w);
  }
  if (n > 0)
    hipLaunchKernelGGL(nl_scan_kernel<Scan::kCount>, dim3(static_cast<unsigned>(ceil_div(n, kScanWaves))), dim3(kScanWaves * kWave), 0, st,
                       w, cutoff, n, static_cast<const int32_t *>(nullptr), int64_t{0}, static_cast<int32_t *>(nullptr), GraphOut{}, 0);
  hipLaunchKernelGGL(nl_offsets_kernel, dim3(1), dim3(kGridThreads), 0, st, w, n, offsets, status, max_degree, counts);
  return check_launch(what);
}

}  // namespace
}  // namespace cm

extern "C" int cm_neighbour_list_count(const double *positions, const double *cell, int pbc_x, int pbc_y, int pbc_z,
                                       double cutoff, int64_t nnodes, int64_t max_cells, void *workspace,
                                       size_t workspace_bytes, int32_t *offsets, int32_t *status, cm_stream_t stream) {
  return cm::search(positions, cell, pbc_x, pbc_y, pbc_z, cutoff, nnodes, max_cells, workspace, workspace_bytes, offsets, status, nullptr,
                    nullptr, cm::as_stream(stream), "cm_neighbour_list_count");
}

extern "C" int cm_neighbour_list_fill(const double *positions, double cutoff, int64_t nnodes, int64_t max_cells,
                                      const void *workspace, const int32_t *offsets, int64_t nedges, int32_t *edge_scratch,
                                      int32_t *row_i, int32_t *row_j, int32_t *unit_shifts, cm_stream_t stream) {
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 4, "cm_neighbour_list_fill: nnodes out of range");
  CM_REQUIRE(max_cells >= 1 && max_cells < INT32_MAX / 2, "cm_neighbour_list_fill: max_cells out of range");
  CM_REQUIRE(nedges >= 0 && nedges < INT32_MAX / 4, "cm_neighbour_list_fill: nedges out of range");
  CM_REQUIRE(cutoff > 0.0 && std::isfinite(cutoff), "cm_neighbour_list_fill: cutoff must be positive and finite");
  if (nnodes == 0 || nedges == 0) return CM_OK;
  CM_REQUIRE(positions && workspace && offsets && edge_scratch && row_i && row_j && unit_shifts,
             "cm_neighbour_list_fill: NULL pointer");
  const cm::Workspace w = cm::carve(const_cast<void *>(workspace), nnodes, max_cells);
  hipStream_t st = cm::as_stream(stream);
  const int n = static_cast<int>(nnodes);
  const dim3 grid(static_cast<unsigned>(cm::ceil_div(n, cm::kScanWaves))), block(cm::kScanWaves * cm::kWave);
  hipLaunchKernelGGL(cm::nl_scan_kernel<cm::Scan::kScratch>, grid, block, 0, st, w, cutoff, n, offsets, nedges, edge_scratch,
                     cm::GraphOut{}, 0);
  hipLaunchKernelGGL(cm::nl_rank_kernel, grid, block, 0, st, offsets, n, nedges, edge_scratch, row_i, row_j, unit_shifts);
  return cm::check_launch("cm_neighbour_list_fill");
}

extern "C" int cm_neighbour_list_search(const double *positions, const double *cell, int pbc_x, int pbc_y, int pbc_z,
                                        double cutoff, int64_t nnodes, int64_t max_cells, void *workspace,
                                        size_t workspace_bytes, int32_t *offsets, int32_t *status, int32_t *max_degree,
                                        cm_stream_t stream) {
  CM_REQUIRE(max_degree != nullptr, "cm_neighbour_list_search: max_degree is NULL");
  return cm::search(positions, cell, pbc_x, pbc_y, pbc_z, cutoff, nnodes, max_cells, workspace, workspace_bytes, offsets, status,
                    max_degree, nullptr, cm::as_stream(stream), "cm_neighbour_list_search");
}

// The host needs three numbers before it can ask for the list's memory.  The kernel writes them into host memory itself and
// the host polls for them: the copy of three words and the wait for it took 12 us longer (2 000 atoms: search, list and step 393
// -> 376 us with this and with what the host allocates before the wait in place of after it).  A search that has not ended after two
// milliseconds sits behind other work of the stream, where that does not matter, and the host waits for the stream.  The call
// returns once the device is done with `counts`, whatever it returns.
extern "C" int cm_neighbour_list_search_counts(const double *positions, const double *cell, int pbc_x, int pbc_y, int pbc_z,
                                               double cutoff, int64_t nnodes, int64_t max_cells, void *workspace,
                                               size_t workspace_bytes, int32_t *offsets, int64_t *counts, int32_t *values,
                                               cm_stream_t stream) {
  static const char *what = "cm_neighbour_list_search_counts";
  CM_REQUIRE(counts != nullptr && values != nullptr, "%s: counts / values is NULL", what);
  hipStream_t st = cm::as_stream(stream);
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  CM_REQUIRE(hipStreamIsCapturing(st, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone,
             "%s: the host has to read the number of pairs, which a stream under capture does not deliver", what);
  uint64_t word[2];
  const auto landed = [&] {
    for (int k = 0; k < 2; ++k) word[k] = static_cast<uint64_t>(__atomic_load_n(counts + k, __ATOMIC_ACQUIRE));
    return (word[0] & word[1] & 1) != 0;
  };
  for (int k = 0; k < 2; ++k) __atomic_store_n(counts + k, int64_t{0}, __ATOMIC_RELEASE);
  int rc = cm::search(positions, cell, pbc_x, pbc_y, pbc_z, cutoff, nnodes, max_cells, workspace, workspace_bytes, offsets, nullptr, nullptr,
                      reinterpret_cast<unsigned long long *>(counts), st, what);
  if (rc == CM_EINVAL || rc == CM_ENOSPC) return rc;  // nothing was launched
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
  while (rc == CM_OK && !landed() && std::chrono::steady_clock::now() < until) {
  }
  if (rc != CM_OK || !landed()) {
    const hipError_t err = hipStreamSynchronize(st);
    if (rc != CM_OK) return rc;
    if (err != hipSuccess || !landed()) {
      cm::set_error("%s: %s", what, hipGetErrorString(err));
      return CM_ELAUNCH;
    }
  }
  values[0] = static_cast<int32_t>(word[0] >> 32);
  values[1] = static_cast<int32_t>(static_cast<uint32_t>(word[1]) >> 1);
  values[2] = static_cast<int32_t>(word[1] >> 32);
  return CM_OK;
}

// A wave keeps a segment's hits in LDS, 12 bytes each: four waves per workgroup up to 512 of them, then one.
static constexpr int kGraphMaxDegree = 8192;

extern "C" int cm_neighbour_list_graph_max_degree(void) { return kGraphMaxDegree; }

extern "C" int cm_neighbour_list_graph(double cutoff, int64_t nnodes, int64_t max_cells, const void *workspace, const int32_t *offsets,
                                       int64_t nedges, int max_degree, int32_t *row_i, int32_t *row_j, int64_t *edge_index,
                                       double *unit_shifts, double *shifts, int32_t *first_occ, int64_t *batch, int64_t *ptr,
                                       int32_t *ptr32, cm_stream_t stream) {
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 4, "cm_neighbour_list_graph: nnodes out of range");
  CM_REQUIRE(max_cells >= 1 && max_cells < INT32_MAX / 2, "cm_neighbour_list_graph: max_cells out of range");
  CM_REQUIRE(nedges >= 0 && nedges < INT32_MAX / 4, "cm_neighbour_list_graph: nedges out of range");
  CM_REQUIRE(max_degree >= 0 && max_degree <= kGraphMaxDegree, "cm_neighbour_list_graph: %d neighbours of one atom, at most %d", max_degree,
             kGraphMaxDegree);
  CM_REQUIRE(cutoff > 0.0 && std::isfinite(cutoff), "cm_neighbour_list_graph: cutoff must be positive and finite");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(workspace && offsets && first_occ, "cm_neighbour_list_graph: NULL pointer");
  CM_REQUIRE(nedges == 0 || (row_i && row_j && edge_index && unit_shifts && shifts), "cm_neighbour_list_graph: NULL edge output");
  const cm::Workspace w = cm::carve(const_cast<void *>(workspace), nnodes, max_cells);
  const int n = static_cast<int>(nnodes);
  const int cap = std::max(kGraphMaxDegree > max_degree ? (max_degree + 63) / 64 * 64 : max_degree, 64);
  const int waves = cap <= 512 ? cm::kScanWaves : 1;
  hipLaunchKernelGGL(cm::nl_scan_kernel<cm::Scan::kGraph>, dim3(static_cast<unsigned>(cm::ceil_div(n, waves))), dim3(waves * cm::kWave),
                     static_cast<unsigned>(waves * cap * 12), cm::as_stream(stream), w, cutoff, n, offsets, nedges,
                     static_cast<int32_t *>(nullptr), cm::GraphOut{row_i, row_j, edge_index, unit_shifts, shifts, first_occ, batch, ptr, ptr32},
                     cap);
  return cm::check_launch("cm_neighbour_list_graph");
}

extern "C" int cm_symmetric_sender_view(const int32_t *row_i, const int32_t *row_j, const double *unit_shifts,
                                        const int32_t *first_occ, int64_t nnodes, int64_t nedges, int32_t *sender_perm,
                                        cm_stream_t stream) {
  CM_REQUIRE(nnodes >= 0 && nnodes < INT32_MAX / 4 && nedges >= 0 && nedges < INT32_MAX / 4, "cm_symmetric_sender_view: sizes out of range");
  if (nedges == 0) return CM_OK;
  CM_REQUIRE(row_i && row_j && unit_shifts && first_occ && sender_perm, "cm_symmetric_sender_view: NULL pointer");
  hipLaunchKernelGGL(cm::nl_sender_view_kernel, dim3(static_cast<unsigned>(cm::ceil_div(nedges, 256))), dim3(256), 0,
                     cm::as_stream(stream), row_i, row_j, unit_shifts, first_occ, static_cast<int>(nnodes), nedges, sender_perm);
  return cm::check_launch("cm_symmetric_sender_view");
}
