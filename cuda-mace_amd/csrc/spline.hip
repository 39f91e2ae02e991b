// Tabulated radial functions (natural cubic spline): evaluation and its derivative-weighted sum.
// The coefficient table ([nknots-1, 4, J], 2 MB at J = 512) stays in L2; the forward is a pure
// write stream of R[E, J], the backward a pure read stream of grad_R[E, J].
#include <algorithm>
#include <initializer_list>

#include "common.hpp"

namespace cm {
namespace {

__device__ __forceinline__ int knot_index(float r, float r_width, int nknots) {
  int idx = static_cast<int>(r / r_width);
  return idx < 0 ? 0 : (idx > nknots - 2 ? nknots - 2 : idx);
}

// One thread per four consecutive outputs of one edge.
template <bool DERIV>
__global__ void spline_forward_kernel(const float *__restrict__ r, const float *__restrict__ r_knots,
                                      const float *__restrict__ coeffs, int64_t nedges, int nknots, int J,
                                      float r_width, float r_max, float *__restrict__ R_out,
                                      float *__restrict__ R_deriv) {
  const int J4 = J / 4;
  const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (t >= nedges * J4) return;
  const int64_t e = t / J4;
  const int j = static_cast<int>(t - e * J4) * 4;
  const float re = r[e];
  f4 val = zero4(), der = zero4();
  if (re <= r_max) {
    const int idx = knot_index(re, r_width, nknots);
    const float x = re - r_knots[idx];
    const float *cp = coeffs + static_cast<int64_t>(idx) * 4 * J + j;
    const f4 a = ld4(cp), b = ld4(cp + J), c = ld4(cp + 2 * J), d = ld4(cp + 3 * J);
    val = a + x * (b + x * (c + x * d));
    if (DERIV) der = b + x * (2.f * c + (3.f * x) * d);
  }
  st4(R_out + e * J + j, val);
  if (DERIV) st4_stream(R_deriv + e * J + j, der);
}

// ---- LDS-table variant of the forward for long edge lists --------------------------------------------------------
// The kernel above pulls the four coefficient vectors of every output through L1 (64 bytes read for 16 written); with
// the 2 MB table spread over all intervals nothing of it stays in a 32 KB L1, so the compute unit's L1 path carries four
// times the bytes of the HBM write stream and sets the pace.  Here a workgroup owns 32 consecutive outputs (one
// 128-byte line of every edge's row) and keeps their coefficients for EVERY interval in LDS ([interval][4][32]
// floats, 512 bytes per interval, a row of zeros behind the last one for edges beyond the cutoff; 139 KB at most); it
// then walks its share of the edges, eight lanes per edge (16 bytes each), eight edges per wave and trip, and each wave
// store writes eight whole lines (4.0 -> 5.2 TB/s at 1.3 million edges x 512 outputs; stores that scatter whole lines
// over rows do not reach what a contiguous stream does).  The workgroups of one
// output slice sit `nslices` apart in the grid, so at any time all slices, hence all parts of a row, are being written.
// The rows are written through the caches: message passing reads them next, from the Infinity Cache as far as they fit there (122 880
// edges x 384 outputs, 189 MB: this kernel 42 -> 37.5 us, the message passing after it 43 -> 39; at 1.6 GB no difference).
constexpr int kSpThreads = 512;
constexpr int kSpSlice = 32;            // outputs per workgroup
constexpr int kSpMaxIntervals = 272;    // rows of the slice, the row of zeros included: 272 * 4 * 32 * 4 B = 139 264 B of LDS
constexpr int64_t kSpMinEdges = 1 << 15;

__global__ __launch_bounds__(kSpThreads) void spline_forward_sliced_kernel(
    const float *__restrict__ r, const float *__restrict__ r_knots, const float *__restrict__ coeffs, int64_t nedges,
    int nknots, int J, float r_width, float r_max, float *__restrict__ R_out, int nslices, int share) {
  __shared__ __attribute__((aligned(16))) float sTab[kSpMaxIntervals * 4 * kSpSlice];
  __shared__ float sKnots[kSpMaxIntervals + 1];
  const int tid = threadIdx.x;
  const int slice = blockIdx.x % nslices;
  const int part = blockIdx.x / nslices;
  const int j0 = slice * kSpSlice;
  // 16-byte pieces: row = 4 * interval + coefficient, eight pieces per row (J is a multiple of 4: a piece is inside the
  // table or beyond it as a whole)
  for (int t = tid; t < (nknots - 1) * 4 * (kSpSlice / 4); t += kSpThreads) {
    const int row = t >> 3, q = t & 7;
    const int j = j0 + 4 * q;
    *reinterpret_cast<f4 *>(sTab + row * kSpSlice + 4 * q) = j < J ? ld4(coeffs + static_cast<int64_t>(row) * J + j) : zero4();
  }
  if (tid < 4 * (kSpSlice / 4)) *reinterpret_cast<f4 *>(sTab + (nknots - 1) * 4 * kSpSlice + 4 * tid) = zero4();  // row of zeros
  for (int t = tid; t < nknots; t += kSpThreads) sKnots[t] = r_knots[t];
  __syncthreads();

  const int lane = tid % kWave;
  const int q = lane & 7;   // 16-byte piece of the slice
  const int g = lane >> 3;  // edge of a trip
  const int j = j0 + 4 * q;
  const bool inside = j < J;  // false in the last slice of a row that is no multiple of 32 wide
  const char *tab = reinterpret_cast<const char *>(sTab) + 16 * q;
  const unsigned zero_row = static_cast<unsigned>(nknots - 1) * (4 * kSpSlice * 4);
  // A wave takes 64 consecutive edges per round: every lane prepares one of them (interval, offset inside it; an edge
  // beyond the cutoff points at the row of zeros), then eight trips of eight edges, each lane fetching its trip's edge
  // from the lane that prepared it.  The radii of the wave's next round are requested before the trips.
  const int64_t rounds = (nedges + kWave - 1) / kWave;
  const int64_t stride = static_cast<int64_t>(share) * (kSpThreads / kWave);
  int64_t round = static_cast<int64_t>(part) * (kSpThreads / kWave) + tid / kWave;
  if (round >= rounds) return;
  const int64_t last = nedges - 1;
  float re = r[min(round * kWave + lane, last)];
  for (; round < rounds; round += stride) {
    const int64_t nxt = round + stride < rounds ? round + stride : round;
    const float re_next = r[min(nxt * kWave + lane, last)];
    const bool live = re <= r_max;
    const int idx = knot_index(re, r_width, nknots);
    const unsigned off = live ? static_cast<unsigned>(idx) * (4 * kSpSlice * 4) : zero_row;
    const float x = live ? re - sKnots[idx] : 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int src = 8 * t + g;
      const char *row = tab + __shfl(off, src);
      const float xs = __shfl(x, src);
      const f4 a = *reinterpret_cast<const f4 *>(row), b = *reinterpret_cast<const f4 *>(row + 128),
               c = *reinterpret_cast<const f4 *>(row + 256), d = *reinterpret_cast<const f4 *>(row + 384);
      const int64_t e = round * kWave + src;
      if (inside && e <= last) st4(R_out + e * J + j, a + xs * (b + xs * (c + xs * d)));
    }
    re = re_next;
  }
}

bool spline_sliced_applies(int64_t nedges, int nknots, int J) {
  return nedges >= kSpMinEdges && nknots - 1 < kSpMaxIntervals && ceil_div(J, kSpSlice) <= device_compute_units();
}

void launch_spline_forward_sliced(const float *r, const float *r_knots, const float *coeffs, int64_t nedges, int nknots, int J,
                                  float r_width, float r_max, float *R_out, hipStream_t st) {
  const int nslices = static_cast<int>(ceil_div(J, kSpSlice));
  const int share = device_compute_units() / nslices;
  hipLaunchKernelGGL(spline_forward_sliced_kernel, dim3(static_cast<unsigned>(nslices * share)), dim3(kSpThreads), 0, st, r,
                     r_knots, coeffs, nedges, nknots, J, r_width, r_max, R_out, nslices, share);
}

// One wavefront per edge: grad_r[e] = sum_j grad_R[e, j] * dR/dr[e, j].
__global__ __launch_bounds__(256) void spline_backward_kernel(
    const float *__restrict__ r, const float *__restrict__ r_knots, const float *__restrict__ coeffs,
    const float *__restrict__ gR, int64_t nedges, int nknots, int J, float r_width, float r_max,
    float *__restrict__ gr) {
  const int lane = threadIdx.x % kWave;
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x / kWave) + threadIdx.x / kWave;
  if (e >= nedges) return;
  const float re = r[e];
  float sum = 0.f;
  if (re <= r_max) {
    const int idx = knot_index(re, r_width, nknots);
    const float x = re - r_knots[idx];
    const float *cp = coeffs + static_cast<int64_t>(idx) * 4 * J;
    const float *gp = gR + e * J;
    f4 acc = zero4();
    for (int j = 4 * lane; j < J; j += 4 * kWave) {
      const f4 b = ld4(cp + J + j), c = ld4(cp + 2 * J + j), d = ld4(cp + 3 * J + j);
      acc += ld4_stream(gp + j) * (b + x * (2.f * c + (3.f * x) * d));
    }
    sum = hsum4(acc);
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if (lane == 0) gr[e] = sum;
}

// ---- backward from 32 768 edges on: edges in the order of their knot intervals --------------------------------------
// The kernel above reads 48 bytes of coefficients for every 16 bytes of the gradient stream, from L2, and that traffic is what
// bounds it.  Here a workgroup of 16 waves, one per compute unit, takes a
// chunk of consecutive edges and serves them in the order of their intervals (a counting sort in LDS): the edges it works
// on at a time share a few rows of the table, which stay in L1.  Half a wave serves an edge, ITER 16-byte pieces of the row
// per lane, all of them requested before the first is used (up to 512 outputs: beyond, 512 at a time; two edges at a time
// where a row is one piece per lane: 122 880 x 128 29.7 -> 18.9 us).  An edge's sum does not depend on its place in the order.
// Which of the two it is from 32 768 edges on: see spline_backward_sliced_from.
constexpr int kSpSortThreads = 1024;
constexpr int kSpSortChunk = 4096;  // edges of a chunk: their place in it takes 12 bits
constexpr int kSpSortBins = 256;
constexpr int kSpSortMaxKnots = 1 << 20;  // the interval takes the other 20 bits of a word

template <int ITER>
__global__ __launch_bounds__(kSpSortThreads) void spline_backward_sorted_kernel(
    const float *__restrict__ r, const float *__restrict__ r_knots, const float *__restrict__ coeffs,
    const float *__restrict__ gR, int64_t nedges, int nknots, int J, float r_width, float r_max, float *__restrict__ gr, int chunk) {
  __shared__ float sX[kSpSortChunk];
  __shared__ unsigned sEdge[kSpSortChunk];  // interval << 12 | place in the chunk
  __shared__ __attribute__((aligned(16))) int sHist[kSpSortBins];
  __shared__ int sCount;
  constexpr int kPer = kSpSortChunk / kSpSortThreads;
  const int tid = threadIdx.x;
  const int lane = tid % 32, slot = tid / 32;  // an edge's lanes
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) * chunk;
  const int n = static_cast<int>(min(static_cast<int64_t>(chunk), nedges - c0));
  if (tid < kSpSortBins) sHist[tid] = 0;
  __syncthreads();
  int bin[kPer];
  unsigned word[kPer];
  float x[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int i = tid + q * kSpSortThreads;
    bin[q] = -1;
    if (i >= n) continue;
    const float re = r[c0 + i];
    if (re <= r_max) {
      const int idx = knot_index(re, r_width, nknots);
      x[q] = re - r_knots[idx];
      word[q] = static_cast<unsigned>(idx) << 12 | static_cast<unsigned>(i);
      bin[q] = idx * kSpSortBins / (nknots - 1);
      atomicAdd(&sHist[bin[q]], 1);
    } else {
      gr[c0 + i] = 0.f;
    }
  }
  __syncthreads();
  if (tid < kWave) {  // places of the bins, four per lane
    int4 c = reinterpret_cast<int4 *>(sHist)[tid];
    const int mine = c.x + c.y + c.z + c.w;
    int upto = mine;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int below = __shfl_up(upto, d);
      upto += tid >= d ? below : 0;
    }
    const int first = upto - mine;
    reinterpret_cast<int4 *>(sHist)[tid] = make_int4(first, first + c.x, first + c.x + c.y, first + c.x + c.y + c.z);
    if (tid == kWave - 1) sCount = upto;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    if (bin[q] < 0) continue;
    const int at = atomicAdd(&sHist[bin[q]], 1);
    sX[at] = x[q];
    sEdge[at] = word[q];
  }
  __syncthreads();

  const int count = sCount;
  if constexpr (ITER > 1) {
    // A row within one trip of the pieces: the next edge's row of the gradient stream is on its way while this one is worked on (two rows
    // ahead were no faster).  us, without -> with: 122 880 x 256 37.2 -> 35.7, x 384 52.9 -> 51.9, x 512 65.2 -> 63.9; 300 000 x 256 76.4 -> 71.6; 450 000 x 512
    // 213 -> 207; 33 000 x 384 21.2 -> 20.3.  Rows of one piece have two edges in flight already, longer ones four pieces.
    if (J <= 128 * ITER) {
      constexpr int kSlots = kSpSortThreads / 32;
      const int first = slot & ~1;  // the wave's first place: its two halves leave together
      if (first >= count) return;
      f4 g[2][ITER];
      auto request = [&](int p, f4 (&into)[ITER]) {  // beyond the last edge: the last one once more
        const float *gp = gR + (c0 + (sEdge[min(p, count - 1)] & (kSpSortChunk - 1))) * J;
#pragma unroll
        for (int i = 0; i < ITER; ++i) {
          const int j = 128 * i + 4 * lane;
          into[i] = ld4_stream(gp + (j < J ? j : 0));
        }
      };
      request(slot, g[0]);
      for (int base = 0; first + base < count; base += 2 * kSlots) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int p = slot + base + u * kSlots;
          if (first + base + u * kSlots >= count) break;
          const unsigned w = sEdge[min(p, count - 1)];
          const float xe = sX[min(p, count - 1)];
          const float *cp = coeffs + (static_cast<int64_t>(w >> 12) * 4 + 1) * J;
          f4 b[ITER], c[ITER], d[ITER], acc = zero4();
#pragma unroll
          for (int i = 0; i < ITER; ++i) {
            const int j = 128 * i + 4 * lane, at = j < J ? j : 0;
            b[i] = ld4(cp + at), c[i] = ld4(cp + J + at), d[i] = ld4(cp + 2 * J + at);
          }
          __builtin_amdgcn_sched_barrier(0);
          request(p + kSlots, g[1 - u]);  // behind this edge's coefficients, which are waited for first
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < ITER; ++i) {
            const f4 v = g[u][i] * (b[i] + xe * (2.f * c[i] + (3.f * xe) * d[i]));
            acc += 128 * i + 4 * lane < J ? v : zero4();
          }
          float sum = hsum4(acc);
#pragma unroll
          for (int off = 16; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
          if (lane == 0 && p < count) gr[c0 + (w & (kSpSortChunk - 1))] = sum;
        }
      }
      return;
    }
  }
  if constexpr (ITER == 2 || ITER == 3) return;  // their rows are never longer
  constexpr int kEdges = ITER == 1 ? 2 : 1;  // of a slot at a time
  for (int p = kEdges * slot; p < count; p += kEdges * (kSpSortThreads / 32)) {
    unsigned w[kEdges];
    float xs[kEdges];
    int64_t e[kEdges];
    f4 acc[kEdges];
#pragma unroll
    for (int u = 0; u < kEdges; ++u) {
      const int at = min(p + u, count - 1);  // beyond the last edge: the last one once more
      w[u] = sEdge[at], xs[u] = sX[at];
      e[u] = c0 + (w[u] & (kSpSortChunk - 1));
      acc[u] = zero4();
    }
    for (int j0 = 0; j0 < J; j0 += 128 * ITER) {
      f4 g[kEdges][ITER], b[kEdges][ITER], c[kEdges][ITER], d[kEdges][ITER];
#pragma unroll
      for (int u = 0; u < kEdges; ++u) {
        const float *cp = coeffs + (static_cast<int64_t>(w[u] >> 12) * 4 + 1) * J, *gp = gR + e[u] * J;
#pragma unroll
        for (int i = 0; i < ITER; ++i) {
          const int j = j0 + 128 * i + 4 * lane, at = j < J ? j : 0;
          g[u][i] = ld4_stream(gp + at), b[u][i] = ld4(cp + at), c[u][i] = ld4(cp + J + at), d[u][i] = ld4(cp + 2 * J + at);
        }
      }
#pragma unroll
      for (int u = 0; u < kEdges; ++u)
#pragma unroll
        for (int i = 0; i < ITER; ++i) {
          const f4 v = g[u][i] * (b[u][i] + xs[u] * (2.f * c[u][i] + (3.f * xs[u]) * d[u][i]));
          acc[u] += j0 + 128 * i + 4 * lane < J ? v : zero4();
        }
    }
#pragma unroll
    for (int u = 0; u < kEdges; ++u) {
      float sum = hsum4(acc[u]);
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
      if (lane == 0) gr[e[u]] = sum;
    }
  }
}

void launch_spline_backward_sorted(const float *r, const float *r_knots, const float *coeffs, const float *gR, int64_t nedges,
                                   int nknots, int J, float r_width, float r_max, float *gr, hipStream_t st) {
  const int64_t cus = device_compute_units();
  const int64_t rounds = ceil_div(nedges, cus * kSpSortChunk);  // chunks per compute unit
  const int chunk = static_cast<int>(ceil_div(nedges, cus * rounds));
  const dim3 grid(static_cast<unsigned>(ceil_div(nedges, chunk))), block(kSpSortThreads);
#define CM_SORTED(ITER_) \
  hipLaunchKernelGGL(spline_backward_sorted_kernel<ITER_>, grid, block, 0, st, r, r_knots, coeffs, gR, nedges, nknots, J, r_width, r_max, gr, chunk)
  switch (std::min<int64_t>(ceil_div(J, 128), 4)) {
    case 1: CM_SORTED(1); break;
    case 2: CM_SORTED(2); break;
    case 3: CM_SORTED(3); break;
    default: CM_SORTED(4); break;
  }
#undef CM_SORTED
}

// ---- LDS-table variant of the backward for the longest lists and for short rows --------------------------------------------------
// Even in the order of the intervals the coefficients pass through L1, 48 bytes for every 16 of the gradient stream.  Here a workgroup owns a chunk of consecutive edges and sums them slice by slice: for each slice of 32
// outputs it loads the derivative's coefficients (b, 2c, 3d per interval: 384 bytes, 104 KB at most) into LDS, streams
// that slice of its edges' gradient rows (one 128-byte line per edge) and adds each edge's partial sum to the edge's
// cell in LDS; after the last slice the cells go to grad_r.  One lane group adds to a cell per slice, and the slices
// follow each other in a fixed order (workgroup b starts at slice b % nslices, so that at any time all parts of the
// rows are being read): the result is reproducible.  The table is re-read from L2 once per slice and chunk, a sixth of
// the bytes of the gradient stream at 5 000 edges per chunk.
constexpr int kSpBwdRow = 3 * kSpSlice;  // floats per interval
constexpr int kSpBwdChunk = 8192;        // edges per chunk at most (their sums: 32 KB of LDS)

__global__ __launch_bounds__(kSpThreads) void spline_backward_sliced_kernel(
    const float *__restrict__ r, const float *__restrict__ r_knots, const float *__restrict__ coeffs,
    const float *__restrict__ gR, int64_t nedges, int nknots, int J, float r_width, float r_max, float *__restrict__ gr,
    int nslices, int chunk) {
  __shared__ __attribute__((aligned(16))) float sTab[kSpMaxIntervals * kSpBwdRow];
  __shared__ float sKnots[kSpMaxIntervals + 1];
  __shared__ float sSum[kSpBwdChunk];
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = tid / kWave;
  const int q = lane & 7;   // 16-byte piece of the slice
  const int g = lane >> 3;  // edge of a trip
  const char *tab = reinterpret_cast<const char *>(sTab) + 16 * q;
  const unsigned zero_row = static_cast<unsigned>(nknots - 1) * (kSpBwdRow * 4);
  for (int t = tid; t < nknots; t += kSpThreads) sKnots[t] = r_knots[t];

  for (int64_t c0 = static_cast<int64_t>(blockIdx.x) * chunk; c0 < nedges; c0 += static_cast<int64_t>(gridDim.x) * chunk) {
    const int n = static_cast<int>(min(static_cast<int64_t>(chunk), nedges - c0));
    for (int t = tid; t < n; t += kSpThreads) sSum[t] = 0.f;
    for (int pass = 0; pass < nslices; ++pass) {
      const int slice = static_cast<int>((blockIdx.x + static_cast<unsigned>(pass)) % static_cast<unsigned>(nslices));
      const int j0 = slice * kSpSlice;
      __syncthreads();  // the table of the previous slice is no longer read (and the sums are cleared)
      for (int t = tid; t < (nknots - 1) * 3 * (kSpSlice / 4); t += kSpThreads) {
        const int row = t >> 3, piece = t & 7;
        const int idx = row / 3, k = row - 3 * idx;  // k = 0, 1, 2: b, 2 c, 3 d
        const int j = j0 + 4 * piece;
        const f4 v = j < J ? ld4(coeffs + (static_cast<int64_t>(idx) * 4 + k + 1) * J + j) : zero4();
        *reinterpret_cast<f4 *>(sTab + row * kSpSlice + 4 * piece) = static_cast<float>(k + 1) * v;
      }
      if (tid < 3 * (kSpSlice / 4)) *reinterpret_cast<f4 *>(sTab + (nknots - 1) * kSpBwdRow + 4 * tid) = zero4();  // row of zeros
      __syncthreads();
      const int j = j0 + 4 * q;
      const bool inside = j < J;
      const int jc = inside ? j : 0;  // lanes beyond the row read its first piece and drop it
      for (int base = wave * kWave; base < n; base += kSpThreads) {
        // every lane prepares one of the round's 64 edges
        const float re = r[c0 + min(base + lane, n - 1)];
        const bool live = re <= r_max;
        const int idx = knot_index(re, r_width, nknots);
        const unsigned off = live ? static_cast<unsigned>(idx) * (kSpBwdRow * 4) : zero_row;
        const float x = live ? re - sKnots[idx] : 0.f;
        f4 gv[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)  // unconditional: an edge beyond the chunk reads the chunk's last edge and is dropped
          gv[t] = ld4_stream(gR + (c0 + min(base + 8 * t + g, n - 1)) * J + jc);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int src = 8 * t + g;
          const unsigned o = __shfl(off, src);
          const float xs = __shfl(x, src);
          const char *row = tab + o;
          const f4 b = *reinterpret_cast<const f4 *>(row), c2 = *reinterpret_cast<const f4 *>(row + 128),
                   d3 = *reinterpret_cast<const f4 *>(row + 256);
          float part = hsum4(gv[t] * (b + xs * (c2 + xs * d3)));
          part = (inside && o != zero_row) ? part : 0.f;  // an edge beyond the cutoff contributes nothing, whatever its gradient
          part += __shfl_xor(part, 1);
          part += __shfl_xor(part, 2);
          part += __shfl_xor(part, 4);
          if (q == 0 && base + src < n) sSum[base + src] += part;  // this lane alone adds to the cell in this slice; slices are barriers apart
        }
      }
    }
    __syncthreads();
    for (int t = tid; t < n; t += kSpThreads) gr[c0 + t] = sSum[t];
    __syncthreads();
  }
}

void launch_spline_backward_sliced(const float *r, const float *r_knots, const float *coeffs, const float *gR, int64_t nedges,
                                   int nknots, int J, float r_width, float r_max, float *gr, hipStream_t st) {
  const int cus = device_compute_units();
  const int64_t per_group = ceil_div(ceil_div(nedges, cus), kSpBwdChunk);  // chunks per workgroup
  const int chunk = static_cast<int>(ceil_div(ceil_div(nedges, cus * per_group), kWave) * kWave);  // <= kSpBwdChunk, whole rounds
  const int groups = static_cast<int>(std::min<int64_t>(cus, ceil_div(nedges, chunk)));
  hipLaunchKernelGGL(spline_backward_sliced_kernel, dim3(static_cast<unsigned>(groups)), dim3(kSpThreads), 0, st, r, r_knots,
                     coeffs, gR, nedges, nknots, J, r_width, r_max, gr, static_cast<int>(ceil_div(J, kSpSlice)), chunk);
}

// Edges from which the LDS-table kernel is the faster one.  It pays a fixed 3 to 6 us per slice of 32 outputs (staging, less with
// fewer knots) and then for the outputs there are; the kernel in the order of the intervals pays for what its lanes span, 128
// outputs or a multiple, beyond 512 a multiple of 512, and half a wave per edge however short the row.  So the line falls with the
// square of the part of the span that a row fills; but not below 2^19 edges where its sums are the longer chains (error against fp64,
// in the order of the intervals / LDS table: 32 outputs 6.89e-8 / 6.64e-8, 128 8.06 / 7.84, 192 8.46 / 8.35, 256 8.54 / 8.89, 512 8.88 /
// 10.2, 1 024 9.62 / 12.6).  Measured, in the order of the intervals / LDS table (us), 256 knots:
//   4 outputs  33 000 5.5 / 6.7, 60 000 7.2 / 6.9, 300 000 29.7 / 11.4      32 40 000 6.9 / 6.8, 300 000 35 / 13    64 90 000 12.9 / 13.5, 110 000 15.3 / 14.0
//   96   200 000 27.6 / 28.7, 250 000 33.2 / 30.1         128 400 000 52.9 / 54.6, 500 000 65.5 / 61.1
//   160  200 000 44.5 / 45.9, 250 000 54 / 48             192 250 000 55.5 / 56.7, 350 000 76 / 73       256 700 000 160 / 162, 800 000 181 / 176
//   320  400 000 126 / 134, 500 000 155 / 152             448 400 000 170 / 184, 500 000 213 / 209       512 700 000 315 / 330, 800 000 362 / 351
//   640  250 000 186 / 191, 350 000 258 / 245             768 400 000 316 / 344, 600 000 476 / 457       1 024 800 000 728 / 748, 900 000 828 / 808
// and with 32 knots 128 200 000 28.5 / 29.5, 400 000 53 / 47; 512 300 000 128 / 141, 600 000 256 / 248; 1 024 600 000 500 / 492.
inline int64_t spline_backward_sliced_from(int nknots, int J) {
  const int span = J <= 512 ? static_cast<int>(ceil_div(J, 128) * 128) : static_cast<int>(ceil_div(J, 512) * 512);
  const double part = 32.0 * static_cast<double>(ceil_div(J, 32)) / span;
  const double most = span == 128 ? 430e3 : (span > 512 ? 850e3 : (part == 1.0 ? 720e3 : 600e3));
  const int64_t line = static_cast<int64_t>(most * part * part * (290 + nknots) / 546.0);
  return std::max<int64_t>(line, span > 256 ? 1 << 19 : 40000);
}

// fp64 variants (the reference dispatches the spline on float and double, jit_wrappers/src/cubic_spline_wrapper.cpp:50,
// :123): same knot lookup and Horner forms as above.
__device__ __forceinline__ int knot_index(double r, double r_width, int nknots) {
  int idx = static_cast<int>(r / r_width);
  return idx < 0 ? 0 : (idx > nknots - 2 ? nknots - 2 : idx);
}

// One thread per output: for short rows and few of them.
template <bool DERIV>
__global__ void spline_forward_f64_kernel(const double *__restrict__ r, const double *__restrict__ r_knots,
                                          const double *__restrict__ coeffs, int64_t nedges, int nknots, int J,
                                          double r_width, double r_max, double *__restrict__ R_out,
                                          double *__restrict__ R_deriv) {
  const int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (t >= nedges * J) return;
  const int64_t e = t / J;
  const int j = static_cast<int>(t - e * J);
  const double re = r[e];
  double val = 0.0, der = 0.0;
  if (re <= r_max) {
    const int idx = knot_index(re, r_width, nknots);
    const double x = re - r_knots[idx];
    const double *cp = coeffs + static_cast<int64_t>(idx) * 4 * J + j;
    const double a = cp[0], b = cp[J], c = cp[2 * J], d = cp[3 * J];
    val = a + x * (b + x * (c + x * d));
    if (DERIV) der = b + x * (2.0 * c + (3.0 * x) * d);
  }
  R_out[t] = val;
  if (DERIV) R_deriv[t] = der;
}

// A wave per edge, VEC consecutive outputs per lane and trip: what depends on the edge alone (the interval, a division in fp64)
// is formed once per edge instead of once per output, which with the split of a flat index into edge and output had been the
// forward's bound, and 16-byte loads and stores halve the L1 path's instructions.  30 000 edges x 256 outputs forward 28.9 ->
// 13.3 us, backward 18.7 -> 13.8 (its stream 11.6), 30 000 x 512 52.5 -> 23.8 and 31.5 -> 24.8, 100 000 x 256 86 -> 39 and 53 -> 43; below some
// two thousand edges the backward with pairs is half a microsecond behind (1 000 x 256 4.5 -> 5.0), so they take one at a time.
// In the forward the edge's number is a scalar: all edges inside the cutoff / half of them, when every lane had formed the edge's
// part and rows were read beyond the cutoff too -> now (us), 30 000 x 256 13.2 / 12.7 -> 12.2 / 11.0, 300 000 x 64 59 / 58 -> 45 / 35,
// 300 000 x 128 68 / 67 -> 57 / 44, 300 000 x 256 124 / 113 -> 114 / 107, 100 000 x 512 78 / 73 -> 77 / 75; with the derivative as a second output, where two streams of
// stores set the pace, 100 000 x 512 143 / 144 -> 142 / 147, 300 000 x 128 91 / 89 -> 92 / 103.
template <int VEC>
struct Doubles {
  typedef double type __attribute__((ext_vector_type(VEC)));
};
template <int VEC>
__device__ __forceinline__ typename Doubles<VEC>::type ldd(const double *p) {
  return *reinterpret_cast<const typename Doubles<VEC>::type *>(p);
}
// KEEP: through the caches, for rows that the next kernel finds in the Infinity Cache (kKeepBytes); else past them
template <int VEC, bool KEEP>
__device__ __forceinline__ void std_out(double *p, typename Doubles<VEC>::type v) {
  typedef typename Doubles<VEC>::type dv;
  if constexpr (KEEP)
    *reinterpret_cast<dv *>(p) = v;
  else
    __builtin_nontemporal_store(v, reinterpret_cast<dv *>(p));
}
// This kernel and the message passing after it, us, past the caches -> through them, 12 and 40 edges per node: 60 MB of rows, 32 channels 48.2 -> 48.2 and 36.1 -> 36.1,
// 64 37.2 -> 36.9 and 36.6 -> 36.2, 128 34.8 -> 34.1 and 37.3 -> 36.1, 192 40.4 -> 38.3 and 40.6 -> 40.0, 256 43.9 -> 40.5 and 43.3 -> 42.6; 20 MB the same to
// 3 less.  The wider the row the more this kernel itself loses (75 MB, 256 channels 21.9 -> 27.1), and from there on it is more than the next one gains: 75 MB, 64 channels
// 44.1 -> 43.4, 160 42.0 -> 45.3, 256 49.3 -> 54.3; 90 MB, 64 43.9 -> 45.5, 128 48.4 -> 50.2, 256 56.2 -> 64.3; 120 MB, 64 62.1 -> 66.4, 256 64.4 -> 75.2; 200 MB,
// 64 84.0 -> 82.3, 128 87.3 -> 90.8, 192 90.7 -> 104.9; 300 MB, 64 127 -> 122, 192 130 -> 145, 256 142 -> 165.
constexpr int64_t kKeepBytes = int64_t{64} << 20;

template <int VEC, bool KEEP>
__global__ __launch_bounds__(256) void spline_forward_f64_wave_kernel(const double *__restrict__ r, const double *__restrict__ r_knots,
                                                                      const double *__restrict__ coeffs, int64_t nedges, int nknots, int J,
                                                                      double r_width, double r_max, double *__restrict__ R_out,
                                                                      double *__restrict__ R_deriv) {
  typedef typename Doubles<VEC>::type dv;
  const int lane = threadIdx.x % kWave;
  // one edge for the whole wave, which the compiler is told: its length comes by a scalar load, the cutoff is a scalar branch
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (e >= nedges) return;
  const double re = r[e];
  if (!(re <= r_max)) {  // beyond the cutoff (or no number): zeros, and no row of the table is read
#pragma unroll 1
    for (int j = VEC * lane; j < J; j += VEC * kWave) {
      std_out<VEC, KEEP>(R_out + e * J + j, dv{});
      if (R_deriv) std_out<VEC, false>(R_deriv + e * J + j, dv{});
    }
    return;
  }
  const int idx = knot_index(re, r_width, nknots);
  const double x = re - r_knots[idx];
  const double *cp = coeffs + static_cast<int64_t>(idx) * 4 * J;
#pragma unroll 1
  for (int j = VEC * lane; j < J; j += VEC * kWave) {
    const dv a = ldd<VEC>(cp + j), b = ldd<VEC>(cp + J + j), c = ldd<VEC>(cp + 2 * J + j), d = ldd<VEC>(cp + 3 * J + j);
    std_out<VEC, KEEP>(R_out + e * J + j, a + x * (b + x * (c + x * d)));
    if (R_deriv) std_out<VEC, false>(R_deriv + e * J + j, b + x * (2.0 * c + (3.0 * x) * d));
  }
}

template <int VEC>
__global__ __launch_bounds__(256) void spline_backward_f64_kernel(
    const double *__restrict__ r, const double *__restrict__ r_knots, const double *__restrict__ coeffs,
    const double *__restrict__ gR, int64_t nedges, int nknots, int J, double r_width, double r_max,
    double *__restrict__ gr) {
  typedef typename Doubles<VEC>::type dv;
  const int lane = threadIdx.x % kWave;
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x / kWave) + threadIdx.x / kWave;
  if (e >= nedges) return;
  const double re = r[e];
  double sum = 0.0;
  if (re <= r_max) {
    const int idx = knot_index(re, r_width, nknots);
    const double x = re - r_knots[idx];
    const double *cp = coeffs + static_cast<int64_t>(idx) * 4 * J;
    const double *gp = gR + e * J;
    dv acc{};
#pragma unroll 1
    for (int j = VEC * lane; j < J; j += VEC * kWave)
      acc += ldd<VEC>(gp + j) * (ldd<VEC>(cp + J + j) + x * (2.0 * ldd<VEC>(cp + 2 * J + j) + (3.0 * x) * ldd<VEC>(cp + 3 * J + j)));
#pragma unroll
    for (int k = 0; k < VEC; ++k) sum += acc[k];
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  if (lane == 0) gr[e] = sum;
}

// whether rows of J doubles behind these pointers are read and written 16 bytes at a time: where their alignment allows it and
// from 2 048 edges on
inline bool pairs_of_doubles(int64_t nedges, int J, std::initializer_list<const void *> pointers) {
  if (J % 2 != 0 || nedges < 2048) return false;
  for (const void *p : pointers)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
  return true;
}

// Whether the forward gives an edge a wave.  A trip of the wave, 64 or 128 outputs, costs what some 45 threads with an output each
// do, and below some 700 000 outputs there are too few waves for their trips, one after the other, to cover each other.  Measured,
// a thread per output -> a wave per edge (us): pairs, one trip, 300 000 x 4 6.6 -> 45, x 24 28 -> 45, x 40 43.5 -> 44.7, x 48 51 -> 45,
// 30 000 x 40 6.6 -> 7.0, x 48 7.8 -> 7.3; single outputs, two trips, 300 000 x 81 84 -> 84, x 97 99 -> 85, 30 000 x 81 11.0 -> 12.0, x 97
// 12.5 -> 12.3; three, 30 000 x 129 15.7 -> 15.9, x 161 19.0 -> 16.2; few rows, 1 000 x 512 4.3 -> 5.4, 2 000 x 225 4.8 -> 5.4, 10 000 x 64
// 4.8 -> 5.3, 10 000 x 97 5.9 -> 6.1, 10 000 x 128 7.0 -> 4.6.  The launch counts its threads in 32 bits: 64 per edge here.
inline bool wave_per_edge_f64(int64_t nedges, int J, bool pairs) {
  const int64_t trips = ceil_div(J, pairs ? 2 * kWave : kWave);
  return J >= 48 * trips - 4 && nedges * J >= 700000 && nedges < (int64_t{1} << 32) / kWave - kWave;
}

}  // namespace
}  // namespace cm

extern "C" int cm_spline_forward(const float *r, const float *r_knots, const float *coeffs, int64_t nedges,
                                 int nknots, int noutputs, float r_width, float r_max, float *R_out,
                                 float *R_deriv, cm_stream_t stream) {
  CM_REQUIRE(nedges >= 0, "cm_spline_forward: negative size");
  CM_REQUIRE(nknots >= 2, "cm_spline_forward: need at least two knots, got %d", nknots);
  CM_REQUIRE(noutputs > 0 && noutputs % 4 == 0, "cm_spline_forward: noutputs=%d must be a positive multiple of 4", noutputs);
  CM_REQUIRE(r_width > 0.f, "cm_spline_forward: r_width must be positive");
  if (nedges == 0) return CM_OK;
  CM_REQUIRE(r && r_knots && coeffs && R_out, "cm_spline_forward: NULL pointer");
  // With the derivative as a second output the direct kernel below writes two streams per set of coefficient loads and
  // reaches 6.3 TB/s at 1.3 million edges x 512 outputs; the LDS-table kernel's line-by-line stores stay at 5.2 TB/s.
  if (!R_deriv && cm::spline_sliced_applies(nedges, nknots, noutputs)) {
    cm::launch_spline_forward_sliced(r, r_knots, coeffs, nedges, nknots, noutputs, r_width, r_max, R_out, cm::as_stream(stream));
    return cm::check_launch("cm_spline_forward");
  }
  const int block = 256;
  const int64_t threads = nedges * (noutputs / 4);
  CM_REQUIRE(cm::ceil_div(threads, block) < INT32_MAX, "cm_spline_forward: problem too large for one launch");
  const dim3 grid(static_cast<unsigned>(cm::ceil_div(threads, block)));
  if (R_deriv)
    hipLaunchKernelGGL(cm::spline_forward_kernel<true>, grid, dim3(block), 0, cm::as_stream(stream), r, r_knots, coeffs,
                       nedges, nknots, noutputs, r_width, r_max, R_out, R_deriv);
  else
    hipLaunchKernelGGL(cm::spline_forward_kernel<false>, grid, dim3(block), 0, cm::as_stream(stream), r, r_knots, coeffs,
                       nedges, nknots, noutputs, r_width, r_max, R_out, R_deriv);
  return cm::check_launch("cm_spline_forward");
}

extern "C" int cm_spline_backward_kernel(int64_t nedges, int nknots, int noutputs) {
  if (nknots < 2 || noutputs < 1) return 0;
  if (cm::spline_sliced_applies(nedges, nknots, noutputs) && nedges >= cm::spline_backward_sliced_from(nknots, noutputs)) return 2;
  return nedges >= cm::kSpMinEdges && nknots <= cm::kSpSortMaxKnots ? 1 : 0;
}

extern "C" int cm_spline_backward(const float *r, const float *r_knots, const float *coeffs, const float *grad_R,
                                  int64_t nedges, int nknots, int noutputs, float r_width, float r_max,
                                  float *grad_r, cm_stream_t stream) {
  CM_REQUIRE(nedges >= 0, "cm_spline_backward: negative size");
  CM_REQUIRE(nknots >= 2, "cm_spline_backward: need at least two knots, got %d", nknots);
  CM_REQUIRE(noutputs > 0 && noutputs % 4 == 0, "cm_spline_backward: noutputs=%d must be a positive multiple of 4", noutputs);
  CM_REQUIRE(r_width > 0.f, "cm_spline_backward: r_width must be positive");
  if (nedges == 0) return CM_OK;
  CM_REQUIRE(r && r_knots && coeffs && grad_R && grad_r, "cm_spline_backward: NULL pointer");
  const int kernel = cm_spline_backward_kernel(nedges, nknots, noutputs);
  if (kernel == 2) {
    cm::launch_spline_backward_sliced(r, r_knots, coeffs, grad_R, nedges, nknots, noutputs, r_width, r_max, grad_r,
                                      cm::as_stream(stream));
    return cm::check_launch("cm_spline_backward");
  }
  if (kernel == 1) {
    cm::launch_spline_backward_sorted(r, r_knots, coeffs, grad_R, nedges, nknots, noutputs, r_width, r_max, grad_r,
                                      cm::as_stream(stream));
    return cm::check_launch("cm_spline_backward");
  }
  const int block = 256;
  const int per = block / cm::kWave;
  hipLaunchKernelGGL(cm::spline_backward_kernel, dim3(static_cast<unsigned>(cm::ceil_div(nedges, per))), dim3(block), 0,
                     cm::as_stream(stream), r, r_knots, coeffs, grad_R, nedges, nknots, noutputs, r_width, r_max, grad_r);
  return cm::check_launch("cm_spline_backward");
}

extern "C" int cm_spline_forward_f64(const double *r, const double *r_knots, const double *coeffs, int64_t nedges,
                                     int nknots, int noutputs, double r_width, double r_max, double *R_out,
                                     double *R_deriv, cm_stream_t stream) {
  CM_REQUIRE(nedges >= 0, "cm_spline_forward_f64: negative size");
  CM_REQUIRE(nknots >= 2, "cm_spline_forward_f64: need at least two knots, got %d", nknots);
  CM_REQUIRE(noutputs > 0, "cm_spline_forward_f64: noutputs=%d must be positive", noutputs);
  CM_REQUIRE(r_width > 0.0, "cm_spline_forward_f64: r_width must be positive");
  if (nedges == 0) return CM_OK;
  CM_REQUIRE(r && r_knots && coeffs && R_out, "cm_spline_forward_f64: NULL pointer");
  const int block = 256;
  const int64_t threads = nedges * noutputs;
  CM_REQUIRE(cm::ceil_div(threads, block) < INT32_MAX, "cm_spline_forward_f64: problem too large for one launch");
  const bool pairs = cm::pairs_of_doubles(nedges, noutputs, {coeffs, R_out, R_deriv});
  const bool waves = cm::wave_per_edge_f64(nedges, noutputs, pairs);
  const dim3 grid(static_cast<unsigned>(cm::ceil_div(waves ? nedges * cm::kWave : threads, block)));
  const bool keep = threads * 8 <= cm::kKeepBytes;
#define CM_FORWARD_F64(KERNEL)                                                                                               \
  hipLaunchKernelGGL(KERNEL, grid, dim3(block), 0, cm::as_stream(stream), r, r_knots, coeffs, nedges, nknots, noutputs, r_width, \
                     r_max, R_out, R_deriv)
  if (waves && pairs && keep) CM_FORWARD_F64((cm::spline_forward_f64_wave_kernel<2, true>));
  else if (waves && pairs) CM_FORWARD_F64((cm::spline_forward_f64_wave_kernel<2, false>));
  else if (waves) CM_FORWARD_F64((cm::spline_forward_f64_wave_kernel<1, false>));
  else if (R_deriv) CM_FORWARD_F64(cm::spline_forward_f64_kernel<true>);
  else CM_FORWARD_F64(cm::spline_forward_f64_kernel<false>);
#undef CM_FORWARD_F64
  return cm::check_launch("cm_spline_forward_f64");
}

extern "C" int cm_spline_backward_f64(const double *r, const double *r_knots, const double *coeffs, const double *grad_R,
                                      int64_t nedges, int nknots, int noutputs, double r_width, double r_max,
                                      double *grad_r, cm_stream_t stream) {
  CM_REQUIRE(nedges >= 0, "cm_spline_backward_f64: negative size");
  CM_REQUIRE(nknots >= 2, "cm_spline_backward_f64: need at least two knots, got %d", nknots);
  CM_REQUIRE(noutputs > 0, "cm_spline_backward_f64: noutputs=%d must be positive", noutputs);
  CM_REQUIRE(r_width > 0.0, "cm_spline_backward_f64: r_width must be positive");
  if (nedges == 0) return CM_OK;
  CM_REQUIRE(r && r_knots && coeffs && grad_R && grad_r, "cm_spline_backward_f64: NULL pointer");
  const int block = 256;
  const int per = block / cm::kWave;
  const dim3 grid(static_cast<unsigned>(cm::ceil_div(nedges, per)));
  if (cm::pairs_of_doubles(nedges, noutputs, {coeffs, grad_R}))
    hipLaunchKernelGGL(cm::spline_backward_f64_kernel<2>, grid, dim3(block), 0, cm::as_stream(stream), r, r_knots, coeffs, grad_R, nedges,
                       nknots, noutputs, r_width, r_max, grad_r);
  else
    hipLaunchKernelGGL(cm::spline_backward_f64_kernel<1>, grid, dim3(block), 0, cm::as_stream(stream), r, r_knots, coeffs, grad_R, nedges,
                       nknots, noutputs, r_width, r_max, grad_r);
  return cm::check_launch("cm_spline_backward_f64");
}
