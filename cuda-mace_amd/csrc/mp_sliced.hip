// Forward message passing from edge vectors with the radial table in LDS.
//
//   out[n, m, c] = sum_{e -> n} X[sender[e], c] * Y_m(vec[e]) * R(|vec[e]|)[l(m), c]
//
// The kernels in mp_spline.hip give a wave one receiver node and all 16 components; per edge a lane fetches its 16
// coefficient pieces of the cubic (8 KB per edge over the wave) through L1, and that path is what bounds them.  Here the work is cut the other way: a workgroup owns two degrees, (0, 3) or (1, 2) -- eight components either
// way, so every workgroup has the same work per edge -- and one slice of 16 channels, and the part of the table it
// needs, (nknots - 1) x 4 coefficients x 2 degrees x 16 channels = 130 KB at 256 knots (147 KB as it is laid out), stays in its LDS for the whole
// launch.  One workgroup per compute unit; the workgroups of a (pair, slice) split the node range evenly.
//
// Inside a workgroup a quad of four lanes serves one receiver node, four channels per lane, so a wave works on 16 nodes
// at once.  Edges are taken four at a time: lane k of the quad loads edge k of the block, computes its length, knot
// interval, offset and the eight harmonics, and in step j of the block the whole quad handles edge j: the X row piece of
// its sender is one contiguous 64 bytes over the quad.  The edge's values reach the other lanes once per block: the
// offset inside the interval and the eight harmonics of the block's four edges are gathered over the quad by one matrix
// instruction each (quad_gather below), after which every lane holds them for all four steps in plain registers; the two
// byte offsets of an edge (table row, X row) come from lane j through a quad permutation of the DPP operand of the
// address addition, once per step.
//
// LDS layout of the table slice: interval idx at 576 idx bytes; inside it the (a, b, c, d) of degree li (0 / 1: first / second of
// the pair), channel 4 k + d of the slice at 256 li + 64 d + 16 k: the four lanes of a quad read 64 contiguous bytes.  A 16-byte
// LDS read is served 16 lanes, i.e. four quads with unrelated intervals, at a time, and takes as many cycles as quads meet
// in a quarter of the banks.  With rows a multiple of the bank span apart all four meet; at 576 bytes the quarter is (d +
// idx) mod 4, and 2.1 meet on average.  Two orders of the channels for quads at odd and even places hold it to two, with X
// rows in two 8-byte loads (which cost the L1 path twice what one of 16 bytes does) or with exchanges in registers, and four
// orders to one: 25 000 x 52 x 128 257 us with two loads, 247 with exchanges, 236 with the rows 576 bytes apart (and the
// table's pieces at constant offsets from one address); 96 channels 202 / 198 / 187, 192 (40 000) 618 / 600 / 582, 64 channels
// with ten neighbours 29.3 / 28.4 / 26.3; four orders by exchanges 256 at 128 channels.
//
// Everything is requested ahead into registers that the step before has just used up, so that none that a load is still on
// its way into has to be copied (a copy would wait for the load): the sender and vector of a lane's edge one block ahead, the X
// piece of an edge when the edge at its place of the block before is done, the table pieces of a channel (both degrees, 32
// bytes) two channels ahead, as soon as those in their place have been multiplied with X.  That is 168 registers, three
// waves per SIMD.  With X rows two blocks ahead, prepared edges and vectors in three rotating sets and all pieces of a step
// together it was 250, and two waves do not cover each other's waits: 25 000 x 52 x 128 246 -> 238 us, 5 000 x 96 50.4 -> 45.9,
// 10 007 x 160 135 -> 128, 40 000 x 192 610 -> 600, 10 752 x 10 x 64 26.1 -> 21.3 (of which 1.5 by the pieces of the table that a
// thread stages being requested four at a time), 2 000 x 52 x 128 28.3 -> 26.0, 12 000 x 256 even; with six neighbours 12 000 x 256
// 63 -> 66.  Of the 238 us 128 channels take 217 with every X row in L1, 231 with edges of one length (no bank conflicts), 188
// with both.  The instruction scheduler, left to itself, moves each request down to the end of the block (it shortens the life
// of the landing registers); scheduling barriers keep every request in its place.
//
// Receiver nodes differ in their edge counts and the 16 nodes of a wave advance together, so a workgroup sorts its nodes
// (2 816 at a time) by their number of edge blocks and its waves draw 16 neighbours of that order at a time from a
// counter in LDS.  Which wave serves a node does not change the node's result: a node's edges are summed in list order, in
// two chains (even and odd places) that are added up at the end; error of the message against fp64 at 52 neighbours, one chain -> two, and of the kernels
// with one wave per node: 96 channels 2.68e-7 -> 2.54e-7 (2.70e-7), 128 2.73 -> 2.59 (2.74), 192 2.67 -> 2.52 (2.69), 256
// 2.81 -> 2.67 (2.83).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mp_common.hpp"
#include "sh_device.hpp"

namespace cm {
namespace mp {
namespace {

constexpr int kSlThreads = 768;       // three waves per SIMD, which 168 registers allow
constexpr unsigned kSlRowBytes = 576;  // of a knot interval: 512 and a quarter of the bank span
constexpr int kSlMaxIntervals = 272;   // 153 KB of table (one row of it is the row of zeros)
constexpr int kSlSub = 2816;          // nodes sorted at a time: what LDS holds next to the largest table
constexpr int kSlBins = 64;           // edge blocks per node that the sort tells apart
// From nearly five rounds of 16 nodes per workgroup on (2 432 nodes at 64 channels, 1 216 at 128; three to four at 160 to 256, see the numbers below); below
// that most of its waves have none.  From there on the edges decide: a workgroup spends 3 us on its slice of the table, and
// nodes with few edges leave it with the fixed part of a round, while the kernel with one wave per node pays per edge.
// Measured, the launch alone, one wave per node -> this one (us), nodes x neighbours:
//   32 channels   2 600 x 52 19.2 -> 22.8, 4 000 x 10 14.7 -> 11.5, 4 000 x 52 25.1 -> 22.7, 12 000 x 2 30.9 -> 17.4: always
//   64            2 000 x 52 22.8 -> 23.3, 2 560 x 10 12.0 -> 12.2, 2 560 x 25 18.2 -> 16.9, 2 560 x 52 29.2 -> 24.9, 4 000 x 10 15.7 -> 13.5
//   96            1 700 x 15 12.1 -> 13.5, 1 700 x 52 27.4 -> 24.9, 3 000 x 4 10.5 -> 12.4, 3 000 x 15 18.8 -> 17.9, 8 000 x 4 19.9 -> 20.4, 8 000
//                 x 15 40.4 -> 30.6
//   128           1 000 x 52 22.6 -> 22.3, 1 300 x 15 12.5 -> 13.9, 1 300 x 25 16.9 -> 16.4, 1 700 x 15 14.4 -> 14.6, 3 000 x 5 13.4 -> 14.7,
//                 3 000 x 10 17.6 -> 17.0, 6 000 x 5 21.2 -> 20.7, 12 000 x 2.8 27.0 -> 29.9, 12 000 x 5 34.9 -> 33.4, 16 000 x 3.8 35.1 -> 37.4
//   160           500 x 52 23.0 -> 22.0, 800 x 7 11.7 -> 11.8, 800 x 15 16.0 -> 13.8, 800 x 52 31.5 -> 24.2, 1 200 x 7 12.7 -> 12.0, 3 000 x 7 20.5 -> 18.4
//   192           500 x 52 19.5 -> 22.7, 800 x 7 11.4 -> 12.2, 800 x 15 16.3 -> 14.3, 1 200 x 7 12.2 -> 13.2, 3 000 x 7 20.6 -> 20.4
//   224           721 x 8 13.9 -> 16.4, 600 x 15 16.0 -> 15.9, 2 000 x 10 22.5 -> 22.2, 12 000 x 4 57.0 -> 53.4 (an earlier form, a few per
//                 cent slower)
//   256           650 x 9.5 13.0 -> 13.7, 650 x 14 16.8 -> 15.2, 700 x 24 23.2 -> 17.6, 700 x 28 (in two parts) 17.6 -> 18.1, 1 000 x 9.3 15.5 -> 15.4, 1 700 x 8
//                 18.2 -> 19.1, 2 500 x 7.3 21.0 -> 21.4, 4 000 x 6 26.2 -> 26.8, 4 000 x 7 29.9 -> 28.1, 8 000 x 6 42.9 -> 44.7, 8 000 x 7 47.4 -> 46.6,
//                 12 000 x 6 60.6 -> 62.8, 12 000 x 7 67.8 -> 66.9
// Launched over and over by itself it finds its output in the last-level cache.  Inside a step it does not, and writes that reach
// memory as the 64-byte pieces of rows that a workgroup's 16 channels are cost more per node than few neighbours win back: from
// several thousand nodes on the line is a number of neighbours, and beyond 256 MB of output, what that cache holds, one that grows
// with the logarithm of the output (up to 64 channels it does not come to that).  Energies alone, the whole call, one wave per node
// -> this one, us:
//   96   25 000 x 4.9 408 -> 409, x 7 425 -> 419, 45 000 x 4.8 712 -> 715, x 7 742 -> 734
//   128  6 000 x 5 169 -> 170, 20 000 x 4.9 416 -> 415, 30 000 x 5 615 -> 623, x 7 646 -> 638, 50 000 x 9.3 1 132 -> 1 187, x 13 1 214 -> 1 205
//   160  12 000 x 2.6 377 -> 382, x 4.8 392 -> 385, 25 000 x 4.9 772 -> 776, 40 000 x 7 1 187 -> 1 228, x 13 1 329 -> 1 278
//   192  6 000 x 6 260 -> 263, x 8.4 272 -> 270, 20 000 x 6 715 -> 750, x 8.3 745 -> 746, 35 000 x 10 1 257 -> 1 297, x 14 1 336 -> 1 323
//   224  6 000 x 2.8 305 -> 311, x 5 316 -> 310, 12 000 x 4.8 528 -> 528, 20 000 x 7 878 -> 881, 35 000 x 7 1 500 -> 1 545, x 13 1 661 -> 1 586
//   256  3 000 x 7 236 -> 240, x 9.5 244 -> 243, 12 000 x 9.3 629 -> 636, x 15 700 -> 677, 20 000 x 7 981 -> 1 031, x 15 1 121 -> 1 100, 35 000 x 11.5 1 825 ->
//        1 889, x 15 1 931 -> 1 902
// With forces:
//   128  35 000 x 6 1 548 -> 1 545, 60 000 x 8.3 2 696 -> 2 752, x 10.5 2 880 -> 2 881, 100 000 x 10.4 4 904 -> 4 990, x 13 5 154 -> 5 133
//   192  20 000 x 8.3 1 509 -> 1 510, 35 000 x 8.2 2 516 -> 2 543, x 10.4 2 670 -> 2 670, 60 000 x 8.3 4 270 -> 4 328, x 13 4 793 -> 4 743, 100 000 x 10.4 7 572 -> 7 700,
//        x 16 8 652 -> 8 485
//   224  35 000 x 6 3 000 -> 3 012, x 8.2 3 206 -> 3 164, 60 000 x 6 5 115 -> 5 130, x 8.3 5 454 -> 5 368
//   256  6 000 x 8.4 765 -> 778, x 16 882 -> 880, 12 000 x 8.2 1 279 -> 1 318, x 13 1 408 -> 1 393, 20 000 x 8.3 2 055 -> 2 076, x 13 2 272 -> 2 249, 60 000 x 10.5 6 442 ->
//        6 559, x 16 7 247 -> 7 153, 80 000 x 13 9 053 -> 9 270, x 19 10 491 -> 10 346
// The lines as they were redrawn when the other kernel's nodes came to be cut into up to six parts, steps with forces, one wave per node (or
// part) -> this one, us: 160 540 x 52 214.9 -> 205.6, x 26 178.4 -> 173.7, 420 x 52 192.6 -> 194.8; 192 560 x 52 224.8 -> 221.8, x 26 185.0 ->
// 186.5; 224 400 x 52 234.7 -> 224.0, x 26 201.1 -> 197.1, 60 molecules of 21 (8.8 neighbours) 277.5 -> 271.8; 256 560 x 52 273.3 -> 266.4, x 26
// 226.1 -> 227.0, 500 x 52 247.4 -> 250.2, molecules of 21: 96 398.9 -> 389.4, 190 (7.3) 513.3 -> 499.1, 240 617 -> 597; 96 190 molecules 216.1 ->
// 211.2, (7.3) 206.9 -> 206.7; 192 190 molecules (7.3) 394.6 -> 385.5.
//
// 256 channels around 5 000 nodes, steps with forces: batches of molecules of 21 with 8.8 neighbours gain at every size (3 150 nodes 528 -> 502, 5 040
// 716 -> 680, 6 006 805 -> 768, 9 996 1 279 -> 1 233), periodic ones from eight to nine neighbours on (3 000 x 7 442 -> 445, 4 000 x 7 493 -> 499, x 8.4
// 556 -> 547, 5 100 x 7 608 -> 615, x 8.4 688 -> 684, 6 000 x 7 692 -> 708, x 8.4 780 -> 787, 8 000 x 7 873 -> 891, x 8.4 984 -> 986): the line rises
// from 6.75 neighbours at 5 000 nodes to 8.25 at 8 000 and 9 at 12 000.
//
// Nodes of a (pair of degrees, slice) that a workgroup has at least.  There are share_of(channels) workgroups for each, so the lines are 3 840
// nodes at 32 channels, 2 432, 1 596 and 1 216 at 64, 96 and 128, and 528, 580, 387 and 552 at 160 to 256; both sides of them are above.
inline int64_t min_nodes_per_workgroup(int channels) {
  switch (channels) {
    case 32: return 60;
    case 160: return 44;
    case 192: return 58;
    case 224: return 43;
    case 256: return 69;
    default: return 76;
  }
}
inline int64_t min_edges(int64_t nnodes, int channels) {
  struct Line {
    int64_t cached;             // edges, while the output fits the last-level cache
    double per_node, doubling;  // beyond: neighbours, and how many more for twice the output
  };
  const Line line = [&]() -> Line {
    switch (channels) {
      case 32: return {0, 0.0, 0.0};
      case 64: return {26000, 0.0, 0.0};
      case 96: return {std::max(28000 + 6 * nnodes / 5, 5 * nnodes), 5.5, 2.0};
      case 128: return {std::max(24000 + 2 * nnodes, 9 * nnodes / 2), 7.0, 3.2};
      case 160: return {std::max(3500 + 7 * nnodes / 2, 21 * nnodes / 5), 6.5, 2.5};
      case 192: return {std::max(4000 + 11 * nnodes / 2, 7 * nnodes), 9.0, 1.9};
      case 224: return {std::max(7000 + 3 * nnodes, 9 * nnodes / 2), 6.0, 1.5};
      default: return {std::max(5000 + 23 * nnodes / 4, 43 * nnodes / 4 - 20000), 11.0, 2.0};
    }
  }();
  const double caches = 64.0 * static_cast<double>(nnodes) * channels / (1 << 28);  // 16 components of 4 bytes in 256 MB
  if (caches <= 1.0) return line.cached;
  return std::max(line.cached, static_cast<int64_t>((line.per_node + line.doubling * std::log2(caches)) * static_cast<double>(nnodes)));
}
inline int share_of(int channels) { return device_compute_units() / (2 * (channels / 16)); }  // workgroups per (pair, slice)

typedef unsigned u4 __attribute__((ext_vector_type(4)));

struct SlicedArgs {
  const float *X, *vec;
  const u4 *records;  // per edge the vector and, as bits, the sender (then vec and sender are not read), or NULL
  const int32_t *sender, *first_occ;
  const float *coeffs, *knots;
  int nknots;
  float r_width, r_max;
  int nnodes;
  int64_t nedges;
  int C;
  float *out;
  int nslices;  // C / 16
  int share;    // workgroups per (pair, slice)
};

// value of `v` in lane J of the reader's quad of four lanes (quad permutation of the DPP operand)
template <int J>
__device__ __forceinline__ unsigned quadu(unsigned v) {
  return static_cast<unsigned>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), J * 0x55, 0xf, 0xf, true));
}

// The value of `v` in each of the four lanes of the reader's quad: element i is lane i's.  One matrix instruction: the
// 4x4x1 form works on 16 independent blocks of four lanes, D_b[i][j] = A_b[i] B_b[j] + C_b[i][j], with A_b[i] taken from
// lane i of the block and row i of D in register i of every lane; B = 1 and C = 0 make it a copy (exact for every
// normal number), 8 cycles of the SIMD instead of the four moves with a DPP operand at 4.4 each.
__device__ __forceinline__ f4 quad_gather(float v) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(v, 1.0f, f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
}

// the two degrees of pair P and their component counts
template <int P>
struct Pair {
  static constexpr int L0 = P == 0 ? 0 : 1, L1 = P == 0 ? 3 : 2;
  static constexpr int M0 = 2 * L0 + 1, M1 = 2 * L1 + 1;
  static_assert(M0 + M1 == 8, "eight components per pair");
  // row of out (component m) that accumulator i stands for
  static constexpr int row(int i) { return i < M0 ? L0 * L0 + i : L1 * L1 + i - M0; }
};

// the eight harmonics of pair P (the unused ones of the full evaluation fall away at compile time)
template <int P>
__device__ __forceinline__ void harmonics(float v0, float v1, float v2, float inv_len, float (&y)[8]) {
  float all[16];
  sh::eval(sh::Direction{v2 * inv_len, v0 * inv_len, v1 * inv_len, inv_len}, all);
#pragma unroll
  for (int i = 0; i < 8; ++i) y[i] = all[Pair<P>::row(i)];
}

// What a lane has prepared for its edge of a block: byte offset of the sender's row in X, byte offset of the knot
// interval in the table slice, offset inside the interval, harmonics.  An edge that does not count (beyond the node's
// range or the cutoff, or with a sender outside the node range) keeps zero harmonics and points at the node's own row
// and at a row of zeros behind the last interval of the table slice.
struct Prepared {
  unsigned xo, io;
  float xr;
  float y[8];
};
// offset inside the interval and harmonics of the four edges of a block, in every lane of the quad
struct Gathered {
  f4 xr;
  f4 y[8];
};
__device__ __forceinline__ Gathered gather(const Prepared &o) {
  Gathered g;
  g.xr = quad_gather(o.xr);
#pragma unroll
  for (int i = 0; i < 8; ++i) g.y[i] = quad_gather(o.y[i]);
  return g;
}
struct Raw {  // what a lane loads for its edge of a block
  int s;
  float v0, v1, v2;
};

template <int J>
__device__ __forceinline__ void request_row(const float *__restrict__ X, unsigned xo, unsigned place, f4 &x) {
  x = *reinterpret_cast<const f4 *>(reinterpret_cast<const char *>(X) + (quadu<J>(xo) + place));
}

// the pieces (a, b, c, d) of channel D of both degrees from the edge's row of the table
template <int D>
__device__ __forceinline__ void request_pieces(const char *row, f4 (&q)[2]) {
  q[0] = *reinterpret_cast<const f4 *>(row + 64 * D);
  q[1] = *reinterpret_cast<const f4 *>(row + 256 + 64 * D);
}

// channel D of step J
template <int P, int J, int D>
__device__ __forceinline__ void channel(const char *ahead, float xr, float xs, const Gathered &all, f4 (&q)[2], float (&acc)[2][8][4]) {
  float t[2];
#pragma unroll
  for (int li = 0; li < 2; ++li) t[li] = xs * fmaf(xr, fmaf(xr, fmaf(xr, q[li].w, q[li].z), q[li].y), q[li].x);
  __builtin_amdgcn_sched_barrier(0);
  request_pieces<(D + 2) % 4>(ahead, q);
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[J & 1][i][D] = fmaf(all.y[i][J], t[i < Pair<P>::M0 ? 0 : 1], acc[J & 1][i][D]);
  __builtin_amdgcn_sched_barrier(0);
}

// Steps J .. 3 of a block whose first table row starts at `row`; behind step j the X values of the next block's edge at
// that place are requested into x[j], and from the third channel on the pieces are those of the step after.
template <int P, int J>
__device__ __forceinline__ void edge_step(const float *__restrict__ X, const char *tab, unsigned io, const Gathered &all, const Prepared &nxt,
                                          unsigned place, const char *row, f4 (&x)[4], f4 (&q)[2][2], float (&acc)[2][8][4]) {
  const char *next_row = tab + (quadu<(J + 1) % 4>(J < 3 ? io : nxt.io) + place);
  channel<P, J, 0>(row, all.xr[J], x[J].x, all, q[0], acc);
  channel<P, J, 1>(row, all.xr[J], x[J].y, all, q[1], acc);
  channel<P, J, 2>(next_row, all.xr[J], x[J].z, all, q[0], acc);
  channel<P, J, 3>(next_row, all.xr[J], x[J].w, all, q[1], acc);
  request_row<J>(X, nxt.xo, place, x[J]);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (J + 1 < 4) edge_step<P, J + 1>(X, tab, io, all, nxt, place, next_row, x, q, acc);
}

// the rounds of one sorted sub-range: nodes lo + order[0 .. cnt)
template <int P, bool RECORDS>
__device__ __forceinline__ void run_rounds(const SlicedArgs &p, const float *sTab, const float *sKnots,
                                           const unsigned short *sOrder, int *sNext, int lo, int cnt, int slice) {
  const int k = threadIdx.x & 3;  // place in the quad: channels 4 k .. 4 k + 3 of the slice
  const unsigned place = 16u * static_cast<unsigned>(k);  // byte offset of the lane's channels in its slice of an X / out row, and of its pieces in a row of the table
  const char *tab = reinterpret_cast<const char *>(sTab);
  const float *X = p.X + 16 * slice;
  float *out = p.out + 16 * slice;
  const int C = p.C;
  const int last_edge = static_cast<int>(p.nedges) - 1;  // the launcher does not come here without edges
  const unsigned zero_row = static_cast<unsigned>(p.nknots - 1) * kSlRowBytes;
  const float inv_width = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, 1.0f / p.r_width)));

  for (;;) {
    int base = 0;
    int lane = threadIdx.x % kWave;
    asm volatile("" : "+v"(lane));  // as above: formed anew for every round
    const int gw = lane >> 2;       // node of the wave's round
    if (lane == 0) base = atomicAdd(sNext, kWave / 4);
    base = __builtin_amdgcn_readfirstlane(base);
    if (base >= cnt) break;
    const int mine = base + gw;
    const int node = mine < cnt ? lo + sOrder[mine] : -1;
    int e0 = 0, e1 = 0;
    if (node >= 0) {
      e0 = p.first_occ[node];
      e1 = p.first_occ[p.nnodes + node];
      clamp_edge_range(e0, e1, p.nedges);
    }
    const int first_mine = e0 + k;
    float acc[2][8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int d = 0; d < 4; ++d) acc[0][i][d] = acc[1][i][d] = 0.f;

    // Unconditional (an edge index beyond the list reads the last edge, and prepare() discards it): loads under a
    // branch would make the later waits cover everything in flight.
    auto request = [&](int blk) {
      const unsigned e = static_cast<unsigned>(min(first_mine + 4 * blk, last_edge));
      if constexpr (RECORDS) {
        const u4 v = *reinterpret_cast<const u4 *>(reinterpret_cast<const char *>(p.records) + 16u * e);
        return Raw{static_cast<int>(v[3]), __uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2])};
      }
      const float *v = reinterpret_cast<const float *>(reinterpret_cast<const char *>(p.vec) + 12u * e);
      return Raw{*reinterpret_cast<const int *>(reinterpret_cast<const char *>(p.sender) + 4u * e), v[0], v[1], v[2]};
    };
    auto prepare = [&](const Raw &r, int blk) {
      Prepared o;
      const bool valid = first_mine + 4 * blk < e1;
      // Direction from one reciprocal square root (the hardware's, one Newton step: within an ulp), the length from it by
      // one more Newton step, whose residual r2 - len^2 is exact in an fma (without it the length is off by 1.4 times the
      // rounding of a square root, and the message by 3 to 8 % more than the other forward kernels' on the same edges), the
      // interval from a product with 1 / width: the square root and the two divisions of the usual form are 40 instructions
      // per edge, and every one of the 16 workgroup types of a piece of the node range prepares every edge.  An edge within
      // rounding of a knot may land in the neighbouring interval, whose cubic continues
      // the spline there (value and two derivatives agree at the knot); one within rounding of the cutoff may be kept
      // or dropped, where the tabulated functions of a model end in zero (their envelope) and a table that does not
      // is cut off at a length that is only known to that rounding anyway.
      const float r2 = fmaf(r.v2, r.v2, fmaf(r.v1, r.v1, r.v0 * r.v0));
      float ir = __builtin_amdgcn_rsqf(r2);
      ir = ir * fmaf(-0.5f * r2 * ir, ir, 1.5f);
      const float near = r2 * ir;
      const float len = fmaf(0.5f * ir, fmaf(-near, near, r2), near);  // NaN for a vector of zeros: such an edge does not count
      // without a branch (the interval of an edge that does not count is looked up and dropped): under a branch the
      // knot's way from LDS is waited for on the spot, here it arrives while the harmonics are formed
      int idx = static_cast<int>(len * inv_width);
      idx = idx < 0 ? 0 : (idx > p.nknots - 2 ? p.nknots - 2 : idx);
      const float knot = sKnots[idx];
      const bool live = valid && len <= p.r_max && static_cast<unsigned>(r.s) < static_cast<unsigned>(p.nnodes);
      harmonics<P>(r.v0, r.v1, r.v2, ir, o.y);
#pragma unroll
      for (int i = 0; i < 8; ++i) o.y[i] = live ? o.y[i] : 0.f;
      o.xr = live ? len - knot : 0.f;
      o.xo = __umul24(static_cast<unsigned>(live ? r.s : max(node, 0)), static_cast<unsigned>(4 * C));  // both below 2^24
      o.io = live ? __umul24(static_cast<unsigned>(idx), kSlRowBytes) : zero_row;
      return o;
    };
    Raw raw = request(0);
    Prepared nxt = prepare(raw, 0);
    raw = request(1);
    f4 x[4], q[2][2];
    request_row<0>(X, nxt.xo, place, x[0]);
    request_row<1>(X, nxt.xo, place, x[1]);
    request_row<2>(X, nxt.xo, place, x[2]);
    request_row<3>(X, nxt.xo, place, x[3]);
    const char *row = tab + (quadu<0>(nxt.io) + place);
    request_pieces<0>(row, q[0]);
    request_pieces<1>(row, q[1]);
    for (int blk = 0;; ++blk) {
      const Prepared cur = nxt;
      nxt = prepare(raw, blk + 1);  // before the gathering: fewer values live at a time
      __builtin_amdgcn_sched_barrier(0);
      raw = request(blk + 2);
      const Gathered all = gather(cur);
      __builtin_amdgcn_sched_barrier(0);
      edge_step<P, 0>(X, tab, cur.io, all, nxt, place, tab + (quadu<0>(cur.io) + place), x, q, acc);
      if (!__any(first_mine + 4 * (blk + 1) < e1)) break;  // the first lane of a quad tells for all four
    }

    if (node >= 0) {
      unsigned at = place;
      asm volatile("" : "+v"(at));  // keeps the address out of the registers of the edge loop
      char *op = reinterpret_cast<char *>(out + static_cast<int64_t>(node) * 16 * C) + at;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        *reinterpret_cast<f4 *>(op + static_cast<int64_t>(Pair<P>::row(i)) * (4 * C)) =
            f4{acc[0][i][0] + acc[1][i][0], acc[0][i][1] + acc[1][i][1], acc[0][i][2] + acc[1][i][2], acc[0][i][3] + acc[1][i][3]};
    }
  }
}

template <bool RECORDS>
__global__ __launch_bounds__(kSlThreads) void mp_edge_forward_sliced_kernel(const SlicedArgs p) {
  __shared__ __attribute__((aligned(16))) float sTab[kSlMaxIntervals * (kSlRowBytes / 4)];
  __shared__ float sKnots[kSlMaxIntervals + 1];
  __shared__ unsigned short sOrder[kSlSub];
  __shared__ int sHist[kSlBins];
  __shared__ int sNext;

  const int tid = threadIdx.x;
  // Which (pair, slice) and which piece j of the node range.  Consecutive workgroups go to consecutive XCDs (eight of
  // them, each with its own L2).  The pieces in order, each with all its types, are cut into eight runs, one per XCD: the edge data
  // and the X rows of neighbouring nodes are fetched into one L2, or two where a piece is cut (share / 8 is no whole number at 96, 160, 192
  // and 224 channels).  With pieces 8 apart on an XCD and the rest of share / 8 spread over all of them every L2 fetched up to a third of
  // the nodes.  Energies alone, us, that -> this in turn on one card (best of three runs): 96 channels 40 000 955.7 -> 941.2; 128 25 000 778.4 ->
  // 773.8; 160 10 007 455.1 -> 449.0; 192 40 000 2 075 -> 2 060; 224 30 000 1 870 -> 1 864; within the runs' spread 32 12 000 134.2 -> 133.8, 96 10 000 259.2 -> 259.4, 128 30 000
  // 934.8 -> 932.8, 192 10 000 538.2 -> 537.2, 160 25 000 1 085 -> 1 091; 64 and 256 the same (the gain differs by the card: 979 -> 931 and 1 088 -> 1 055 have been
  // seen for 96 x 40 000 and 160 x 25 000).  Sixteen workgroups more at 160 and 192 channels, each with its share of the nodes of one or two types, gave
  // 0 to 0.8 % in place of that (the second slice of the table, the rounds at the end of both parts).
  int type, j;
  {
    const int types = 2 * p.nslices;
    const int total = types * p.share, xcd = blockIdx.x % 8;
    const int rank = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
    type = rank % types;
    j = rank / types;
  }
  const int slice = type >> 1;
  const int pair = type & 1;
  const int lo = static_cast<int>(static_cast<int64_t>(p.nnodes) * j / p.share);
  const int hi = static_cast<int>(static_cast<int64_t>(p.nnodes) * (j + 1) / p.share);

  // the slice of the table: coeffs[idx][coef][l C + 16 slice + 4 k + d] -> byte kSlRowBytes idx + 256 li + 64 d + 16 k of sTab,
  // (a, b, c, d) together
  constexpr int kRow = kSlRowBytes / 4;
  const int intervals = p.nknots - 1;
  constexpr int kAhead = 4;  // pieces of a thread requested together
  for (int i0 = tid; i0 < intervals * 32; i0 += kAhead * kSlThreads) {
    f4 v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int i = min(i0 + u * kSlThreads, intervals * 32 - 1);
      const int idx = i >> 5, coef = (i >> 3) & 3, li = (i >> 2) & 1, k = i & 3;
      const int l = pair == 0 ? (li == 0 ? 0 : 3) : (li == 0 ? 1 : 2);
      v[u] = ld4(p.coeffs + (static_cast<int64_t>(idx * 4 + coef) * 4 + l) * p.C + slice * 16 + 4 * k);
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int i = min(i0 + u * kSlThreads, intervals * 32 - 1);  // beyond the table: the last piece once more
      const int idx = i >> 5, coef = (i >> 3) & 3, li = (i >> 2) & 1, k = i & 3;
      float *dst = sTab + idx * kRow + 64 * li + 4 * k + coef;
      dst[0] = v[u].x;
      dst[16] = v[u].y;
      dst[32] = v[u].z;
      dst[48] = v[u].w;
    }
  }
  for (int i = tid; i < 128; i += kSlThreads) sTab[intervals * kRow + i] = 0.f;  // the row of edges that do not count
  for (int i = tid; i < p.nknots; i += kSlThreads) sKnots[i] = p.knots[i];

  for (int sub = lo; sub < hi; sub += kSlSub) {
    const int cnt = min(kSlSub, hi - sub);
    int here = tid;  // opaque: what the sort derives from it is formed anew for every sub-range, not kept through the rounds
    asm volatile("" : "+v"(here));
    __syncthreads();  // every wave has left the previous sub-range (and the table is staged)
    if (here < kSlBins) sHist[here] = 0;
    if (here == 0) sNext = 0;
    __syncthreads();
    // counting sort by the number of edge blocks, most blocks first
    constexpr int kPerThread = (kSlSub + kSlThreads - 1) / kSlThreads;
    int bin[kPerThread];
#pragma unroll
    for (int q = 0; q < kPerThread; ++q) {
      const int i = here + q * kSlThreads;
      bin[q] = -1;
      if (i < cnt) {
        int e0 = p.first_occ[sub + i], e1 = p.first_occ[p.nnodes + sub + i];
        clamp_edge_range(e0, e1, p.nedges);
        bin[q] = kSlBins - 1 - min((e1 - e0 + 3) >> 2, kSlBins - 1);
        atomicAdd(&sHist[bin[q]], 1);
      }
    }
    __syncthreads();
    if (here == 0) {
      int run = 0;
      for (int b = 0; b < kSlBins; ++b) {
        const int n = sHist[b];
        sHist[b] = run;
        run += n;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPerThread; ++q)
      if (bin[q] >= 0) sOrder[atomicAdd(&sHist[bin[q]], 1)] = static_cast<unsigned short>(here + q * kSlThreads);
    __syncthreads();
    if (pair == 0)
      run_rounds<0, RECORDS>(p, sTab, sKnots, sOrder, &sNext, sub, cnt, slice);
    else
      run_rounds<1, RECORDS>(p, sTab, sKnots, sOrder, &sNext, sub, cnt, slice);
  }
}

}  // namespace

bool sliced_forward_applies(int64_t nnodes, int64_t nedges, int channels, int nknots) {
  if (channels % 16 != 0 || share_of(channels) < 2 || nedges == 0) return false;
  if (nedges < min_edges(nnodes, channels)) return false;
  return nnodes > share_of(channels) * min_nodes_per_workgroup(channels) && nnodes < (1 << 24) &&
         nnodes * channels < (int64_t{1} << 30) && nedges <= UINT32_MAX / 12 && nknots >= 2 && nknots - 1 < kSlMaxIntervals;
}

int launch_sliced_forward(const float *X, const float *vec, const void *records, const float *knots, const float *coeffs, int nknots,
                          float r_width, float r_max, const int32_t *sender, const int32_t *first_occ, int64_t nnodes, int64_t nedges,
                          int channels, float *out, hipStream_t st) {
  SlicedArgs a{X, vec, static_cast<const u4 *>(records), sender, first_occ, coeffs, knots, nknots, r_width, r_max, static_cast<int>(nnodes), nedges,
               channels, out, channels / 16, 0};
  a.share = share_of(channels);
  const dim3 grid(static_cast<unsigned>(a.share * 2 * a.nslices));
  if (records)
    hipLaunchKernelGGL(mp_edge_forward_sliced_kernel<true>, grid, dim3(kSlThreads), 0, st, a);
  else
    hipLaunchKernelGGL(mp_edge_forward_sliced_kernel<false>, grid, dim3(kSlThreads), 0, st, a);
  return check_launch("cm_mp_edge_forward");
}

}  // namespace mp
}  // namespace cm
