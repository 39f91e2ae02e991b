// Invariant message passing with the radial weights evaluated inside the kernels from the cubic-spline
// table, so that R[E, 4, C], its derivative and grad_R never exist in HBM.
//
//   out[n, m, c] = sum_{e -> n} X[sender[e], c] * Y[m, e] * R(r[e])[l(m), c],
//   R(r)[j] = a + b x + c x^2 + d x^3,  (a, b, c, d) = coeffs[idx, :, j],  x = r - r_knots[idx]
//
// Same decomposition as the tabulated-radial kernels (one wave per receiver node, lane = 4 channels,
// node-resident accumulators / gradients in registers, Y and sender staged in LDS); the per-edge knot
// interval and offset are staged next to them.  The coefficient table (2 MB at C = 128) lives in L2:
// per edge and l a lane reads its four 16-byte coefficient pieces, evaluates R_l (and dR_l/dr in the
// backward) and drops them, so only 16 registers of radial data are live at a time.  The backward
// returns the gradient with respect to the edge length directly:
//   g_r[e] = sum_{l, c} X[s, c] * q_l[c] * dR_l/dr[c],   q_l = sum_{m in l} Y[m, e] * grad_out[n, m, c].
//
// The FROM_VEC variants go one step further and take the fp32 edge vectors instead of Y and r: the 16 harmonics and the
// length are computed per edge while the chunk is staged, and the backward turns the reduced gY and g_r of an edge
// straight into the gradient with respect to its vector (harmonics Jacobian + radial part), so Y[16, E], grad_Y and
// grad_r never exist either.  Beyond a thousand or two of receiver nodes the forward from edge vectors runs on the kernel of
// mp_sliced.hip, which keeps a workgroup's part of the table in LDS (same arithmetic per edge, sums in list order).
#include <algorithm>
#include <cmath>

#include "mp_spline_device.hpp"

// waves per SIMD the register allocator must leave room for.  The backward edge pass runs with a rotated edge loop (the
// next edge's loads are requested before the current edge's reductions), which needs the registers of two waves per SIMD.
#ifndef CM_FUSED_FWD_WAVES
#define CM_FUSED_FWD_WAVES 3
#endif
#ifndef CM_FUSED_BWD_WAVES
#define CM_FUSED_BWD_WAVES 2
#endif

namespace cm {
namespace {

using namespace mp;

// -----------------------------------------------------------------------------------------------
// forward
// -----------------------------------------------------------------------------------------------
// MULTI: a workgroup of up to six waves per node, each on a part of the node's edge range (launched for few nodes)
template <int C, bool FROM_VEC, bool MULTI>
__global__ __launch_bounds__(MULTI ? 8 * kWave : kWave, (MULTI || Cfg<C, true>::V > 5 ? 2 : CM_FUSED_FWD_WAVES)) void mp_spline_forward_kernel(const float *__restrict__ X,
                                                                 const float *__restrict__ Y, Spline sp,
                                                                 const int32_t *__restrict__ sender,
                                                                 const int32_t *__restrict__ first_occ, int nnodes,
                                                                 int64_t nedges, float *__restrict__ out) {
  using K = Cfg<C, true>;
  using vec = typename K::vec;
  // A workgroup is one wave per part of the node's edge range (MULTI; otherwise one wave and one part: see forward_parts).
  // Every wave stages its own edges in its own piece of LDS; the waves meet once, at the end.
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_lds[];
  const int wave = MULTI ? threadIdx.x / kWave : 0;
  const int parts = MULTI ? blockDim.x / kWave : 1;
  unsigned char *mine = dyn_lds + wave * kStageBytes;
  float *sY = reinterpret_cast<float *>(mine);
  int *sS = reinterpret_cast<int *>(mine + kChunk * 64);
  int *sIdx = sS + kChunk;
  float *sXr = reinterpret_cast<float *>(sIdx + kChunk);
  int *sOrig = reinterpret_cast<int *>(sXr + kChunk);

  const int node = blockIdx.x;
  const int lane = threadIdx.x % kWave;
  const int slot = lane / K::SW;
  const int cl = lane % K::SW;
  const bool active = cl < K::LPE;
  int e0 = first_occ[node];
  int e1 = first_occ[nnodes + node];
  clamp_edge_range(e0, e1, nedges);
  if (parts > 1) {
    const int64_t len = e1 - e0;
    const int lo = e0 + static_cast<int>(len * wave / parts);
    e1 = e0 + static_cast<int>(len * (wave + 1) / parts);
    e0 = lo;
  }

  vec acc[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) acc[m] = zerov<vec>();

  for (int base = e0; base < e1;) {
    wave_lds_fence();  // the staged edges belong to this wave alone
    const int nlive = stage_edges<FROM_VEC>(Y, sender, sp, nnodes, nedges, base, e1, lane, sY, sS, sIdx, sXr, sOrig,
                                            [](int, int, unsigned long long, bool) {});
    wave_lds_fence();
    if (active) {
      // what one edge brings in: the sender's row piece, the 16 coefficient pieces of its knot interval, its harmonics
      struct Edge {
        vec x, coef[16];
        float y[16], xr;
      };
      auto fetch = [&](int j, Edge &e) {
        const int s = sS[j];
        const int idx = sIdx[j];
        e.xr = sXr[j];
        e.x = K::ld(X + (static_cast<unsigned>(s) * C + unsigned(K::off(cl))));
        const f4 *yp = reinterpret_cast<const f4 *>(sY + j * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f4 v = yp[q];
          e.y[4 * q] = v.x, e.y[4 * q + 1] = v.y, e.y[4 * q + 2] = v.z, e.y[4 * q + 3] = v.w;
        }
        const unsigned co = static_cast<unsigned>(idx) * (16u * C) + unsigned(K::off(cl));  // 32-bit offset from the uniform table base
        // addressed from the middle of the interval's 16C-float row: all 16 pieces lie within +-8C floats of it, which
        // up to C = 128 fits the signed immediate offset of a load, so one address serves them all
        const float *mid = sp.coeffs + (co + 8 * C);
#pragma unroll
        for (int q = 0; q < 16; ++q) e.coef[q] = K::ld(mid + (q * C - 8 * C));  // piece q: coefficient q / 4 of degree q % 4
      };
      auto accumulate = [&](const Edge &e) {
        auto per_l = [&](auto lc) {
          constexpr int L = decltype(lc)::value;
          const vec t = e.x * (e.coef[L] + e.xr * (e.coef[4 + L] + e.xr * (e.coef[8 + L] + e.xr * e.coef[12 + L])));
#pragma unroll
          for (int m = MRange<L>::lo; m < MRange<L>::hi; ++m) acc[m] += e.y[m] * t;
        };
        per_l(std::integral_constant<int, 0>{});
        per_l(std::integral_constant<int, 1>{});
        per_l(std::integral_constant<int, 2>{});
        per_l(std::integral_constant<int, 3>{});
      };
      if constexpr (MULTI && K::V <= 4) {
        // few nodes: a wave's part is a dozen edges, and what it waits for is one memory round trip per trip of this
        // loop, so two edges per slot are requested per trip (same order of the sums; registers for it up to four
        // channels per lane)
        for (int j = slot; j < nlive; j += 2 * K::EPW) {
          Edge e0, e1;
          const bool two = j + K::EPW < nlive;
          fetch(j, e0);
          fetch(two ? j + K::EPW : j, e1);
          __builtin_amdgcn_sched_barrier(0);  // both edges' loads stay ahead of the first edge's arithmetic
          accumulate(e0);
          if (two) accumulate(e1);
        }
      } else if constexpr (MULTI && K::V == 5) {
        // five channels per lane: one edge's 85 registers (degree by degree, as below, an edge is four round trips)
        for (int j = slot; j < nlive; j += K::EPW) {
          Edge e0;
          fetch(j, e0);
          __builtin_amdgcn_sched_barrier(0);
          accumulate(e0);
        }
      } else {
        // one edge per trip; per degree the four coefficient pieces are loaded, used and dropped (16 registers of
        // radial data live at a time)
        for (int j = slot; j < nlive; j += K::EPW) {
          const int s = sS[j];
          const int idx = sIdx[j];
          const float xr = sXr[j];
          const vec x = K::ld(X + (static_cast<unsigned>(s) * C + unsigned(K::off(cl))));
          float y[16];
          {
            const f4 *yp = reinterpret_cast<const f4 *>(sY + j * 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f4 v = yp[q];
              y[4 * q] = v.x, y[4 * q + 1] = v.y, y[4 * q + 2] = v.z, y[4 * q + 3] = v.w;
            }
          }
          const unsigned co = static_cast<unsigned>(idx) * (16u * C) + unsigned(K::off(cl));
          const float *__restrict__ tab = sp.coeffs;
          auto per_l = [&](auto lc) {
            constexpr int L = decltype(lc)::value;
            const float *mid = tab + (co + 8 * C);
            const vec a = K::ld(mid + (L * C - 8 * C)), b = K::ld(mid + (L * C - 4 * C)), c = K::ld(mid + L * C),
                      d = K::ld(mid + (L * C + 4 * C));
            const vec t = x * (a + xr * (b + xr * (c + xr * d)));
#pragma unroll
            for (int m = MRange<L>::lo; m < MRange<L>::hi; ++m) acc[m] += y[m] * t;
          };
          per_l(std::integral_constant<int, 0>{});
          per_l(std::integral_constant<int, 1>{});
          per_l(std::integral_constant<int, 2>{});
          per_l(std::integral_constant<int, 3>{});
        }
      }
    }
  }

#pragma unroll
  for (int off = kWave / 2; off >= K::SW; off >>= 1) {
#pragma unroll
    for (int m = 0; m < 16; ++m) acc[m] += shfl_downv(acc[m], off);
  }
  if (parts > 1) {
    // sums of the parts, added up by the first wave in the order of the parts (the same on every run)
    float *comb = reinterpret_cast<float *>(dyn_lds + parts * kStageBytes);
    if (wave > 0 && slot == 0 && active) {
      float *cp = comb + (wave - 1) * (16 * C) + K::off(cl);
#pragma unroll
      for (int m = 0; m < 16; ++m) K::st(cp + m * C, acc[m]);
    }
    __syncthreads();
    if (wave > 0) return;
    if (slot == 0 && active) {
      for (int w = 1; w < parts; ++w) {
        const float *cp = comb + (w - 1) * (16 * C) + K::off(cl);
#pragma unroll
        for (int m = 0; m < 16; ++m) acc[m] += K::ld(cp + m * C);
      }
    }
  }
  if (slot == 0 && active) {
    float *op = out + static_cast<int64_t>(node) * (16 * C) + K::off(cl);
#pragma unroll
    for (int m = 0; m < 16; ++m) K::st(op + m * C, acc[m]);
  }
}

// -----------------------------------------------------------------------------------------------
// backward, edge pass: gY, g_r and the per-edge contribution to gX
// -----------------------------------------------------------------------------------------------
// Up to 64 channels three waves per SIMD on one operand set (168 registers): a trip's chain of lane exchanges is as long there as
// at 128 channels for half or a quarter of the arithmetic, and a third wave fills it (11 000 x 52 x 64 100.6 -> 95.8 us, 3 000 x
// 52 x 64 31.2 -> 27.6, 11 000 x 10 x 32 27.8 -> 24.4).  From 96 on the L1 path is the limit (25 000 x 52 x 128 389 against 394).
template <int C, bool FROM_VEC>
constexpr bool kOneOperandSet = FROM_VEC && C <= 64;

template <int C, bool FROM_VEC, bool WANT_GY, bool WANT_GR, bool WANT_GX>
__global__ __launch_bounds__(kWave, (kOneOperandSet<C, FROM_VEC> ? 3 : CM_FUSED_BWD_WAVES)) void mp_spline_backward_edge_kernel(
    const float *__restrict__ X, const float *__restrict__ Y, Spline sp, const float *__restrict__ G,
    const int32_t *__restrict__ sender, const int32_t *__restrict__ first_occ, int nnodes, int64_t nedges,
    float *__restrict__ gY, float *__restrict__ g_r, float *__restrict__ gXe, int parts) {
  using K = Cfg<C>;
  using vec = typename K::vec;
  // From edge vectors, the harmonic m = 0 is the constant 1: q_0 is the gradient row itself, and nothing needs the gradient
  // of that harmonic, so its place in the reduction over the slot carries the radial sum (which had a reduction, a lane
  // exchange through LDS and an array of its own next to the unused sixteenth dot product).  us, without / with gX and its
  // sender pass: 25 000 x 52 x 128 445 / 635 -> 414 / 632, 12 000 x 52 x 96 196 / 268 -> 181 / 264, 12 000 x 52 x 256
  // 430 / 596 -> 388 / 581, 11 000 x 10 x 64 42 / 55 -> 39 / 53.
  constexpr bool kRadialInFirst = FROM_VEC && WANT_GY && WANT_GR;
  // Every slot needs all of the node's 16 rows: loaded row by row, each of the two, four or eight slots fetches them for itself,
  // and 16 load instructions are as many as an edge per slot takes.  The rows are one piece of memory: fetched once, 16 bytes
  // per lane, and handed out through LDS, they are C / 16 instructions.
  constexpr bool kRowsThroughLds = FROM_VEC && K::EPW > 1;
  __shared__ __attribute__((aligned(16))) float sY[kChunk * 16];
  __shared__ int sS[kChunk];
  __shared__ int sIdx[kChunk];
  __shared__ float sXr[kChunk];
  __shared__ int sOrig[kChunk];
  // The node's gradient rows on their way into registers, then the reduced gY, [m][edge].
  __shared__ __attribute__((aligned(16))) float sRows[kRowsThroughLds && 16 * C > 16 * kChunk ? 16 * C : 16 * kChunk];
  float *const sGY = sRows;
  __shared__ float sGr[kChunk];
  // The knots, where there are at most kKnotsInLds of them: the staging looks one up per edge, and a lookup in memory is
  // waited for behind everything the wave has in flight (the gradient rows from HBM first of all).
  __shared__ float sKnots[kKnotsInLds];

  // one wave per node, or (backward_parts) per part of a node's edge range: every output of this pass belongs to
  // one edge, so the parts share nothing but the node's gradient rows, which each of them reads
  const int node = parts == 1 ? blockIdx.x : blockIdx.x / parts;
  const int lane = threadIdx.x;
  const int slot = lane / K::SW;
  const int cl = lane % K::SW;
  const bool active = cl < K::LPE;
  const unsigned cla = active ? cl : 0;  // lanes beyond the channel count read lane 0's addresses; their g is zero
  const bool knots_in_lds = KnotCopy<>::applies(sp);
  KnotCopy<> knots;
  knots.request(sp, lane);
  __builtin_amdgcn_sched_barrier(0);
  int e0 = first_occ[node];
  int e1 = first_occ[nnodes + node];
  clamp_edge_range(e0, e1, nedges);
  if (parts > 1) {
    const int part = blockIdx.x % parts;
    const int64_t len = e1 - e0;
    const int lo = e0 + static_cast<int>(len * part / parts);
    e1 = e0 + static_cast<int>(len * (part + 1) / parts);
    e0 = lo;
  }
  if (e0 >= e1) return;

  // Order of the first requests: the raw edges of the first chunk (from L2, and the staging waits for them), then the
  // node's gradient rows (from HBM, read once, not needed before the first edge's arithmetic).  Memory operations retire
  // in issue order, so with the rows in front the staging would wait for them as well.
  RawEdge ahead{-1, 0.f, 0.f, 0.f};
  if constexpr (FROM_VEC) {
    const int64_t e = min(static_cast<int64_t>(e0) + lane, nedges - 1);  // unconditional; lanes beyond the range drop it
    ahead.s = sender[e];
    ahead.v0 = sp.vec[3 * e + 0], ahead.v1 = sp.vec[3 * e + 1], ahead.v2 = sp.vec[3 * e + 2];
    __builtin_amdgcn_sched_barrier(0);
  }
  vec g[16];
  f4 rows[kRowsThroughLds ? C / 16 : 1];
  if constexpr (kRowsThroughLds) {
    const float *gp = G + static_cast<int64_t>(node) * (16 * C) + 4 * lane;
#pragma unroll
    for (int q = 0; q < C / 16; ++q) rows[q] = ld4_stream(gp + 256 * q);
  } else {
    const float *gp = G + static_cast<int64_t>(node) * (16 * C) + K::off(cl);
#pragma unroll
    for (int m = 0; m < 16; ++m) g[m] = active ? K::ld_stream(gp + m * C) : zerov<vec>();  // read once
  }
  __builtin_amdgcn_sched_barrier(0);
  if (knots_in_lds) knots.store(sp, lane, sKnots);

  // The first chunk is written out ahead of the loop over the others (most nodes have no others): at a loop's head the
  // compiler has to assume that the loads a previous iteration left in flight (a slot's last, unused look-ahead) are still
  // on their way into registers the staging reuses, and waits for everything, the gradient rows included.
  int cursor = e0;
  auto chunk = [&](auto first_chunk) {
    const int base = cursor;  // sOrig counts from here
    // (the workgroup is this one wave: ordering its own LDS traffic is all that is needed, and a workgroup barrier would
    // wait for everything in flight first, the gradient rows and the previous chunk's stores included)
    wave_lds_fence();
    // consumed edges that are not live: their gradients are zeros (their rows of gXe stay unwritten: the sender pass
    // reads the rows of live edges only)
    auto dead = [&](int pass_base, int, unsigned long long, bool lane_is_dead) {
      if constexpr (WANT_GY || WANT_GR) {
        if (lane_is_dead) {
          const int64_t e = pass_base + lane;
          if constexpr (FROM_VEC) {
            gY[3 * e + 0] = g_r ? g_r[3 * e + 0] : 0.f;
            gY[3 * e + 1] = g_r ? g_r[3 * e + 1] : 0.f;
            gY[3 * e + 2] = g_r ? g_r[3 * e + 2] : 0.f;
          } else {
            if constexpr (WANT_GY) {
#pragma unroll
              for (int m = 0; m < 16; ++m) gY[m * nedges + e] = 0.f;
            }
            if constexpr (WANT_GR) g_r[e] = 0.f;
          }
        }
      }
    };
    const int nlive = stage_edges<FROM_VEC, FROM_VEC && decltype(first_chunk)::value>(
        Y, sender, sp, nnodes, nedges, cursor, e1, lane, sY, sS, sIdx, sXr, sOrig, dead, ahead, sKnots, knots_in_lds);
    if constexpr (kRowsThroughLds && decltype(first_chunk)::value) {
#pragma unroll
      for (int q = 0; q < C / 16; ++q) st4(sRows + 4 * lane + 256 * q, rows[q]);
    }
    wave_lds_fence();
    if constexpr (kRowsThroughLds && decltype(first_chunk)::value) {
#pragma unroll
      for (int m = 0; m < 16; ++m) g[m] = active ? K::ld(sRows + m * C + K::off(cla)) : zerov<vec>();
      wave_lds_fence();  // the rows' place is the reduced sums' from here on
    }
    // Every lane of a slot takes part in the reductions, so the loop bound is slot-uniform; only live edges are staged.
    // The loop is rotated: the sender row and the 16 coefficient pieces of the NEXT edge are requested right after the
    // arithmetic of the current one, so they travel while the cross-lane reductions (a chain of dependent lane
    // exchanges) run.
    // Two operand sets used in turn (the loop body is written out twice), so that the set being loaded is never copied
    // into the set being consumed; or one set (kOneOperandSet), whose values are used up when the next edge's are requested.
    auto fetch = [&](Operands<K> &o, int j) { fetch_operands<C>(o, X, sp.coeffs, sS[j], sIdx[j], sXr[j], cla); };
    auto edge = [&](Operands<K> &o, int j, Operands<K> &next) {
      float y[16];
      staged_harmonics(sY, j, y);
      float p[16];
      vec gxe = zerov<vec>();
      vec grq = zerov<vec>();
      edge_products<K, FROM_VEC, WANT_GY, WANT_GR, WANT_GX>(o, y, g, p, gxe, grq);
      float grv = 0.f;
      if constexpr (kRadialInFirst) p[0] = dotv(o.x, grq);
      else if constexpr (WANT_GR) grv = hsumv(o.x * grq);

      if constexpr (WANT_GX) {
        // streamed out: 666 MB at the headline size, read once by the sender pass (measured 2 % on the whole step).
        // Issued before the loads of the next edge: memory operations retire in issue order, so a store that is
        // younger than those loads would have to be complete wherever the loop waits for all of them.
        if (active) K::st_stream(gXe + static_cast<int64_t>(base + sOrig[j]) * C + K::off(cl), gxe);
        __builtin_amdgcn_sched_barrier(0);  // keeps the instruction scheduler from sinking the store below the loads
      }
      if constexpr (kOneOperandSet<C, FROM_VEC>) __builtin_amdgcn_sched_barrier(0);  // no request before its landing registers are free
      // Unconditional (the last edge of a slot fetches itself again): loads under a branch would make every later wait
      // assume that they were not issued, i.e. wait for all but the oldest few of them.
      fetch(next, j + K::EPW < nlive ? j + K::EPW : j);
      if constexpr (WANT_GR && !kRadialInFirst) {
        const float tot = slot_sum<K::SW>(grv);
        if (cl == 0) sGr[j] = tot;
      }
      if constexpr (WANT_GY) {
        slot_reduce16<K::SW>(p, cl);
        store_reduced16<K::SW>(p, cl, j, sGY);
      }
    };
    Operands<K> opa;
    if (slot < nlive) fetch(opa, slot);
    if constexpr (kOneOperandSet<C, FROM_VEC>) {
#pragma unroll 1
      for (int j = slot; j < nlive; j += K::EPW) edge(opa, j, opa);
    } else {
      Operands<K> opb;
      for (int j = slot; j < nlive; j += 2 * K::EPW) {
        edge(opa, j, opb);
        if (j + K::EPW >= nlive) break;
        edge(opb, j + K::EPW, opa);
      }
    }
    if constexpr (WANT_GY || WANT_GR) {
      wave_lds_fence();
      // lane k < nlive finishes the k-th staged edge
      int k = lane;
      asm volatile("; addresses formed from here, not carried through the loops" : "+v"(k));
      if (k < nlive) {
        const int64_t e = base + sOrig[k];
        if constexpr (FROM_VEC) {
          float sums[16];
#pragma unroll
          for (int m = 0; m < 16; ++m) sums[m] = sGY[m * kChunk + k];
          finish_vector_gradient(sp.vec, e, sums, g_r, gY);  // gY is the [E, 3] output in this variant, g_r its addend
        } else {
          if constexpr (WANT_GY) {
#pragma unroll
            for (int m = 0; m < 16; ++m) gY[m * nedges + e] = sGY[m * kChunk + k];
          }
          if constexpr (WANT_GR) g_r[e] = sGr[k];
        }
      }
    }
  };
  chunk(std::true_type{});
  while (cursor < e1) chunk(std::false_type{});
}

// -----------------------------------------------------------------------------------------------
// backward, edge pass from edge vectors at 160, 192 and 224 channels (most sizes: steps_of_four_edges): four edges side by side, the channels in steps of 64
// -----------------------------------------------------------------------------------------------
// In the kernel above an edge of 160, 192 or 224 channels takes a whole wave, and its 17 load instructions move 40 or 56 lanes of
// 16 bytes or 64 of 12 where 64 of 16 cost the L1 path the same (16 cycles for any load of 8 to 16 bytes per lane).  Here a row of 16 lanes serves an edge, four channels per lane, a group
// of four edges takes C / 64 steps of 17 full-width loads, and the sixteen sums of an edge go through one reduction
// over 16 lanes instead of 64.  The node's gradient rows of a step would be 64 registers for each of the steps: they stay in
// LDS, from where a degree's rows are read as the degree is worked on (all rows of lanes read the same 256 bytes, at a
// quarter of what the same bytes cost through L1).  The table's pieces for degree l of the next step are requested as soon as
// this step's are used up (one operand set).
//
// The contractions over m stay on the vector ALU: the fp32 matrix instruction computes no faster than plain multiply-adds (32
// cycles for 1 024 of them, 2.3 to 2.8 per 64) and takes the SIMD's time from them, and the kernel that had
// q_l and the gradient with respect to the direction on it, with every product padded to four m, spent 640 cycles per four
// edges and step there against the 370 of the sums here.  Against that kernel and, where it did not run, the one above, us
// without / with gX and its sender pass: 192 channels 100 nodes x 52 11.8 / 19.6 -> 11.1 / 18.3, 1 100 56 / 80 -> 39 / 64,
// 11 000 314 / 442 -> 276 / 414, 40 000 1 089 / 1 598 -> 1 003 / 1 522; 160 channels 100 15.5 / 23.9 -> 11.1 / 18.5,
// 11 000 319 / 428 -> 262 / 381, 4 000 x 4 24.6 -> 20.4; 224 channels 3 000 127 / 161 -> 112 / 147, 30 000 913 / 1 366 -> 909 / 1 358.
// Not at the widths that fill the lanes of the kernel above: 256 357 / 524 -> 359 / 535, 96 170 / 242 -> 176 / 247, 128 (25 000)
// 406 / 616 -> 399 / 612; and not everywhere at 192 and 224: see steps_of_four_edges.
template <int C, bool WANT_GV, bool WANT_GX>
__global__ __launch_bounds__(kWave, CM_FUSED_BWD_WAVES) void mp_edge_backward_steps_kernel(
    const float *__restrict__ X, Spline sp, const float *__restrict__ G, const int32_t *__restrict__ sender,
    const int32_t *__restrict__ first_occ, int nnodes, int64_t nedges, float *__restrict__ gvec,
    const float *__restrict__ addend, float *__restrict__ gXe, int parts) {
  static_assert(C % 32 == 0, "channel count");
  constexpr int H = (C + 63) / 64;
  __shared__ __attribute__((aligned(16))) float sY[kChunk * 16];  // harmonics of an edge, then its reduced sums
  __shared__ __attribute__((aligned(16))) float sRows[16 * C];    // the node's gradient rows
  __shared__ int sS[kChunk];
  __shared__ int sIdx[kChunk];
  __shared__ float sXr[kChunk];
  __shared__ int sOrig[kChunk];
  // 160 KB hold eight waves' arrays at every width.  At 224 channels that leaves room for 256 knots; more are read from memory, which
  // costs less than a place for 512 and seven waves (400 knots, us without / with gX: 1 000 x 52 49.8 / 68.0 -> 39.4 / 56.3, 3 000 x 52
  // 112 / 158 -> 105 / 148, 6 000 x 12 62.2 / 87.8 -> 61.4 / 86.4, 216 x 52 14.4 / 22.9 -> 15.2 / 23.7).
  constexpr int kKnots = C == 224 ? 256 : kKnotsInLds;
  __shared__ float sKnots[kKnots];

  // Runs of 128 workgroups, a node's parts in order, on an XCD: where the X rows are more than one L2 holds, a neighbour's rows come from there more
  // often (step, us, with the forces' runs: 40 000 x 160 4 810 -> 4 776 and 4 736 -> 4 720 by the card, 100 000 x 192 by the card 13 987 -> 13 849 or 13 985 -> 13 968; runs of 32
  // and 512 the same; 10 007 x 160 and 20 000 x 224 equal).  The kernel above gains nothing from it (25 000 x 128, 40 000 x 96,
  // 12 000 x 256; 25 000 x 128 without gX 448 -> 459 alone).
  const int place = place_on_xcd<128>(blockIdx.x, nnodes * parts);
  const int node = parts == 1 ? place : place / parts;
  const int lane = threadIdx.x;
  const int row = lane / 16;  // which edge of a group
  const int cl = lane % 16;
  // The last step of a channel count that is an odd multiple of 32 has work for half of a row's lanes; the others repeat
  // it with the sender's row taken as zero, which leaves them out of the sums over channels.
  constexpr bool kHalf = C % 64 != 0;
  const bool twin = kHalf && cl >= 8;
  const auto step_offset = [&](int h) { return 64 * h - (twin && h == H - 1 ? 32 : 0); };
  const bool knots_in_lds = KnotCopy<kKnots>::applies(sp);
  KnotCopy<kKnots> knots;
  knots.request(sp, lane);
  __builtin_amdgcn_sched_barrier(0);
  int e0 = first_occ[node];
  int e1 = first_occ[nnodes + node];
  clamp_edge_range(e0, e1, nedges);
  if (parts > 1) {
    const int part = place % parts;
    const int64_t len = e1 - e0;
    const int lo = e0 + static_cast<int>(len * part / parts);
    e1 = e0 + static_cast<int>(len * (part + 1) / parts);
    e0 = lo;
  }
  if (e0 >= e1) return;

  // order of the first requests: as in the kernel above
  RawEdge ahead;
  {
    const int64_t e = min(static_cast<int64_t>(e0) + lane, nedges - 1);
    ahead.s = sender[e];
    ahead.v0 = sp.vec[3 * e + 0], ahead.v1 = sp.vec[3 * e + 1], ahead.v2 = sp.vec[3 * e + 2];
    __builtin_amdgcn_sched_barrier(0);
  }
  f4 rows[C / 16];
  {
    const float *gp = G + static_cast<int64_t>(node) * (16 * C) + 4 * lane;
#pragma unroll
    for (int q = 0; q < C / 16; ++q) rows[q] = ld4_stream(gp + 256 * q);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (knots_in_lds) knots.store(sp, lane, sKnots);

  int cursor = e0;
  auto chunk = [&](auto first_chunk) {
    const int base = cursor;
    wave_lds_fence();
    auto dead = [&](int pass_base, int, unsigned long long, bool lane_is_dead) {
      if (WANT_GV && lane_is_dead) {
        const int64_t e = pass_base + lane;
#pragma unroll
        for (int k = 0; k < 3; ++k) gvec[3 * e + k] = addend ? addend[3 * e + k] : 0.f;
      }
    };
    const int nlive = stage_edges<true, decltype(first_chunk)::value>(nullptr, sender, sp, nnodes, nedges, cursor, e1, lane, sY, sS, sIdx,
                                                                     sXr, sOrig, dead, ahead, sKnots, knots_in_lds);
    if constexpr (decltype(first_chunk)::value) {
#pragma unroll
      for (int q = 0; q < C / 16; ++q) st4(sRows + 4 * lane + 256 * q, rows[q]);
    }
    wave_lds_fence();
    if (nlive == 0) return;

    f4 ca[4], cb[4], cc[4], cd[4], x, xnext;
    float xr;
    unsigned co, xo;  // element offsets of the lane's pieces of the edge's table row and of its sender's row
    const auto locate_group = [&](int s, unsigned &o_tab, unsigned &o_x, float &o_xr) {
      const int j = min(4 * s + row, nlive - 1);
      o_tab = static_cast<unsigned>(sIdx[j]) * (16u * C) + 4u * cl;
      o_x = static_cast<unsigned>(sS[j]) * C + 4u * cl;
      o_xr = sXr[j];
    };
    const auto request = [&](int L, unsigned o_tab) {
      const float *mid = sp.coeffs + (o_tab + 8 * C);
      ca[L] = ld4(mid + (L * C - 8 * C));
      cb[L] = ld4(mid + (L * C - 4 * C));
      cc[L] = ld4(mid + L * C);
      cd[L] = ld4(mid + (L * C + 4 * C));
    };
    locate_group(0, co, xo, xr);
    // in the loop's order: the waits in the loop count from the end of whichever way leads into it
    x = ld4(X + (xo + step_offset(0)));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int L = 0; L < 4; ++L) {
      request(L, co + step_offset(0));
      __builtin_amdgcn_sched_barrier(0);
    }

    const int ngroups = (nlive + 3) / 4;
    for (int s = 0; s < ngroups; ++s) {
      unsigned co_next, xo_next;
      float xr_next;
      locate_group(min(s + 1, ngroups - 1), co_next, xo_next, xr_next);
      const int j = min(4 * s + row, nlive - 1);
      const int orig = sOrig[j];
      // Two chains per sum over m >= 1, a lane's first and last two channels (the radial sum has one, of a product per step: its
      // four channels are added up first).  Error of the vector gradient against fp64, mean of four graphs, one edge per wave or
      // matrix products / one chain / two: 160 channels 2.504e-7 / - / 2.500e-7, 192 2.514 / 2.52 / 2.513, 224 2.560 / 2.57 / 2.563 (the
      // graphs differ by 0.04e-7; a second chain for the radial sum: 2.498, 2.511, 2.565).
      float y[16], p[16], r[16];
      staged_harmonics(sY, j, y);
#pragma unroll
      for (int m = 0; m < 16; ++m) p[m] = r[m] = 0.f;
      const float xr2 = 2.f * xr, xr3 = 3.f * xr * xr;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const bool last = h == H - 1;
        const int next_step = last ? step_offset(0) : step_offset(h + 1);
        const unsigned next_tab = (last ? co_next : co) + next_step;
        xnext = ld4(X + ((last ? xo_next : xo) + next_step));
        if (kHalf && last && twin) x = zero4();
        const float *rows_of_step = sRows + step_offset(h) + 4 * cl;
        f4 gxe = zero4(), grq = zero4();
        const auto degree = [&](auto lc) {
          constexpr int L = decltype(lc)::value;
          f4 g[2 * L + 1];
#pragma unroll
          for (int m = 0; m < 2 * L + 1; ++m) g[m] = ld4(rows_of_step + (L * L + m) * C);
          const f4 ra = ca[L], rb = cb[L], rc = cc[L], rd = cd[L];
          const f4 rl = ra + xr * (rb + xr * (rc + xr * rd));
          const f4 dr = rb + xr2 * rc + xr3 * rd;
          __builtin_amdgcn_sched_barrier(0);  // keeps the scheduler from collecting loads
          request(L, next_tab);
          f4 q = g[0];
          if constexpr (L > 0) {
            q = y[L * L] * g[0];
#pragma unroll
            for (int m = 1; m < 2 * L + 1; ++m) q += y[L * L + m] * g[m];
            if constexpr (WANT_GV) {
              const f4 t = x * rl;
#pragma unroll
              for (int m = 0; m < 2 * L + 1; ++m) {
                p[L * L + m] = fmaf(g[m].y, t.y, fmaf(g[m].x, t.x, p[L * L + m]));
                r[L * L + m] = fmaf(g[m].w, t.w, fmaf(g[m].z, t.z, r[L * L + m]));
              }
            }
          }
          if constexpr (WANT_GX) gxe += rl * q;
          if constexpr (WANT_GV) grq += q * dr;
          __builtin_amdgcn_sched_barrier(0);
        };
        degree(std::integral_constant<int, 0>{});
        degree(std::integral_constant<int, 1>{});
        degree(std::integral_constant<int, 2>{});
        degree(std::integral_constant<int, 3>{});
        if constexpr (WANT_GV) p[0] += dot4(x, grq);  // the radial sum in the place of m = 0, as above
        // unconditional: rows of lanes beyond the last edge have worked on the last edge and store its values again
        if constexpr (WANT_GX) st4_stream(gXe + static_cast<int64_t>(base + orig) * C + step_offset(h) + 4 * cl, gxe);
        x = xnext;
      }
      co = co_next, xo = xo_next, xr = xr_next;
      if constexpr (WANT_GV) {
#pragma unroll
        for (int m = 1; m < 16; ++m) p[m] += r[m];
        slot_reduce16<16>(p, cl);
        sY[j * 16 + reduced_index16<16>(cl)] = p[0];  // (a row beyond the last edge: the last edge's value again)
      }
    }
    if constexpr (!WANT_GV) return;
    wave_lds_fence();
    if (lane < nlive) {
      float sums[16];
      staged_harmonics(sY, lane, sums);
      finish_vector_gradient(sp.vec, base + sOrig[lane], sums, addend, gvec);
    }
  };
  chunk(std::true_type{});
  while (cursor < e1) chunk(std::false_type{});
}

// Parts of a receiver's edges in the forward pass, a wave each, all of one node in a workgroup.  A part is worth its place in the sum of the
// parts from four edges per slot on (three at eight slots), and a compute unit holds eight such waves: more nodes than one round of
// workgroups of p waves take fewer parts.  us at p = 1 2 3 4 5 6 8, the rule's p in brackets: 128 channels 216 x 52 18.9 12.1 11.2 10.8
// 10.6 [10.6] 11.7, 400 x 52 19.4 14.5 13.9 [14.2] 18.4 19.0 20.1, 60 x 30 11.0 8.3 [8.2] 8.4 8.3 8.7 9.8; 64 216 x 52 11.8 8.8 [8.5] 9.0 9.2 9.7
// 10.7, 1 000 x 30 [10.2] 11.6 15.7 17.5 28 30 34; 256 21 x 12 14.0 8.2 [7.5] 7.7 7.6 7.8 8.0, 300 x 9 12.8 [8.6] 8.6 8.9 11.9 12.1 12.9, 216 x 52
// 43.5 20.5 17.2 16.1 15.1 [15.1] 15.7; 192 672 x 9 14.7 [10.7] 11.6 12.2 15.7 15.9 17.4.
// At 160 channels a part is worth it from two edges per slot on, and up to one round of waves the kernel with parts also where there is one: a whole
// step, us, with parts from four edges per slot on and degree by degree -> as it is: 20 x 8 120 -> 108, 50 x 11 134 -> 119, 200 x 15 145 -> 135, 420 x 9 156 ->
// 150, 200 x 52 161 -> 156, 700 x 52 the same; at 224 channels, where 17 pieces of seven do not fit, no gain, and where two edges per slot are fetched at
// once one part is better off alone (1 260 x 9 x 32 channels 84 -> 86, 1 500 x 128 154 -> 156).
// With lengths and harmonics given a wave has less to wait for, and beyond two nodes per unit a part takes twelve edges (128 channels 1 000 x 20
// 13.3 in one, 14.5 in two).
template <int C, bool FROM_VEC>
int forward_parts(int64_t nnodes, int64_t nedges) {
  constexpr int kSlots = Cfg<C, true>::EPW, kLeast = kSlots >= 8 ? 24 : (Cfg<C, true>::V == 5 ? 2 : 4) * kSlots;
  if (nnodes <= 0) return 1;
  const int64_t least = !FROM_VEC && nnodes > 2 * device_compute_units() ? std::max(12, kLeast) : kLeast;
  int parts = static_cast<int>(std::min<int64_t>(6, std::max<int64_t>(1, nedges / (least * nnodes))));
  while (parts > 1 && nnodes > static_cast<int64_t>(device_compute_units()) * (8 / parts)) --parts;
  return parts;
}

// Parts of a receiver's edges in the backward edge pass, waves that share nothing: the number that takes the least time if a wave costs its
// edges and eight more (the gradient rows, the staging), waves run in rounds of what the chip holds, and a round that is
// filled by a share f takes 0.55 + 0.45 f of a full one.  us without / with gX at p = 1 2 3 4 6 8, the rule's p in brackets: 128 channels 216 x
// 52 26.1 / 40 16.2 / 24 12.3 / 19 10.4 / 17 9.3 / 15.6 [9.3 / 15.7], 700 x 52 28.7 / 43 [20.2 / 31] 22.3 / 33 21.8 / 33 23.8 / 36 25.2 / 37, 1 200 x 52
// 33.4 / 49 31.5 / 47 [28.5 / 43], 2 200 x 52 58 / 81 [53.5 / 75] 55.3 / 79, 3 300 x 52 [68.9 / 98.7] 67.5 / 98.5 72 / 106, 5 000 x 52 [105.6 / 149]
// 107 / 150 116 / 162, 2 500 x 12 [20.3 / 29.9] 22.1 / 32.4; 256 21 x 12 16.2 / 24 10.1 / 15.6 7.7 / 12.7 7.1 / 11.5 5.8 / 9.9 [5.3 / 9.5], 1 200 x 52 64 / 98 59 / 85
// [55 / 78]; 160 2 200 x 52 76 / 109 [67 / 98] 68 / 101.
// Up to 64 channels a wave's loads are a quarter or half of that, its start-up is not, and more than a round of waves never pays: eight
// waves per compute unit, five parts at most (400 x 52 x 64 five 8.1, eight 10.9), of two edges each, beyond two nodes per unit of 256 / C;
// two parts of 16 edges while they fit twelve waves.  (From lengths, two sets of operands and eight waves: no such two parts, 1 500 x 52 x 32 23.5
// in one, 26.0 in two, and twelve edges per part beyond two nodes per unit.)  us without gX at p = 1 2 3 4 5: 64 channels 21 x 9 6.2 5.3 4.8 4.6 [4.3], 120 x 52
// 17.1 10.1 8.4 7.4 [7.0], 500 x 52 17.3 10.7 9.8 [9.4] 10.4, 1 000 x 52 17.9 [13.4] 14.3 16.6 17.2, 1 500 x 52 21.9 [18.9] 20.9, 1 800 x 52 [23.3] 23.9
// 24.7, 2 000 x 52 [25.3] 26.6 26.4, 800 x 20 10.5 [8.6] 9.1, 1 200 x 20 [10.6] 10.5, 300 x 9 6.9 6.2 6.0 5.6 [5.8], 500 x 9 7.0 6.5 6.2 [6.4], 1 000 x
// 9 7.5 [7.4]; 32 channels 500 x 52 11.5 7.8 7.5 [7.4], 1 500 x 52 14.1 [12.2] 14.1, 2 000 x 52 [15.4] 16.8 17.6, 800 x 20 7.2 [6.8], 1 500 x 20 [8.2] 9.0,
// 1 000 x 9 [6.0] 6.6 7.6.
template <int C, bool FROM_VEC>
int backward_parts(int64_t nnodes, int64_t nedges) {
  if (nnodes <= 0) return 1;
  if constexpr (C <= 64) {
    const int64_t units = device_compute_units(), each = nedges / nnodes, least = nnodes <= 2 * units ? 2 : (FROM_VEC ? 256 / C : 12);
    const int64_t parts = std::min<int64_t>(5, std::min(8 * units / nnodes, (each + 1) / least));
    return static_cast<int>(FROM_VEC && parts < 2 && nnodes <= 6 * units && each >= 32 ? 2 : std::max<int64_t>(1, parts));
  }
  constexpr int kMost = 8;
  const double slots = device_compute_units() * 8.0;
  const double edges = static_cast<double>(nedges) / static_cast<double>(nnodes);
  int best = 1;
  double least = 0.0;
  for (int p = 1; p <= kMost && (p == 1 || edges >= p); ++p) {
    const double rounds = static_cast<double>(nnodes) * p / slots, full = std::floor(rounds);
    const double time = (full + (rounds > full ? 0.55 + 0.45 * (rounds - full) : 0.0)) * (edges / p + 8.0);
    if (p == 1 || time < least) best = p, least = time;
  }
  return best;
}

template <int C, bool FROM_VEC>
int launch_forward(const float *X, const float *Y, const Spline &sp, const int32_t *sender, const int32_t *first_occ,
                   int64_t nnodes, int64_t nedges, float *out, hipStream_t st) {
  const int parts = forward_parts<C, FROM_VEC>(nnodes, nedges);
  const size_t lds = static_cast<size_t>(parts) * kStageBytes + static_cast<size_t>(parts - 1) * 16 * C * sizeof(float);
  const int64_t one_round = 8 * device_compute_units();
  if (parts > 1 || (Cfg<C, true>::V == 5 && nnodes <= one_round))
    hipLaunchKernelGGL((mp_spline_forward_kernel<C, FROM_VEC, true>), dim3(static_cast<unsigned>(nnodes)), dim3(kWave * parts), lds, st,
                       X, Y, sp, sender, first_occ, static_cast<int>(nnodes), nedges, out);
  else
    hipLaunchKernelGGL((mp_spline_forward_kernel<C, FROM_VEC, false>), dim3(static_cast<unsigned>(nnodes)), dim3(kWave), lds, st, X, Y,
                       sp, sender, first_occ, static_cast<int>(nnodes), nedges, out);
  return check_launch(FROM_VEC ? "cm_mp_edge_forward" : "cm_mp_spline_forward");
}

// Whether the edge pass from edge vectors takes a group of four edges per step (mp_edge_backward_steps_kernel) or an edge per wave.
// At 160 channels always.  At 192 and 224 a receiver with few edges leaves most of its last group empty, and the rows of its
// gradient pass through LDS for nothing; at 224 the two are level as long as every SIMD has both its waves (the kernel with an
// edge per wave keeps the gradient rows in registers, the other reads them from LDS, which eight waves share), and the steps gain
// where a chip is partly filled.  us without / with gX, steps -> an edge per wave:
//   192  60 x 2.6 6.4 / 10.6 -> 5.6 / 10.1, 60 x 5 6.6 / 10.8 -> 7.1 / 11.6, 500 x 4.9 8.3 / 13.1 -> 7.9 / 12.7, 500 x 7 8.8 / 14.5 -> 9.2 / 15.0, 3 000 x 0.9 11.8 / 16.4 -> 9.6 / 14.3,
//        3 000 x 5 20.3 / 28.4 -> 19.7 / 27.8, 3 000 x 9.5 26.9 / 38.2 -> 28.1 / 39.7, 20 000 x 0.9 49 / 66 -> 42 / 58, 20 000 x 7 116 / 163 -> 118 / 164
//   224  500 x 1.7 7.8 / 12.4 -> 7.2 / 11.5, 1 000 x 2.6 8.7 / 13.5 -> 9.5 / 13.6, 500 x 3.8 8.2 / 12.8 -> 8.7 / 13.4, 3 000 x 5 24.0 / 33.7 -> 22.9 / 31.8, 3 000 x 9.5 32 / 45 -> 32.5 / 45,
//        20 000 x 1.7 77 / 99 -> 74 / 95, 20 000 x 2.7 87 / 114 -> 89 / 116, 20 000 x 3.8 99 / 132 -> 102 / 136; one round of waves: 500 x 52 (four parts) 23.5 / 34.4 -> 22.7 / 32.8,
//        1 000 x 52 (two) 38.4 / 55.1 -> 36.8 / 53.3, 2 048 x 12 24.9 / 35.9 -> 23.7 / 34.2; part of one: 216 x 52 13.8 / 22.2 -> 18.2 / 23.6,
//        1 200 x 52 50 / 77 -> 58 / 83
template <int C>
bool steps_of_four_edges(int64_t nnodes, int64_t nedges, int parts) {
  if constexpr (C == 160) return true;
  if constexpr (C == 192) return nedges >= 5 * nnodes;
  if constexpr (C == 224) {
    const int64_t waves = nnodes * parts;
    if (waves > 1536 && waves <= 2048) return false;
    return 2 * nedges >= (waves > 2048 && waves <= 8192 ? 10 : 5) * nnodes;
  }
  return false;
}

template <int C, bool FROM_VEC, bool GY, bool GR, bool GX>
void launch_edge(const float *X, const float *Y, const Spline &sp, const float *G, const int32_t *sender,
                 const int32_t *first_occ, int64_t nnodes, int64_t nedges, float *gY, float *g_r, float *gXe,
                 hipStream_t st) {
  const int parts = backward_parts<C, FROM_VEC>(nnodes, nedges);
  const dim3 grid(static_cast<unsigned>(nnodes * parts));
  if constexpr (FROM_VEC && (C == 160 || C == 192 || C == 224)) {
    if (steps_of_four_edges<C>(nnodes, nedges, parts)) {
      hipLaunchKernelGGL((mp_edge_backward_steps_kernel<C, GY, GX>), grid, dim3(kWave), 0, st, X, sp, G, sender, first_occ,
                         static_cast<int>(nnodes), nedges, gY, g_r, gXe, parts);
      return;
    }
  }
  if constexpr (!FROM_VEC || C != 160)
    hipLaunchKernelGGL((mp_spline_backward_edge_kernel<C, FROM_VEC, GY, GR, GX>), grid, dim3(kWave), 0, st, X, Y, sp, G, sender,
                       first_occ, static_cast<int>(nnodes), nedges, gY, g_r, gXe, parts);
}

// gY / g_r: outputs of the Y-and-r variant; in the FROM_VEC variant gY is the [E, 3] vector gradient and g_r, when given,
// an [E, 3] addend to it (read only).
template <int C, bool FROM_VEC>
int launch_backward(const float *X, const float *Y, const Spline &sp, const float *G, const int32_t *sender,
                    const int32_t *first_occ, const int32_t *perm, const int32_t *offsets, int64_t nnodes, int64_t nedges,
                    float *gX, float *gY, float *g_r, float *gXe, hipStream_t st) {
  if constexpr (FROM_VEC) {
    if (gY && gX) launch_edge<C, true, true, true, true>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st);
    else if (gY) launch_edge<C, true, true, true, false>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st);
    else if (gX) launch_edge<C, true, false, false, true>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st);
    else return CM_OK;
  } else {
    const int key = (gY ? 4 : 0) | (g_r ? 2 : 0) | (gX ? 1 : 0);
    switch (key) {
      case 7: launch_edge<C, false, true, true, true>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      case 6: launch_edge<C, false, true, true, false>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      case 5: launch_edge<C, false, true, false, true>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      case 4: launch_edge<C, false, true, false, false>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      case 3: launch_edge<C, false, false, true, true>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      case 2: launch_edge<C, false, false, true, false>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      case 1: launch_edge<C, false, false, false, true>(X, Y, sp, G, sender, first_occ, nnodes, nedges, gY, g_r, gXe, st); break;
      default: return CM_OK;
    }
  }
  int rc = check_launch(FROM_VEC ? "cm_mp_edge_backward (edge pass)" : "cm_mp_spline_backward (edge pass)");
  if (rc != CM_OK) return rc;
  if (gX) rc = mp::launch_sender_pass(C, gXe, perm, offsets, nnodes, nedges, gX, st, FROM_VEC ? sp.vec : nullptr,
                                      FROM_VEC ? nullptr : sp.r, sp.r_max, sp.live_bits);
  return rc;
}

int check_spline(const char *who, const float *r_or_vec, const float *r_knots, const float *coeffs, int nknots,
                 float r_width, int64_t nedges, int64_t nnodes, int channels) {
  // the kernels address X rows and table rows with 32-bit element offsets
  CM_REQUIRE(nnodes * channels < (int64_t{1} << 31) && static_cast<int64_t>(nknots) * 16 * channels < (int64_t{1} << 31),
             "%s: nnodes * channels or the spline table exceeds 32-bit element offsets", who);
  CM_REQUIRE(nknots >= 2, "%s: need at least two knots, got %d", who, nknots);
  CM_REQUIRE(r_width > 0.f, "%s: r_width must be positive", who);
  CM_REQUIRE(nedges == 0 || (r_or_vec && r_knots && coeffs), "%s: NULL spline operand", who);
  return CM_OK;
}

}  // namespace
}  // namespace cm

extern "C" int cm_mp_spline_forward(const float *X, const float *Y, const float *r, const float *r_knots,
                                    const float *coeffs, int nknots, float r_width, float r_max, const int32_t *sender,
                                    const int32_t *first_occ, int64_t nnodes, int64_t nedges, int channels, float *out,
                                    cm_stream_t stream) {
  CM_REQUIRE(cm_channels_supported(channels), "cm_mp_spline_forward: channels=%d must be a multiple of 32 in [32, 256]", channels);
  CM_REQUIRE(nedges >= 0 && nnodes >= 0, "cm_mp_spline_forward: negative size");
  CM_REQUIRE(nedges < INT32_MAX && nnodes < INT32_MAX / 2, "cm_mp_spline_forward: sizes exceed int32 indexing");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && first_occ && out, "cm_mp_spline_forward: NULL pointer");
  CM_REQUIRE(nedges == 0 || (Y && sender), "cm_mp_spline_forward: NULL edge operand");
  int rc = cm::check_spline("cm_mp_spline_forward", r, r_knots, coeffs, nknots, r_width, nedges, nnodes, channels);
  if (rc != CM_OK) return rc;
  const cm::Spline sp{nullptr, r, r_knots, coeffs, nknots, r_width, r_max};
  rc = CM_EINVAL;
  CM_DISPATCH_C(channels, rc = (cm::launch_forward<C_, false>(X, Y, sp, sender, first_occ, nnodes, nedges, out, cm::as_stream(stream))));
  return rc;
}

extern "C" int cm_mp_spline_backward(const float *X, const float *Y, const float *r, const float *r_knots,
                                     const float *coeffs, int nknots, float r_width, float r_max, const float *grad_out,
                                     const int32_t *sender, const int32_t *first_occ, const int32_t *sender_perm,
                                     const int32_t *sender_offsets, int64_t nnodes, int64_t nedges, int channels,
                                     float *gX, float *gY, float *grad_r, float *edge_scratch, cm_stream_t stream) {
  CM_REQUIRE(cm_channels_supported(channels), "cm_mp_spline_backward: channels=%d must be a multiple of 32 in [32, 256]", channels);
  CM_REQUIRE(nedges >= 0 && nnodes >= 0, "cm_mp_spline_backward: negative size");
  CM_REQUIRE(nedges < INT32_MAX && nnodes < INT32_MAX / 2, "cm_mp_spline_backward: sizes exceed int32 indexing");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && grad_out && first_occ, "cm_mp_spline_backward: NULL pointer");
  CM_REQUIRE(nedges == 0 || (Y && sender), "cm_mp_spline_backward: NULL edge operand");
  CM_REQUIRE(!gX || (sender_offsets && (nedges == 0 || (sender_perm && edge_scratch))),
             "cm_mp_spline_backward: gX wanted but sender_perm / sender_offsets / edge_scratch missing");
  int rc = cm::check_spline("cm_mp_spline_backward", r, r_knots, coeffs, nknots, r_width, nedges, nnodes, channels);
  if (rc != CM_OK) return rc;
  const cm::Spline sp{nullptr, r, r_knots, coeffs, nknots, r_width, r_max};
  rc = CM_EINVAL;
  CM_DISPATCH_C(channels, rc = (cm::launch_backward<C_, false>(X, Y, sp, grad_out, sender, first_occ, sender_perm, sender_offsets,
                                                               nnodes, nedges, gX, gY, grad_r, edge_scratch, cm::as_stream(stream))));
  return rc;
}

extern "C" int cm_mp_edge_forward_kernel(int64_t nnodes, int64_t nedges, int channels, int nknots) {
  return cm_channels_supported(channels) && nnodes > 0 && cm::mp::sliced_forward_applies(nnodes, nedges, channels, nknots) ? 1 : 0;
}

extern "C" int cm_mp_edge_backward_kernel(int64_t nnodes, int64_t nedges, int channels) {
  if (nnodes <= 0) return 0;
  bool steps = false;
  CM_DISPATCH_C(channels, steps = cm::steps_of_four_edges<C_>(nnodes, nedges, (cm::backward_parts<C_, true>(nnodes, nedges))));
  return steps ? 1 : 0;
}

extern "C" int cm_mp_edge_forward(const float *X, const float *vectors, const float *r_knots, const float *coeffs, int nknots,
                                  float r_width, float r_max, const int32_t *sender, const int32_t *first_occ,
                                  int64_t nnodes, int64_t nedges, int channels, float *out, cm_stream_t stream) {
  CM_REQUIRE(cm_channels_supported(channels), "cm_mp_edge_forward: channels=%d must be a multiple of 32 in [32, 256]", channels);
  CM_REQUIRE(nedges >= 0 && nnodes >= 0, "cm_mp_edge_forward: negative size");
  CM_REQUIRE(nedges < INT32_MAX / 3 && nnodes < INT32_MAX / 2, "cm_mp_edge_forward: sizes exceed int32 indexing");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && first_occ && out, "cm_mp_edge_forward: NULL pointer");
  CM_REQUIRE(nedges == 0 || sender, "cm_mp_edge_forward: NULL edge operand");
  int rc = cm::check_spline("cm_mp_edge_forward", vectors, r_knots, coeffs, nknots, r_width, nedges, nnodes, channels);
  if (rc != CM_OK) return rc;
  if (cm::mp::sliced_forward_applies(nnodes, nedges, channels, nknots))
    return cm::mp::launch_sliced_forward(X, vectors, nullptr, r_knots, coeffs, nknots, r_width, r_max, sender, first_occ, nnodes, nedges,
                                         channels, out, cm::as_stream(stream));
  const cm::Spline sp{vectors, nullptr, r_knots, coeffs, nknots, r_width, r_max};
  rc = CM_EINVAL;
  CM_DISPATCH_C(channels, rc = (cm::launch_forward<C_, true>(X, nullptr, sp, sender, first_occ, nnodes, nedges, out, cm::as_stream(stream))));
  return rc;
}

namespace cm {
namespace mp {

int edge_forward_parts(int channels, int64_t nnodes, int64_t nedges) {
  int parts = 1;
  CM_DISPATCH_C(channels, parts = (forward_parts<C_, true>(nnodes, nedges)));
  return parts;
}

int edge_forward_from_records(const float *X, const void *records, const float *r_knots, const float *coeffs, int nknots, float r_width,
                              float r_max, const int32_t *first_occ, int64_t nnodes, int64_t nedges, int channels, float *out, hipStream_t st) {
  const int rc = check_spline("cm_mace_step", static_cast<const float *>(records), r_knots, coeffs, nknots, r_width, nedges, nnodes, channels);
  if (rc != CM_OK) return rc;
  return launch_sliced_forward(X, nullptr, records, r_knots, coeffs, nknots, r_width, r_max, nullptr, first_occ, nnodes, nedges, channels, out, st);
}

int edge_backward_with_live_bits(const float *X, const float *vectors, const float *r_knots, const float *coeffs, int nknots, float r_width,
                                 float r_max, const float *grad_out, const int32_t *sender, const int32_t *first_occ, const int32_t *sender_perm,
                                 const int32_t *sender_offsets, int64_t nnodes, int64_t nedges, int channels, float *gX, float *grad_vectors,
                                 float *edge_scratch, const uint32_t *live_bits, hipStream_t st) {
  if (nnodes == 0) return CM_OK;
  int rc = check_spline("cm_mace_step", vectors, r_knots, coeffs, nknots, r_width, nedges, nnodes, channels);
  if (rc != CM_OK) return rc;
  const Spline sp{vectors, nullptr, r_knots, coeffs, nknots, r_width, r_max, live_bits};
  rc = CM_EINVAL;
  CM_DISPATCH_C(channels, rc = (launch_backward<C_, true>(X, nullptr, sp, grad_out, sender, first_occ, sender_perm, sender_offsets, nnodes, nedges,
                                                          gX, grad_vectors, nullptr, edge_scratch, st)));
  return rc;
}

// cm_mp_edge_backward without gX whose vector gradient is written as (this layer's gradient + addend[e]): saves the pass
// that adds two layers' gradients of the same edge vectors.  Arguments as checked by the caller (cm_mace_step).
int edge_backward_onto(const float *X, const float *vectors, const float *r_knots, const float *coeffs, int nknots, float r_width,
                       float r_max, const float *grad_out, const int32_t *sender, const int32_t *first_occ, int64_t nnodes,
                       int64_t nedges, int channels, float *grad_vectors, const float *addend, hipStream_t st) {
  if (nnodes == 0) return CM_OK;
  const Spline sp{vectors, nullptr, r_knots, coeffs, nknots, r_width, r_max};
  int rc = CM_EINVAL;
  CM_DISPATCH_C(channels, rc = (launch_backward<C_, true>(X, nullptr, sp, grad_out, sender, first_occ, nullptr, nullptr, nnodes, nedges,
                                                          nullptr, grad_vectors, const_cast<float *>(addend), nullptr, st)));
  return rc;
}

}  // namespace mp
}  // namespace cm

extern "C" int cm_mp_edge_backward(const float *X, const float *vectors, const float *r_knots, const float *coeffs, int nknots,
                                   float r_width, float r_max, const float *grad_out, const int32_t *sender,
                                   const int32_t *first_occ, const int32_t *sender_perm, const int32_t *sender_offsets,
                                   int64_t nnodes, int64_t nedges, int channels, float *gX, float *grad_vectors,
                                   float *edge_scratch, cm_stream_t stream) {
  CM_REQUIRE(cm_channels_supported(channels), "cm_mp_edge_backward: channels=%d must be a multiple of 32 in [32, 256]", channels);
  CM_REQUIRE(nedges >= 0 && nnodes >= 0, "cm_mp_edge_backward: negative size");
  CM_REQUIRE(nedges < INT32_MAX / 3 && nnodes < INT32_MAX / 2, "cm_mp_edge_backward: sizes exceed int32 indexing");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && grad_out && first_occ, "cm_mp_edge_backward: NULL pointer");
  CM_REQUIRE(nedges == 0 || sender, "cm_mp_edge_backward: NULL edge operand");
  CM_REQUIRE(!gX || (sender_offsets && (nedges == 0 || (sender_perm && edge_scratch))),
             "cm_mp_edge_backward: gX wanted but sender_perm / sender_offsets / edge_scratch missing");
  int rc = cm::check_spline("cm_mp_edge_backward", vectors, r_knots, coeffs, nknots, r_width, nedges, nnodes, channels);
  if (rc != CM_OK) return rc;
  const cm::Spline sp{vectors, nullptr, r_knots, coeffs, nknots, r_width, r_max};
  rc = CM_EINVAL;
  CM_DISPATCH_C(channels, rc = (cm::launch_backward<C_, true>(X, nullptr, sp, grad_out, sender, first_occ, sender_perm,
                                                              sender_offsets, nnodes, nedges, gX, grad_vectors, nullptr,
                                                              edge_scratch, cm::as_stream(stream))));
  return rc;
}
