// Device code of the spline-fused message passing (mp_spline.hip, whose head has the formulas) and of the kernels that take a node
// through a whole layer (few_nodes.hip).  Both use the staging of a node's edges, the operands and products of one edge of the backward pass and
// the end of its vector gradient.  Staged, SlotSums and forward_wave are few_nodes.hip's alone: a second writing of the loop of
// mp_spline_forward_kernel, which reads its knots and lays out its LDS otherwise and has variants that this one does not need.  Both sum in
// the same order and must stay alike: the step of few nodes is compared with the separate launches bit for bit in the tests.
#pragma once

#include <type_traits>

#include "mp_common.hpp"
#include "sh_device.hpp"

namespace cm {
namespace mp {

struct Spline {
  const float *vec;     // [E, 3] edge vectors (FROM_VEC variants; then r is unused)
  const float *r;       // [E]
  const float *knots;   // [nknots]
  const float *coeffs;  // [nknots - 1, 4, 4C]
  int nknots;
  float r_width;
  float r_max;
  const uint32_t *live_bits = nullptr;  // backward with gX: a bit per edge within r_max, or NULL (the sender pass then looks at vec or r)
};

// Knot interval (or -1 beyond the cutoff) and offset inside it for one edge length.  lds_knots: a copy of the knots in LDS,
// read instead of the one in memory if use_lds.
__device__ __forceinline__ void locate(const Spline &sp, float re, int &idx, float &x, const float *lds_knots = nullptr,
                                       bool use_lds = false) {
  idx = -1;
  x = 0.f;
  if (re <= sp.r_max) {
    idx = static_cast<int>(re / sp.r_width);
    idx = idx < 0 ? 0 : (idx > sp.nknots - 2 ? sp.nknots - 2 : idx);
    // The markers keep each read and its use inside its branch: merged, the two become one read through a generic
    // address, or one subtraction behind a wait for the read of memory, on the path that reads LDS as well.
    if (use_lds) {
      x = re - lds_knots[idx];
      asm volatile("; offset from the knot in LDS" : "+v"(x));
    } else {
      x = re - sp.knots[idx];
      asm volatile("; offset from the knot in memory" : "+v"(x));
    }
  }
}

// Stages up to kChunk LIVE edges of a node -- those inside the cutoff whose sender index is valid -- densely, in their
// original order: sender, Y (as [edge][16]), knot interval, offset inside it, and the position of the edge counted from
// `first` (the value of `base` on entry).  Raw edges are read kChunk at a time until kChunk live ones are staged or the
// node's edges are used up, so a neighbour list with a skin (a quarter of its pairs beyond the cutoff) fills the chunk
// all the same, and the edges beyond the cutoff cost nothing after this point.  `base` advances past every raw edge that
// was consumed; `dead(pass_base, consumed, live_mask, lane_is_dead)` is called once per pass for the consumed edges that
// are not live (the backward writes their zeros there).  Returns the number of staged edges (the same in every lane).
// FROM_VEC: Y and the length come from the edge vector; otherwise from the Y and r arrays.
// `ahead` (AHEAD, FROM_VEC only): sender and vector of edge base + lane, which the caller asked for before it
// called (so that loads it issued in between do not stand in front of them in the queue); used by the first pass.
struct RawEdge {
  int s;
  float v0, v1, v2;
};
template <bool FROM_VEC, bool AHEAD = false, class DeadFn>
__device__ __forceinline__ int stage_edges(const float *__restrict__ Y, const int32_t *__restrict__ sender, const Spline &sp,
                                           int nnodes, int64_t nedges, int &base, int e1, int lane, float *sY, int *sS,
                                           int *sIdx, float *sXr, int *sOrig, DeadFn dead,
                                           RawEdge ahead = RawEdge{-1, 0.f, 0.f, 0.f}, const float *lds_knots = nullptr,
                                           bool use_lds_knots = false) {
  static_assert(FROM_VEC || !AHEAD, "raw edges are handed in for the edge-vector variant only");
  const int first = base;
  int nlive = 0;
  // one pass over up to kChunk raw edges; the first one is written out on its own where its raw edges are handed in, so
  // that its waits are not those of a pass that has just issued its loads
  auto pass = [&](auto use_ahead) {
    const int cnt = min(kChunk, e1 - base);
    int s = -1, idx = -1;
    float x = 0.f;
    float y[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) y[m] = 0.f;
    if (lane < cnt) {
      const int64_t e = base + lane;
      if constexpr (FROM_VEC) {
        float v0, v1, v2;
        if constexpr (decltype(use_ahead)::value) {
          s = ahead.s, v0 = ahead.v0, v1 = ahead.v1, v2 = ahead.v2;
        } else {
          s = sender[e], v0 = sp.vec[3 * e + 0], v1 = sp.vec[3 * e + 1], v2 = sp.vec[3 * e + 2];
        }
        locate(sp, edge_length(v0, v1, v2), idx, x, lds_knots, use_lds_knots);
        sh::eval(sh::direction(v0, v1, v2), y);
      } else {
        s = sender[e];
        locate(sp, sp.r[e], idx, x, lds_knots, use_lds_knots);
#pragma unroll
        for (int m = 0; m < 16; ++m) y[m] = Y[m * nedges + e];
      }
    }
    const bool live = lane < cnt && idx >= 0 && static_cast<unsigned>(s) < static_cast<unsigned>(nnodes);
    const unsigned long long live_mask = __ballot(live);
    const int pos = nlive + __popcll(live_mask & ((1ull << lane) - 1ull));
    const int nlive_pass = __popcll(live_mask);
    // raw edges consumed by this pass: all of them, or those up to the live edge that fills the last place
    int consumed = cnt;
    if (nlive + nlive_pass > kChunk) consumed = __ffsll(static_cast<long long>(__ballot(live && pos == kChunk - 1)));
    if (live && pos < kChunk) {
      sS[pos] = s;
      sIdx[pos] = idx;
      sXr[pos] = x;
      sOrig[pos] = base - first + lane;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f4 *>(sY + pos * 16 + 4 * q) = f4{y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]};
    }
    dead(base, consumed, live_mask, lane < consumed && !live);
    nlive = min(kChunk, nlive + nlive_pass);
    base += consumed;
  };
  if constexpr (AHEAD) {
    if (base < e1) pass(std::true_type{});
  }
  while (nlive < kChunk && base < e1) pass(std::false_type{});
  return nlive;
}

constexpr int kKnotsInLds = 512;  // knots the backward edge pass keeps in LDS (more, or fewer than four, are read from memory)

// A wave's copy of the knots on its way to LDS, four per lane and load (a load instruction occupies the L1 path for 16 cycles
// whatever its width; one dword per lane took eight of them, as many as half an edge does).
template <int kMost = kKnotsInLds>
struct KnotCopy {
  static constexpr int kLoads = kMost / (4 * kWave);
  typedef float Four __attribute__((ext_vector_type(4), aligned(4)));  // the caller's array may start at any float
  Four v[kLoads];
  __device__ __forceinline__ static bool applies(const Spline &sp) { return sp.nknots >= 4 && sp.nknots <= kMost; }
  __device__ __forceinline__ static int at(const Spline &sp, int lane, int q) { return min(4 * (lane + kWave * q), sp.nknots - 4); }
  __device__ __forceinline__ void request(const Spline &sp, int lane) {
    if (!applies(sp)) return;
#pragma unroll
    for (int q = 0; q < kLoads; ++q)
      if (q == 0 || sp.nknots > 4 * kWave * q) v[q] = *reinterpret_cast<const Four *>(sp.knots + at(sp, lane, q));
  }
  __device__ __forceinline__ void store(const Spline &sp, int lane, float *lds) const {
#pragma unroll
    for (int q = 0; q < kLoads; ++q)
      if (q == 0 || sp.nknots > 4 * kWave * q) {
        float *to = lds + at(sp, lane, q);
        to[0] = v[q].x, to[1] = v[q].y, to[2] = v[q].z, to[3] = v[q].w;
      }
  }
};

template <int L>
struct MRange {
  static constexpr int lo = L * L;
  static constexpr int hi = (L + 1) * (L + 1);
};

// LDS of one wave's staged chunk: harmonics [kChunk][16], then sender, knot interval, offset in it and position of every edge
constexpr int kStageBytes = kChunk * 64 + 4 * kChunk * 4;
struct Staged {
  float *sY;
  int *sS, *sIdx;
  float *sXr;
  int *sOrig;
  __device__ __forceinline__ explicit Staged(unsigned char *at)
      : sY(reinterpret_cast<float *>(at)), sS(reinterpret_cast<int *>(at + kChunk * 64)), sIdx(sS + kChunk),
        sXr(reinterpret_cast<float *>(sIdx + kChunk)), sOrig(reinterpret_cast<int *>(sXr + kChunk)) {}
};

// The slots of a wave have sums of their own (a vector per row m and lane); total() adds them up, (s0 + s2) + (s1 + s3) for four slots, and
// leaves every lane with kRows of the node's 16 rows, from first_row on: a stage swaps half of the rows against the other half of the
// lanes, so that it adds where a plain exchange of all 16 rows through LDS (ds_bpermute, one per value) took as many again.
template <class K>
struct SlotSums {
  using vec = typename K::vec;
  static constexpr int kRows = K::SW >= 64 ? 16 : (K::SW == 32 ? 8 : 4);
  __device__ static __forceinline__ int first_row(int lane) { return K::SW >= 64 ? 0 : (K::SW == 32 ? 8 * (lane / 32) : 4 * (2 * (lane / 32) + lane / 16 % 2)); }
  // the lane has a share of the result (each share is held once)
  __device__ static __forceinline__ bool holds(int lane) { return lane % K::SW < K::LPE && (K::SW > 8 || (lane & 8) == 0); }
  template <int N, class Swap>
  __device__ static __forceinline__ void halve(vec (&acc)[16], Swap swap) {
#pragma unroll
    for (int m = 0; m < N; ++m)
#pragma unroll
      for (int i = 0; i < K::V; ++i) {
        const auto both = swap(__float_as_uint(acc[m][i]), __float_as_uint(acc[N + m][i]));
        const unsigned first = both[0], second = both[1];  // element-wise copies, as in slot_reduce16
        acc[m][i] = __uint_as_float(first) + __uint_as_float(second);
      }
  }
  __device__ static __forceinline__ void total(vec (&acc)[16]) {
    if constexpr (K::SW <= 32) halve<8>(acc, [](unsigned p, unsigned q) { return __builtin_amdgcn_permlane32_swap(p, q, false, false); });
    if constexpr (K::SW <= 16) halve<4>(acc, [](unsigned p, unsigned q) { return __builtin_amdgcn_permlane16_swap(p, q, false, false); });
    if constexpr (K::SW == 8) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int i = 0; i < K::V; ++i) acc[m][i] += dpp_move<0x128>(acc[m][i]);
    }
  }
};

// A wave's sums over the edges e0 .. e1 - 1 of a node, in each slot: acc[m] for the lane's channels.  The loop of mp_spline_forward_kernel's
// several waves per node (up to four channels per lane).  lds_knots: a copy of the knots in LDS, or NULL.
template <int C>
__device__ __forceinline__ void forward_wave(const float *__restrict__ X, const Spline &sp,
                                             const int32_t *__restrict__ sender, int nnodes, int64_t nedges, int e0, int e1, const Staged &st,
                                             typename Cfg<C, true>::vec (&acc)[16], const float *lds_knots = nullptr) {
  using K = Cfg<C, true>;
  using vec = typename K::vec;
  const int lane = threadIdx.x % kWave;
  const int slot = lane / K::SW;
  const int cl = lane % K::SW;
  const bool active = cl < K::LPE;
  float *const sY = st.sY;
  int *const sS = st.sS, *const sIdx = st.sIdx;
  float *const sXr = st.sXr;
  int *const sOrig = st.sOrig;
#pragma unroll
  for (int m = 0; m < 16; ++m) acc[m] = zerov<vec>();

  for (int base = e0; base < e1;) {
    wave_lds_fence();  // the staged edges belong to this wave alone
    const int nlive = stage_edges<true>(nullptr, sender, sp, nnodes, nedges, base, e1, lane, sY, sS, sIdx, sXr, sOrig,
                                            [](int, int, unsigned long long, bool) {}, RawEdge{-1, 0.f, 0.f, 0.f}, lds_knots,
                                            lds_knots != nullptr);
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
    }
  }
}

// what an edge brings in: the sender's row piece and the 16 pieces of its knot interval
template <class K>
struct Operands {
  typename K::vec x, ca[4], cb[4], cc[4], cd[4];
  float xr;
};

template <int C, class K>
__device__ __forceinline__ void fetch_operands(Operands<K> &o, const float *__restrict__ X, const float *__restrict__ tab, int s, int idx,
                                               float xr, unsigned cla) {
  o.xr = xr;
  o.x = K::ld(X + (static_cast<unsigned>(s) * C + unsigned(K::off(cla))));
  const unsigned co = static_cast<unsigned>(idx) * (16u * C) + unsigned(K::off(cla));
#pragma unroll
  for (int L = 0; L < 4; ++L) {
    // addressed from the middle of the interval's 16C-float row (offsets within +-8C floats: one address and
    // immediate offsets, up to C = 128)
    const float *mid = tab + (co + 8 * C);
    o.ca[L] = K::ld(mid + (L * C - 8 * C));
    o.cb[L] = K::ld(mid + (L * C - 4 * C));
    o.cc[L] = K::ld(mid + L * C);
    o.cd[L] = K::ld(mid + (L * C + 4 * C));
  }
}

// A lane's part of one edge: p[m] = sum over its channels of X R_l(m) g_m, gxe = sum_l R_l q_l and grq = sum_l q_l dR_l/dr.
// kConstantFirst: the harmonic m = 0 is the constant 1 and its gradient is not wanted (p[0] is left alone).
template <class K, bool kConstantFirst, bool WANT_GY, bool WANT_GR, bool WANT_GX>
__device__ __forceinline__ void edge_products(const Operands<K> &o, const float (&y)[16], const typename K::vec (&g)[16], float (&p)[16],
                                              typename K::vec &gxe, typename K::vec &grq) {
  using vec = typename K::vec;
  const float xr = o.xr;
  const float xr2 = 2.f * xr, xr3 = 3.f * xr * xr;
  auto per_l = [&](auto lc) {
    constexpr int L = decltype(lc)::value;
    const vec a = o.ca[L], b = o.cb[L], c = o.cc[L], d = o.cd[L];
    const vec rl = a + xr * (b + xr * (c + xr * d));
    vec q = zerov<vec>();
    if constexpr (kConstantFirst && L == 0) {
      q = g[0];
    } else {
#pragma unroll
      for (int m = MRange<L>::lo; m < MRange<L>::hi; ++m) q += y[m] * g[m];
    }
    if constexpr (WANT_GY && !(kConstantFirst && L == 0)) {
      const vec t = o.x * rl;
#pragma unroll
      for (int m = MRange<L>::lo; m < MRange<L>::hi; ++m) p[m] = dotv(g[m], t);
    }
    if constexpr (WANT_GX) gxe += rl * q;
    if constexpr (WANT_GR) grq += q * (b + xr2 * c + xr3 * d);  // q_l * dR_l/dr
  };
  per_l(std::integral_constant<int, 0>{});
  per_l(std::integral_constant<int, 1>{});
  per_l(std::integral_constant<int, 2>{});
  per_l(std::integral_constant<int, 3>{});
}

// the 16 staged harmonics of edge j
__device__ __forceinline__ void staged_harmonics(const float *sY, int j, float (&y)[16]) {
  const f4 *yp = reinterpret_cast<const f4 *>(sY + j * 16);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f4 v = yp[q];
    y[4 * q] = v.x, y[4 * q + 1] = v.y, y[4 * q + 2] = v.z, y[4 * q + 3] = v.w;
  }
}

// Gradient with respect to the vector of edge e: harmonics Jacobian applied to the reduced sums gy, plus the radial sum (in the
// place of m = 0) along the direction.  addend: an optional [E, 3] array (another layer's gradient of the same
// vectors) to write the sum with; formed from the rounded value, as a separate addition pass would form it.
__device__ __forceinline__ void finish_vector_gradient(const float *vec, int64_t e, const float (&gy)[16], const float *addend, float *gvec) {
  const float v0 = vec[3 * e + 0], v1 = vec[3 * e + 1], v2 = vec[3 * e + 2];
  const sh::Direction d = sh::direction(v0, v1, v2);
  float gin[3];
  sh::vjp(d, gy, gin);
  const float gr = gy[0];
  float o0 = gin[0] + gr * d.y, o1 = gin[1] + gr * d.z, o2 = gin[2] + gr * d.x;
  if (addend) {
    o0 = __fadd_rn(o0, addend[3 * e + 0]);
    o1 = __fadd_rn(o1, addend[3 * e + 1]);
    o2 = __fadd_rn(o2, addend[3 * e + 2]);
  }
  gvec[3 * e + 0] = o0;
  gvec[3 * e + 1] = o1;
  gvec[3 * e + 2] = o2;
}

}  // namespace mp
}  // namespace cm
