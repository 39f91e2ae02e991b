// Invariant message passing in fp64: forward and backward.
//
// The reference dispatches its message-passing kernels on float and double
// (jit_wrappers/src/invariant_message_passing_wrapper.cpp:102, :189); the model runs them in fp32, the double path
// serves accuracy studies and gradient checks.  Same operands and outputs as the fp32 entry points, in double.
//
// Work decomposition: a lane owns four channels (two pairs, 2 cl and C / 2 + 2 cl, so that each of its two 16-byte accesses
// of a row is contiguous over the lanes), an edge occupies C / 4 lanes, and a wavefront is split into 64 / pow2ceil(C / 4)
// slots that walk the node's edge range interleaved (the forward two edges per slot and trip, their rows requested
// together).  The node's 16 x C accumulator (forward) or incoming gradient (backward) stays in registers; Y and sender of
// up to 64 edges are staged in LDS.  Where the nodes are few, a node's range is cut into parts of one wave each.  Sums run in a fixed
// order with no atomics: results are reproducible bit for bit.
//
// Bound: latency of a wave's trip at the sizes this path is used at (1 000 nodes x 30 edges x 64 channels: 155 MB of
// operands, 30 us at the rate of a copy).  With one lane per channel, one edge per trip and Y read through 16 dependent
// line look-ups the backward edge pass took 228 us there, 7.6 us per edge, the forward 32, the sender pass 17; now 34, 22
// and 7.
#include "mp_common.hpp"

namespace cm {
namespace {

using mp::kChunk;

typedef double d2 __attribute__((ext_vector_type(2)));

// The four channels of a lane in a row of C doubles: channels 2 cl, 2 cl + 1, C / 2 + 2 cl, C / 2 + 2 cl + 1.
struct Quad {
  d2 a, b;
  __device__ __forceinline__ Quad operator*(const Quad &o) const { return {a * o.a, b * o.b}; }
  __device__ __forceinline__ Quad operator*(double y) const { return {a * y, b * y}; }
};
__device__ __forceinline__ Quad fma(Quad x, double y, Quad z) {
  return {d2{::fma(x.a.x, y, z.a.x), ::fma(x.a.y, y, z.a.y)}, d2{::fma(x.b.x, y, z.b.x), ::fma(x.b.y, y, z.b.y)}};
}
__device__ __forceinline__ Quad fma(Quad x, Quad y, Quad z) {
  return {d2{::fma(x.a.x, y.a.x, z.a.x), ::fma(x.a.y, y.a.y, z.a.y)}, d2{::fma(x.b.x, y.b.x, z.b.x), ::fma(x.b.y, y.b.y, z.b.y)}};
}
__device__ __forceinline__ double dot(Quad x, Quad y) { return ::fma(x.b.y, y.b.y, ::fma(x.b.x, y.b.x, ::fma(x.a.y, y.a.y, x.a.x * y.a.x))); }
__device__ __forceinline__ Quad zero_quad() { return {d2{0.0, 0.0}, d2{0.0, 0.0}}; }
__device__ __forceinline__ Quad ld_quad(const double *row, int cl, int C) {
  return {*reinterpret_cast<const d2 *>(row + 2 * cl), *reinterpret_cast<const d2 *>(row + C / 2 + 2 * cl)};
}
__device__ __forceinline__ Quad ld_quad_stream(const double *row, int cl, int C) {
  return {__builtin_nontemporal_load(reinterpret_cast<const d2 *>(row + 2 * cl)),
          __builtin_nontemporal_load(reinterpret_cast<const d2 *>(row + C / 2 + 2 * cl))};
}
__device__ __forceinline__ void st_quad(double *row, int cl, int C, Quad v) {
  *reinterpret_cast<d2 *>(row + 2 * cl) = v.a;
  *reinterpret_cast<d2 *>(row + C / 2 + 2 * cl) = v.b;
}

// Value of `v` in the lane OFF away (lane ^ OFF); inside a quad by a DPP move, else through the LDS crossbar.
template <int OFF>
__device__ __forceinline__ double from_lane_xor(double v) {
  if constexpr (OFF <= 2) {
    constexpr int ctrl = OFF == 1 ? 0xB1 : 0x4E;
    const unsigned long long w = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(w), ctrl, 0xf, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(w >> 32), ctrl, 0xf, 0xf, false);
    return __builtin_bit_cast(double, static_cast<unsigned long long>(hi) << 32 | lo);
  } else {
    return __shfl_xor(v, OFF);
  }
}

template <int OFF, int HALF>
__device__ __forceinline__ void halve(double (&p)[16], int cl) {
  const bool up = (cl & OFF) != 0;
#pragma unroll
  for (int i = 0; i < HALF; ++i) {
    const double keep = up ? p[HALF + i] : p[i];
    const double give = up ? p[i] : p[HALF + i];
    p[i] = keep + from_lane_xor<OFF>(give);
  }
}

// Sums p[m] over the SW lanes of a slot by a butterfly that halves what a lane holds: 8 + 4 + 2 + 1 exchanges.  The lane
// then holds in p[0] (and p[1] where the slot has eight lanes) the totals of the components reduced_index(cl) + {0, 1}.
template <int SW>
__device__ __forceinline__ void slot_reduce16_f64(double (&p)[16], int cl) {
  halve<1, 8>(p, cl);
  halve<2, 4>(p, cl);
  halve<4, 2>(p, cl);
  if constexpr (SW >= 16) halve<8, 1>(p, cl);
  if constexpr (SW >= 32) p[0] += from_lane_xor<16>(p[0]);
  if constexpr (SW >= 64) p[0] += from_lane_xor<32>(p[0]);
}
template <int SW>
__device__ __forceinline__ int reduced_index_f64(int cl) {
  return ((cl & 1) << 3) | ((cl & 2) << 1) | ((cl & 4) >> 1) | (SW >= 16 ? (cl & 8) >> 3 : 0);
}

// Y[0:16, base:base+cnt] transposed to [edge][16] and sender[base:base+cnt] into LDS (one wave)
__device__ __forceinline__ void stage_chunk_f64(const double *__restrict__ Y, const int32_t *__restrict__ sender, int64_t nedges,
                                                int base, int cnt, int lane, double *sY, int *sS) {
  if (lane < cnt) {
    const int64_t e = base + lane;
    sS[lane] = sender[e];
    double y[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) y[m] = Y[m * nedges + e];
#pragma unroll
    for (int m = 0; m < 16; m += 2) *reinterpret_cast<d2 *>(sY + lane * 16 + m) = d2{y[m], y[m + 1]};
  }
}

// The rows a slot needs for one edge: the four radial rows (streamed) and the sender's features.
struct EdgeRows {
  Quad r[4], x;
};
template <bool WANT_R>
__device__ __forceinline__ EdgeRows load_rows(const double *__restrict__ X, const double *__restrict__ R, int64_t e, int s, int nnodes,
                                              int cl, int C) {
  EdgeRows o;
#pragma unroll
  for (int l = 0; l < 4; ++l) o.r[l] = WANT_R ? ld_quad_stream(R + e * (4 * C) + l * C, cl, C) : zero_quad();
  o.x = static_cast<unsigned>(s) < static_cast<unsigned>(nnodes) ? ld_quad(X + static_cast<int64_t>(s) * C, cl, C) : zero_quad();
  return o;
}

// Part `part` of `parts` of a node's edge range.
__device__ __forceinline__ void take_part(int &e0, int &e1, int part, int parts) {
  const int64_t len = e1 - e0;
  const int lo = e0 + static_cast<int>(len * part / parts);
  e1 = e0 + static_cast<int>(len * (part + 1) / parts);
  e0 = lo;
}

// One workgroup per receiver node, one wave per part of its edges; the parts' sums are added by the first wave in the
// order of the parts.
constexpr size_t kForwardLdsPerWave = kChunk * 16 * sizeof(double) + kChunk * sizeof(int);
template <int SW>
__global__ __launch_bounds__(4 * kWave) void mp_forward_f64_kernel(const double *__restrict__ X, const double *__restrict__ Y,
                                                                  const double *__restrict__ R, const int32_t *__restrict__ sender,
                                                                  const int32_t *__restrict__ first_occ, int nnodes, int64_t nedges,
                                                                  int C, double *__restrict__ out) {
  constexpr int EPW = kWave / SW;
  extern __shared__ __attribute__((aligned(16))) double lds[];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, parts = blockDim.x / kWave;
  double *sY = lds + wave * (kForwardLdsPerWave / sizeof(double));
  int *sS = reinterpret_cast<int *>(sY + kChunk * 16);
  const int slot = lane / SW, cl = lane % SW;
  const bool active = cl < C / 4;
  const int node = blockIdx.x;
  int e0 = first_occ[node];
  int e1 = first_occ[nnodes + node];
  clamp_edge_range(e0, e1, nedges);
  take_part(e0, e1, wave, parts);
  Quad acc[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) acc[m] = zero_quad();

  for (int base = e0; base < e1; base += kChunk) {
    const int cnt = min(kChunk, e1 - base);
    wave_lds_fence();
    stage_chunk_f64(Y, sender, nedges, base, cnt, lane, sY, sS);
    wave_lds_fence();
    if (active) {
      auto add = [&](const EdgeRows &o, int j) {
        const d2 *yp = reinterpret_cast<const d2 *>(sY + j * 16);
        const Quad t[4] = {o.x * o.r[0], o.x * o.r[1], o.x * o.r[2], o.x * o.r[3]};
#pragma unroll
        for (int m = 0; m < 16; m += 2) {
          const d2 y = yp[m / 2];
          acc[m] = fma(t[l_of_m(m)], y.x, acc[m]);
          acc[m + 1] = fma(t[l_of_m(m + 1)], y.y, acc[m + 1]);
        }
      };
      int j = slot;
      for (; j + EPW < cnt; j += 2 * EPW) {
        const EdgeRows o0 = load_rows<true>(X, R, base + j, sS[j], nnodes, cl, C);
        const EdgeRows o1 = load_rows<true>(X, R, base + j + EPW, sS[j + EPW], nnodes, cl, C);
        add(o0, j);
        add(o1, j + EPW);
      }
      if (j < cnt) add(load_rows<true>(X, R, base + j, sS[j], nnodes, cl, C), j);
    }
  }
#pragma unroll
  for (int off = kWave / 2; off >= SW; off >>= 1) {
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      acc[m].a.x += __shfl_down(acc[m].a.x, off), acc[m].a.y += __shfl_down(acc[m].a.y, off);
      acc[m].b.x += __shfl_down(acc[m].b.x, off), acc[m].b.y += __shfl_down(acc[m].b.y, off);
    }
  }
  if (parts > 1) {
    // four components at a time through LDS (the staging area is free by then): 4 C doubles per part
    double *comb = lds;
    for (int m0 = 0; m0 < 16; m0 += 4) {
      __syncthreads();
      if (wave > 0 && slot == 0 && active) {
#pragma unroll
        for (int m = 0; m < 16; ++m)
          if (m / 4 == m0 / 4) st_quad(comb + ((wave - 1) * 4 + m % 4) * C, cl, C, acc[m]);
      }
      __syncthreads();
      if (wave == 0 && slot == 0 && active) {
#pragma unroll
        for (int m = 0; m < 16; ++m) {
          if (m / 4 != m0 / 4) continue;
          for (int w = 1; w < parts; ++w) {
            const Quad v = ld_quad(comb + ((w - 1) * 4 + m % 4) * C, cl, C);
            acc[m].a += v.a;
            acc[m].b += v.b;
          }
        }
      }
    }
  }
  if (wave == 0 && slot == 0 && active) {
#pragma unroll
    for (int m = 0; m < 16; ++m) st_quad(out + (static_cast<int64_t>(node) * 16 + m) * C, cl, C, acc[m]);
  }
}

// One wave per (receiver node, part of its edges): every output is per edge.
template <int SW, bool WANT_GY, bool WANT_GR, bool WANT_GX>
__global__ __launch_bounds__(kWave, 2) void mp_backward_edge_f64_kernel(
    const double *__restrict__ X, const double *__restrict__ Y, const double *__restrict__ R, const double *__restrict__ G,
    const int32_t *__restrict__ sender, const int32_t *__restrict__ first_occ, int nnodes, int64_t nedges, int C,
    double *__restrict__ gY, double *__restrict__ gR, double *__restrict__ gXe) {
  constexpr int EPW = kWave / SW;
  __shared__ __attribute__((aligned(16))) double sY[kChunk * 16];
  __shared__ int sS[kChunk];
  __shared__ double sGY[WANT_GY ? 16 * kChunk : 1];
  const int lane = threadIdx.x, slot = lane / SW, cl = lane % SW;
  const bool active = cl < C / 4;
  const int node = blockIdx.x;
  int e0 = first_occ[node];
  int e1 = first_occ[nnodes + node];
  clamp_edge_range(e0, e1, nedges);
  take_part(e0, e1, blockIdx.y, gridDim.y);
  if (e0 >= e1) return;

  Quad g[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) g[m] = active ? ld_quad(G + (static_cast<int64_t>(node) * 16 + m) * C, cl, C) : zero_quad();

  for (int base = e0; base < e1; base += kChunk) {
    const int cnt = min(kChunk, e1 - base);
    wave_lds_fence();  // the workgroup is this one wave
    stage_chunk_f64(Y, sender, nedges, base, cnt, lane, sY, sS);
    wave_lds_fence();
    auto load = [&](int j) -> EdgeRows {
      if (active) return load_rows<WANT_GY || WANT_GX>(X, R, base + j, sS[j], nnodes, cl, C);
      return {{zero_quad(), zero_quad(), zero_quad(), zero_quad()}, zero_quad()};
    };
    auto one = [&](const EdgeRows &o, int j) {
      const int64_t e = base + j;
      if constexpr (WANT_GR || WANT_GX) {
        const d2 *yp = reinterpret_cast<const d2 *>(sY + j * 16);
        Quad q[4] = {zero_quad(), zero_quad(), zero_quad(), zero_quad()};
#pragma unroll
        for (int m = 0; m < 16; m += 2) {
          const d2 y = yp[m / 2];
          q[l_of_m(m)] = fma(g[m], y.x, q[l_of_m(m)]);
          q[l_of_m(m + 1)] = fma(g[m + 1], y.y, q[l_of_m(m + 1)]);
        }
        if (active) {
          if constexpr (WANT_GR) {
#pragma unroll
            for (int l = 0; l < 4; ++l) st_quad(gR + e * (4 * C) + l * C, cl, C, o.x * q[l]);
          }
          if constexpr (WANT_GX)
            st_quad(gXe + e * C, cl, C, fma(o.r[3], q[3], fma(o.r[2], q[2], fma(o.r[1], q[1], o.r[0] * q[0]))));
        }
      }
      if constexpr (WANT_GY) {
        const Quad t[4] = {o.x * o.r[0], o.x * o.r[1], o.x * o.r[2], o.x * o.r[3]};
        double p[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) p[m] = dot(g[m], t[l_of_m(m)]);
        slot_reduce16_f64<SW>(p, cl);
        const int m = reduced_index_f64<SW>(cl);
        if (cl < 16) sGY[m * kChunk + j] = p[0];
        if constexpr (SW == 8) sGY[(m + 1) * kChunk + j] = p[1];
      }
    };
    // Every lane of a slot takes part in the reduction, so the loop bound is slot-uniform.  One edge per slot and trip: two
    // with their rows requested together do not fit the 256 registers that two waves per SIMD leave (39 us instead of 34,
    // with spills at two waves per SIMD and without at one alike).
    for (int j = slot; j < cnt; j += EPW) one(load(j), j);
    if constexpr (WANT_GY) {
      wave_lds_fence();
      if (lane < cnt) {
#pragma unroll
        for (int m = 0; m < 16; ++m) gY[m * nedges + base + lane] = sGY[m * kChunk + lane];
      }
    }
  }
}

// gX[n, :] = sum, in the order of the sender-sorted view, of the per-edge rows gXe[e, :] of the edges sent by n.  Lane i
// owns channels i, i + 64, ...; the rows of eight edges are requested together and added in order.
template <int KS>
__global__ __launch_bounds__(kWave) void mp_backward_sender_f64_kernel(const double *__restrict__ gXe,
                                                                      const int32_t *__restrict__ perm,
                                                                      const int32_t *__restrict__ offsets, int64_t nedges,
                                                                      int C, double *__restrict__ gX) {
  constexpr int B = 8;
  const int lane = threadIdx.x;
  const int node = blockIdx.x;
  double acc[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k) acc[k] = 0.0;
  const int q1 = offsets[node + 1];
  for (int q = offsets[node]; q < q1; q += B) {
    int e[B];
    double row[B][KS];
#pragma unroll
    for (int j = 0; j < B; ++j) e[j] = q + j < q1 ? perm[q + j] : -1;
#pragma unroll
    for (int j = 0; j < B; ++j) {
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const int c = lane + kWave * k;
        const bool take = static_cast<unsigned>(e[j]) < static_cast<uint64_t>(nedges) && c < C;
        row[j][k] = take ? gXe[static_cast<int64_t>(e[j]) * C + c] : 0.0;
      }
    }
#pragma unroll
    for (int j = 0; j < B; ++j)
#pragma unroll
      for (int k = 0; k < KS; ++k) acc[k] += row[j][k];
  }
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    const int c = lane + kWave * k;
    if (c < C) gX[static_cast<int64_t>(node) * C + c] = acc[k];
  }
}

// Parts a node's edge range is cut into where one wave per node would leave most of the device idle (a 216-atom cell is
// 216 waves for 1 024 SIMDs, each walking its ~90 edges one after the other): as many as fill about 2 048 wave slots
// and leave a part a dozen edges on average, at most 8.
inline int parts_for(int64_t nnodes, int64_t nedges) {
  if (nnodes <= 0) return 1;
  const int64_t by_slots = 2048 / nnodes, by_edges = nedges / (12 * nnodes);
  const int64_t parts = by_slots < by_edges ? by_slots : by_edges;
  return parts < 1 ? 1 : (parts > 8 ? 8 : static_cast<int>(parts));
}

template <int SW>
void launch_forward(const double *X, const double *Y, const double *R, const int32_t *sender, const int32_t *first_occ, int64_t nnodes,
                    int64_t nedges, int C, double *out, hipStream_t st) {
  const int parts = std::min(parts_for(nnodes, nedges), 4);  // a wave's 16 x 4 fp64 sums leave room for four waves per workgroup
  hipLaunchKernelGGL(mp_forward_f64_kernel<SW>, dim3(static_cast<unsigned>(nnodes)), dim3(parts * kWave),
                     static_cast<unsigned>(parts * kForwardLdsPerWave), st, X, Y, R, sender, first_occ, static_cast<int>(nnodes), nedges,
                     C, out);
}

template <int SW, bool GY, bool GR, bool GX>
void launch_edge(const double *X, const double *Y, const double *R, const double *G, const int32_t *sender,
                 const int32_t *first_occ, int64_t nnodes, int64_t nedges, int C, double *gY, double *gR, double *gXe,
                 hipStream_t st) {
  const int parts = parts_for(nnodes, nedges);
  hipLaunchKernelGGL((mp_backward_edge_f64_kernel<SW, GY, GR, GX>), dim3(static_cast<unsigned>(nnodes), parts), dim3(kWave), 0, st,
                     X, Y, R, G, sender, first_occ, static_cast<int>(nnodes), nedges, C, gY, gR, gXe);
}

template <int SW>
int launch_backward(const double *X, const double *Y, const double *R, const double *G, const int32_t *sender,
                    const int32_t *first_occ, const int32_t *perm, const int32_t *offsets, int64_t nnodes, int64_t nedges,
                    int C, double *gX, double *gY, double *gR, double *gXe, hipStream_t st) {
  const int key = (gY ? 4 : 0) | (gR ? 2 : 0) | (gX ? 1 : 0);
  switch (key) {
    case 7: launch_edge<SW, true, true, true>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    case 6: launch_edge<SW, true, true, false>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    case 5: launch_edge<SW, true, false, true>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    case 4: launch_edge<SW, true, false, false>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    case 3: launch_edge<SW, false, true, true>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    case 2: launch_edge<SW, false, true, false>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    case 1: launch_edge<SW, false, false, true>(X, Y, R, G, sender, first_occ, nnodes, nedges, C, gY, gR, gXe, st); break;
    default: return CM_OK;
  }
  int rc = check_launch("cm_mp_backward_f64 (edge pass)");
  if (rc != CM_OK || !gX) return rc;
  const dim3 grid(static_cast<unsigned>(nnodes)), block(kWave);
  switch (static_cast<int>(ceil_div(C, kWave))) {
    case 1: hipLaunchKernelGGL(mp_backward_sender_f64_kernel<1>, grid, block, 0, st, gXe, perm, offsets, nedges, C, gX); break;
    case 2: hipLaunchKernelGGL(mp_backward_sender_f64_kernel<2>, grid, block, 0, st, gXe, perm, offsets, nedges, C, gX); break;
    case 3: hipLaunchKernelGGL(mp_backward_sender_f64_kernel<3>, grid, block, 0, st, gXe, perm, offsets, nedges, C, gX); break;
    default: hipLaunchKernelGGL(mp_backward_sender_f64_kernel<4>, grid, block, 0, st, gXe, perm, offsets, nedges, C, gX); break;
  }
  return check_launch("cm_mp_backward_f64 (sender pass)");
}

}  // namespace
}  // namespace cm

// SW_: lanes of a slot, the power of two that holds channels / 4
#define CM_DISPATCH_SW(channels, ...)                         \
  switch (cm::mp::pow2ceil((channels) / 4)) {                 \
    case 8: { constexpr int SW_ = 8; __VA_ARGS__; break; }    \
    case 16: { constexpr int SW_ = 16; __VA_ARGS__; break; }  \
    case 32: { constexpr int SW_ = 32; __VA_ARGS__; break; }  \
    default: { constexpr int SW_ = 64; __VA_ARGS__; break; }  \
  }

extern "C" int cm_mp_forward_f64(const double *X, const double *Y, const double *R, const int32_t *sender,
                                 const int32_t *first_occ, int64_t nnodes, int64_t nedges, int channels, double *out,
                                 cm_stream_t stream) {
  CM_REQUIRE(cm_channels_supported(channels), "cm_mp_forward_f64: channels=%d must be a multiple of 32 in [32, 256]", channels);
  CM_REQUIRE(nedges >= 0 && nnodes >= 0, "cm_mp_forward_f64: negative size");
  CM_REQUIRE(nedges < INT32_MAX && nnodes < INT32_MAX / 2, "cm_mp_forward_f64: sizes exceed int32 indexing");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && first_occ && out, "cm_mp_forward_f64: NULL pointer");
  CM_REQUIRE(nedges == 0 || (Y && R && sender), "cm_mp_forward_f64: NULL edge operand");
  CM_DISPATCH_SW(channels, cm::launch_forward<SW_>(X, Y, R, sender, first_occ, nnodes, nedges, channels, out, cm::as_stream(stream)));
  return cm::check_launch("cm_mp_forward_f64");
}

extern "C" int cm_mp_backward_f64(const double *X, const double *Y, const double *R, const double *grad_out,
                                  const int32_t *sender, const int32_t *first_occ, const int32_t *sender_perm,
                                  const int32_t *sender_offsets, int64_t nnodes, int64_t nedges, int channels, double *gX,
                                  double *gY, double *gR, double *edge_scratch, cm_stream_t stream) {
  CM_REQUIRE(cm_channels_supported(channels), "cm_mp_backward_f64: channels=%d must be a multiple of 32 in [32, 256]", channels);
  CM_REQUIRE(nedges >= 0 && nnodes >= 0, "cm_mp_backward_f64: negative size");
  CM_REQUIRE(nedges < INT32_MAX && nnodes < INT32_MAX / 2, "cm_mp_backward_f64: sizes exceed int32 indexing");
  if (nnodes == 0) return CM_OK;
  CM_REQUIRE(X && grad_out && first_occ, "cm_mp_backward_f64: NULL pointer");
  CM_REQUIRE(nedges == 0 || (Y && R && sender), "cm_mp_backward_f64: NULL edge operand");
  CM_REQUIRE(!gX || (sender_offsets && (nedges == 0 || (sender_perm && edge_scratch))),
             "cm_mp_backward_f64: gX wanted but sender_perm / sender_offsets / edge_scratch missing");
  int rc = CM_EINVAL;
  CM_DISPATCH_SW(channels, rc = cm::launch_backward<SW_>(X, Y, R, grad_out, sender, first_occ, sender_perm, sender_offsets, nnodes,
                                                         nedges, channels, gX, gY, gR, edge_scratch, cm::as_stream(stream)));
  return rc;
}
