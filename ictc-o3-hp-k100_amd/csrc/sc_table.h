// Symmetric-contraction kernels over per-species coefficient tables, for the shapes of ScTab
// (generated/ictc_sc.h).  Layouts and outputs are those of sc_kernels.h.
//
// The per-node kernels form the weight combination of every (output, monomial) pair per node and channel, and
// are bound by VALU issue: 10,817 multiply-adds per node and channel for (3,2,3), of which all but 1,503 (one
// per pair) and about 1,000 (the monomials) depend on the species alone.  Here table_kernel forms the pairs'
// coefficients once per call, [S][groups][PAIRS][64] (64 channels a group, zero past C), and a wave evaluates
// B nodes of one species at a time from the species-sorted order, one table row of 256 bytes per pair: the
// four waves of a block take nodes of the same species, so three of their four reads of a row hit in L1.
// The weight gradient sums go[k] m(x) per pair over a chunk of nodes (one multiply-add per pair and node
// instead of one per term), adds the chunks in order, and contracts pairs with weights once at the end.
// Deterministic: every sum runs in a fixed order.
#pragma once
#include <algorithm>

#include "sc_kernels.h"

namespace ictc {
namespace sc {

constexpr int kPairBlock = 64;   // pairs per weight-gradient wave (PAIR_BLOCK in gen_sc.py)
constexpr int kTabDwWaves = 4096;   // about this many waves per weight gradient

struct TabArgs {
  const float* x;
  const float* table;     // [S][groups][PAIRS][64]
  const int32_t* ptr;     // [S+2] species-sorted CSR: nodes of species s at order[ptr[s] .. ptr[s+1]), others last
  const int32_t* order;   // [N]
  int64_t nodes;
  int num_species;
  int channels;
};

// Nodes per weight-gradient chunk (at least 32): the chunks, channel groups and pair blocks together make about
// kTabDwWaves waves.
inline int64_t tab_chunks(int64_t pairs, int channels) {
  const int64_t waves = ((channels + 63) / 64) * ((pairs + kPairBlock - 1) / kPairBlock);
  return (kTabDwWaves + waves - 1) / waves;
}
inline int64_t tab_chunk(int64_t nodes, int64_t pairs, int channels) {
  const int64_t chunks = tab_chunks(pairs, channels);
  const int64_t c = ((nodes + chunks - 1) / chunks + 31) / 32 * 32;
  return c < 32 ? 32 : c;
}
inline int64_t tab_max_chunks(int64_t nodes, int64_t pairs, int channels, int species) {
  const int64_t c = tab_chunk(nodes, pairs, channels);
  return (nodes + c - 1) / c + species;
}
// As many or more, and never fewer for more nodes (the chunks of a call fall where their nodes step up by 32).
inline int64_t tab_most_chunks(int64_t nodes, int64_t pairs, int channels, int species) {
  return std::min((nodes + 31) / 32, tab_chunks(pairs, channels)) + species;
}
inline int64_t tab_floats(int64_t pairs, int channels, int species) {
  return (int64_t)species * ((channels + 63) / 64) * pairs * 64;
}

template <class T, class Tab>
__global__ __launch_bounds__(256) void table_kernel(ScWeights w, int C, float* __restrict__ table) {
  const int r = (int)blockIdx.x * kWaves + wave_id(), g = blockIdx.y, s = blockIdx.z, l = lane_id();
  if (r >= Tab::PAIRS) return;
  const int c = 64 * g + l;
  float acc = 0.f;
  if (c < C) {
    // all terms of a pair have its degree and output degree, so one weight block: only the path varies
    const int beg = Tab::TERM_PTR[r], end = Tab::TERM_PTR[r + 1];
    const int q0 = Tab::TERM_Q[beg], L = T::WQ[q0][0], nu = T::WQ[q0][1], p0 = T::WQ[q0][2];
    const float* row = w.w[L][nu] + ((int64_t)s * T::P[L][nu] + p0) * C + c;
#pragma unroll 8
    for (int t = beg; t < end; ++t) acc = fmaf(Tab::TERM_V[t], row[(int64_t)(Tab::TERM_Q[t] - q0) * C], acc);
  }
  table[(((int64_t)s * gridDim.y + g) * Tab::PAIRS + r) * 64 + l] = acc;
}

// Tiles of `per` nodes that species t (0 .. S, S the out-of-range tail) takes; 0 past S.
__device__ __forceinline__ int32_t species_tiles(const int32_t* __restrict__ ptr, int S, int t, int32_t per, int32_t& beg,
                                                 int32_t& end) {
  beg = end = 0;
  if (t <= S) beg = ptr[t], end = ptr[t + 1];
  return (end - beg + per - 1) / per;
}

// Species and sorted range of node tile `blk` (`per` nodes a tile, tiles never straddle a species; species S is the
// out-of-range tail): false past the last tile.  Up to kWalk species a walk over them, a chain of scalar loads ((3,2),
// 8,191 nodes of 128 channels and 10 species, feature gradient: 125 us); above that the wave's 64
// lanes take 64 species at a time and scan their tile counts (with the walk alone, forward and feature gradient of
// (2,2) over 131,072 nodes took 2,404 us with 1,000 species; 755 with the scan).
constexpr int kWalk = 32;
__device__ __forceinline__ bool species_tile(const int32_t* __restrict__ ptr, int S, int64_t blk, int32_t per, int& s,
                                             int32_t& beg, int32_t& end) {
  if (S <= kWalk) {
    int64_t k = blk;
    for (s = 0; s <= S; ++s) {
      const int32_t b = ptr[s], e = ptr[s + 1], n = (e - b + per - 1) / per;
      if (k < n) {
        beg = b + (int32_t)k * per;
        end = min(e, beg + per);
        return true;
      }
      k -= n;
    }
    return false;
  }
  int64_t k = blk;
  for (int s0 = 0; s0 <= S; s0 += 64) {
    int32_t b, e;
    const int32_t n = species_tiles(ptr, S, s0 + lane_id(), per, b, e);
    int32_t incl = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t v = __shfl_up(incl, d, 64);
      if (lane_id() >= d) incl += v;
    }
    // (lane reads, not shuffles: the result stays in scalar registers, and with it the table's base address)
    const int32_t total = __builtin_amdgcn_readlane(incl, 63);
    if (k < total) {
      const int f = __ffsll((unsigned long long)__ballot(k < incl)) - 1;
      s = s0 + f;
      beg = __builtin_amdgcn_readlane(b, f) + (int32_t)(k - __builtin_amdgcn_readlane(incl - n, f)) * per;
      end = min(__builtin_amdgcn_readlane(e, f), beg + per);
      return true;
    }
    k -= total;
  }
  return false;
}

// First tile and tile count of species s, in the same way (all 64 lanes call it).
__device__ __forceinline__ void tiles_of(const int32_t* __restrict__ ptr, int S, int s, int32_t per, int32_t& first,
                                         int32_t& count) {
  int32_t before = 0, b, e;
  for (int t = lane_id(); t < s; t += 64) before += species_tiles(ptr, S, t, per, b, e);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) before += __shfl_xor(before, d, 64);
  first = __builtin_amdgcn_readfirstlane(before);
  count = species_tiles(ptr, S, s, per, b, e);
}

// MODE 0: out = SC(x); 1: out = J(x) h; 2: out = grad (go . SC); 3: out = Hess(go . SC) h.
template <class T, class Tab, int MODE, int B, int WAVES>
__global__ __launch_bounds__(256, WAVES) void tab_kernel(TabArgs a, const float* __restrict__ go,
                                                         const float* __restrict__ h, float* __restrict__ out) {
  constexpr bool kDx = MODE >= 2, kTan = MODE == 1 || MODE == 3;
  constexpr int NOUT = kDx ? T::NX : T::NO;
  int s;
  int32_t beg, end;
  if (!species_tile(a.ptr, a.num_species, blockIdx.x, B * kWaves, s, beg, end)) return;
  beg += B * wave_id();
  const int nb = min(end - beg, B);
  if (nb <= 0) return;
  const int C = a.channels, g = blockIdx.y;
  const int c = min(64 * g + lane_id(), C - 1);   // idle lanes read the last channel and store nothing
  const bool active = 64 * g + lane_id() < C;
  int64_t n[B];
#pragma unroll
  for (int b = 0; b < B; ++b) n[b] = a.order[beg + (b < nb ? b : 0)];
  float o[B][NOUT];
#pragma unroll
  for (int b = 0; b < B; ++b)
#pragma unroll
    for (int k = 0; k < NOUT; ++k) o[b][k] = 0.f;
  if (s < a.num_species) {
    float x[B][T::NX];
#pragma unroll
    for (int b = 0; b < B; ++b) load<T::NX>(a.x + n[b] * (int64_t)(T::NX * C), C, c, x[b]);
    const float* t = a.table + ((int64_t)s * gridDim.y + g) * (Tab::PAIRS * 64);
    const uint32_t off = sc_lane_offset(lane_id());
    if constexpr (MODE == 0) {
      Tab::template fwd<B>(x, t, off, o);
    } else {
      float hv[kTan ? B : 1][T::NX], gv[kDx ? B : 1][T::NO];
      if constexpr (kTan) {
#pragma unroll
        for (int b = 0; b < B; ++b) load<T::NX>(h + n[b] * (int64_t)(T::NX * C), C, c, hv[b]);
      }
      if constexpr (kDx) {
#pragma unroll
        for (int b = 0; b < B; ++b) load<T::NO>(go + n[b] * (int64_t)(T::NO * C), C, c, gv[b]);
      }
      if constexpr (MODE == 1) Tab::template jvp<B>(x, hv, t, off, o);
      if constexpr (MODE == 2) Tab::template dx<B>(x, gv, t, off, o);
      if constexpr (MODE == 3) Tab::template hvp<B>(x, hv, gv, t, off, o);
    }
  }
#pragma unroll
  for (int b = 0; b < B; ++b)
    if (active && b < nb) store<NOUT>(out + n[b] * (int64_t)(NOUT * C), C, c, o[b]);
}

template <class T, class Tab, int MODE, int Q>
__device__ __forceinline__ void tab_dw_block(const TabArgs& a, const float* __restrict__ go,
                                             const float* __restrict__ h, int32_t beg, int32_t end, int c,
                                             float* __restrict__ prow) {
  constexpr int R0 = Q * kPairBlock, NR = Tab::PAIRS - R0 < kPairBlock ? Tab::PAIRS - R0 : kPairBlock;
  const int C = a.channels;
  float acc[kPairBlock];
#pragma unroll
  for (int r = 0; r < kPairBlock; ++r) acc[r] = 0.f;
  // the next node's rows load while this node's products run
  float x0[T::NX], g0[T::NO], h0[MODE ? T::NX : 1], x1[T::NX], g1[T::NO], h1[MODE ? T::NX : 1];
  auto fetch = [&](int32_t k, float* xv, float* gv, float* hv) {
    const int64_t n = a.order[k];
    load<T::NX>(a.x + n * (int64_t)(T::NX * C), C, c, xv);
    load<T::NO>(go + n * (int64_t)(T::NO * C), C, c, gv);
    if constexpr (MODE == 1) load<T::NX>(h + n * (int64_t)(T::NX * C), C, c, hv);
  };
  auto add = [&](const float* xv, const float* gv, const float* hv) {
    if constexpr (MODE == 0) Tab::template dw<Q>(xv, gv, acc);
    else Tab::template dwjvp<Q>(xv, hv, gv, acc);
  };
  fetch(beg, x0, g0, h0);
  for (int32_t k = beg; k < end; k += 2) {
    if (k + 1 < end) fetch(k + 1, x1, g1, h1);
    add(x0, g0, h0);
    if (k + 1 >= end) break;
    if (k + 2 < end) fetch(k + 2, x0, g0, h0);
    add(x1, g1, h1);
  }
  store<NR>(prow + R0 * (int64_t)C, C, c, acc);
}

template <class T, class Tab, int MODE, int Q = 0>
__device__ __forceinline__ void tab_dw_blocks(int q, const TabArgs& a, const float* __restrict__ go,
                                              const float* __restrict__ h, int32_t beg, int32_t end, int c,
                                              float* __restrict__ prow) {
  if constexpr (Q < Tab::NB) {
    if (q == Q) tab_dw_block<T, Tab, MODE, Q>(a, go, h, beg, end, c, prow);
    else tab_dw_blocks<T, Tab, MODE, Q + 1>(q, a, go, h, beg, end, c, prow);
  }
}

// Pair sums of one chunk, one channel group and one block of pairs per wave: partial [chunk][PAIRS][C].
// blockIdx.x = chunk * ceil(NB / 4) + quarter: the blocks of one chunk run together and share its rows in L2.
template <class T, class Tab, int MODE>
__global__ __launch_bounds__(256) void tab_dw_kernel(TabArgs a, const float* __restrict__ go,
                                                     const float* __restrict__ h, int32_t per,
                                                     float* __restrict__ partial) {
  constexpr int kQuarters = (Tab::NB + kWaves - 1) / kWaves;
  const int64_t chunk = blockIdx.x / kQuarters;
  const int q = (int)(blockIdx.x % kQuarters) * kWaves + wave_id();
  int s;
  int32_t beg, end;
  if (q >= Tab::NB || !species_tile(a.ptr, a.num_species, chunk, per, s, beg, end) || s >= a.num_species) return;
  const int c = 64 * (int)blockIdx.y + lane_id();
  if (c >= a.channels) return;
  tab_dw_blocks<T, Tab, MODE>(q, a, go, h, beg, end, c, partial + chunk * (int64_t)(Tab::PAIRS * a.channels));
}

// The chunks of each species added in order, into its first (partial [chunk][PAIRS][C], `row` floats a chunk).
template <int = 0>
__global__ __launch_bounds__(256) void tab_dw_sum_kernel(const int32_t* __restrict__ ptr, int S, int32_t per, int64_t row,
                                                         float* __restrict__ partial) {
  int32_t k, n;
  tiles_of(ptr, S, blockIdx.y, per, k, n);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= row || n < 2) return;
  float* p = partial + k * row + i;
  float acc = *p;
  for (int32_t j = 1; j < n; ++j) acc += p[j * row];
  *p = acc;
}

// dW(L, nu)[s, p, c] = sum over the pairs of weight q of factor * (the species' sums)[pair][c]; 0 without nodes.
template <class T, class Tab>
__global__ __launch_bounds__(256) void tab_dw_weights_kernel(const int32_t* __restrict__ ptr, int S, int32_t per,
                                                             const float* __restrict__ partial, int C, WeightGrads g) {
  const int q = (int)blockIdx.x * kWaves + wave_id(), s = blockIdx.z, c = 64 * (int)blockIdx.y + lane_id();
  int32_t k, n;
  tiles_of(ptr, S, s, per, k, n);
  if (q >= T::NW || c >= C) return;
  float acc = 0.f;
  if (n > 0) {
    const float* row = partial + k * ((int64_t)Tab::PAIRS * C) + c;
#pragma unroll 8
    for (int t = Tab::WEIGHT_PTR[q]; t < Tab::WEIGHT_PTR[q + 1]; ++t)
      acc = fmaf(Tab::WEIGHT_V[t], row[(int64_t)Tab::WEIGHT_R[t] * C], acc);
  }
  const int L = T::WQ[q][0], nu = T::WQ[q][1], p = T::WQ[q][2];
  float* dst = g.w[L][nu];
  if (dst) dst[((int64_t)s * T::P[L][nu] + p) * C + c] = acc;
}

// Launchers (one specialisation per sc_part_tab_*.hip).
template <class T>
struct TabLaunch {
  static hipError_t table(const ScWeights& w, int S, int C, float* table, hipStream_t st);
  static hipError_t apply(const TabArgs& a, const float* go, const float* h, float* out, int mode, hipStream_t st);
  static hipError_t dw(const TabArgs& a, const float* go, const float* h, float* const* dw, float* partial,
                       hipStream_t st);
};

// Nodes per wave (B) and waves per SIMD of each mode.  More nodes share a table row's load but need the
// registers of their features and sums.  Measured (us; per-node kernels in brackets, forward / J h / feature
// gradient / Hess h): (3,2) over 8,191 nodes of 128 channels (384 / 603 / 438 / 464) 121 / 151 / 144 / 176 with
// three nodes, 149 / 159 / 158 / 181 with two, 120 / 162 / 159 / 297 with four; (3,1) over 8,191 of 64 channels
// (78 / 102 / 97 / 101) 34 / 46 / 45 / 65 with three.  (2,2) over 131,072 of 64 channels (266 / 346 / 329 / 340)
// 190 / 245 / 240 with four, Hess h 303 with three; three nodes 228 / 263 / 251.
template <class T, int MODE>
struct TabTile {
  static constexpr bool wide = T::NX > 9;
  static constexpr int B = wide || MODE == 3 ? 3 : 4;
  static constexpr int WAVES = MODE == 0 || (wide && MODE == 2) ? 3 : 2;
};

template <class T, class Tab, int MODE>
inline hipError_t tab_apply(const TabArgs& a, const float* go, const float* h, float* out, hipStream_t st) {
  constexpr int B = TabTile<T, MODE>::B, WAVES = TabTile<T, MODE>::WAVES;
  const int64_t per = B * kWaves;
  const dim3 grid((unsigned)((a.nodes + per - 1) / per + a.num_species + 1), (a.channels + 63) / 64);
  hipLaunchKernelGGL((tab_kernel<T, Tab, MODE, B, WAVES>), grid, dim3(256), 0, st, a, go, h, out);
  return hipGetLastError();
}

#define ICTC_SC_TAB_DEFINE(A, B, C)                                                                                   \
  template <>                                                                                                         \
  hipError_t TabLaunch<Sc<A, B, C>>::table(const ScWeights& w, int S, int ch, float* table, hipStream_t st) {         \
    using Tab = ScTab<A, B, C>;                                                                                       \
    const dim3 grid((Tab::PAIRS + kWaves - 1) / kWaves, (ch + 63) / 64, S);                                           \
    hipLaunchKernelGGL((table_kernel<Sc<A, B, C>, Tab>), grid, dim3(256), 0, st, w, ch, table);                       \
    return hipGetLastError();                                                                                         \
  }                                                                                                                   \
  template <>                                                                                                         \
  hipError_t TabLaunch<Sc<A, B, C>>::apply(const TabArgs& a, const float* go, const float* h, float* out, int mode,   \
                                           hipStream_t st) {                                                          \
    using T = Sc<A, B, C>;                                                                                            \
    using Tab = ScTab<A, B, C>;                                                                                       \
    if (mode == 0) return tab_apply<T, Tab, 0>(a, go, h, out, st);                                          \
    if (mode == 1) return tab_apply<T, Tab, 1>(a, go, h, out, st);                                          \
    if (mode == 2) return tab_apply<T, Tab, 2>(a, go, h, out, st);                                          \
    return tab_apply<T, Tab, 3>(a, go, h, out, st);                                                         \
  }

#define ICTC_SC_TAB_DEFINE_DW(A, B, C)                                                                                \
  template <>                                                                                                         \
  hipError_t TabLaunch<Sc<A, B, C>>::dw(const TabArgs& a, const float* go, const float* h, float* const* dwp,         \
                                        float* partial, hipStream_t st) {                                             \
    using T = Sc<A, B, C>;                                                                                            \
    using Tab = ScTab<A, B, C>;                                                                                       \
    const int64_t per = tab_chunk(a.nodes, Tab::PAIRS, a.channels),                                                    \
                  chunks = tab_max_chunks(a.nodes, Tab::PAIRS, a.channels, a.num_species);                            \
    const int64_t row = (int64_t)Tab::PAIRS * a.channels;                                                             \
    const unsigned G = (a.channels + 63) / 64;                                                                        \
    const dim3 grid((unsigned)(chunks * ((Tab::NB + kWaves - 1) / kWaves)), G);                                       \
    if (!h) hipLaunchKernelGGL((tab_dw_kernel<T, Tab, 0>), grid, dim3(256), 0, st, a, go, h, (int32_t)per, partial);  \
    else hipLaunchKernelGGL((tab_dw_kernel<T, Tab, 1>), grid, dim3(256), 0, st, a, go, h, (int32_t)per, partial);     \
    hipLaunchKernelGGL(tab_dw_sum_kernel<0>, dim3((unsigned)((row + 255) / 256), a.num_species), dim3(256), 0, st,    \
                       a.ptr, a.num_species, (int32_t)per, row, partial);                                             \
    WeightGrads g;                                                                                                    \
    for (int L = 0; L < 4; ++L)                                                                                       \
      for (int n = 0; n < 3; ++n) g.w[L][n] = T::P[L][n] > 0 ? dwp[L * 3 + n] : nullptr;                              \
    hipLaunchKernelGGL((tab_dw_weights_kernel<T, Tab>), dim3((T::NW + kWaves - 1) / kWaves, G, a.num_species),        \
                       dim3(256), 0, st, a.ptr, a.num_species, (int32_t)per, partial, a.channels, g);                 \
    return hipGetLastError();                                                                                         \
  }

#define ICTC_SC_TAB_DECLARE(A, B, C)                                                                                  \
  template <>                                                                                                         \
  hipError_t TabLaunch<Sc<A, B, C>>::table(const ScWeights&, int, int, float*, hipStream_t);                          \
  template <>                                                                                                         \
  hipError_t TabLaunch<Sc<A, B, C>>::apply(const TabArgs&, const float*, const float*, float*, int, hipStream_t);     \
  template <>                                                                                                         \
  hipError_t TabLaunch<Sc<A, B, C>>::dw(const TabArgs&, const float*, const float*, float* const*, float*,            \
                                        hipStream_t);
ICTC_FOR_EACH_SC_TAB(ICTC_SC_TAB_DECLARE)

}  // namespace sc
}  // namespace ictc
