// gb_sssp_small.hpp -- delta-stepping inside one workgroup, distances in LDS.
//
// A graph whose distances fit the 160 KB LDS of a CU (32768 vertices with
// 4-byte distances, 16384 with 8-byte ones) is solved by one workgroup of
// 1024 threads per source: distances, the set of vertices waiting to be
// expanded (one bit each) and the queue of a round live in LDS, so a round is
// a few block barriers instead of two kernel launches, and relaxing an edge
// is an LDS atomic instead of an L2 one.  Only row bounds and edges come from
// memory.  A round moves the waiting vertices below the current threshold to
// the queue, then spreads their edges evenly over the 1024 lanes (block-wide
// prefix sum of the degrees, one bit per edge slot where a vertex's edges begin).  When nothing waits
// below the threshold it moves to the smallest waiting distance plus a width.
// The width starts at the caller's delta and doubles while a threshold's
// rounds hold too few edges to keep the lanes busy: the distances are exact
// for any sequence of thresholds, and a round of few edges costs its barriers
// and memory latencies whatever it relaxes.
// What bounds it: one CU's memory parallelism, about 1 ns per edge (R-MAT 12,
// one source: 112 K relaxations in 20 rounds, 170 us, where the engine took
// 1360 us in 96 phases of two launches); LDS reads and atomics are not the
// limit (fewer of them measured the same).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gb_device.hpp"

constexpr int SM_BLOCK = 1024;
constexpr int SM_WAVES = SM_BLOCK / GB_WAVE;
constexpr int SM_QCAP = 8192;  // queued vertices per round; the rest wait on
constexpr int SM_U = 4;        // edge slots per lane in flight
constexpr int SM_SWEEP = SM_U * SM_BLOCK;
static_assert(SM_SWEEP / 64 == GB_WAVE, "a lane holds one word of a sweep's start bits");
// fewer edges than this under one threshold: double the width
constexpr uint32_t SM_FEW_EDGES = 4096;

// u32: saturating sums flag the overflow; f64: non-negative doubles order like
// their bit patterns
struct SmU32 {
  using D = uint32_t;
  using W = uint32_t;
  using T = uint64_t;  // thresholds and widths
  using Bits = unsigned int;
  static constexpr D INF = 0xFFFFFFFFu;
  static __device__ __forceinline__ Bits bits(D d) { return d; }
  static __device__ __forceinline__ D val(Bits b) { return b; }
  static __device__ __forceinline__ Bits inf_bits() { return 0xFFFFFFFFu; }
  static __device__ __forceinline__ D add(D du, W w, bool &ovf) {
    const uint64_t s = (uint64_t)du + w;
    ovf = s >= 0xFFFFFFFFull;
    return ovf ? 0xFFFFFFFEu : (uint32_t)s;
  }
  static __device__ __forceinline__ bool below(D d, T t) { return (uint64_t)d < t; }
  static __device__ __forceinline__ T next(D lo, T width) { return (uint64_t)lo + width; }
  static __device__ __forceinline__ T widen(T width) {
    return width < (1ull << 32) ? width * 2 : width;
  }
  // whether d + w stays in d's bucket of width delta (< 2^32); magic:
  // floor((2^64 - 1) / delta) + 1, which makes the quotient exact (0: delta is 1)
  static __device__ __forceinline__ bool stays(D d, W w, T delta, uint64_t magic) {
    const uint32_t dl = (uint32_t)delta;
    if (w >= dl) return false;
    return magic == 0 || w < dl - (d - (uint32_t)__umul64hi(d, magic) * dl);
  }
  static uint64_t host_magic(T delta) { return delta > 1 ? (~0ull / delta) + 1 : 0; }
};
struct SmF64 {
  using D = double;
  using W = double;
  using T = double;
  using Bits = unsigned long long;
  static __device__ __forceinline__ Bits bits(D d) {
    return (unsigned long long)__double_as_longlong(d);
  }
  static __device__ __forceinline__ D val(Bits b) { return __longlong_as_double((long long)b); }
  static __device__ __forceinline__ Bits inf_bits() { return 0x7FF0000000000000ull; }
  static __device__ __forceinline__ D add(D du, W w, bool &ovf) {
    ovf = false;
    return __dadd_rn(du, w);
  }
  static __device__ __forceinline__ bool below(D d, T t) { return d < t; }
  // a threshold above lo even where the width vanishes against it
  static __device__ __forceinline__ T next(D lo, T width) {
    const D t = lo + width;
    return t > lo ? t : __longlong_as_double(__double_as_longlong(lo) + 1);
  }
  static __device__ __forceinline__ T widen(T width) { return width * 2.0; }
  static __device__ __forceinline__ bool stays(D d, W w, T delta, uint64_t) {
    return (uint64_t)(long long)(__dadd_rn(d, w) / delta) == (uint64_t)(long long)(d / delta);
  }
  static uint64_t host_magic(T) { return 0; }
};

// W void: no weights
template <class W>
struct SmGraph {
  const int32_t *rp;
  const int32_t *col;
  const W *w;
  int32_t V;
};
template <class W>
using sm_weight = std::conditional_t<std::is_void<W>::value, uint32_t, W>;

struct SmStats {
  unsigned long long buckets, phases, relax, imp_near, imp_far, reached, traversed, ovf;
};

// LDS of the edge spreading
struct SmShare {
  // of a batch's vertices with edges: edge index minus edge slot, vertex
  uint2 own[SM_BLOCK];
  unsigned long long start[3][SM_SWEEP / 64];  // slots where a vertex's edges begin
  uint32_t wsum[SM_WAVES], wcnt[SM_WAVES];
};
// LDS of one workgroup; VCAP a multiple of 2048.
template <class Tr, int VCAP>
struct SmLds : SmShare {
  typename Tr::Bits dist[VCAP];
  uint32_t pend[VCAP / 32];
  uint16_t queue[SM_QCAP];
  uint32_t n, lim, edges;
  unsigned long long lo;  // bits of the smallest waiting distance
  unsigned long long acc[6];
};

// Edge slots [k0, k0 + U * SM_BLOCK) of a batch, U per lane, to
// f(in, v, x, w), arrays of U (in: below total; v -> x the edge), so that f can
// keep its LDS reads in flight together.  bits: this lane's word of the start
// bits; pre: the start bits before that word plus those of earlier sweeps.
// The owner of slot k is the last start at or before k: the wave's 64
// consecutive slots are one word, held by one lane.
template <int U, class W, class F>
__device__ __forceinline__ void sm_edges(const SmShare &s, const SmGraph<W> &G, uint32_t k0,
                                         uint32_t total, uint64_t bits, uint32_t pre, F f) {
  const int wv = threadIdx.x >> 6;
  const uint64_t upto = ~0ull >> (63 - gb_lane());
  uint32_t v[U], x[U];
  sm_weight<W> w[U];
  bool in[U];
  uint2 o[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int q = u * SM_WAVES + wv;
    const uint64_t word = gb_shfl_u64(bits, q);
    const uint32_t first = __shfl(pre, q, GB_WAVE);
    o[u] = s.own[first + (uint32_t)__popcll(word & upto) - 1u];  // slot 0 is a start
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    const uint32_t k = k0 + (uint32_t)(u * SM_BLOCK) + threadIdx.x;
    in[u] = k < total;
    const int32_t e = (int32_t)k + (int32_t)o[u].x;
    v[u] = o[u].y;
    x[u] = in[u] ? (uint32_t)G.col[e] : 0u;
    w[u] = 0;
    if constexpr (!std::is_void<W>::value) w[u] = in[u] ? G.w[e] : (W)0;
  }
  f(in, v, x, w);
}

// Spreads the out-edges of vertices vert(0 .. n) over the block's lanes and
// calls f for them (see sm_edges).  Block-uniform n.  sweep counts the sweeps
// of all calls (block-uniform): start bits rotate through three buffers, so
// that a sweep needs one barrier (set this sweep's, clear the next one's).
// Every lane searching the batch's first slots instead (10 LDS reads per edge)
// measured 3 to 10% slower (32768 vertices, 31 edges each, 32 sources: 1762
// against 1608 us).
template <class W, class Vert, class F>
__device__ __forceinline__ void sm_expand(SmShare &s, const SmGraph<W> &G, uint32_t n,
                                          uint32_t &sweep, Vert vert, F f) {
  const int tid = threadIdx.x, lane = gb_lane(), wv = tid >> 6;
  for (uint32_t b = 0; b < n; b += SM_BLOCK) {
    int32_t beg = 0;
    uint32_t deg = 0, v = 0;
    if (b + tid < n) {
      v = vert(b + tid);
      beg = G.rp[v];
      deg = (uint32_t)(G.rp[v + 1] - beg);
    }
    uint32_t wt;
    uint32_t ex = gb_wave_excl_sum(deg, &wt);
    const uint64_t some = __ballot(deg > 0);
    uint32_t c = (uint32_t)__popcll(some & ((1ull << lane) - 1));
    if (lane == 0) {
      s.wsum[wv] = wt;
      s.wcnt[wv] = (uint32_t)__popcll(some);
    }
    __syncthreads();
    uint32_t total = 0;
#pragma unroll
    for (int q = 0; q < SM_WAVES; q++) {
      const uint32_t x = s.wsum[q];
      ex += q < wv ? x : 0u;
      c += q < wv ? s.wcnt[q] : 0u;
      total += x;
    }
    if (deg > 0) s.own[c] = make_uint2((uint32_t)(beg - (int32_t)ex), v);
    if (total == 0) __syncthreads();  // wsum is read before the next batch
    uint32_t seen = 0;                // starts of earlier sweeps
    for (uint32_t k0 = 0; k0 < total; k0 += SM_SWEEP) {
      if (deg > 0 && ex - k0 < SM_SWEEP)  // ex >= k0 (unsigned)
        atomicOr(&s.start[sweep % 3][(ex - k0) >> 6], 1ull << (ex & 63));
      if (tid < SM_SWEEP / 64) s.start[(sweep + 1) % 3][tid] = 0;
      __syncthreads();
      const uint64_t bits = s.start[sweep % 3][lane];
      uint32_t st;
      const uint32_t pre = seen + gb_wave_excl_sum((uint32_t)__popcll(bits), &st);
      if (total - k0 > SM_BLOCK)
        sm_edges<SM_U>(s, G, k0, total, bits, pre, f);
      else
        sm_edges<1>(s, G, k0, total, bits, pre, f);
      seen += st;
      sweep++;
    }
  }
  __syncthreads();
}

// Distances from src into s.dist (bits); every thread of the block.  The
// thresholds start `width` apart.  COUNT: the improvements by whether they leave
// the bucket of the caller's width delta, whatever the thresholds.
template <bool COUNT, class Tr, int VCAP>
__device__ __forceinline__ void sm_solve(SmLds<Tr, VCAP> &s, const SmGraph<typename Tr::W> &G,
                                         int32_t src, typename Tr::T width,
                                         const typename Tr::T delta, uint64_t magic,
                                         uint32_t &sweep, SmStats &st) {
  using D = typename Tr::D;
  using Bits = typename Tr::Bits;
  const int tid = threadIdx.x, lane = gb_lane();
  const int V = G.V;
  for (int v = tid; v < V; v += SM_BLOCK) s.dist[v] = Tr::inf_bits();
  for (int i = tid; i < VCAP / 32; i += SM_BLOCK) s.pend[i] = 0;
  if (tid < SM_SWEEP / 64) s.start[sweep % 3][tid] = 0;
  // FP64 weights: no wider than the plain rule's width, twice the mean weight over
  // the mean degree, by a sample (the caller bounds the width of whole ones)
  if constexpr (std::is_same<typename Tr::W, double>::value) {
    const int64_t E = G.rp[V];
    double *sum = (double *)s.own;
    const double w = gb_wave_sum_f64(E > 0 ? G.w[tid * E / SM_BLOCK] : 0.0);
    if (lane == 0) sum[tid >> 6] = w;
    __syncthreads();
    double mean = 0.0;
    for (int q = 0; q < SM_WAVES; q++) mean += sum[q] / SM_BLOCK;
    const double plain = E > 0 ? 2.0 * mean * V / E : 0.0;
    if (plain > 0.0 && plain < width) width = plain;
  }
  __syncthreads();
  if (tid == 0) {
    s.dist[src] = 0;
    s.pend[src >> 5] = 1u << (src & 31);
  }
  typename Tr::T T = Tr::next((D)0, width);
  uint32_t edges = 0;  // under the current threshold
  uint32_t relax = 0, near = 0, imp = 0;
  bool ovf = false;
  st.buckets = 1;
  st.phases = 0;
  for (;;) {
    if (tid == 0) {
      s.n = 0;
      s.lim = ~0u;
      s.lo = ~0ull;
    }
    __syncthreads();
    // waiting vertices below the threshold to the queue, as far as it holds
    // them; the smallest of the others
    unsigned long long lo = ~0ull;
    for (int v0 = tid & ~63; v0 < V; v0 += SM_BLOCK) {  // wave-uniform
      const uint64_t p = (uint64_t)s.pend[v0 >> 5] | ((uint64_t)s.pend[(v0 >> 5) + 1] << 32);
      if (p == 0) continue;
      const bool on = (p >> lane) & 1u;
      Bits d = Tr::inf_bits();
      if (on) d = s.dist[v0 + lane];
      const bool take = on && Tr::below(Tr::val(d), T);
      const uint64_t m = __ballot(take);
      uint64_t left = p;
      if (m) {
        const uint32_t c = (uint32_t)__popcll(m);
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&s.n, c);
        base = __shfl(base, 0, GB_WAVE);
        if (base + c <= SM_QCAP) {
          if (take)
            s.queue[base + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = (uint16_t)(v0 + lane);
          left = p & ~m;
          if (lane == 0) {
            s.pend[v0 >> 5] = (uint32_t)left;
            s.pend[(v0 >> 5) + 1] = (uint32_t)(left >> 32);
          }
        } else if (lane == 0) {
          atomicMin(&s.lim, base);  // every later reservation fails too
        }
      }
      if (on && !take) lo = d < lo ? (unsigned long long)d : lo;
    }
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) {
      const unsigned long long o = gb_shfl_u64(lo, lane ^ dd);
      lo = o < lo ? o : lo;
    }
    if (lane == 0 && lo != ~0ull) atomicMin(&s.lo, lo);
    __syncthreads();
    const uint32_t n = s.n < s.lim ? s.n : s.lim;
    const unsigned long long wait = s.lo;
    __syncthreads();  // read before the next round clears them
    if (n == 0) {
      if (wait == ~0ull) break;
      if (edges < SM_FEW_EDGES) width = Tr::widen(width);
      edges = 0;
      T = Tr::next(Tr::val((Bits)wait), width);
      st.buckets++;
      continue;
    }
    st.phases++;
    uint32_t mine = 0;
    sm_expand(
        s, G, n, sweep, [&](uint32_t i) { return (uint32_t)s.queue[i]; },
        [&](auto &in, auto &v, auto &x, auto &w) {
          constexpr int U = sizeof(in) / sizeof(in[0]);
          Bits du[U], old[U];
#pragma unroll
          for (int u = 0; u < U; u++) {
            du[u] = s.dist[v[u]];
            old[u] = s.dist[x[u]];
          }
          // improvement is judged on the value read, so that nothing waits for
          // an atomic's return; a smaller distance written meanwhile costs one
          // idle expansion at most
#pragma unroll
          for (int u = 0; u < U; u++) {
            bool o;
            const D nd = Tr::add(Tr::val(du[u]), w[u], o);
            const Bits nb = Tr::bits(nd);
            mine += in[u];
            ovf |= in[u] & o;
            if (in[u] & (nb < old[u])) {
              atomicMin(&s.dist[x[u]], nb);
              atomicOr(&s.pend[x[u] >> 5], 1u << (x[u] & 31));
              if (COUNT) {
                imp++;
                near += Tr::stays(Tr::val(du[u]), w[u], delta, magic);
              }
            }
          }
        });
    relax += mine;
    uint32_t tot;
    (void)gb_wave_excl_sum(mine, &tot);
    if (tid == 0) s.edges = 0;
    __syncthreads();
    if (lane == 0) atomicAdd(&s.edges, tot);
    __syncthreads();
    edges += s.edges;
  }
  // totals
  uint32_t reached = 0;
  unsigned long long trav = 0;
  for (int v = tid; v < V; v += SM_BLOCK)
    if (s.dist[v] != Tr::inf_bits()) {
      reached++;
      trav += (unsigned long long)(G.rp[v + 1] - G.rp[v]);
    }
  if (tid < 6) s.acc[tid] = 0;
  __syncthreads();
  const unsigned long long mine[6] = {relax, near, imp - near, reached, trav, ovf ? 1ull : 0ull};
#pragma unroll
  for (int i = 0; i < 6; i++) {
    unsigned long long t = mine[i];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) t += gb_shfl_u64(t, lane ^ d);
    if (lane == 0 && t) atomicAdd(&s.acc[i], t);
  }
  __syncthreads();
  st.relax = s.acc[0];
  st.imp_near = s.acc[1];
  st.imp_far = s.acc[2];
  st.reached = s.acc[3];
  st.traversed = s.acc[4];
  st.ovf = s.acc[5];
}
