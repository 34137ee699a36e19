// gb_bc.hip -- weighted Brandes betweenness (f64 weights) for gfx950.
//
// Replaces the weighted form of run_bc (btwcentral/csr_bc.c:16-130): the
// per-source run_sspath with predecessor lists, the distance sort
// (q_sort_double) and the comp_num_spath / comp_delta loops become kernels over
// a batch of sources on the tight-edge DAG of the exact distances.  An edge
// u->x is tight when fl(d[u] + w) == d[x] (the '<=' predecessor rule of
// csr_sspath.c:101-118 with each edge recorded once).  Every (source slot,
// vertex) pair is an entry of one `order` array, grouped by DAG depth, which
// is also Brandes' stack.
//   indeg     count of tight in-edges per (slot, vertex)
//   expand    one wave per depth-d entry, lanes over its out-edges: the last
//             tight in-edge to be processed assigns depth d+1 (Kahn order).
//   sigma     one wave per depth-(d+1) entry, pull over its tight in-edges
//             (FP64; integer values are exact below 2^53).
//   delta     backwards, one wave per depth-d entry, pull over tight out-edges:
//             delta[v] = sum ((1+delta[w])*sigma[v])/sigma[w] (the operand
//             order of csr_bc.c:116), fixed-order wave sum.
//   accum     bc[v] += delta[slot][v] for v != source, slots in order
//             (csr_bc.c:57-61, sums not halved).
// Unweighted BC and BFS levels are the batched kernels of gb_msbc.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "gb_device.hpp"
#include "gb_internal.hpp"
#include "gb_sssp_small.hpp"

namespace {

constexpr int BC_BLOCK = 256;

__global__ void bc_fill_kernel(int64_t n, int32_t *__restrict__ level, double *__restrict__ sigma,
                               double *__restrict__ delta) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    level[i] = -1;
    if (sigma) sigma[i] = 0.0;
    if (delta) delta[i] = 0.0;
  }
}

__global__ void bc_seed_kernel(int32_t V, int32_t nslots, const int32_t *__restrict__ src,
                               int32_t *__restrict__ level, double *__restrict__ sigma,
                               uint64_t *__restrict__ order) {
  int32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nslots) return;
  const int64_t base = (int64_t)s * V;
  level[base + src[s]] = 0;
  if (sigma) sigma[base + src[s]] = 1.0;
  order[s] = ((uint64_t)s << 32) | (uint32_t)src[s];
}

// Tight-DAG discovery (weighted): decrement the count of unprocessed tight
// in-edges of each tight successor; the last one assigns depth d+1.
__global__ __launch_bounds__(BC_BLOCK) void bcw_expand_kernel(
    int32_t V, const int32_t *__restrict__ rp, const int32_t *__restrict__ col,
    const double *__restrict__ w, const double *__restrict__ dist, int32_t *__restrict__ indeg,
    uint64_t *__restrict__ order, uint64_t lo, uint64_t hi, int32_t d, int32_t *__restrict__ level,
    unsigned long long *n_order) {
  const int lane = gb_lane();
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint64_t nwaves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
  for (uint64_t i = lo + wave; i < hi; i += nwaves) {
    const uint64_t ent = order[i];
    const uint32_t s = (uint32_t)(ent >> 32);
    const int32_t u = (int32_t)(uint32_t)ent;
    const int64_t base = (int64_t)s * V;
    const double du = dist[base + u];
    const int32_t beg = rp[u], end = rp[u + 1];
    for (int32_t b0 = beg; b0 < end; b0 += GB_WAVE) {
      const int32_t e = b0 + lane;
      bool push = false;
      int32_t x = 0;
      if (e < end) {
        x = col[e];
        if (__dadd_rn(du, w[e]) == dist[base + x] && level[base + x] != 0) {
          if (atomicSub(&indeg[base + x], 1) == 1) {
            level[base + x] = d + 1;
            push = true;
          }
        }
      }
      const uint64_t pb = gb_wave_reserve(n_order, push ? 1u : 0u);
      if (push) order[pb] = ((uint64_t)s << 32) | (uint32_t)x;
    }
  }
}

// Count tight in-edges per (slot, vertex) for the weighted form.
__global__ __launch_bounds__(BC_BLOCK) void bcw_indeg_kernel(
    int32_t V, int32_t nslots, const int32_t *__restrict__ rrp, const int32_t *__restrict__ rcol,
    const double *__restrict__ rw, const double *__restrict__ dist, int32_t *__restrict__ indeg) {
  const int64_t n = (int64_t)nslots * V;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t s = i / V;
    const int32_t v = (int32_t)(i - s * V);
    const double dv = dist[i];
    int32_t c = 0;
    if (dv != __longlong_as_double(0x7FF0000000000000ll)) {
      const double *ds = dist + s * V;
      for (int32_t e = rrp[v]; e < rrp[v + 1]; e++) {
        const double du = ds[rcol[e]];
        if (__dadd_rn(du, rw[e]) == dv) c++;
      }
    }
    indeg[i] = c;
  }
}

// Reached (slot, vertex) pairs: finite distances, one atomic per block.
__global__ void bcw_reached_kernel(int64_t n, const double *__restrict__ dist,
                                   unsigned long long *__restrict__ count) {
  unsigned long long c = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    c += dist[i] != __longlong_as_double(0x7FF0000000000000ll) ? 1ull : 0ull;
  __shared__ unsigned long long s_c[256 / GB_WAVE];
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, GB_WAVE);
  if (gb_lane() == 0) s_c[threadIdx.x / GB_WAVE] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int k = 0; k < (int)(blockDim.x / GB_WAVE); k++) t += s_c[k];
    atomicAdd(count, t);
  }
}

struct PredTight {
  const double *dist;
  const double *w;   // forward weights
  const double *rw;  // reverse weights
  __device__ __forceinline__ bool in_edge(int64_t base, int32_t u, int32_t v, int32_t e,
                                          int32_t) const {
    return __dadd_rn(dist[base + u], rw[e]) == dist[base + v];
  }
  __device__ __forceinline__ bool out_edge(int64_t base, int32_t v, int32_t x, int32_t e,
                                           int32_t) const {
    return __dadd_rn(dist[base + v], w[e]) == dist[base + x];
  }
};

// sigma pull for the entries [lo, hi) at level d (d >= 1)
template <class P>
__global__ __launch_bounds__(BC_BLOCK) void bc_sigma_kernel(
    int32_t V, const int32_t *__restrict__ rrp, const int32_t *__restrict__ rcol,
    const uint64_t *__restrict__ order, uint64_t lo, uint64_t hi, int32_t d, P pred,
    double *__restrict__ sigma) {
  const int lane = gb_lane();
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint64_t nwaves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
  for (uint64_t i = lo + wave; i < hi; i += nwaves) {
    const uint64_t ent = order[i];
    const int64_t base = (int64_t)(ent >> 32) * V;
    const int32_t v = (int32_t)(uint32_t)ent;
    double acc = 0.0;
    for (int32_t e = rrp[v] + lane; e < rrp[v + 1]; e += GB_WAVE) {
      const int32_t u = rcol[e];
      if (pred.in_edge(base, u, v, e, d)) acc += sigma[base + u];
    }
    acc = gb_wave_sum_f64(acc);
    if (lane == 0) sigma[base + v] = acc;
  }
}

// delta pull for the entries [lo, hi) at level d
template <class P>
__global__ __launch_bounds__(BC_BLOCK) void bc_delta_kernel(
    int32_t V, const int32_t *__restrict__ rp, const int32_t *__restrict__ col,
    const uint64_t *__restrict__ order, uint64_t lo, uint64_t hi, int32_t d, P pred,
    const double *__restrict__ sigma, double *__restrict__ delta) {
  const int lane = gb_lane();
  const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint64_t nwaves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
  for (uint64_t i = lo + wave; i < hi; i += nwaves) {
    const uint64_t ent = order[i];
    const int64_t base = (int64_t)(ent >> 32) * V;
    const int32_t v = (int32_t)(uint32_t)ent;
    const double sv = sigma[base + v];
    double acc = 0.0;
    for (int32_t e = rp[v] + lane; e < rp[v + 1]; e += GB_WAVE) {
      const int32_t x = col[e];
      if (pred.out_edge(base, v, x, e, d))
        acc += __ddiv_rn(__dmul_rn(__dadd_rn(1.0, delta[base + x]), sv), sigma[base + x]);
    }
    acc = gb_wave_sum_f64(acc);
    if (lane == 0) delta[base + v] = acc;
  }
}

__global__ void bc_accum_kernel(int32_t V, int32_t nslots, const int32_t *__restrict__ src,
                                const double *__restrict__ delta, double *__restrict__ bc) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  double acc = bc[v];
  for (int32_t s = 0; s < nslots; s++)
    if (src[s] != (int32_t)v) acc += delta[(int64_t)s * V + v];
  bc[v] = acc;
}

// ---- a source's whole solve in one workgroup -------------------------------
// Graphs whose FP64 distances fit the LDS of a CU (gb_sssp_small.hpp): one
// workgroup per source finds the distances, the tight in-degree counts, the
// DAG depths with the path counts, and the dependencies, with block barriers
// between the levels.  The engine's form below launches three kernels and
// waits for the host twice per level, after thousands of launches for the
// distances: R-MAT 13 with 16 sources 22.5 ms, now 0.6 ms; 16384 vertices with
// 196 K edges and 32 sources 28 ms, now 1.3 ms.  The steps and the operand
// order of the dependencies are the kernels' above; sigma is added
// instead of pulled (exact in any order below 2^53; beyond, the last bits follow
// the order in which lanes arrive, and vary between runs), a dependency is summed by
// 8 lanes, or by a wave from BCS_HUB out-edges on, in a fixed order.
constexpr int BCS_G = 8;        // lanes per vertex in the backward pass
constexpr int BCS_HUB = 128;
constexpr int BCS_SOURCES = 256;  // sources per launch, passed by value
struct BcsSources {
  int32_t s[BCS_SOURCES];
};
// what a workgroup reports: reached vertices, ordered vertices, levels
struct BcsOut {
  uint32_t reached, ordered, depth, pad;
};
struct BcsCtx {
  double *sigma, *delta;  // [slot][V]
  int32_t *indeg;         // [slot][V]
  uint32_t *order;        // [slot][V] vertices by depth
  uint32_t *loff;         // [slot][V + 1] first entry of each level
  BcsOut *out;
};

template <int VCAP>
__global__ __launch_bounds__(SM_BLOCK) void bcw_small_kernel(SmGraph<double> G, BcsSources src,
                                                             double width, BcsCtx c) {
  __shared__ SmLds<SmF64, VCAP> s;
  __shared__ uint32_t s_n;
  const int tid = threadIdx.x, lane = gb_lane(), wv = tid >> 6;
  const int64_t base = (int64_t)blockIdx.x * G.V;
  double *sigma = c.sigma + base, *delta = c.delta + base;
  int32_t *indeg = c.indeg + base;
  uint32_t *order = c.order + base, *loff = c.loff + (int64_t)blockIdx.x * (G.V + 1);
  const int32_t s0 = src.s[blockIdx.x];
  SmStats st;
  uint32_t sweep = 0;
  sm_solve<false>(s, G, s0, width, width, 0, sweep, st);
  // s.dist is only read from here on
  for (int v = tid; v < G.V; v += SM_BLOCK) {
    sigma[v] = 0.0;
    delta[v] = 0.0;
    indeg[v] = 0;
  }
  if (tid == 0) s_n = 0;
  __syncthreads();
  // the reached vertices, in any order, and their tight in-degrees
  for (int v0 = tid & ~63; v0 < G.V; v0 += SM_BLOCK) {
    const int v = v0 + lane;
    const bool on = v < G.V && s.dist[v] != SmF64::inf_bits();
    const uint64_t m = __ballot(on);
    uint32_t b = 0;
    if (lane == 0 && m) b = atomicAdd(&s_n, (uint32_t)__popcll(m));
    b = __shfl(b, 0, GB_WAVE);
    if (on) order[b + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = (uint32_t)v;
  }
  __syncthreads();
  const uint32_t reached = s_n;
  auto tight = [&](uint32_t u, uint32_t x, double w) {
    return SmF64::bits(__dadd_rn(SmF64::val(s.dist[u]), w)) == s.dist[x];
  };
  // an infinite weight is tight to a vertex that is not reached, as in the
  // kernels above, but counts for no order
  auto leads = [&](uint32_t u, uint32_t x, double w) {
    return tight(u, x, w) && s.dist[x] != SmF64::inf_bits();
  };
  sm_expand(
      s, G, reached, sweep, [&](uint32_t i) { return order[i]; },
      [&](auto &in, auto &u, auto &x, auto &w) {
        constexpr int U = sizeof(in) / sizeof(in[0]);
#pragma unroll
        for (int k = 0; k < U; k++)
          if (in[k] && leads(u[k], x[k], w[k]))
            __hip_atomic_fetch_add(&indeg[x[k]], 1, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
      });
  if (tid == 0) {
    order[0] = (uint32_t)s0;
    sigma[s0] = 1.0;
    loff[0] = 0;
    loff[1] = 1;
    s_n = 1;
  }
  __syncthreads();
  // Kahn's order: the last tight in-edge of a vertex appends it to the next level
  uint32_t lo = 0, hi = 1, depth = 1;
  for (;;) {
    sm_expand(
        s, G, hi - lo, sweep, [&](uint32_t i) { return order[lo + i]; },
        [&](auto &in, auto &u, auto &x, auto &w) {
          constexpr int U = sizeof(in) / sizeof(in[0]);
          double su[U];
          int32_t left[U];
#pragma unroll
          for (int k = 0; k < U; k++) su[k] = sigma[u[k]];
#pragma unroll
          for (int k = 0; k < U; k++) {
            left[k] = 0;
            if (in[k] && x[k] != (uint32_t)s0 && leads(u[k], x[k], w[k])) {
              __hip_atomic_fetch_add(&sigma[x[k]], su[k], __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
              left[k] = __hip_atomic_fetch_add(&indeg[x[k]], -1, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
            }
          }
#pragma unroll
          for (int k = 0; k < U; k++)
            if (left[k] == 1) order[atomicAdd(&s_n, 1u)] = x[k];
        });
    lo = hi;
    hi = s_n;
    __syncthreads();  // s_n is read before the next level appends
    if (hi == lo) break;
    depth++;
    if (tid == 0) loff[depth] = hi;
  }
  if (tid == 0) c.out[blockIdx.x] = BcsOut{reached, hi, depth, 0};
  if (hi != reached) return;  // a cycle of tight edges: the caller refuses
  // dependencies, deepest level first
  const int sub = lane / BCS_G, sl = lane % BCS_G;
  constexpr int PER = GB_WAVE / BCS_G;
  for (int32_t d = (int32_t)depth - 1; d >= 0; d--) {
    const uint32_t l0 = loff[d], l1 = loff[d + 1];
    for (uint32_t i0 = l0 + wv * PER; i0 < l1; i0 += SM_WAVES * PER) {
      const bool on = i0 + sub < l1;
      const uint32_t v = on ? order[i0 + sub] : 0u;
      const int32_t beg = on ? G.rp[v] : 0, end = on ? G.rp[v + 1] : 0;
      const double sv = on ? sigma[v] : 0.0;
      const bool hub = end - beg >= BCS_HUB;
      auto sum = [&](uint32_t vv, double svv, int32_t e0, int32_t e1, int step) {
        double acc = 0.0;
        for (int32_t e = e0; e < e1; e += 4 * step) {
          int32_t x[4];
          double w[4];
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const int32_t ee = min(e + k * step, e1 - 1);
            x[k] = G.col[ee];
            w[k] = G.w[ee];
          }
#pragma unroll
          for (int k = 0; k < 4; k++)
            if (e + k * step < e1 && tight(vv, (uint32_t)x[k], w[k]))
              acc += __ddiv_rn(__dmul_rn(__dadd_rn(1.0, delta[x[k]]), svv), sigma[x[k]]);
        }
        return acc;
      };
      double acc = hub ? 0.0 : sum(v, sv, beg + sl, end, BCS_G);
#pragma unroll
      for (int k = BCS_G / 2; k >= 1; k >>= 1) acc += __shfl_xor(acc, k, GB_WAVE);
      if (on && !hub && sl == 0) delta[v] = acc;
      uint64_t hubs = __ballot(hub && sl == 0);
      while (hubs) {
        const int l = __ffsll((unsigned long long)hubs) - 1;
        hubs &= hubs - 1;
        const uint32_t hv = __shfl(v, l, GB_WAVE);
        const double a = gb_wave_sum_f64(sum(hv, __shfl(sv, l, GB_WAVE),
                                             __shfl(beg, l, GB_WAVE) + lane,
                                             __shfl(end, l, GB_WAVE), GB_WAVE));
        if (lane == 0) delta[hv] = a;
      }
    }
    __syncthreads();
  }
}

struct BcWork {
  DevBuf level, sigma, delta, order, src, cnt, indeg, dist, loff;
  void release() {
    for (DevBuf *b : {&level, &sigma, &delta, &order, &src, &cnt, &indeg, &dist, &loff}) b->release();
  }
};
// Heap singleton, never destroyed: device memory must not be freed from a
// static destructor, which can run after the HIP runtime has shut down.
BcWork &g_bcw_ref() {
  static BcWork *w = new BcWork();
  return *w;
}
#define g_bcw (g_bcw_ref())

int wave_grid(uint64_t n) {
  uint64_t blocks = (n + 3) / 4;
  uint64_t cap = (uint64_t)gb_num_cus() * 16;
  if (blocks > cap) blocks = cap;
  return blocks < 1 ? 1 : (int)blocks;
}

int fill_grid(int64_t n) {
  int64_t b = (n + 255) / 256;
  int64_t cap = (int64_t)gb_num_cus() * 32;
  if (b > cap) b = cap;
  return b < 1 ? 1 : (int)b;
}

gb_status bcw_refuse(uint64_t n) {
  return gb_fail(GB_ERR_INVALID,
                 "gb_bc_weighted: %llu reached vertices lie on a cycle of tight edges "
                 "(weights must be positive and not vanish against the distances)",
                 (unsigned long long)n);
}

// Forward levels for nslots sources; returns level offsets (size depth+2).
gb_status forward_levels(gb_graph g, int32_t nslots, hipStream_t st,
                         std::vector<uint64_t> &off, bool with_sigma, int32_t *level) {
  BcWork &w = g_bcw;
  const int32_t V = g->V;
  unsigned long long *cnt = w.cnt.as<unsigned long long>();
  uint64_t *order = w.order.as<uint64_t>();
  double *sigma = with_sigma ? w.sigma.as<double>() : nullptr;
  off.assign(1, 0);
  off.push_back((uint64_t)nslots);
  unsigned long long h = nslots;
  GB_HIP(hipMemcpyAsync(cnt, &h, sizeof(h), hipMemcpyHostToDevice, st));
  int32_t d = 0;
  PredTight pt{w.dist.as<double>(), g->w64, g->rw64};
  for (;;) {
    const uint64_t lo = off[d], hi = off[d + 1];
    if (hi == lo) break;
    hipLaunchKernelGGL(bcw_expand_kernel, dim3(wave_grid(hi - lo)), dim3(BC_BLOCK), 0, st, V,
                         g->rp, g->col, g->w64, w.dist.as<double>(), w.indeg.as<int32_t>(), order,
                         lo, hi, d, level, cnt);
    GB_HIP(hipGetLastError());
    GB_HIP(hipMemcpyAsync(&h, cnt, sizeof(h), hipMemcpyDeviceToHost, st));
    GB_HIP(hipStreamSynchronize(st));
    off.push_back(h);
    d++;
    if (with_sigma && h > hi) {
      const int32_t *rrp = g->rrp ? g->rrp : g->rp;
      const int32_t *rcol = g->rcol ? g->rcol : g->col;
      hipLaunchKernelGGL(bc_sigma_kernel<PredTight>, dim3(wave_grid(h - hi)), dim3(BC_BLOCK), 0,
                         st, V, rrp, rcol, order, hi, (uint64_t)h, d, pt, sigma);
      GB_HIP(hipGetLastError());
    }
  }
  return GB_OK;
}

// Where the workgroup form serves: distances in LDS, and edges that one CU
// reads in about the time of the engine's launches.  The engine's time follows the
// depth of the tight edges and the longest rows (a wave each), one workgroup's the
// edges.  Measured, workgroups against engine (ms), 1 M edges, 1 / 16 / 64 sources:
// uniform, 4000 vertices 2.56 / 2.58 / 2.63 against 1.15 / 2.14 / 5.36, 16384 vertices
// 3.26 / 3.30 / 3.37 against 1.46 / 3.92 / 12.2; R-MAT 16384 3.39 / 3.49 / 3.61 against
// 6.3 / 12.4 / 26.5; two thirds of the edges at one vertex 4.6 / 4.8 / 4.7 against 61 /
// 94 / 142; 262 K edges, every graph and number of sources, 2 to 40 times.  Past 2^18
// edges few sources of a uniform graph lose up to a factor of 2 by this line, what
// others win by it is larger.
constexpr int32_t BCS_MAX_V = 16384;
constexpr int64_t BCS_MAX_E = (int64_t)1 << 20;

// The dependencies of one batch, w.delta[slot][V], by one workgroup per source.
gb_status bcs_batch(gb_graph g, const int32_t *h_sources, int32_t ns, int32_t *max_depth,
                    hipStream_t st) {
  static BcsOut *res = nullptr;  // pinned, kept for the process's life
  if (!res)
    GB_HIP(hipHostMalloc((void **)&res, sizeof(BcsOut) * BCS_SOURCES, hipHostMallocDefault));
  BcWork &w = g_bcw;
  const int32_t V = g->V;
  const double width = g->split64_valid ? g->split64_delta : 0.1;
  GB_TRY(w.loff.ensure(sizeof(uint32_t) * (size_t)std::min(ns, BCS_SOURCES) * (V + 1)));
  for (int32_t g0 = 0; g0 < ns; g0 += BCS_SOURCES) {
    const int n = std::min<int32_t>(BCS_SOURCES, ns - g0);
    BcsSources src{};
    for (int i = 0; i < n; i++) src.s[i] = h_sources[g0 + i];
    const int64_t o = (int64_t)g0 * V;
    const BcsCtx c{w.sigma.as<double>() + o,  w.delta.as<double>() + o,
                   w.indeg.as<int32_t>() + o, w.order.as<uint32_t>() + o,
                   w.loff.as<uint32_t>(),     res};
    const SmGraph<double> G{g->rp, g->col, g->w64, V};
    if (V <= BCS_MAX_V / 4)
      hipLaunchKernelGGL(bcw_small_kernel<BCS_MAX_V / 4>, dim3(n), dim3(SM_BLOCK), 0, st, G, src,
                         width, c);
    else
      hipLaunchKernelGGL(bcw_small_kernel<BCS_MAX_V>, dim3(n), dim3(SM_BLOCK), 0, st, G, src,
                         width, c);
    GB_HIP(hipGetLastError());
    GB_HIP(hipStreamSynchronize(st));
    for (int i = 0; i < n; i++) {
      if (res[i].reached != res[i].ordered) return bcw_refuse(res[i].reached - res[i].ordered);
      *max_depth = std::max(*max_depth, (int32_t)res[i].depth);
    }
  }
  return GB_OK;
}

gb_status bc_run(gb_graph g, const int32_t *h_sources, int32_t nsrc, int32_t batch, double *d_bc,
                 gb_bc_stats *stats, void *stream) {
  if (!g || (!h_sources && nsrc > 0) || nsrc < 0 || !d_bc)
    return gb_fail(GB_ERR_INVALID, "gb_bc: null argument");
  const int32_t V = g->V;
  for (int32_t i = 0; i < nsrc; i++)
    if (h_sources[i] < 0 || h_sources[i] >= V)
      return gb_fail(GB_ERR_INVALID, "gb_bc: source %d out of range", h_sources[i]);
  if (!g->w64 || (g->rrp && !g->rw64))
    return gb_fail(GB_ERR_INVALID, "gb_bc_weighted: graph needs f64 weights (forward and reverse)");
  hipStream_t st = gb_stream(stream);
  if (batch <= 0 || batch > nsrc) batch = nsrc;
  if (batch > 65535) batch = 65535;
  BcWork &w = g_bcw;
  const int64_t n = (int64_t)batch * V;
  GB_TRY(w.level.ensure(sizeof(int32_t) * (n + 1)));
  GB_TRY(w.sigma.ensure(sizeof(double) * (n + 1)));
  GB_TRY(w.delta.ensure(sizeof(double) * (n + 1)));
  GB_TRY(w.order.ensure(sizeof(uint64_t) * (n + 1)));
  GB_TRY(w.src.ensure(sizeof(int32_t) * batch));
  GB_TRY(w.cnt.ensure(2 * sizeof(unsigned long long)));
  GB_TRY(w.indeg.ensure(sizeof(int32_t) * (n + 1)));
  GB_TRY(w.dist.ensure(sizeof(double) * (n + 1)));
  hipEvent_t e0, e1;
  GB_HIP(hipEventCreate(&e0));
  GB_HIP(hipEventCreate(&e1));
  GB_HIP(hipEventRecord(e0, st));
  GB_HIP(hipMemsetAsync(d_bc, 0, sizeof(double) * V, st));
  int32_t max_depth = 0, batches = 0;
  const bool small = V <= BCS_MAX_V && g->E <= BCS_MAX_E && gb_sssp_small_enabled();
  std::vector<uint64_t> off;
  for (int32_t b0 = 0; b0 < nsrc; b0 += batch) {
    const int32_t ns = std::min(batch, nsrc - b0);
    const int64_t nn = (int64_t)ns * V;
    GB_HIP(hipMemcpyAsync(w.src.p, h_sources + b0, sizeof(int32_t) * ns, hipMemcpyHostToDevice, st));
    if (small) {
      GB_TRY(bcs_batch(g, h_sources + b0, ns, &max_depth, st));
      hipLaunchKernelGGL(bc_accum_kernel, dim3((V + 255) / 256), dim3(256), 0, st, V, ns,
                         w.src.as<int32_t>(), w.delta.as<double>(), d_bc);
      GB_HIP(hipGetLastError());
      batches++;
      continue;
    }
    // exact distances of the batch, then tight in-degree counts; bucket
    // width: the last f64 split of this graph, else the reference's BC
    // constant (run_sspath(gs, pred, source, 0.1), csr_bc.c:43)
    GB_TRY(gb_sssp_f64(g, g->split64_valid ? g->split64_delta : 0.1, h_sources + b0, ns,
                       w.dist.as<double>(), nullptr, stream));
    const int32_t *rrp = g->rrp ? g->rrp : g->rp;
    const int32_t *rcol = g->rcol ? g->rcol : g->col;
    const double *rw = g->rrp ? g->rw64 : g->w64;
    hipLaunchKernelGGL(bcw_indeg_kernel, dim3(fill_grid(nn)), dim3(256), 0, st, V, ns, rrp, rcol,
                       rw, w.dist.as<double>(), w.indeg.as<int32_t>());
    GB_HIP(hipGetLastError());
    hipLaunchKernelGGL(bc_fill_kernel, dim3(fill_grid(nn)), dim3(256), 0, st, nn,
                       w.level.as<int32_t>(), w.sigma.as<double>(), w.delta.as<double>());
    hipLaunchKernelGGL(bc_seed_kernel, dim3((ns + 255) / 256), dim3(256), 0, st, V, ns,
                       w.src.as<int32_t>(), w.level.as<int32_t>(), w.sigma.as<double>(),
                       w.order.as<uint64_t>());
    GB_HIP(hipGetLastError());
    GB_TRY(forward_levels(g, ns, st, off, true, w.level.as<int32_t>()));
    // Every reached pair must have been given a depth.  A cycle of tight edges
    // (a zero weight, or a weight below half an ulp of the distance it is
    // added to) never lets Kahn's count reach zero: its vertices would keep
    // sigma 0 and divide by it below.
    {
      unsigned long long *rc = w.cnt.as<unsigned long long>() + 1;
      GB_HIP(hipMemsetAsync(rc, 0, sizeof(unsigned long long), st));
      hipLaunchKernelGGL(bcw_reached_kernel, dim3(fill_grid(nn)), dim3(256), 0, st, nn,
                         (const double *)w.dist.as<double>(), rc);
      GB_HIP(hipGetLastError());
      unsigned long long reached = 0;
      GB_HIP(hipMemcpyAsync(&reached, rc, sizeof(reached), hipMemcpyDeviceToHost, st));
      GB_HIP(hipStreamSynchronize(st));
      if (reached != off.back()) return bcw_refuse(reached - off.back());
    }
    const int32_t depth = (int32_t)off.size() - 2;  // number of non-empty levels
    max_depth = std::max(max_depth, depth);
    PredTight pt{w.dist.as<double>(), g->w64, g->rw64};
    for (int32_t d = depth - 1; d >= 0; d--) {
      const uint64_t lo = off[d], hi = off[d + 1];
      if (hi == lo) continue;
      hipLaunchKernelGGL(bc_delta_kernel<PredTight>, dim3(wave_grid(hi - lo)), dim3(BC_BLOCK), 0,
                         st, V, g->rp, g->col, w.order.as<uint64_t>(), lo, hi, d, pt,
                         w.sigma.as<double>(), w.delta.as<double>());
      GB_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(bc_accum_kernel, dim3((V + 255) / 256), dim3(256), 0, st, V, ns,
                       w.src.as<int32_t>(), w.delta.as<double>(), d_bc);
    GB_HIP(hipGetLastError());
    batches++;
  }
  GB_HIP(hipEventRecord(e1, st));
  GB_HIP(hipEventSynchronize(e1));
  float ms = 0;
  GB_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (stats) {
    stats->max_depth = max_depth;
    stats->batches = batches;
    stats->ms = ms;
  }
  return GB_OK;
}

}  // namespace

void gb_bc_release() { g_bcw.release(); }

extern "C" gb_status gb_bc_weighted(gb_graph g, const int32_t *h_sources, int32_t nsrc,
                                    int32_t batch, double *d_bc, gb_bc_stats *st, void *stream) {
  return bc_run(g, h_sources, nsrc, batch, d_bc, st, stream);
}
