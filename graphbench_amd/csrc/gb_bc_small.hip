// gb_bc_small.hip -- unweighted Brandes, one workgroup per source.
//
// The batched engine (gb_msbc.hip) replays 16 levels of ten launches whatever
// the depth, captures two hipGraphs and waits for the host six times per
// call: on a graph of a few thousand vertices that is all of its time (R-MAT
// 12 symmetrised, 50 sources: 1.98 ms, 0.6 ms of it kernels that had work).
// A graph whose path counts fit the LDS of a CU is solved by one workgroup of
// 1024 threads per source, all sources side by side, with block barriers
// between levels: path counts (later psi = (1 + delta) / sigma), the order of
// discovery and the level masks in LDS, edges spread evenly over the lanes
// (gb_sssp_small.hpp).  R-MAT 12, 50 sources: 220 us in all, 182 us of it the
// kernel, which one CU's memory parallelism bounds (131 K edges twice).
//
// Replaces comp_num_spath / comp_delta (csr_bc.c:70-96, 98-123) per source and
// the accumulation of csr_bc.c:57-61, as gb_msbc.hip does; the sums of a
// vertex's successors run in a fixed order (8 lanes, or a wave for a vertex
// of 128 out-edges or more, then a butterfly), so results do not vary with the
// batch, nor between runs while path counts stay below 2^53 (they are whole
// numbers added in the order the lanes arrive: exact up to there, rounded in that
// order beyond, as in the pushes of gb_msbc.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "gb_device.hpp"
#include "gb_internal.hpp"
#include "gb_sssp_small.hpp"

namespace {

constexpr int SB_G = 8;           // lanes per vertex in the backward pass
constexpr int SB_HUB = 128;       // out-edges from which a wave takes a vertex
constexpr int SB_SOURCES = 256;   // sources per launch, passed by value
constexpr int SB_MAX_V = 14336;   // 157 KB of LDS

struct SbSources {
  int32_t s[SB_SOURCES];
};

template <int VCAP>
struct SbLds : SmShare {
  double sigma[VCAP];       // path counts, then psi
  uint16_t order[VCAP];     // vertices by level
  uint32_t vis[VCAP / 32];  // forward: levels <= d; backward: level d + 1
  uint32_t nxt[VCAP / 32];  // forward: level d + 1
  uint32_t n;
};

// delta[slot][V]: dependencies (0 for vertices not reached); loff[slot][V + 2]:
// scratch, the levels' first entries in `order`; depth[slot]: non-empty levels.
template <int VCAP>
__global__ __launch_bounds__(SM_BLOCK) void bc_small_kernel(SmGraph<void> G, SbSources src,
                                                            double *__restrict__ delta,
                                                            uint32_t *__restrict__ loff,
                                                            uint32_t *__restrict__ depth_out) {
  __shared__ SbLds<VCAP> s;
  const int tid = threadIdx.x, lane = gb_lane(), wv = tid >> 6;
  const int V = G.V;
  double *dl = delta + (int64_t)blockIdx.x * V;
  uint32_t *lo = loff + (int64_t)blockIdx.x * (V + 2);
  const int32_t s0 = src.s[blockIdx.x];
  uint32_t sweep = 0;
  for (int v = tid; v < V; v += SM_BLOCK) {
    s.sigma[v] = 0.0;
    dl[v] = 0.0;
  }
  for (int i = tid; i < VCAP / 32; i += SM_BLOCK) s.vis[i] = s.nxt[i] = 0;
  if (tid < SM_SWEEP / 64) s.start[0][tid] = 0;
  __syncthreads();
  if (tid == 0) {
    s.sigma[s0] = 1.0;
    s.order[0] = (uint16_t)s0;
    s.vis[s0 >> 5] = 1u << (s0 & 31);
    s.n = 1;
    lo[0] = 0;
    lo[1] = 1;
  }
  __syncthreads();
  // forward: level [a, b) of the order discovers the next one.  sigma holds
  // whole numbers, so its adds are exact in any order (below 2^53).
  uint32_t a = 0, b = 1, depth = 1;
  for (;;) {
    sm_expand(
        s, G, b - a, sweep, [&](uint32_t i) { return (uint32_t)s.order[a + i]; },
        [&](auto &in, auto &v, auto &x, auto &) {
          constexpr int U = sizeof(in) / sizeof(in[0]);
          double sv[U];
          bool fresh[U];
#pragma unroll
          for (int u = 0; u < U; u++) {
            sv[u] = s.sigma[v[u]];
            fresh[u] = in[u] & !((s.vis[x[u] >> 5] >> (x[u] & 31)) & 1u);
          }
#pragma unroll
          for (int u = 0; u < U; u++)
            if (fresh[u]) {
              atomicAdd(&s.sigma[x[u]], sv[u]);
              const uint32_t bit = 1u << (x[u] & 31);
              if (!(s.nxt[x[u] >> 5] & bit) && !(atomicOr(&s.nxt[x[u] >> 5], bit) & bit))
                s.order[atomicAdd(&s.n, 1u)] = (uint16_t)x[u];
            }
        });
    a = b;
    b = s.n;
    __syncthreads();  // s.n is read before the next level appends
    if (a == b) break;
    for (int i = tid; i < VCAP / 32; i += SM_BLOCK) {
      s.vis[i] |= s.nxt[i];
      s.nxt[i] = 0;
    }
    depth++;
    if (tid == 0) lo[depth] = b;
    __syncthreads();
  }
  if (tid == 0) depth_out[blockIdx.x] = depth;
  // backward: delta[v] = sigma[v] * sum of psi over the successors one level
  // deeper, psi over sigma once delta is known.  The deepest level has none.
  const int sub = lane / SB_G, sl = lane % SB_G;
  constexpr int PER = GB_WAVE / SB_G;
  for (int32_t d = (int32_t)depth - 1; d >= 0; d--) {
    const uint32_t l0 = lo[d], l1 = lo[d + 1];
    for (int i = tid; i < VCAP / 32; i += SM_BLOCK) s.vis[i] = 0;
    __syncthreads();
    if (d < (int32_t)depth - 1) {
      const uint32_t l2 = lo[d + 2];
      for (uint32_t i = l1 + tid; i < l2; i += SM_BLOCK) {
        const uint32_t x = s.order[i];
        atomicOr(&s.vis[x >> 5], 1u << (x & 31));
      }
    }
    __syncthreads();
    auto sum = [&](int32_t e0, int32_t e1, int step) {
      double acc = 0.0;
      for (int32_t e = e0; e < e1; e += 8 * step) {
        int32_t x[8];
#pragma unroll
        for (int k = 0; k < 8; k++) x[k] = G.col[min(e + k * step, e1 - 1)];
#pragma unroll
        for (int k = 0; k < 8; k++)
          if (e + k * step < e1 && ((s.vis[x[k] >> 5] >> (x[k] & 31)) & 1u)) acc += s.sigma[x[k]];
      }
      return acc;
    };
    auto store = [&](uint32_t v, double acc) {
      const double sv = s.sigma[v];
      const double dv = sv * acc;
      dl[v] = dv;
      s.sigma[v] = (1.0 + dv) / sv;
    };
    const bool leaf = d == (int32_t)depth - 1;
    for (uint32_t i0 = l0 + wv * PER; i0 < l1; i0 += SM_WAVES * PER) {
      const bool on = i0 + sub < l1;
      const uint32_t v = on ? s.order[i0 + sub] : 0u;
      const int32_t beg = on && !leaf ? G.rp[v] : 0, end = on && !leaf ? G.rp[v + 1] : 0;
      const bool hub = end - beg >= SB_HUB;
      double acc = hub ? 0.0 : sum(beg + sl, end, SB_G);
#pragma unroll
      for (int k = SB_G / 2; k >= 1; k >>= 1) acc += __shfl_xor(acc, k, GB_WAVE);
      if (on && !hub && sl == 0) store(v, acc);
      uint64_t hubs = __ballot(hub && sl == 0);
      while (hubs) {
        const int l = __ffsll((unsigned long long)hubs) - 1;
        hubs &= hubs - 1;
        const double h = gb_wave_sum_f64(
            sum(__shfl(beg, l, GB_WAVE) + lane, __shfl(end, l, GB_WAVE), GB_WAVE));
        if (lane == l) store(v, h);
      }
    }
    __syncthreads();
  }
}

// bc[v] += delta[slot][v], slots in order, except where v is the source
__global__ void bc_small_accum_kernel(int32_t V, int32_t n, SbSources src,
                                      const double *__restrict__ delta, double *__restrict__ bc) {
  const int32_t v = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  if (v >= V) return;
  double acc = bc[v];
  int32_t s = 0;
  for (; s + 8 <= n; s += 8) {
    double d[8];
#pragma unroll
    for (int k = 0; k < 8; k++) d[k] = delta[(int64_t)(s + k) * V + v];
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (src.s[s + k] != v) acc += d[k];
  }
  for (; s < n; s++)
    if (src.s[s] != v) acc += delta[(int64_t)s * V + v];
  bc[v] = acc;
}

struct SbWork {
  DevBuf delta, loff;
  void release() {
    delta.release();
    loff.release();
  }
};
SbWork &sbw() {
  static SbWork *w = new SbWork();  // never destroyed (no frees at exit)
  return *w;
}

}  // namespace

void gb_bc_small_release() { sbw().release(); }

// A launch of up to SB_SOURCES sources takes 1 to 2 ns an edge, as long as its
// slowest CU, however few they are; the engine 0.3 to 0.5 ms of phases and less per
// edge and source the more there are.  So the line lies at a product of launches and
// edges.  Measured, workgroups against engine (us): uniform, R-MAT and a graph with
// one vertex in two thirds of its edges; 4096 vertices, 131 K edges, 256 sources 181
// / 243 / 281 against 579 / 828 / 468, 1024 sources 628 / 861 / 1026 against 1131 /
// 1436 / 814; 262 K edges, 512 sources 464 / 678 / 946 against 829 / 984 / 661; 524 K
// edges, 256 sources 553 / 586 / 896 against 721 / 930 / 633, 1024 sources 2082 / 2209
// / 3504 against 1594 / 1681 / 1146.  14336 vertices, 524 K edges, 1024 sources 2014
// / 2478 / 4137 against 2461 / 2137 / 1244.
bool gb_bc_small_fits(gb_graph g, int32_t nsrc) {
  for (const char *k : {"GB_BC_GRID", "GB_BC_ALPHA", "GB_BC_HUB", "GB_BC_BCHUNK"}) {
    const char *e = getenv(k);
    if (e && e[0]) return false;
  }
  const char *e = getenv("GB_BC_SMALL");
  return !(e && e[0] == '0') && g->V <= SB_MAX_V &&
         g->E * (((int64_t)nsrc + SB_SOURCES - 1) / SB_SOURCES) <= ((int64_t)1 << 19);
}

gb_status gb_bc_small_run(gb_graph g, const int32_t *h_sources, int32_t nsrc, double *d_bc,
                          int32_t *depth, hipStream_t st) {
  static uint32_t *res = nullptr;  // pinned, kept for the process's life
  if (!res)
    GB_HIP(hipHostMalloc((void **)&res, sizeof(uint32_t) * SB_SOURCES, hipHostMallocDefault));
  SbWork &w = sbw();
  const int32_t V = g->V;
  const int32_t most = std::min(nsrc, SB_SOURCES);
  GB_TRY(w.delta.ensure(sizeof(double) * (size_t)most * V));
  GB_TRY(w.loff.ensure(sizeof(uint32_t) * (size_t)most * (V + 2)));
  const SmGraph<void> G{g->rp ? g->rp : g->rrp, g->rp ? g->col : g->rcol, nullptr, V};
  for (int32_t g0 = 0; g0 < nsrc; g0 += SB_SOURCES) {
    const int n = std::min<int32_t>(SB_SOURCES, nsrc - g0);
    SbSources src{};
    for (int i = 0; i < n; i++) src.s[i] = h_sources[g0 + i];
    if (V <= 4096)
      hipLaunchKernelGGL(bc_small_kernel<4096>, dim3(n), dim3(SM_BLOCK), 0, st, G, src,
                         w.delta.as<double>(), w.loff.as<uint32_t>(), res);
    else
      hipLaunchKernelGGL(bc_small_kernel<SB_MAX_V>, dim3(n), dim3(SM_BLOCK), 0, st, G, src,
                         w.delta.as<double>(), w.loff.as<uint32_t>(), res);
    hipLaunchKernelGGL(bc_small_accum_kernel, dim3((V + 63) / 64), dim3(64), 0, st, V, n, src,
                       w.delta.as<double>(), d_bc);
    GB_HIP(hipGetLastError());
    GB_HIP(hipStreamSynchronize(st));
    for (int i = 0; i < n; i++) *depth = std::max(*depth, (int32_t)res[i]);
  }
  return GB_OK;
}
