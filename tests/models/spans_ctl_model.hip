// Host model of both engines' phases over ranges of buckets (SpanCtl): queue
// entries counted per phase and handed to the next advance the way the
// one-launch phases do, against Dijkstra on random graphs.
#include "gb_sssp_ctl.hpp"
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <queue>
#include <random>
#include <vector>
using u64 = uint64_t;
struct Csr {
  int V;
  std::vector<int> rp, le, col;
  std::vector<uint32_t> w;
};
static std::mt19937_64 rng(4242);
static Csr graph(int tr, uint32_t wmax, uint32_t lmax) {
  Csr g;
  g.V = 1 + rng() % 200;
  std::vector<std::vector<std::pair<uint32_t, int>>> adj(g.V);
  const int E = rng() % (g.V * 6 + 1);
  for (int e = 0; e < E; e++) adj[rng() % g.V].push_back({(uint32_t)(rng() % (wmax + 1)), (int)(rng() % g.V)});
  if (tr % 4 == 0)  // a long path: many buckets, few entries each
    for (int v = 0; v + 1 < g.V; v++) adj[v].push_back({1 + (uint32_t)(rng() % (wmax + 1)), v + 1});
  g.rp.assign(1, 0);
  for (auto &a : adj) {
    std::stable_sort(a.begin(), a.end(), [&](auto x, auto y) { return (x.first <= lmax) > (y.first <= lmax); });
    int l = 0;
    for (auto &p : a) {
      g.w.push_back(p.first);
      g.col.push_back(p.second);
      l += p.first <= lmax;
    }
    g.le.push_back(g.rp.back() + l);
    g.rp.push_back((int)g.col.size());
  }
  return g;
}
static std::vector<u64> dijkstra(const Csr &g, int s) {
  std::vector<u64> d(g.V, ~0ull);
  std::priority_queue<std::pair<u64, int>, std::vector<std::pair<u64, int>>, std::greater<>> q;
  d[s] = 0;
  q.push({0, s});
  while (!q.empty()) {
    auto [x, u] = q.top();
    q.pop();
    if (x > d[u]) continue;
    for (int e = g.rp[u]; e < g.rp[u + 1]; e++)
      if (x + g.w[e] < d[g.col[e]]) q.push({d[g.col[e]] = x + g.w[e], g.col[e]});
  }
  return d;
}
static SpanCtl spans() {
  SpanCtl c{};
  c.adapt = 1;
  c.few = 1 + rng() % 200;
  c.many = c.few * (1 + rng() % 8);
  c.leap = 2 + rng() % 15;
  return c;
}
// one source, light / heavy phases, "all" ranges
static bool per_source(const Csr &g, uint32_t delta, int src, std::vector<u64> &d, long &phases) {
  d.assign(g.V, ~0ull);
  std::vector<uint32_t> nst(g.V), sst(g.V), fst(g.V);
  std::vector<int> q[5];
  unsigned long long n[C_MINB + 1] = {0};
  u64 minb = ~0ull;
  SsspCtl s{};
  s.gen = 1;
  s.fepoch = 1;
  s.max_phases = 1 << 30;
  s.state = ST_BUCKET;
  s.sp = spans();
  d[src] = 0;
  q[0] = {src};
  n[C_NEAR0] = 1;
  for (long k = 0; k < 4000000; k++) {
    n[C_MINB] = minb;
    sssp_ctl_advance(s, n, 256);
    if (s.done) {
      phases += s.phases;
      return true;
    }
    minb = ~0ull;
    const std::vector<int> in = q[s.a_in];
    if (in.size() != n[s.a_in]) return false;
    q[s.a_near].clear();
    if (s.action == ACT_FAR) q[s.a_far].clear();
    q[C_S].resize(n[C_S]);
    if (q[s.a_far].size() != n[s.a_far]) return false;
    for (int u : in) {
      if (s.action == ACT_FAR) {
        const u64 b = d[u] / delta;
        if (b >= s.a_first && b <= s.a_bucket) {
          if (nst[u] != s.a_gen) q[s.a_near].push_back(u);
          nst[u] = s.a_gen;
        } else if (b > s.a_bucket) {
          if (fst[u] != s.a_fepoch) q[s.a_far].push_back(u);
          fst[u] = s.a_fepoch;
          minb = std::min(minb, b);
        }
        continue;
      }
      const bool heavy = s.action == ACT_HEAVY, all = !heavy && s.a_all;
      if (!heavy && !all && g.rp[u + 1] > g.le[u] && sst[u] != s.a_sround) {
        sst[u] = s.a_sround;
        q[C_S].push_back(u);
      }
      for (int e = heavy ? g.le[u] : g.rp[u]; e < (heavy || all ? g.rp[u + 1] : g.le[u]); e++) {
        const int x = g.col[e];
        const u64 nd = d[u] + g.w[e];
        if (nd >= d[x]) continue;
        d[x] = nd;
        const bool far = nd / delta > s.a_bucket;
        uint32_t &st = far ? fst[x] : nst[x];
        const uint32_t now = far ? s.a_fepoch : s.a_gen;
        if (st != now) q[far ? s.a_far : s.a_near].push_back(x);
        st = now;
      }
    }
    n[s.a_near] = q[s.a_near].size();
    n[s.a_far] = q[s.a_far].size();
    n[C_S] = q[C_S].size();
  }
  return false;
}
// up to 8 sources as masks; masks and near queues rotate through three buffers
static bool batched(const Csr &g, uint32_t delta, const std::vector<int> &src,
                    std::vector<std::vector<u64>> &d, long &phases) {
  const int T = (int)src.size();
  d.assign(T, std::vector<u64>(g.V, ~0ull));
  std::vector<uint32_t> mask[3], far(g.V, 0);
  for (auto &m : mask) m.assign(g.V, 0);
  std::vector<int> qn[3], qf[2];
  unsigned long long n[MS_MINB + 1] = {0};
  u64 minb = ~0ull;
  for (int t = 0; t < T; t++) {
    d[t][src[t]] = 0;
    if (!mask[0][src[t]]) qn[0].push_back(src[t]);
    mask[0][src[t]] |= 1u << t;
  }
  n[MS_NEAR0] = qn[0].size();
  MsCtl s{};
  s.max_phases = 1 << 30;
  s.state = MS_ST_LIGHT;
  s.sp = spans();
  for (long k = 0; k < 4000000; k++) {
    const bool was_light = s.action == ACT_LIGHT;
    const u64 old_n = s.a_in_n;
    n[MS_MINB] = minb;
    ms_ctl_advance(s, n);
    if (s.done) {
      phases += s.phases;
      return true;
    }
    minb = ~0ull;
    const int in = k % 3, out = (k + 1) % 3, old = (k + 2) % 3;
    if (was_light) {
      if (qn[old].size() != old_n) return false;
      for (int v : qn[old]) mask[old][v] = 0;
    }
    qn[out].clear();
    auto mark = [&](int x, uint32_t m) {
      if (m && !mask[out][x]) qn[out].push_back(x);
      mask[out][x] |= m;
    };
    std::vector<int> &fo = qf[s.a_far - MS_FAR0];
    if (s.action == ACT_FAR) {
      fo.clear();
      const std::vector<int> &fi = qf[s.a_in - MS_FAR0];
      if (fi.size() != n[s.a_in]) return false;
      for (int x : fi) {
        uint32_t nm = 0, km = 0;
        for (int t = 0; t < T; t++) {
          if (!((far[x] >> t) & 1)) continue;
          const u64 b = d[t][x] / delta;
          if (b >= s.a_first && b <= s.a_bucket) nm |= 1u << t;
          if (b > s.a_bucket) {
            km |= 1u << t;
            minb = std::min(minb, b);
          }
        }
        far[x] = km;
        mark(x, nm);
        if (km) fo.push_back(x);
      }
    } else {
      if (qn[in].size() != n[s.a_in]) return false;
      for (int u : qn[in])
        for (int e = g.rp[u]; e < g.rp[u + 1]; e++) {
          const int x = g.col[e];
          uint32_t nm = 0, fm = 0;
          for (int t = 0; t < T; t++) {
            if (!((mask[in][u] >> t) & 1)) continue;
            const u64 nd = d[t][u] + g.w[e];
            if (nd >= d[t][x]) continue;
            d[t][x] = nd;
            (nd / delta <= s.a_bucket ? nm : fm) |= 1u << t;
          }
          mark(x, nm);
          if (fm && !far[x]) fo.push_back(x);
          far[x] |= fm;
        }
    }
    n[s.a_near] = qn[out].size();
    n[s.a_far] = fo.size();
  }
  return false;
}
int main(int argc, char **argv) {
  const int trials = argc > 1 ? atoi(argv[1]) : 200;
  long one = 0, many = 0;
  for (int tr = 0; tr < trials; tr++) {
    const uint32_t wmax = 1 + rng() % 1000, delta = 1 + rng() % (wmax / 4 + 2);
    const Csr g = graph(tr, wmax, tr % 3 ? delta : delta / 2);
    std::vector<int> src(1 + rng() % 8);
    for (int &x : src) x = rng() % g.V;
    std::vector<u64> d;
    std::vector<std::vector<u64>> dm;
    if (!per_source(g, delta, src[0], d, one) || !batched(g, delta, src, dm, many)) {
      printf("loop or counts wrong in trial %d\n", tr);
      return 1;
    }
    if (d != dijkstra(g, src[0])) {
      printf("per-source mismatch in trial %d\n", tr);
      return 1;
    }
    for (size_t t = 0; t < src.size(); t++)
      if (dm[t] != dijkstra(g, src[t])) {
        printf("batched mismatch in trial %d\n", tr);
        return 1;
      }
  }
  printf("ok: %d trials, %ld and %ld phases\n", trials, one, many);
  return 0;
}
