// gb_csr_build.hip -- CSR construction on the device from an edge list.
//
// The reference builds its CSRs on the host from the edge files: a counting
// pass (scan_csr_idx, graph/csr.c:133-202) and a scatter in file order
// (read_graph_csr, graph/csr.c:4-66; read_csr_bin, graph/csr.c:211-299).  Here
// the edge list is on the device and the CSR is one stable radix sort of the
// edges by row (edges of a row keep their input order, as the reference's
// scatter does) that carries the other endpoint and the weight along, and a
// search of the sorted rows for the row offsets.  The transpose of a CSR is
// the same construction with the endpoints swapped.
//
// What bounds it: bytes.  A pass reads and writes an edge once (12 bytes with
// 4-byte weights each way) and reads its key once more for the histogram.
// Against a sort of (row, index) pairs, a gather of the payload through the
// sorted indices and one atomic per edge for the row counts, a CSR of R-MAT 20
// (16.8 M edges) takes 0.53 ms instead of 5.4 ms: the row counts took 2.6 ms
// of it, serialised on the hubs' counters, the gather 0.64 ms, a 64-byte line
// per 4-byte value, and allocations 1.5 ms.
#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>
#include <hipcub/device/device_scan.hpp>

#include <algorithm>
#include <atomic>
#include <thread>

#include "gb_device.hpp"
#include "graphbench.h"
#include "gb_internal.hpp"

namespace {

// ---- stable radix sort by row, payload carried -----------------------------
// Least significant digit first, digits of at most RS_MAX_BITS bits, a tile of
// RS_TILE consecutive edges per block.  A pass is four launches: the tiles'
// digit counts, two levels of scan over the tiles (groups of RS_GROUP), and
// the scatter.  Tile-major counts keep every access of the scans coalesced.
constexpr int RS_BLOCK = 256;
constexpr int RS_WAVES = RS_BLOCK / GB_WAVE;
constexpr int RS_TILE = 8192;
constexpr int RS_ITEMS = RS_TILE / RS_BLOCK;       // edges per thread
// the scatter: 16 waves per tile, each over RS_SEG consecutive edges
constexpr int RS_SBLOCK = 1024;
constexpr int RS_SWAVES = RS_SBLOCK / GB_WAVE;
constexpr int RS_SITEMS = RS_TILE / RS_SBLOCK;
constexpr int RS_SEG = RS_TILE / RS_SWAVES;
constexpr int RS_MAX_BITS = 11;
constexpr int RS_GROUP = 64;                       // tiles per scan group

// Digit counts of every tile: hist[tile * D + digit].  The first pass also
// checks the endpoints: a bad one sets *bad, which makes every later kernel
// of the build return at once (nothing is written); its digit is masked, so
// the count stays inside the table.
template <bool CHECK>
__global__ __launch_bounds__(RS_BLOCK) void rs_hist_kernel(
    int64_t E, int32_t V, const int32_t *__restrict__ key, const int32_t *__restrict__ other,
    int shift, int bits, uint32_t *__restrict__ hist, int *__restrict__ bad) {
  __shared__ uint32_t s_cnt[1 << RS_MAX_BITS];
  if (!CHECK && *bad) return;
  const int D = 1 << bits;
  for (int d = threadIdx.x; d < D; d += RS_BLOCK) s_cnt[d] = 0;
  __syncthreads();
  const int64_t t0 = (int64_t)blockIdx.x * RS_TILE;
  bool wrong = false;
  for (int k0 = 0; k0 < RS_ITEMS; k0 += 8) {
    int32_t a[8], b[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {  // clamped: the reads stay one batch
      const int64_t e = min(t0 + (int64_t)(k0 + k) * RS_BLOCK + threadIdx.x, E - 1);
      a[k] = key[e];
      if (CHECK) b[k] = other[e];
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const bool in = t0 + (int64_t)(k0 + k) * RS_BLOCK + threadIdx.x < E;
      if (CHECK) wrong |= a[k] < 0 || a[k] >= V || b[k] < 0 || b[k] >= V;
      if (in) atomicAdd(&s_cnt[((uint32_t)a[k] >> shift) & (D - 1)], 1u);
    }
  }
  if (CHECK && wrong) *bad = 1;
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += RS_BLOCK)
    hist[(int64_t)blockIdx.x * D + d] = s_cnt[d];
}

// Exclusive scan of the counts over the RS_GROUP tiles of a group, in place;
// the group's totals to gsum[group * D + digit].  A block takes 64 digits, a
// wave 16 of the tiles.
__global__ __launch_bounds__(RS_BLOCK) void rs_scan_kernel(int64_t ntiles, int D,
                                                           uint32_t *__restrict__ hist,
                                                           uint32_t *__restrict__ gsum,
                                                           const int *__restrict__ bad) {
  constexpr int PER = RS_GROUP / RS_WAVES;
  __shared__ uint32_t s_sum[RS_WAVES][GB_WAVE];
  if (*bad) return;
  const int w = threadIdx.x >> 6, lane = gb_lane();
  const int d = blockIdx.x * GB_WAVE + lane;
  const int64_t t0 = (int64_t)blockIdx.y * RS_GROUP + w * PER;
  uint32_t x[PER], sum = 0;
#pragma unroll
  for (int k = 0; k < PER; k++)
    x[k] = d < D && t0 + k < ntiles ? hist[(t0 + k) * D + d] : 0u;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const uint32_t v = x[k];
    x[k] = sum;
    sum += v;
  }
  s_sum[w][lane] = sum;
  __syncthreads();
  uint32_t base = 0, tot = 0;
  for (int q = 0; q < RS_WAVES; q++) {
    if (q < w) base += s_sum[q][lane];
    tot += s_sum[q][lane];
  }
#pragma unroll
  for (int k = 0; k < PER; k++)
    if (d < D && t0 + k < ntiles) hist[(t0 + k) * D + d] = base + x[k];
  if (w == 0 && d < D) gsum[(int64_t)blockIdx.y * D + d] = tot;
}

// Exclusive scan of the groups' totals over the groups, in place; the digits'
// totals to total[digit].
__global__ __launch_bounds__(GB_WAVE) void rs_groups_kernel(int64_t ngroups, int D,
                                                            uint32_t *__restrict__ gsum,
                                                            uint32_t *__restrict__ total,
                                                            const int *__restrict__ bad) {
  if (*bad) return;
  const int d = blockIdx.x * GB_WAVE + threadIdx.x;
  if (d >= D) return;
  uint32_t sum = 0;
  for (int64_t g0 = 0; g0 < ngroups; g0 += 16) {
    uint32_t x[16];
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = g0 + k < ngroups ? gsum[(g0 + k) * D + d] : 0u;
#pragma unroll
    for (int k = 0; k < 16; k++) {
      if (g0 + k < ngroups) gsum[(g0 + k) * D + d] = sum;
      sum += x[k];
    }
  }
  total[d] = sum;
}

// Exclusive scan of s[0 .. N) by a block of NB threads (N a power of two).
template <int NB, int N>
__device__ __forceinline__ void rs_block_scan(uint32_t *s) {
  constexpr int PER = N > NB ? N / NB : 1, NW = NB / GB_WAVE;
  __shared__ uint32_t s_w[NW];
  const int b = threadIdx.x * PER;
  uint32_t x[PER], sum = 0;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    x[k] = b + k < N ? s[b + k] : 0u;
    sum += x[k];
  }
  uint32_t wt;
  uint32_t ex = gb_wave_excl_sum(sum, &wt);
  if (gb_lane() == 0) s_w[threadIdx.x >> 6] = wt;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NW; q++) ex += q < (int)(threadIdx.x >> 6) ? s_w[q] : 0u;
#pragma unroll
  for (int k = 0; k < PER; k++) {
    if (b + k < N) s[b + k] = ex;
    ex += x[k];
  }
  __syncthreads();
}

// Moves a tile's edges to their digits' places, keeping their order.  A wave
// owns RS_SEG consecutive edges and ranks them 64 at a time: the lanes with
// the same digit find each other with one ballot per digit bit, and the
// wave's own counter of the digit (LDS, one writer) gives the rank of the
// first.  The tile is then put in digit order in LDS, one array after the
// other, so that a digit's edges leave as one run of consecutive addresses:
// written straight from the ranking lanes, each edge was a write request of
// its own and a pass over 16.8 M edges took 426 us instead of
// 173 us (2.3 TB/s).
// Digits have BITS bits; LDS is 34, 40 or 80 KiB at 8, 10 or 11.  At 10 and 11
// bits the kernel keeps its 89 registers (one block of 16 waves per CU): held
// to 64 for two blocks it spills, 205 us a pass.  At 8 bits it spills little
// and two blocks win (R-MAT 24 with 134 M edges, a CSR and its reverse: 8.4
// against 9.2 ms).
template <int WB, int BITS>
__global__ __launch_bounds__(RS_SBLOCK)
__attribute__((amdgpu_waves_per_eu(BITS == 8 ? 8 : 4))) void rs_scatter_kernel(
    int64_t E, const int32_t *__restrict__ key, const int32_t *__restrict__ val,
    const void *__restrict__ w, int shift, const uint32_t *__restrict__ hist,
    const uint32_t *__restrict__ gsum, const uint32_t *__restrict__ total,
    int32_t *__restrict__ key_out, int32_t *__restrict__ val_out, void *__restrict__ w_out,
    const int *__restrict__ bad) {
  constexpr int D = 1 << BITS;
  __shared__ uint32_t s_delta[D];  // global minus tile place of a digit
  __shared__ uint32_t s_place[D];  // tile place of a digit
  // the tile takes the counters' place once the ranks are known
  constexpr int CNT_WORDS = RS_SWAVES * D / 2;
  __shared__ uint32_t s_tile[RS_TILE > CNT_WORDS ? RS_TILE : CNT_WORDS];
  uint16_t *s_cnt = (uint16_t *)s_tile;  // [RS_SWAVES][D]
  if (*bad) return;
  for (int d = threadIdx.x; d < D; d += RS_SBLOCK) s_delta[d] = total[d];
  for (int d = threadIdx.x; d < RS_SWAVES * D / 2; d += RS_SBLOCK) ((uint32_t *)s_cnt)[d] = 0;
  __syncthreads();
  rs_block_scan<RS_SBLOCK, D>(s_delta);
  const int wv = threadIdx.x >> 6, lane = gb_lane();
  const uint64_t below = (1ull << lane) - 1;
  const int64_t t0 = (int64_t)blockIdx.x * RS_TILE;
  const int n = (int)min((int64_t)RS_TILE, E - t0);
  const int32_t *tkey = key + t0, *tval = val + t0;
  const int i0 = wv * RS_SEG + lane;  // this lane's first edge in the tile
  volatile uint16_t *cnt = s_cnt + wv * D;
  uint32_t at[RS_SITEMS];  // digit | rank << 16, then the place in the tile
  int32_t kk[RS_SITEMS];
#pragma unroll
  for (int r = 0; r < RS_SITEMS; r++) kk[r] = tkey[(uint32_t)min(i0 + r * GB_WAVE, n - 1)];
#pragma unroll
  for (int r = 0; r < RS_SITEMS; r++) {
    const bool in = i0 + r * GB_WAVE < n;
    const uint32_t d = ((uint32_t)kk[r] >> shift) & (D - 1);
    uint64_t peers = __ballot(in);
#pragma unroll
    for (int b = 0; b < BITS; b++) {
      const bool one = (d >> b) & 1u;
      const uint64_t m = __ballot(one);
      peers &= one ? m : ~m;
    }
    uint32_t old = 0;
    if (in) old = cnt[d];
    __builtin_amdgcn_wave_barrier();
    if (in && (peers & below) == 0) cnt[d] = (uint16_t)(old + (uint32_t)__popcll(peers));
    __builtin_amdgcn_wave_barrier();
    at[r] = d | (old + (uint32_t)__popcll(peers & below)) << 16;
  }
  __syncthreads();
  // the tile's counts of each digit, their scan, and each wave's first place
  for (int d = threadIdx.x; d < D; d += RS_SBLOCK) {
    uint32_t c = 0;
    for (int q = 0; q < RS_SWAVES; q++) c += s_cnt[q * D + d];
    s_place[d] = c;
  }
  __syncthreads();
  rs_block_scan<RS_SBLOCK, D>(s_place);
  const int64_t g = blockIdx.x / RS_GROUP;
  for (int d = threadIdx.x; d < D; d += RS_SBLOCK) {
    uint32_t p = s_place[d];
    s_delta[d] += gsum[g * D + d] + hist[(int64_t)blockIdx.x * D + d] - p;
    for (int q = 0; q < RS_SWAVES; q++) {
      const uint32_t c = s_cnt[q * D + d];
      s_cnt[q * D + d] = (uint16_t)p;  // < RS_TILE where c > 0
      p += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RS_SITEMS; r++) at[r] = s_cnt[wv * D + (at[r] & 0xFFFFu)] + (at[r] >> 16);
  __syncthreads();  // the counters give way to the tile
  // the keys give every place its address; the other arrays follow
  uint32_t dest[RS_SITEMS];
#pragma unroll
  for (int r = 0; r < RS_SITEMS; r++)
    if (i0 + r * GB_WAVE < n) s_tile[at[r]] = (uint32_t)kk[r];
  __syncthreads();
  int32_t x[RS_SITEMS];
#pragma unroll
  for (int r = 0; r < RS_SITEMS; r++) x[r] = tval[(uint32_t)min(i0 + r * GB_WAVE, n - 1)];
#pragma unroll
  for (int r = 0; r < RS_SITEMS; r++) {
    const int i = r * RS_SBLOCK + threadIdx.x;
    if (i < n) {
      const uint32_t k = s_tile[i];
      dest[r] = (uint32_t)i + s_delta[(k >> shift) & (D - 1)];
      key_out[dest[r]] = (int32_t)k;
    }
  }
  // one 4-byte array through the tile: out word dest * step + off
  auto move = [&](uint32_t *out, int step, int off) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_SITEMS; r++)
      if (i0 + r * GB_WAVE < n) s_tile[at[r]] = (uint32_t)x[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_SITEMS; r++) {
      const int i = r * RS_SBLOCK + threadIdx.x;
      if (i < n) out[(uint64_t)dest[r] * step + off] = s_tile[i];
    }
  };
  move((uint32_t *)val_out, 1, 0);
  for (int h = 0; h < WB / 4; h++) {
    const int32_t *ws = (const int32_t *)w + t0 * (WB / 4) + h;
#pragma unroll
    for (int r = 0; r < RS_SITEMS; r++)
      x[r] = ws[(uint32_t)(min(i0 + r * GB_WAVE, n - 1) * (WB / 4))];
    move((uint32_t *)w_out, WB / 4, h);
  }
}

// row_ptr[r] = first index whose row is >= r, for r in [0, V]: a binary search
// per row in the sorted rows, inside the edges that share its high digit
// (total: the last pass's digit counts, `shift` its shift).
__global__ __launch_bounds__(RS_BLOCK) void rs_rows_kernel(int32_t V, int64_t E,
                                                           const int32_t *__restrict__ row,
                                                           int shift, int bits,
                                                           const uint32_t *__restrict__ total,
                                                           int32_t *__restrict__ row_ptr,
                                                           const int *__restrict__ bad) {
  constexpr int MAXD = 1 << RS_MAX_BITS;
  __shared__ uint32_t s_base[MAXD + 1];
  if (*bad) return;
  const int D = 1 << bits;
  for (int d = threadIdx.x; d < MAXD; d += RS_BLOCK) s_base[d] = d < D ? total[d] : 0u;
  __syncthreads();
  rs_block_scan<RS_BLOCK, MAXD>(s_base);
  if (threadIdx.x == 0) s_base[D] = (uint32_t)E;
  __syncthreads();
  for (int64_t r = (int64_t)blockIdx.x * RS_BLOCK + threadIdx.x; r <= V;
       r += (int64_t)gridDim.x * RS_BLOCK) {
    const int64_t d = r >> shift;  // r = V may lie past the last digit
    uint32_t lo = d < D ? s_base[d] : (uint32_t)E, hi = d < D ? s_base[d + 1] : (uint32_t)E;
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (row[mid] < r)
        lo = mid + 1;
      else
        hi = mid;
    }
    row_ptr[r] = (int32_t)lo;
  }
}

// Row id of every edge of a CSR.  A block takes EX_TILE consecutive edges:
// the rows that begin inside the tile leave their ids at their first edges
// (the largest where several begin at one edge: all but the last are empty),
// and a running maximum over the tile fills the rest.  The first edge's row
// is found by binary search.  One wave per row had left hub rows to one wave
// (R-MAT 20: 201 us, now 48 us).
constexpr int EX_ITEMS = 16;
constexpr int EX_TILE = RS_BLOCK * EX_ITEMS;
__global__ __launch_bounds__(RS_BLOCK) void expand_rows_kernel(int32_t V, int64_t E,
                                                               const int32_t *__restrict__ rp,
                                                               int32_t *__restrict__ row) {
  __shared__ int32_t s_row[EX_TILE];
  __shared__ int32_t s_wmax[RS_WAVES];
  __shared__ int32_t s_lim[2];
  const int64_t t0 = (int64_t)blockIdx.x * EX_TILE;
  const int64_t t1 = min(t0 + EX_TILE, E);
  for (int i = threadIdx.x; i < EX_TILE; i += RS_BLOCK) s_row[i] = 0;
  if (threadIdx.x < 2) {
    // thread 0: last row with rp <= t0 (the first edge's row); thread 1: last
    // row with rp < t1
    const int64_t x = threadIdx.x ? t1 - 1 : t0;
    int32_t lo = 0, hi = V;  // rp[lo] <= x < rp[hi] = E
    while (hi - lo > 1) {
      const int32_t mid = lo + (hi - lo) / 2;
      if (rp[mid] <= x)
        lo = mid;
      else
        hi = mid;
    }
    s_lim[threadIdx.x] = lo;
  }
  __syncthreads();
  const int32_t first = s_lim[0], last = s_lim[1];
  if (last - first > 8 * EX_TILE) {
    // mostly empty rows: a search per edge instead of a visit per row
    for (int64_t e = t0 + threadIdx.x; e < t1; e += RS_BLOCK) {
      int32_t lo = first, hi = last + 1;
      while (hi - lo > 1) {
        const int32_t mid = lo + (hi - lo) / 2;
        if (rp[mid] <= e)
          lo = mid;
        else
          hi = mid;
      }
      row[e] = lo;
    }
    return;
  }
  for (int64_t v = (int64_t)first + 1 + threadIdx.x; v <= last; v += RS_BLOCK) {
    // rp[v] in (t0, t1) or, for an empty row, at the tile's first edge or
    // equal to a later row's
    const int64_t o = rp[v] - t0;
    if (o >= 0 && o < EX_TILE) atomicMax(&s_row[o], (int32_t)v);
  }
  if (threadIdx.x == 0) atomicMax(&s_row[0], first);
  __syncthreads();
  // thread i holds EX_ITEMS consecutive edges
  int32_t m = 0, x[EX_ITEMS];
#pragma unroll
  for (int k = 0; k < EX_ITEMS; k++) {
    m = max(m, s_row[threadIdx.x * EX_ITEMS + k]);
    x[k] = m;
  }
  int32_t incl = m;
#pragma unroll
  for (int d = 1; d < GB_WAVE; d <<= 1) {
    const int32_t y = __shfl_up(incl, d, GB_WAVE);
    if (gb_lane() >= d) incl = max(incl, y);
  }
  if (gb_lane() == GB_WAVE - 1) s_wmax[threadIdx.x >> 6] = incl;
  int32_t before = __shfl_up(incl, 1, GB_WAVE);
  if (gb_lane() == 0) before = 0;
  __syncthreads();
  for (int q = 0; q < (int)(threadIdx.x >> 6); q++) before = max(before, s_wmax[q]);
#pragma unroll
  for (int k = 0; k < EX_ITEMS; k++) s_row[threadIdx.x * EX_ITEMS + k] = max(x[k], before);
  __syncthreads();
  for (int64_t e = t0 + threadIdx.x; e < t1; e += RS_BLOCK) row[e] = s_row[e - t0];
}

// Scratch of the builds, kept between calls up to CSR_KEEP bytes (allocating
// and freeing it took 1.5 ms of a 5.4 ms build).  One build uses it at a time,
// on any thread, stream and device: a build waits for its stream before it lets
// go of the scratch, and one on another device starts with none.  An allocation
// that would fail elsewhere in the library takes it back first (gb_csr_trim), a
// build whose own allocations fail gives up what it does not use;
// gb_release_workspaces returns it to other allocators.
constexpr size_t CSR_KEEP = (size_t)4 << 30;
struct CsrWork {
  std::atomic<int> busy{0};
  int device = -1;  // where the buffers are
  DevBuf rows, k[2], v, w, hist, gsum, total, flag;
  size_t held() const {
    return rows.bytes + k[0].bytes + k[1].bytes + v.bytes + w.bytes + hist.bytes + gsum.bytes +
           total.bytes + flag.bytes;
  }
  void release() {
    rows.release();
    release_sort();
  }
  void release_sort() {  // all but the row ids of a transpose
    for (DevBuf *b : {&k[0], &k[1], &v, &w, &hist, &gsum, &total, &flag}) b->release();
  }
};
// Holds the scratch for one build; at most CSR_KEEP bytes outlive it.
struct CsrHold {
  CsrWork &k;
  explicit CsrHold(CsrWork &work) : k(work) {
    int idle = 0;
    while (!k.busy.compare_exchange_weak(idle, 1)) {
      idle = 0;
      std::this_thread::yield();
    }
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (dev != k.device) k.release();
    k.device = dev;
  }
  ~CsrHold() {
    if (k.held() > CSR_KEEP) k.release();
    k.busy.store(0);
  }
};
// Heap singleton, never destroyed (no device memory freed from a static
// destructor).
CsrWork &csr_work() {
  static CsrWork *w = new CsrWork();
  return *w;
}

// Whether [a, a + na) and [b, b + nb) share a byte.
bool overlap(const void *a, size_t na, const void *b, size_t nb) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return a && b && x < y + nb && y < x + na;
}

int grid_for(int64_t n) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, (int64_t)gb_num_cus() * 16));
}

// ---- duplicate edges ------------------------------------------------------
__global__ void pair_keys_kernel(int64_t E, const int32_t *__restrict__ src,
                                 const int32_t *__restrict__ dst, uint64_t *__restrict__ key,
                                 int32_t *__restrict__ ids, int *__restrict__ bad) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int32_t s = src[e], d = dst[e];
    if (s < 0 || d < 0) *bad = 1;
    key[e] = ((uint64_t)(uint32_t)s << 32) | (uint32_t)d;
    ids[e] = (int32_t)e;
  }
}

// keep[e] = 1 for the first index of each run of equal keys (the sort is
// stable, so that is the pair's first occurrence in input order)
__global__ void first_of_run_kernel(int64_t E, const uint64_t *__restrict__ skey,
                                    const int32_t *__restrict__ sid, int32_t *__restrict__ keep) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < E;
       i += (int64_t)gridDim.x * blockDim.x)
    keep[sid[i]] = (i == 0 || skey[i] != skey[i - 1]) ? 1 : 0;
}

__global__ void compact_pairs_kernel(int64_t E, const int32_t *__restrict__ keep,
                                     const int32_t *__restrict__ pos,
                                     const int32_t *__restrict__ src,
                                     const int32_t *__restrict__ dst, int32_t *__restrict__ src_out,
                                     int32_t *__restrict__ dst_out) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < E;
       e += (int64_t)gridDim.x * blockDim.x)
    if (keep[e]) {
      src_out[pos[e]] = src[e];
      dst_out[pos[e]] = dst[e];
    }
}

}  // namespace

// Keeps the first occurrence of every (src, dst) pair, in input order, as
// remove_duplicate (partition/csr_partition_bin_mpi.c:31-106) does with a hash
// set over the file order: a stable radix sort of the 64-bit pair keys with
// their indices marks the first index of each run; a scan compacts.
extern "C" gb_status gb_edges_unique(int64_t E, const int32_t *d_src, const int32_t *d_dst,
                                     int32_t *d_src_out, int32_t *d_dst_out, int64_t *h_kept,
                                     void *stream) {
  if (E < 0 || E >= ((int64_t)1 << 31) || !h_kept ||
      (E > 0 && (!d_src || !d_dst || !d_src_out || !d_dst_out)))
    return gb_fail(GB_ERR_INVALID, "gb_edges_unique: bad arguments");
  *h_kept = 0;
  if (E == 0) return GB_OK;
  hipStream_t st = gb_stream(stream);
  DevBuf key, skey, ids, sids, keep, pos, flag, tmp;
  GB_TRY(key.ensure(sizeof(uint64_t) * E));
  GB_TRY(skey.ensure(sizeof(uint64_t) * E));
  GB_TRY(ids.ensure(sizeof(int32_t) * E));
  GB_TRY(sids.ensure(sizeof(int32_t) * E));
  GB_TRY(keep.ensure(sizeof(int32_t) * E));
  GB_TRY(pos.ensure(sizeof(int32_t) * (E + 1)));
  GB_TRY(flag.ensure(sizeof(int)));
  GB_HIP(hipMemsetAsync(flag.p, 0, sizeof(int), st));
  hipLaunchKernelGGL(pair_keys_kernel, dim3(grid_for(E)), dim3(256), 0, st, E, d_src, d_dst,
                     key.as<uint64_t>(), ids.as<int32_t>(), flag.as<int>());
  GB_HIP(hipGetLastError());
  int bad = 0;
  GB_HIP(hipMemcpyAsync(&bad, flag.p, sizeof(int), hipMemcpyDeviceToHost, st));
  GB_HIP(hipStreamSynchronize(st));
  if (bad) return gb_fail(GB_ERR_INVALID, "gb_edges_unique: negative vertex id");
  size_t tb_sort = 0, tb_scan = 0;
  GB_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb_sort, key.as<uint64_t>(),
                                            skey.as<uint64_t>(), ids.as<int32_t>(),
                                            sids.as<int32_t>(), (int)E, 0, 64, st));
  GB_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb_scan, keep.as<int32_t>(),
                                          pos.as<int32_t>(), (int)E, st));
  GB_TRY(tmp.ensure(std::max(tb_sort, tb_scan) + 16));
  GB_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb_sort, key.as<uint64_t>(),
                                            skey.as<uint64_t>(), ids.as<int32_t>(),
                                            sids.as<int32_t>(), (int)E, 0, 64, st));
  hipLaunchKernelGGL(first_of_run_kernel, dim3(grid_for(E)), dim3(256), 0, st, E,
                     skey.as<uint64_t>(), sids.as<int32_t>(), keep.as<int32_t>());
  GB_HIP(hipcub::DeviceScan::ExclusiveSum(tmp.p, tb_scan, keep.as<int32_t>(), pos.as<int32_t>(),
                                          (int)E, st));
  hipLaunchKernelGGL(compact_pairs_kernel, dim3(grid_for(E)), dim3(256), 0, st, E,
                     keep.as<int32_t>(), pos.as<int32_t>(), d_src, d_dst, d_src_out, d_dst_out);
  GB_HIP(hipGetLastError());
  int32_t last_pos = 0, last_keep = 0;
  GB_HIP(hipMemcpyAsync(&last_pos, pos.as<int32_t>() + (E - 1), sizeof(int32_t),
                        hipMemcpyDeviceToHost, st));
  GB_HIP(hipMemcpyAsync(&last_keep, keep.as<int32_t>() + (E - 1), sizeof(int32_t),
                        hipMemcpyDeviceToHost, st));
  GB_HIP(hipStreamSynchronize(st));  // scratch buffers are freed on return
  *h_kept = (int64_t)last_pos + last_keep;
  return GB_OK;
}

namespace {

// The build on the workspace (its lock held): edges sorted by d_src.
template <int WB>
gb_status csr_build(CsrWork &k, int32_t V, int64_t E, const int32_t *d_src, const int32_t *d_dst,
                    const void *d_w, int32_t *d_row_ptr, int32_t *d_col, void *d_w_out,
                    hipStream_t st) {
  GB_TRY(k.flag.ensure(sizeof(int)));
  if (E == 0) {
    GB_HIP(hipMemsetAsync(d_row_ptr, 0, sizeof(int32_t) * ((size_t)V + 1), st));
    GB_HIP(hipStreamSynchronize(st));
    return GB_OK;
  }
  int bits = 1;
  while (bits < 31 && ((int64_t)1 << bits) < (int64_t)V) bits++;
  // as few passes as 11-bit digits allow, with the smallest of 8, 10 and 11
  // bits that needs no more: a pass costs about as much at each (13, 16 and 10
  // us per million edges at 10, 11 and 8 bits on R-MAT 20, 22 and 24)
  const int passes = (bits + RS_MAX_BITS - 1) / RS_MAX_BITS;
  const int even = (bits + passes - 1) / passes;
  const int db = even <= 8 ? 8 : even <= 10 ? 10 : 11;
  const int D = 1 << db;
  const int64_t ntiles = (E + RS_TILE - 1) / RS_TILE;
  const int64_t ngroups = (ntiles + RS_GROUP - 1) / RS_GROUP;
  // the endpoints and weights alternate between the scratch and the caller's
  // arrays so that the last pass ends in the latter
  GB_TRY(k.k[0].ensure(sizeof(int32_t) * E));
  if (passes > 1) {
    GB_TRY(k.k[1].ensure(sizeof(int32_t) * E));
    GB_TRY(k.v.ensure(sizeof(int32_t) * E));
    if (WB) GB_TRY(k.w.ensure((size_t)WB * E));
  }
  GB_TRY(k.hist.ensure(sizeof(uint32_t) * ntiles * D));
  GB_TRY(k.gsum.ensure(sizeof(uint32_t) * ngroups * D));
  GB_TRY(k.total.ensure(sizeof(uint32_t) * D));
  // An output may take the place of the keys (d_src; a transpose in place:
  // d_tcol == d_col).  Where the first pass writes the caller's arrays, tiles
  // would write them while others read their keys: the keys move away first.
  const bool aside = passes % 2 == 1 && (overlap(d_src, sizeof(int32_t) * E, d_col, sizeof(int32_t) * E) ||
                                         overlap(d_src, sizeof(int32_t) * E, d_w_out, (size_t)WB * E));
  if (aside) GB_TRY(k.k[1].ensure(sizeof(int32_t) * E));
  int *bad = k.flag.as<int>();
  uint32_t *hist = k.hist.as<uint32_t>(), *gsum = k.gsum.as<uint32_t>(),
           *total = k.total.as<uint32_t>();
  GB_HIP(hipMemsetAsync(bad, 0, sizeof(int), st));
  const int32_t *key = d_src, *val = d_dst;
  const void *w = d_w;
  if (aside) {
    GB_HIP(hipMemcpyAsync(k.k[1].p, d_src, sizeof(int32_t) * E, hipMemcpyDeviceToDevice, st));
    key = k.k[1].as<int32_t>();  // pass 0 writes k[0], and pass 1, if any, reads that
  }
  for (int p = 0; p < passes; p++) {
    const int shift = p * db;
    const bool to_caller = (passes - 1 - p) % 2 == 0;
    if (p == 0)
      hipLaunchKernelGGL(rs_hist_kernel<true>, dim3((unsigned)ntiles), dim3(RS_BLOCK), 0, st, E, V,
                         key, val, shift, db, hist, bad);
    else
      hipLaunchKernelGGL(rs_hist_kernel<false>, dim3((unsigned)ntiles), dim3(RS_BLOCK), 0, st, E,
                         V, key, val, shift, db, hist, bad);
    hipLaunchKernelGGL(rs_scan_kernel, dim3((D + GB_WAVE - 1) / GB_WAVE, (unsigned)ngroups),
                       dim3(RS_BLOCK), 0, st, ntiles, D, hist, gsum, bad);
    hipLaunchKernelGGL(rs_groups_kernel, dim3((D + GB_WAVE - 1) / GB_WAVE), dim3(GB_WAVE), 0, st,
                       ngroups, D, gsum, total, bad);
    int32_t *ko = k.k[p & 1].as<int32_t>();
    int32_t *vo = to_caller ? d_col : k.v.as<int32_t>();
    void *wo = to_caller ? d_w_out : k.w.p;
    auto scatter = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)ntiles), dim3(RS_SBLOCK), 0, st, E, key, val, w,
                         shift, hist, gsum, total, ko, vo, wo, bad);
    };
    if (db == 8)
      scatter(rs_scatter_kernel<WB, 8>);
    else if (db == 10)
      scatter(rs_scatter_kernel<WB, 10>);
    else
      scatter(rs_scatter_kernel<WB, 11>);
    GB_HIP(hipGetLastError());
    key = ko;
    val = vo;
    w = wo;
  }
  hipLaunchKernelGGL(rs_rows_kernel, dim3(grid_for((int64_t)V + 1)), dim3(RS_BLOCK), 0, st, V, E,
                     key, (passes - 1) * db, db, total, d_row_ptr, bad);
  GB_HIP(hipGetLastError());
  int h_bad = 0;
  GB_HIP(hipMemcpyAsync(&h_bad, bad, sizeof(int), hipMemcpyDeviceToHost, st));
  GB_HIP(hipStreamSynchronize(st));  // the scratch is idle from here on
  if (h_bad) return gb_fail(GB_ERR_INVALID, "gb_csr_from_edges: endpoint outside [0, V)");
  return GB_OK;
}

gb_status csr_build_any(CsrWork &k, int32_t V, int64_t E, const int32_t *d_src,
                        const int32_t *d_dst, const void *d_w, int32_t w_bytes, int32_t *d_row_ptr,
                        int32_t *d_col, void *d_w_out, hipStream_t st) {
  auto build = [&]() {
    return w_bytes == 8   ? csr_build<8>(k, V, E, d_src, d_dst, d_w, d_row_ptr, d_col, d_w_out, st)
           : w_bytes == 4 ? csr_build<4>(k, V, E, d_src, d_dst, d_w, d_row_ptr, d_col, d_w_out, st)
                          : csr_build<0>(k, V, E, d_src, d_dst, d_w, d_row_ptr, d_col, d_w_out, st);
  };
  gb_status s = build();
  if (s == GB_ERR_NOMEM) {
    // nothing is queued yet but a transpose's row ids: without what earlier
    // builds left, once more
    k.release_sort();
    if (d_dst != k.rows.p) k.rows.release();
    s = build();
  }
  if (s != GB_OK) (void)hipStreamSynchronize(st);  // launches before an error end first
  return s;
}

}  // namespace

// Gives the kept scratch back unless a build is using it; returns whether it
// held anything.
bool gb_csr_trim() {
  CsrWork &k = csr_work();
  int idle = 0;
  if (!k.busy.compare_exchange_strong(idle, 2)) return false;
  const bool had = k.held() > 0;
  k.release();
  k.busy.store(0);
  return had;
}

extern "C" gb_status gb_csr_from_edges(int32_t V, int64_t E, const int32_t *d_src,
                                       const int32_t *d_dst, const void *d_w, int32_t w_bytes,
                                       int32_t *d_row_ptr, int32_t *d_col, void *d_w_out,
                                       void *stream) {
  if (V < 0 || E < 0 || E >= ((int64_t)1 << 31) || !d_row_ptr || (E > 0 && (!d_src || !d_dst || !d_col)))
    return gb_fail(GB_ERR_INVALID, "gb_csr_from_edges: bad arguments");
  if (w_bytes != 0 && w_bytes != 4 && w_bytes != 8)
    return gb_fail(GB_ERR_INVALID, "gb_csr_from_edges: w_bytes must be 0, 4 or 8");
  if (w_bytes && E > 0 && (!d_w || !d_w_out))
    return gb_fail(GB_ERR_INVALID, "gb_csr_from_edges: weights without a weight buffer");
  CsrHold hold(csr_work());
  CsrWork &k = hold.k;
  return csr_build_any(k, V, E, d_src, d_dst, d_w, w_bytes, d_row_ptr, d_col, d_w_out,
                       gb_stream(stream));
}

extern "C" gb_status gb_csr_transpose(int32_t V, int64_t E, const int32_t *d_row_ptr,
                                      const int32_t *d_col, const void *d_w, int32_t w_bytes,
                                      int32_t *d_trow_ptr, int32_t *d_tcol, void *d_tw,
                                      void *stream) {
  if (V < 0 || E < 0 || !d_row_ptr || !d_trow_ptr || (E > 0 && (!d_col || !d_tcol)))
    return gb_fail(GB_ERR_INVALID, "gb_csr_transpose: bad arguments");
  if (E >= ((int64_t)1 << 31) || (w_bytes != 0 && w_bytes != 4 && w_bytes != 8) ||
      (w_bytes && E > 0 && (!d_w || !d_tw)))
    return gb_fail(GB_ERR_INVALID, "gb_csr_transpose: bad arguments");
  hipStream_t st = gb_stream(stream);
  CsrHold hold(csr_work());
  CsrWork &k = hold.k;
  gb_status rs = k.rows.ensure(sizeof(int32_t) * ((size_t)E + 1));
  if (rs == GB_ERR_NOMEM) {
    k.release();
    rs = k.rows.ensure(sizeof(int32_t) * ((size_t)E + 1));
  }
  GB_TRY(rs);
  if (E > 0 && V > 0) {
    hipLaunchKernelGGL(expand_rows_kernel, dim3((unsigned)((E + EX_TILE - 1) / EX_TILE)),
                       dim3(RS_BLOCK), 0, st, V, E, d_row_ptr, k.rows.as<int32_t>());
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return gb_fail(GB_ERR_HIP, "expand_rows: %s", hipGetErrorString(e));
  }
  // transposed rows are keyed by the column; edges of a transposed row keep
  // the order of their source rows
  return csr_build_any(k, V, E, d_col, k.rows.as<int32_t>(), d_w, w_bytes, d_trow_ptr, d_tcol,
                       d_tw, st);
}
