// construct.hip -- symmetrize, degree-descending relabel and CSR build on GPU.
//
// Semantics follow the reference's single-rank construction:
//  - self loops dropped, both directions kept, vertex space = 2^(msb(OR of
//    endpoint IDs)+1)          (mpi/benchmark_helper.hpp:389-497)
//  - degree = symmetric edge count including duplicates, vertices renumbered
//    by descending degree      (mpi/graph_constructor.hpp:572-761)
//  - each row sorted by renumbered target, duplicates merged
//    (mpi/graph_constructor.hpp:1968-2101)
// Ties in degree are broken by ascending original ID (the reference's
// std::sort leaves them unspecified), which makes the whole CSR a pure
// function of the edge list.
//
// Pipeline: degrees counted in LDS (csrsort.hip) -> IDs radix-sorted by
// inverted degree -> relabel maps -> rows by bucket partition and LDS sort
// (csrsort.hip).  Lists that partition cannot handle take the general form:
// (new_src, new_dst) keys, loops as a max-value sentinel -> radix sort ->
// flag/scan/scatter dedupe into row offsets + uint32 columns.
#include <algorithm>

#include "internal.hpp"

namespace g500 {

namespace {

constexpr int kT = 256;

// stats[2] = max degree, stats[3] = #vertices with degree > 0,
// stats[4] = max vertex with degree > 0.  Three atomics a block: on one
// address they take ~12 ns each in turn (one set per wave of 8 192 blocks cost
// 1.14 ms at SCALE 24, now 0.03).
__global__ __launch_bounds__(kT) void k_deg_stats(const uint32_t* __restrict__ deg,
                                                 int64_t n,
                                                 unsigned long long* stats) {
  __shared__ uint64_t part[3][kT / kWave];
  uint64_t x[3] = {0, 0, 0};
  for (int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * kT) {
    const uint32_t d = deg[v];
    x[0] = d > x[0] ? d : x[0];
    if (d) {
      ++x[1];
      x[2] = (uint64_t)v;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t a = __shfl_xor(x[0], o, kWave), c = __shfl_xor(x[2], o, kWave);
    x[0] = a > x[0] ? a : x[0];
    x[1] += __shfl_xor(x[1], o, kWave);
    x[2] = c > x[2] ? c : x[2];
  }
  if (lane_id() == 0)
    for (int j = 0; j < 3; ++j) part[j][threadIdx.x / kWave] = x[j];
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kT / kWave; ++w) {
      x[0] = part[0][w] > x[0] ? part[0][w] : x[0];
      x[1] += part[1][w];
      x[2] = part[2][w] > x[2] ? part[2][w] : x[2];
    }
    if (x[0]) atomicMax(&stats[2], (unsigned long long)x[0]);
    if (x[1]) atomicAdd(&stats[3], (unsigned long long)x[1]);
    if (x[2]) atomicMax(&stats[4], (unsigned long long)x[2]);
  }
}

__global__ __launch_bounds__(kT) void k_vertex_keys(const uint32_t* __restrict__ deg,
                                                   int64_t n, int lg,
                                                   uint64_t maxdeg,
                                                   uint64_t* __restrict__ keys) {
  const int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (v < n) keys[v] = ((maxdeg - deg[v]) << lg) | (uint64_t)v;
}

__global__ __launch_bounds__(kT) void k_relabel(const uint64_t* __restrict__ keys,
                                               int64_t n, int lg, uint64_t maxdeg,
                                               uint32_t* __restrict__ n2o,
                                               uint32_t* __restrict__ o2n,
                                               uint32_t* __restrict__ deg_new) {
  const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (i >= n) return;
  const uint64_t k = keys[i];
  const uint32_t o = (uint32_t)(k & ((1ull << lg) - 1));
  n2o[i] = o;
  o2n[o] = (uint32_t)i;
  deg_new[i] = (uint32_t)(maxdeg - (k >> lg));
}

// Two keys per input edge ((a,b) and (b,a)), or one when the input is
// already symmetric; self loops become the sentinel (sorts last).
__global__ __launch_bounds__(kT) void k_sym_keys(const uint2* __restrict__ e,
                                                int64_t ne, int symmetric,
                                                const uint32_t* __restrict__ o2n,
                                                int lg, uint64_t sentinel,
                                                uint64_t* __restrict__ keys) {
  const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (i >= ne) return;
  const uint2 x = e[i];
  uint64_t k0 = sentinel, k1 = sentinel;
  if (x.x != x.y) {
    const uint64_t a = o2n[x.x], b = o2n[x.y];
    k0 = (a << lg) | b;
    k1 = (b << lg) | a;
  }
  if (symmetric) {
    keys[i] = k0;
  } else {
    keys[2 * i] = k0;
    keys[2 * i + 1] = k1;
  }
}

constexpr int kDedupItems = 16;
constexpr int kDedupTile = kT * kDedupItems;

__device__ inline uint64_t block_excl_scan_u64(uint64_t v, uint64_t* wsum,
                                               uint64_t* total) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  uint64_t x = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint64_t y = __shfl_up(x, o, kWave);
    if (lane >= o) x += y;
  }
  if (lane == kWave - 1) wsum[wave] = x;
  __syncthreads();
  uint64_t off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kT / kWave; ++w) {
    off += (w < wave) ? wsum[w] : 0;
    tot += wsum[w];
  }
  __syncthreads();
  *total = tot;
  return x - v + off;
}

// Per tile: number of keys that differ from their predecessor.
__global__ __launch_bounds__(kT) void k_dedup_count(const uint64_t* __restrict__ k,
                                                   int64_t n,
                                                   uint32_t* __restrict__ cnt) {
  __shared__ uint64_t wsum[kT / kWave];
  const int64_t base = (int64_t)blockIdx.x * kDedupTile + threadIdx.x * kDedupItems;
  uint32_t c = 0;
  for (int j = 0; j < kDedupItems; ++j) {
    const int64_t i = base + j;
    if (i < n && (i == 0 || k[i] != k[i - 1])) ++c;
  }
  uint64_t tot;
  (void)block_excl_scan_u64(c, wsum, &tot);
  if (threadIdx.x == 0) cnt[blockIdx.x] = (uint32_t)tot;
}

__global__ __launch_bounds__(kT) void k_dedup_write(
    const uint64_t* __restrict__ k, int64_t n, int lg,
    const uint64_t* __restrict__ tile_off, uint32_t* __restrict__ col,
    int64_t* __restrict__ row_off) {
  __shared__ uint64_t wsum[kT / kWave];
  const int64_t base = (int64_t)blockIdx.x * kDedupTile + threadIdx.x * kDedupItems;
  const uint64_t mask = (1ull << lg) - 1;
  uint32_t c = 0;
  for (int j = 0; j < kDedupItems; ++j) {
    const int64_t i = base + j;
    if (i < n && (i == 0 || k[i] != k[i - 1])) ++c;
  }
  uint64_t tot;
  uint64_t pos = tile_off[blockIdx.x] + block_excl_scan_u64(c, wsum, &tot);
  for (int j = 0; j < kDedupItems; ++j) {
    const int64_t i = base + j;
    if (i >= n) break;
    const uint64_t cur = k[i];
    const uint64_t prev = i ? k[i - 1] : ~cur;
    if (cur == prev) continue;
    col[pos] = (uint32_t)(cur & mask);
    if (i == 0 || (cur >> lg) != (prev >> lg)) row_off[cur >> lg] = (int64_t)pos;
    ++pos;
  }
}

__global__ void k_set_i64(int64_t* p, int64_t v) { *p = v; }

// Copy of each row's first entry with its original ID, stored densely so that
// the bottom-up sweep reads both coalesced (the reference keeps the same
// "isolated first edge", mpi/graph_constructor.hpp:1387-1557), and bit v of
// `multi`: row v has more than one entry (a bottom-up vertex whose first
// neighbour is unvisited has nothing else to scan otherwise).
__global__ __launch_bounds__(kT) void k_first_nbr(const int64_t* __restrict__ row_off,
                                                 const uint32_t* __restrict__ col,
                                                 const uint32_t* __restrict__ n2o,
                                                 int64_t n_c, uint2* __restrict__ first,
                                                 uint64_t* __restrict__ multi) {
  const int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x;
  bool more = false;
  if (v < n_c) {
    const int64_t beg = row_off[v];
    const uint32_t u = col[beg];
    first[v] = make_uint2(u, n2o[u]);
    more = row_off[v + 1] - beg > 1;
  }
  // 64 consecutive vertices from a multiple of 64: one word
  const uint64_t word = __ballot(more);
  if (lane_id() == 0 && v < n_c) multi[v >> 6] = word;
}

// Bit o: original ID o has a CSR edge.  The host keeps these n bits to answer
// has_edge and to place a run's root; the map itself (32 times as much, the
// earlier form) took 15 of an engine's first 57 ms to copy at SCALE 24.
__global__ __launch_bounds__(kT) void k_edge_bits(const uint32_t* __restrict__ o2n, int64_t n,
                                                 int64_t n_c, uint64_t* __restrict__ bits) {
  const int64_t o = (int64_t)blockIdx.x * kT + threadIdx.x;
  const uint64_t word = __ballot(o < n && (int64_t)o2n[o] < n_c);
  if (lane_id() == 0 && o < n) bits[o >> 6] = word;
}

int bitlen(uint64_t x) { return x ? 64 - __builtin_clzll(x) : 0; }

// The general form: any list, the symmetric (new_src, new_dst) keys radix
// sorted and then deduplicated (80 ms at SCALE 24, where the buckets take 22).
void sort_rows(g500_graph* g, const uint2* edges, int64_t ne, bool symmetric) {
  hipStream_t s = g->stream;
  const int lg = g->log_n;
  const int64_t n = g->n;
  const int64_t nk = symmetric ? ne : 2 * ne;
  IdleReleases released;
  DevBuf<uint64_t> ek, ek_alt;
  ek.alloc_raw((size_t)nk);
  ek_alt.alloc_raw((size_t)nk);
  const uint64_t sentinel = ((uint64_t)(n - 1) << lg) | (uint64_t)(n - 1);
  if (ne > 0) {
    hipLaunchKernelGGL(k_sym_keys, dim3((unsigned)ceil_div(ne, kT)), dim3(kT), 0,
                       s, edges, ne, (int)symmetric, g->orig2new.get(), lg, sentinel,
                       ek.get());
    G500_CHECK_LAUNCH();
  }
  uint64_t* sorted = radix_sort_u64(ek.get(), ek_alt.get(), nk, 0, 2 * lg,
                                    g->radix_ws, s);
  const int64_t ms = g->m_sym;  // sentinels sort to the end
  const int64_t tiles = std::max<int64_t>(1, ceil_div(ms, kDedupTile));
  DevBuf<uint32_t> tcnt;
  DevBuf<uint64_t> toff;
  tcnt.alloc_raw((size_t)tiles);
  toff.alloc_raw((size_t)tiles + 1);
  hipLaunchKernelGGL(k_dedup_count, dim3((unsigned)tiles), dim3(kT), 0, s,
                     sorted, ms, tcnt.get());
  G500_CHECK_LAUNCH();
  exclusive_scan<uint32_t>(tcnt.get(), toff.get(), tiles, g->scan_ws, s);
  uint64_t m_total = 0;
  G500_CHECK_HIP(hipMemcpyAsync(&m_total, toff.get() + tiles, sizeof(uint64_t),
                                hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  g->m = (int64_t)m_total;
  // padding: bottom-up scans read aligned 16-byte groups, which may run a
  // few entries past the last row
  g->col.alloc((size_t)g->m + kColPad, s);
  g->row_off.alloc((size_t)g->n_c + 1, s);
  hipLaunchKernelGGL(k_dedup_write, dim3((unsigned)tiles), dim3(kT), 0, s,
                     sorted, ms, lg, toff.get(), g->col.get(), g->row_off.get());
  G500_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_set_i64, dim3(1), dim3(1), 0, s, g->row_off.get() + g->n_c,
                     g->m);
  G500_CHECK_LAUNCH();
  G500_CHECK_HIP(hipStreamSynchronize(s));  // the scratch is freed on return
  released.now();
}

}  // namespace

void build_csr(g500_graph* g, const uint2* edges, int64_t ne, DegreeMode mode,
               int force_log_n) {
  hipStream_t s = g->stream;
  const bool symmetric = mode != DegreeMode::kBothEnds;
  const int64_t nv = (int64_t)1 << g->id_bits;  // covers every input ID

  DevBuf<unsigned long long> stats;
  stats.alloc(8, s);
  G500_CHECK_HIP(hipMemsetAsync(stats.get(), 0, 8 * sizeof(unsigned long long), s));
  DevBuf<uint32_t> deg;
  deg.alloc_raw((size_t)nv);
  G500_CHECK_HIP(hipMemsetAsync(deg.get(), 0, nv * sizeof(uint32_t), s));
  if (ne > 0)
    count_degrees(edges, ne, mode, nv, deg.get(), stats.get(), s);
  {
    const int64_t blocks = std::min<int64_t>(ceil_div(nv, kT * 8), 1024);
    hipLaunchKernelGGL(k_deg_stats, dim3((unsigned)blocks), dim3(kT), 0, s,
                       deg.get(), nv, stats.get());
    G500_CHECK_LAUNCH();
  }
  unsigned long long h[8];
  G500_CHECK_HIP(hipMemcpyAsync(h, stats.get(), sizeof(h), hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  const uint64_t ormask = h[0];
  const int64_t nonloop = (int64_t)h[1];
  const uint64_t maxdeg = h[2];
  const int lg = force_log_n >= 0 ? force_log_n : bitlen(ormask);  // msb + 1
  const int64_t n = (int64_t)1 << lg;
  g->log_n = lg;
  g->n = n;
  g->n_c = (int64_t)h[3];
  g->max_used = (int64_t)h[4];
  g->max_deg = (int64_t)maxdeg;
  g->m_sym = symmetric ? nonloop : 2 * nonloop;

  // ---- relabel by (degree desc, id asc)
  g->new2orig.alloc_raw((size_t)n);
  g->orig2new.alloc_raw((size_t)n);
  g->deg_new.alloc_raw((size_t)n);
  IdleReleases released;
  {
    DevBuf<uint64_t> vk, vk_alt;
    vk.alloc_raw((size_t)n);
    vk_alt.alloc_raw((size_t)n);
    const int64_t blocks = ceil_div(n, kT);
    hipLaunchKernelGGL(k_vertex_keys, dim3((unsigned)blocks), dim3(kT), 0, s,
                       deg.get(), n, lg, (uint64_t)maxdeg, vk.get());
    G500_CHECK_LAUNCH();
    // the IDs start in ascending order and the sort is stable: the degree bits
    // alone decide
    uint64_t* sorted = radix_sort_u64(vk.get(), vk_alt.get(), n, lg,
                                      lg + std::max(1, bitlen(maxdeg)),
                                      g->radix_ws, s);
    hipLaunchKernelGGL(k_relabel, dim3((unsigned)blocks), dim3(kT), 0, s, sorted,
                       n, lg, (uint64_t)maxdeg, g->new2orig.get(),
                       g->orig2new.get(), g->deg_new.get());
    G500_CHECK_LAUNCH();
    G500_CHECK_HIP(hipStreamSynchronize(s));
    released.now();
  }
  deg.release();
  released.over();

  if (!build_rows(g, edges, ne, symmetric)) sort_rows(g, edges, ne, symmetric);
  {
    g->first.alloc_raw((size_t)std::max<int64_t>(g->n_c, 1));
    g->multi.alloc_raw((size_t)ceil_div(std::max<int64_t>(g->n_c, 1), 64));
    if (g->n_c > 0) {
      hipLaunchKernelGGL(k_first_nbr, dim3((unsigned)ceil_div(g->n_c, kT)), dim3(kT), 0, s,
                         g->row_off.get(), g->col.get(), g->new2orig.get(), g->n_c,
                         g->first.get(), g->multi.get());
      G500_CHECK_LAUNCH();
    }
    G500_CHECK_HIP(hipStreamSynchronize(s));
  }
  g->h_edge_bits.clear();
}

void construct_graph(g500_graph* g, int corebfs) {
  build_csr(g, g->edges.get(), g->nedges,
            g->symmetric_input ? DegreeMode::kSourceNoLoops : DegreeMode::kBothEnds, -1);
  g->corebfs = corebfs;
  g->constructed = true;
}

void ensure_edge_bits(g500_graph* g) {
  if (!g->h_edge_bits.empty() || g->n == 0) return;
  const int64_t words = ceil_div(g->n, 64);
  DevBuf<uint64_t> bits;
  bits.alloc_raw((size_t)words);
  hipLaunchKernelGGL(k_edge_bits, dim3((unsigned)ceil_div(g->n, kT)), dim3(kT), 0, g->stream,
                     g->orig2new.get(), g->n, g->n_c, bits.get());
  G500_CHECK_LAUNCH();
  std::vector<uint64_t> h((size_t)words);
  G500_CHECK_HIP(hipMemcpyAsync(h.data(), bits.get(), words * sizeof(uint64_t),
                                hipMemcpyDeviceToHost, g->stream));
  G500_CHECK_HIP(hipStreamSynchronize(g->stream));
  g->h_edge_bits.swap(h);
}

}  // namespace g500

int64_t g500_graph::device_bytes() const {
  int64_t order = 0;
  {
    std::lock_guard<std::mutex> lock(order_mu);
    if (ordered)
      order = (int64_t)(ordered->keys.n * sizeof(uint64_t) +
                        ordered->chunks.n * sizeof(g500::EdgeChunk));
  }
  return order + (int64_t)(edges.n * sizeof(uint2) + row_off.n * sizeof(int64_t) +
                   col.n * sizeof(uint32_t) + first.n * sizeof(uint2) +
                   multi.n * sizeof(uint64_t) +
                   (deg_new.n + new2orig.n + orig2new.n) * sizeof(uint32_t) +
                   tree_parent.n * sizeof(uint32_t) + has_parent.n * sizeof(uint64_t));
}
