// corebfs.hip -- CoreBFS forest pruning on the GPU.
//
// Preprocess (corebfs_adaptor::preprocess, mpi/corebfs_adaptor.hpp:328-357 ->
// prune_trees, external/indexed_bfs/bfs/corebfs/decomposition.hpp:350-572):
// on the deduplicated symmetric CSR, repeatedly take the vertices of live
// degree 1 ("leaves"); each leaf's parent is its one neighbour that was live
// when the round started; leaves then drop to degree 0 and each parent loses
// one degree, dying when it reaches 0.  What stays live is the 2-core; its
// edges are rebuilt into the CSR the BFS runs on (same vertex space).
//
// reset_unreachable (corebfs_adaptor.hpp:228-249, postprocess.hpp:106-154):
// after one BFS over the core from its highest-degree vertex, a forest vertex
// keeps its parent only if following parents leads into that component.
#include <algorithm>

#include "internal.hpp"

namespace g500 {

namespace {

constexpr int kT = 256;

// One atomic per block: atomics on one address take ~12 ns each in turn, so
// one per wave of a launch over 2^22 vertices cost ~0.8 ms (SCALE 22; the
// kernels' own memory time is below 0.02 ms).  All threads of the block call.
__device__ inline void block_add(uint64_t v, unsigned long long* cnt) {
  __shared__ uint64_t part[kT / kWave];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  if (lane_id() == 0) part[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kT / kWave; ++w) v += part[w];
    if (v) atomicAdd(cnt, (unsigned long long)v);
  }
}

__global__ __launch_bounds__(kT) void k_core_init(const int64_t* __restrict__ row_off,
                                                 int64_t n_c, uint32_t* __restrict__ deg,
                                                 uint8_t* __restrict__ alive,
                                                 uint32_t* __restrict__ par) {
  const int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (v >= n_c) return;
  const uint32_t d = (uint32_t)(row_off[v + 1] - row_off[v]);
  deg[v] = d;
  alive[v] = d > 0;
  par[v] = kNoParent;
}

// leaves (live degree 1) appended to `leaves`; cnt[0] = count
__global__ __launch_bounds__(kT) void k_core_leaves(const uint32_t* __restrict__ deg,
                                                   int64_t n_c,
                                                   uint32_t* __restrict__ leaves,
                                                   unsigned long long* cnt) {
  const int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x;
  const bool leaf = v < n_c && deg[v] == 1;
  const uint64_t mask = __ballot(leaf);
  if (!mask) return;
  unsigned long long base = 0;
  if (lane_id() == 0) base = atomicAdd(cnt, (unsigned long long)__popcll(mask));
  base = __shfl(base, 0, kWave);
  if (leaf) leaves[base + __popcll(mask & lanemask_lt())] = (uint32_t)v;
}

// twig of each leaf: first neighbour live at the start of the round
__global__ __launch_bounds__(kT) void k_core_twigs(const uint32_t* __restrict__ leaves,
                                                  int64_t nl,
                                                  const int64_t* __restrict__ row_off,
                                                  const uint32_t* __restrict__ col,
                                                  const uint8_t* __restrict__ alive,
                                                  uint32_t* __restrict__ twig) {
  const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (i >= nl) return;
  const uint32_t s = leaves[i];
  uint32_t t = kNoParent;
  for (int64_t e = row_off[s]; e < row_off[s + 1]; ++e)
    if (alive[col[e]]) {
      t = col[e];
      break;
    }
  twig[i] = t;
}

__global__ __launch_bounds__(kT) void k_core_by_source(const uint32_t* __restrict__ leaves,
                                                      const uint32_t* __restrict__ twig,
                                                      int64_t nl, uint32_t* __restrict__ deg,
                                                      uint8_t* __restrict__ alive,
                                                      uint32_t* __restrict__ par) {
  const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (i >= nl || twig[i] == kNoParent) return;
  const uint32_t s = leaves[i];
  deg[s] = 0;
  par[s] = twig[i];
  alive[s] = 0;
}

// A target loses one degree per twig; targets zeroed as leaves this round
// are skipped (a twig can only reach a zero-degree target when both ends
// were leaves, so the decrements never underflow).
__global__ __launch_bounds__(kT) void k_core_by_target(const uint32_t* __restrict__ twig,
                                                      int64_t nl, uint32_t* __restrict__ deg,
                                                      uint8_t* __restrict__ alive) {
  const int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (i >= nl) return;
  const uint32_t t = twig[i];
  if (t == kNoParent || deg[t] == 0) return;
  if (atomicSub(&deg[t], 1u) == 1u) alive[t] = 0;
}

// Core edges, taken from the CSR's entries in tiles of kFilterTile, one block
// a tile, so that a row's length never decides how long a lane works: with a
// thread a row (the earlier form) the hub rows, 10^5 entries and more at SCALE
// 22, were walked by single lanes, and counting and writing took 42 and 85 ms
// there; the tiles take 0.47 and 1.18 ms, bound by the random reads of the
// targets' flags and original IDs.
// kCount: kept entries per tile; kWrite: the kept entries as (original ID,
// original ID) pairs in entry order from tile_off[tile] on.  tile_row[t] is
// the row that holds entry t * kFilterTile.
constexpr int kFilterItems = 8;
constexpr int kFilterTile = kT * kFilterItems;
enum { kCount = 0, kWrite = 1 };

__global__ __launch_bounds__(kT) void k_core_tile_rows(const int64_t* __restrict__ row_off,
                                                      int64_t n_c,
                                                      uint32_t* __restrict__ tile_row) {
  const int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (v >= n_c) return;
  const int64_t end = row_off[v + 1];
  for (int64_t t = ceil_div(row_off[v], kFilterTile); t * kFilterTile < end; ++t)
    tile_row[t] = (uint32_t)v;
}

template <int kPass>
__global__ __launch_bounds__(kT) void k_core_filter(
    const int64_t* __restrict__ row_off, const uint32_t* __restrict__ col,
    const uint8_t* __restrict__ alive, const uint32_t* __restrict__ n2o,
    const uint32_t* __restrict__ tile_row, int64_t n_c, int64_t m,
    uint32_t* __restrict__ tile_cnt, const uint64_t* __restrict__ tile_off,
    uint2* __restrict__ out) {
  // start of each row of the tile, relative to the tile; every row holds an
  // entry, so at most kFilterTile rows start inside it
  __shared__ int rstart[kFilterTile + 1];
  __shared__ uint32_t kept[kFilterItems][kT / kWave];
  const int t = threadIdx.x, wave = t / kWave;
  const int64_t base = (int64_t)blockIdx.x * kFilterTile;
  const int64_t last = (m - base < kFilterTile ? m : base + kFilterTile) - 1;
  const int64_t r0 = tile_row[blockIdx.x];
  // the row of the tile's last entry: the owner of the next tile's first
  // entry, or the row before it
  int64_t r1 = n_c - 1;
  if (last + 1 < m) {
    r1 = tile_row[blockIdx.x + 1];
    if (row_off[r1] > last) --r1;
  }
  const int rows = (int)(r1 - r0) + 1;
  for (int i = t; i < rows; i += kT) {
    const int64_t d = row_off[r0 + i] - base;
    rstart[i] = d < 0 ? 0 : (int)d;
  }
  __syncthreads();
  uint32_t src[kFilterItems], dst[kFilterItems];
  uint64_t mask[kFilterItems];
#pragma unroll
  for (int k = 0; k < kFilterItems; ++k) {
    const int li = k * kT + t;
    const bool in = base + li <= last;
    const uint32_t u = in ? col[base + li] : 0u;
    int lo = 0, hi = rows;  // last row that starts at or before li
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (rstart[mid] <= li) lo = mid;
      else hi = mid;
    }
    src[k] = (uint32_t)(r0 + lo);
    dst[k] = u;
    mask[k] = __ballot(in && alive[u] && alive[r0 + lo]);
    if (lane_id() == 0) kept[k][wave] = (uint32_t)__popcll(mask[k]);
  }
  __syncthreads();
  uint32_t run = 0;
  if (kPass == kCount) {
    if (t == 0) {
      for (int k = 0; k < kFilterItems; ++k)
        for (int w = 0; w < kT / kWave; ++w) run += kept[k][w];
      tile_cnt[blockIdx.x] = run;
    }
    return;
  }
  uint2* o = out + tile_off[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kFilterItems; ++k) {
    uint32_t before = run;
#pragma unroll
    for (int w = 0; w < kT / kWave; ++w) {
      const uint32_t c = kept[k][w];
      before += w < wave ? c : 0u;
      run += c;
    }
    if ((mask[k] >> lane_id()) & 1ull)
      o[before + __popcll(mask[k] & lanemask_lt())] = make_uint2(n2o[src[k]], n2o[dst[k]]);
  }
}

// forest parents by original ID + the has-parent bitmap
__global__ __launch_bounds__(kT) void k_core_forest(const uint32_t* __restrict__ par,
                                                   const uint32_t* __restrict__ n2o,
                                                   int64_t n_c, uint32_t* __restrict__ tp,
                                                   unsigned long long* __restrict__ hp,
                                                   unsigned long long* cnt) {
  uint64_t c = 0;
  for (int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x; v < n_c;
       v += (int64_t)gridDim.x * kT) {
    if (par[v] == kNoParent) continue;
    const uint32_t o = n2o[v];
    tp[o] = n2o[par[v]];
    atomicOr(&hp[o >> 6], 1ull << (o & 63));
    ++c;
  }
  block_add(c, cnt);
}

// reach[o] = o is a core vertex the hd_root BFS visited
__global__ __launch_bounds__(kT) void k_reach_init(const uint32_t* __restrict__ o2n,
                                                  const uint64_t* __restrict__ vis,
                                                  int64_t n, int64_t n_c,
                                                  uint8_t* __restrict__ reach) {
  const int64_t o = (int64_t)blockIdx.x * kT + threadIdx.x;
  if (o >= n) return;
  const uint32_t v = o2n[o];
  reach[o] = vis && ((int64_t)v < n_c) && ((vis[v >> 6] >> (v & 63)) & 1ull);
}

// one sweep of "reachable parent -> reachable child"; cnt += changes
__global__ __launch_bounds__(kT) void k_reach_sweep(const uint32_t* __restrict__ tp,
                                                   int64_t n, uint8_t* reach,
                                                   unsigned long long* cnt) {
  uint64_t c = 0;
  for (int64_t o = (int64_t)blockIdx.x * kT + threadIdx.x; o < n;
       o += (int64_t)gridDim.x * kT) {
    if (reach[o]) continue;
    const uint32_t p = tp[o];
    if (p != kNoParent && __atomic_load_n(&reach[p], __ATOMIC_RELAXED)) {
      reach[o] = 1;
      ++c;
    }
  }
  block_add(c, cnt);
}

__global__ __launch_bounds__(kT) void k_reach_reset(uint32_t* __restrict__ tp,
                                                   const uint8_t* __restrict__ reach,
                                                   int64_t n, unsigned long long* cnt) {
  uint64_t c = 0;
  for (int64_t o = (int64_t)blockIdx.x * kT + threadIdx.x; o < n;
       o += (int64_t)gridDim.x * kT) {
    if (tp[o] == kNoParent || reach[o]) continue;
    tp[o] = kNoParent;
    ++c;
  }
  block_add(c, cnt);
}

// largest original ID that is a core vertex or has a parent
__global__ __launch_bounds__(kT) void k_max_used(const uint32_t* __restrict__ o2n,
                                                int64_t n, int64_t n_c,
                                                const uint64_t* __restrict__ hp,
                                                unsigned long long* mx) {
  unsigned long long best = 0;
  for (int64_t o = (int64_t)blockIdx.x * kT + threadIdx.x; o < n;
       o += (int64_t)gridDim.x * kT)
    if ((int64_t)o2n[o] < n_c || ((hp[o >> 6] >> (o & 63)) & 1ull)) best = (unsigned long long)o;
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    const unsigned long long x = __shfl_xor(best, s, kWave);
    best = x > best ? x : best;
  }
  if (lane_id() == 0 && best) atomicMax(mx, best);
}

unsigned blocks(int64_t n) { return (unsigned)std::max<int64_t>(1, ceil_div(n, kT)); }
// grid of the kernels that end with an atomic (grid-stride): four blocks a CU
unsigned few_blocks(int64_t n) { return std::min(blocks(n), 1024u); }

uint64_t read_u64(const unsigned long long* d, hipStream_t s) {
  unsigned long long h = 0;
  G500_CHECK_HIP(hipMemcpyAsync(&h, d, sizeof(h), hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  return h;
}

}  // namespace

void corebfs_prune(g500_graph* g) {
  hipStream_t s = g->stream;
  // 1. full deduplicated symmetric CSR of the input
  build_csr(g, g->edges.get(), g->nedges,
            g->symmetric_input ? DegreeMode::kSourceNoLoops : DegreeMode::kBothEnds, -1);
  const int64_t n = g->n, n_c = g->n_c;
  const int log_n = g->log_n;

  // 2. peel leaves
  DevBuf<uint32_t> deg, par, leaves, twig;
  DevBuf<uint8_t> alive;
  DevBuf<unsigned long long> cnt;
  const int64_t nn = std::max<int64_t>(n_c, 1);
  deg.alloc_raw((size_t)nn);
  par.alloc_raw((size_t)nn);
  leaves.alloc_raw((size_t)nn);
  twig.alloc_raw((size_t)nn);
  alive.alloc_raw((size_t)nn);
  cnt.alloc(4, s);
  if (n_c > 0) {
    hipLaunchKernelGGL(k_core_init, dim3(blocks(n_c)), dim3(kT), 0, s, g->row_off.get(),
                       n_c, deg.get(), alive.get(), par.get());
    G500_CHECK_LAUNCH();
  }
  for (int iter = 0; n_c > 0; ++iter) {
    // Kronecker graphs have a small diameter; the reference gives up past 32
    if (iter > 64) fail(G500_ERR_STATE, "CoreBFS pruning did not converge");
    G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long), s));
    hipLaunchKernelGGL(k_core_leaves, dim3(blocks(n_c)), dim3(kT), 0, s, deg.get(), n_c,
                       leaves.get(), cnt.get());
    G500_CHECK_LAUNCH();
    const int64_t nl = (int64_t)read_u64(cnt.get(), s);
    if (nl == 0) break;
    hipLaunchKernelGGL(k_core_twigs, dim3(blocks(nl)), dim3(kT), 0, s, leaves.get(), nl,
                       g->row_off.get(), g->col.get(), alive.get(), twig.get());
    G500_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_core_by_source, dim3(blocks(nl)), dim3(kT), 0, s, leaves.get(),
                       twig.get(), nl, deg.get(), alive.get(), par.get());
    G500_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_core_by_target, dim3(blocks(nl)), dim3(kT), 0, s, twig.get(), nl,
                       deg.get(), alive.get());
    G500_CHECK_LAUNCH();
  }
  deg.release();
  leaves.release();
  twig.release();

  // 3. forest parents by original ID
  g->tree_parent.alloc_raw((size_t)n);
  g->has_parent.alloc_raw((size_t)ceil_div(n, 64));
  G500_CHECK_HIP(hipMemsetAsync(g->tree_parent.get(), 0xFF, n * sizeof(uint32_t), s));
  G500_CHECK_HIP(hipMemsetAsync(g->has_parent.get(), 0, ceil_div(n, 64) * sizeof(uint64_t), s));
  G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long), s));
  if (n_c > 0) {
    hipLaunchKernelGGL(k_core_forest, dim3(few_blocks(n_c)), dim3(kT), 0, s, par.get(),
                       g->new2orig.get(), n_c, g->tree_parent.get(),
                       (unsigned long long*)g->has_parent.get(), cnt.get());
    G500_CHECK_LAUNCH();
  }
  g->tree_vertices = (int64_t)read_u64(cnt.get(), s);
  par.release();

  // 4. core edge list (original IDs) -> core CSR in the same vertex space
  const int64_t tiles = ceil_div(g->m, kFilterTile);
  DevBuf<uint32_t> tile_row, tile_cnt;
  DevBuf<uint64_t> tile_off;
  tile_row.alloc_raw((size_t)tiles);
  tile_cnt.alloc_raw((size_t)tiles);
  tile_off.alloc_raw((size_t)tiles + 1);
  if (tiles > 0) {
    hipLaunchKernelGGL(k_core_tile_rows, dim3(blocks(n_c)), dim3(kT), 0, s, g->row_off.get(),
                       n_c, tile_row.get());
    G500_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_core_filter<kCount>, dim3((unsigned)tiles), dim3(kT), 0, s,
                       g->row_off.get(), g->col.get(), alive.get(), g->new2orig.get(),
                       tile_row.get(), n_c, g->m, tile_cnt.get(), (const uint64_t*)nullptr,
                       (uint2*)nullptr);
    G500_CHECK_LAUNCH();
  }
  exclusive_scan<uint32_t>(tile_cnt.get(), tile_off.get(), tiles, g->scan_ws, s);
  uint64_t m_core = 0;
  G500_CHECK_HIP(hipMemcpyAsync(&m_core, tile_off.get() + tiles, sizeof(uint64_t),
                                hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  DevBuf<uint2> core_edges;
  core_edges.alloc_raw((size_t)std::max<uint64_t>(m_core, 1));
  if (tiles > 0) {
    hipLaunchKernelGGL(k_core_filter<kWrite>, dim3((unsigned)tiles), dim3(kT), 0, s,
                       g->row_off.get(), g->col.get(), alive.get(), g->new2orig.get(),
                       tile_row.get(), n_c, g->m, tile_cnt.get(), tile_off.get(),
                       core_edges.get());
    G500_CHECK_LAUNCH();
  }
  G500_CHECK_HIP(hipStreamSynchronize(s));
  IdleReleases released;
  released.now();
  alive.release();
  tile_row.release();
  tile_cnt.release();
  tile_off.release();
  // drop the full CSR before building the core one
  g->col.release();
  g->first.release();
  g->multi.release();
  g->row_off.release();
  released.over();
  build_csr(g, core_edges.get(), (int64_t)m_core, DegreeMode::kSourceRuns, log_n);
  released.now();  // build_csr waited for its stream
  core_edges.release();
  released.over();
  g->core_vertices = g->n_c;

  // find_max_used_vertex over has_edge = core vertex or forest vertex
  G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long), s));
  hipLaunchKernelGGL(k_max_used, dim3(few_blocks(n)), dim3(kT), 0, s, g->orig2new.get(), n,
                     g->n_c, g->has_parent.get(), cnt.get());
  G500_CHECK_LAUNCH();
  g->max_used = (int64_t)read_u64(cnt.get(), s);

  g->h_has_parent.resize((size_t)ceil_div(n, 64));
  copy_to_host(g->h_has_parent.data(), g->has_parent.get(), (int64_t)g->h_has_parent.size(), s);
  g->corebfs = 1;
  g->core_reset_done = false;
  g->hd_root = g->n_c > 0 ? -2 : -1;  // resolved after the new2orig copy below
  if (g->n_c > 0) {
    uint32_t r = 0;
    copy_to_host(&r, g->new2orig.get(), 1, s);
    g->hd_root = r;  // new ID 0: highest core degree, ties by lowest original ID
  }
  g->constructed = true;
}

void corebfs_reset_unreachable(g500_graph* g, const uint64_t* visited, hipStream_t s) {
  const int64_t n = g->n;
  DevBuf<uint8_t> reach;
  DevBuf<unsigned long long> cnt;
  reach.alloc_raw((size_t)n);
  cnt.alloc(1, s);
  hipLaunchKernelGGL(k_reach_init, dim3(blocks(n)), dim3(kT), 0, s, g->orig2new.get(),
                     visited, n, g->n_c, reach.get());
  G500_CHECK_LAUNCH();
  for (int iter = 0;; ++iter) {
    if (iter > (1 << 16)) fail(G500_ERR_STATE, "forest reachability did not converge");
    G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long), s));
    hipLaunchKernelGGL(k_reach_sweep, dim3(few_blocks(n)), dim3(kT), 0, s,
                       g->tree_parent.get(), n, reach.get(), cnt.get());
    G500_CHECK_LAUNCH();
    if (read_u64(cnt.get(), s) == 0) break;
  }
  G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long), s));
  hipLaunchKernelGGL(k_reach_reset, dim3(few_blocks(n)), dim3(kT), 0, s, g->tree_parent.get(),
                     reach.get(), n, cnt.get());
  G500_CHECK_LAUNCH();
  g->removed_parents = (int64_t)read_u64(cnt.get(), s);
  g->h_tree_parent.resize((size_t)n);
  copy_to_host(g->h_tree_parent.data(), g->tree_parent.get(), n, s);
  g->core_reset_done = true;
}

}  // namespace g500
