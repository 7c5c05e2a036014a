// validate.hip -- the Graph500 result validator on the GPU.
//
// Same checks, same order and the same early exits as
// BfsValidation::validate (mpi/validate.hpp:608-976): parent range, root is
// its own parent, no other self-parent, depth map (or, with CoreBFS, the
// depth rebuild of validate.hpp:1040-1141), then one pass over every input
// edge (tree/non-tree mix, depth gap, parent-edge depth, traversed-edge
// count) and finally "every reached vertex has an edge to its parent".
// One difference: the reference stops its edge pass at the first 8 Mi-edge
// chunk that has errors; this pass always covers all edges, so error totals
// (never the verdict or the count of a valid tree) can differ.
//
// The edge pass looks two vertices up per edge.  As random 8-byte reads of
// pred that ran at 65 G reads/s, 8.2 ms for the 2^28 edges of SCALE 24.  The
// ordered edges (order_edges) keep the lookups near: a block holds one byte
// (depth, low bits of the parent) for each source of its slice in LDS and
// walks the targets' window part by part, so that the lanes of a step share a
// few lines, the window staying in the L2; pred itself is read only where those
// bits say an edge may be a tree edge.  1.2 ms at SCALE 24, bound by the
// L2 requests still left (with parts of 16 KB instead of 1 KB, which leaves
// nearly one per edge: 1.9).  The second edge pass over a graph orders the
// edges, the first is direct: ordering takes 6 ms at SCALE 24, so a program that
// validates one tree of a graph would lose by it.  The first, second and third
// call take 8.0, 7.6 and 1.4 ms there (8.4 each when all are direct), 1.5, 2.0 and
// 0.45 at SCALE 22 (1.6 each).  From 2^28 edges on ordering at once would cost the
// first call no more than the direct pass (33 against 38 ms at SCALE 26) while its 16
// bytes an edge are at hand; where the driver has to clear them first it took 124
// and 184 ms, which one tree does not earn back.
// Graphs of fewer edges, or trees deeper than a byte's four bits hold, take
// the direct form.
#include "engine.hpp"

namespace g500 {

namespace {

constexpr int kT = 256;
enum {
  kTE = G500_VERR_NUM,
  kChanged,
  kDeep,  // vertices deeper than a code holds
  kRoot,  // the root's entry
  kCounters
};
// code of a vertex: depth << 4 | low bits of its parent
constexpr uint32_t kCodeNone = 15;  // the depth of a vertex without one

__host__ __device__ inline int64_t pe_parent(int64_t e) {
  return (int64_t)((uint64_t)e << 16) >> 16;
}
__host__ __device__ inline uint32_t pe_depth(int64_t e) {
  return (uint32_t)(((uint64_t)e >> 48) & 0xFFFF);
}

// Adds v to cnt[k] with one atomic per block (on one address they take ~12 ns
// each in turn).  All threads of a block of kThreads call.
template <int kThreads>
__device__ inline void block_count(unsigned long long* cnt, int k, uint64_t v) {
  __shared__ uint64_t part[kThreads / kWave];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
  if (lane_id() == 0) part[threadIdx.x / kWave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / kWave; ++w) v += part[w];
    if (v) atomicAdd(&cnt[k], (unsigned long long)v);
  }
  __syncthreads();
}

// One pass over the vertices: parents out of range, vertices that are their
// own parent, the depth map (validate.hpp:1145-1255; not with CoreBFS, whose
// depths are rebuilt first), the root's entry, and the codes.  Counts mean
// something only up to the first kind that is not zero, in that order: a
// parent out of range is not looked up.
__global__ __launch_bounds__(kT) void k_v_tree(const int64_t* __restrict__ pred, int64_t nlocal,
                                              int64_t nglobal, int64_t root, int check_depth,
                                              uint8_t* __restrict__ code,
                                              unsigned long long* cnt) {
  uint64_t range = 0, self = 0, bad = 0, deep = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < nlocal;
       i += (int64_t)gridDim.x * kT) {
    const int64_t e = pred[i];
    const int64_t p = pe_parent(e);
    const uint32_t d = pe_depth(e);
    const bool out = p < -1 || p >= nglobal;
    if (out) ++range;
    if (i != root && p != -1 && p == i) ++self;
    if (d >= kCodeNone && d != 0xFFFF) ++deep;
    if (code) code[i] = (uint8_t)((d < kCodeNone ? d : kCodeNone) << 4 | ((uint32_t)p & 15u));
    if (!check_depth) continue;
    if (p == -1 && d != 0xFFFF) ++bad;
    else if (p != -1 && d == 0xFFFF) ++bad;
    if (i == root || p == -1 || out) continue;
    const uint32_t dp = pe_depth(pred[p]);
    if (dp == 0xFFFF) ++bad;
    if (d != dp + 1) ++bad;
  }
  block_count<kT>(cnt, G500_VERR_RANGE, range);
  block_count<kT>(cnt, G500_VERR_SELF_PARENT, self);
  block_count<kT>(cnt, G500_VERR_DEPTH_MAP, bad);
  block_count<kT>(cnt, kDeep, deep);
  if (blockIdx.x == 0 && threadIdx.x == 0 && root >= 0 && root < nlocal)
    cnt[kRoot] = (unsigned long long)pred[root];
}

// validate.hpp:1040-1141: depth[v] = depth[parent]+1 where unknown; one sweep.
__global__ __launch_bounds__(kT) void k_v_depth_build(int64_t* __restrict__ pred,
                                                     int64_t nlocal, int64_t root,
                                                     unsigned long long* cnt) {
  uint64_t changed = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < nlocal;
       i += (int64_t)gridDim.x * kT) {
    if (i == root) continue;
    const int64_t e = pred[i];
    const int64_t p = pe_parent(e);
    if (p < 0 || pe_depth(e) != 0xFFFF) continue;
    const uint32_t dp = pe_depth(__atomic_load_n(&pred[p], __ATOMIC_RELAXED));
    if (dp == 0xFFFF) continue;
    pred[i] = (int64_t)(((uint64_t)e & 0xFFFFFFFFFFFFull) | ((uint64_t)((dp + 1) & 0xFFFF) << 48));
    ++changed;
  }
  block_count<kT>(cnt, kChanged, changed);
}

__global__ void k_v_set_root_depth0(int64_t* pred, int64_t root) {
  pred[root] = (int64_t)((uint64_t)pred[root] & 0xFFFFFFFFFFFFull);
}

__device__ inline int64_t pred_at(const int64_t* pred, int64_t nlocal, int64_t v) {
  return (v >= 0 && v < nlocal) ? pred[v] : (int64_t)-1;
}

// validate.hpp:834-916
__global__ __launch_bounds__(kT) void k_v_edges(const uint2* __restrict__ edges,
                                               int64_t ne,
                                               const int64_t* __restrict__ pred,
                                               int64_t nlocal,
                                               uint8_t* __restrict__ pred_valid,
                                               unsigned long long* cnt) {
  uint64_t te = 0, tree = 0, gap = 0, pdep = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < ne;
       i += (int64_t)gridDim.x * kT) {
    const uint2 x = edges[i];
    const int64_t s = x.x, t = x.y;
    const int64_t ps = pred_at(pred, nlocal, s), pt = pred_at(pred, nlocal, t);
    const int ds = (int)pe_depth(ps), dt = (int)pe_depth(pt);
    if (ds != 0xFFFF && dt == 0xFFFF) ++tree;
    else if (ds == 0xFFFF && dt != 0xFFFF) ++tree;
    else if (ds - dt < -1 || ds - dt > 1) ++gap;
    else if (ds != 0xFFFF) ++te;
    const bool s_to_t = pe_parent(ps) == t, t_to_s = pe_parent(pt) == s;
    if ((s_to_t || t_to_s) && s != t &&
        ((s_to_t && dt + 1 != ds) || (t_to_s && ds + 1 != dt)))
      pdep += (uint64_t)s_to_t + (uint64_t)t_to_s;
    if (s_to_t) pred_valid[s] = 1;
    if (t_to_s) pred_valid[t] = 1;
  }
  block_count<kT>(cnt, kTE, te);
  block_count<kT>(cnt, G500_VERR_EDGE_TREE, tree);
  block_count<kT>(cnt, G500_VERR_EDGE_GAP, gap);
  block_count<kT>(cnt, G500_VERR_PRED_DEPTH, pdep);
}

// Orders a wave's LDS accesses (its lanes read what other lanes wrote).
__device__ inline void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The same over the ordered edges, one block a chunk.  checked: the depth map
// holds (every vertex but the root is one deeper than its parent), so only an
// edge to a vertex one level up can be a tree edge.  Edges that may be one, a
// few of every 64, wait in LDS until a wave has 64 of them: looked up at once
// they would put dependent reads into nearly every step.
constexpr int kTileT = 1024;
constexpr int kTileIlp = 8;
constexpr uint32_t kEdgeIndex = 0x7FFFFFFFu;  // the top bit: the target is the child

__global__ __launch_bounds__(kTileT) void k_v_tiles(
    const uint64_t* __restrict__ ordered, const EdgeChunk* __restrict__ chunks, int part_bits,
    const uint8_t* __restrict__ code, const int64_t* __restrict__ pred, int64_t nlocal,
    int checked, uint8_t* __restrict__ pred_valid, unsigned long long* cnt) {
  __shared__ uint4 slice4[(1 << kEdgeSliceBits) / 16];
  __shared__ uint32_t waiting[kTileT / kWave][2 * kWave];
  const uint8_t* slice = reinterpret_cast<const uint8_t*>(slice4);
  const EdgeChunk c = chunks[blockIdx.x];
  const int64_t s0 = (int64_t)c.slice << kEdgeSliceBits;
  const int64_t t0 = (int64_t)c.window << kEdgeWindowBits;
  const uint4* from = reinterpret_cast<const uint4*>(code + s0);
  for (int i = threadIdx.x; i < (1 << kEdgeSliceBits) / 16; i += kTileT) slice4[i] = from[i];
  __syncthreads();
  const uint8_t* window = code + t0;
  const uint64_t* e = ordered + c.first;
  const int lane = lane_id();
  uint32_t* wait = waiting[threadIdx.x / kWave];
  uint32_t waits = 0;  // the wave's edges that may be tree edges
  uint32_t te = 0, tree = 0, gap = 0, pdep = 0;
  // looks at pred for the last n of them
  auto settle = [&](uint32_t n) {
    waits -= n;
    if ((uint32_t)lane < n) {
      const uint32_t w = wait[waits + lane];
      uint32_t sp, tp;
      edge_places(e[w & kEdgeIndex], part_bits, &sp, &tp);
      const int64_t s = s0 + sp, t = t0 + tp;
      if (checked) {
        const int64_t child = w & ~kEdgeIndex ? t : s;
        if (pe_parent(pred_at(pred, nlocal, child)) == s + t - child) pred_valid[child] = 1;
        return;
      }
      const int64_t ps = pred_at(pred, nlocal, s), pt = pred_at(pred, nlocal, t);
      const bool st = pe_parent(ps) == t, ts = pe_parent(pt) == s;
      const int ds = (int)pe_depth(ps), dt = (int)pe_depth(pt);
      if ((st || ts) && s != t && ((st && dt + 1 != ds) || (ts && ds + 1 != dt)))
        pdep += (uint32_t)st + (uint32_t)ts;
      if (st) pred_valid[s] = 1;
      if (ts) pred_valid[t] = 1;
    }
  };
  for (uint32_t i0 = threadIdx.x & ~(kWave - 1u); i0 < c.count; i0 += kTileT * kTileIlp) {
    uint32_t si[kTileIlp], ti[kTileIlp], cs[kTileIlp], ct[kTileIlp];
#pragma unroll
    for (int k = 0; k < kTileIlp; ++k) {
      const uint32_t i = i0 + k * kTileT + lane;
      const uint64_t x = i < c.count ? __builtin_nontemporal_load(e + i) : 0;
      edge_places(x, part_bits, &si[k], &ti[k]);
    }
#pragma unroll
    for (int k = 0; k < kTileIlp; ++k) {
      ct[k] = window[ti[k]];
      cs[k] = slice[si[k]];
    }
#pragma unroll
    for (int k = 0; k < kTileIlp; ++k) {
      const uint32_t i = i0 + k * kTileT + lane;
      bool may = i < c.count, down = false;
      if (may) {
        const uint32_t ds = cs[k] >> 4, dt = ct[k] >> 4;
        if ((ds == kCodeNone) != (dt == kCodeNone)) ++tree;
        else if (ds > dt + 1 || dt > ds + 1) ++gap;
        else if (ds != kCodeNone) ++te;
        const bool st = (cs[k] & 15u) == (ti[k] & 15u), ts = (ct[k] & 15u) == (si[k] & 15u);
        down = ts && (!checked || dt == ds + 1);
        may = down || (st && (!checked || ds == dt + 1));
      }
      const uint64_t mask = __ballot(may);
      if (may) wait[waits + (uint32_t)__popcll(mask & lanemask_lt())] =
                 i | (down ? ~kEdgeIndex : 0u);
      waits += (uint32_t)__popcll(mask);
      if (waits >= kWave) {
        wave_order();
        settle(kWave);
        wave_order();
      }
    }
  }
  wave_order();
  settle(waits);
  block_count<kTileT>(cnt, kTE, te);
  block_count<kTileT>(cnt, G500_VERR_EDGE_TREE, tree);
  block_count<kTileT>(cnt, G500_VERR_EDGE_GAP, gap);
  block_count<kTileT>(cnt, G500_VERR_PRED_DEPTH, pdep);
}

__global__ __launch_bounds__(kT) void k_v_parent_edges(const int64_t* __restrict__ pred,
                                                      int64_t nlocal, int64_t root,
                                                      const uint8_t* __restrict__ pv,
                                                      unsigned long long* cnt) {
  uint64_t bad = 0;
  for (int64_t i = (int64_t)blockIdx.x * kT + threadIdx.x; i < nlocal;
       i += (int64_t)gridDim.x * kT) {
    if (pe_parent(pred[i]) == -1) continue;
    if (!pv[i] && i != root) ++bad;
  }
  block_count<kT>(cnt, G500_VERR_NO_PARENT_EDGE, bad);
}

unsigned grid(int64_t n) {
  const int64_t b = ceil_div(n, kT);
  return (unsigned)(b < 1 ? 1 : (b > 2048 ? 2048 : b));
}

// The engine's codes; IDs past the last vertex (loops may name them) have no
// depth.  False where there is no room.
bool code_room(g500_bfs* b) {
  if (b->vcode.get()) return true;
  const int64_t ids = ceil_div((int64_t)1 << b->g->id_bits, 1 << kEdgeWindowBits)
                      << kEdgeWindowBits;
  if (!b->vcode.try_raw((size_t)ids)) return false;
  G500_CHECK_HIP(hipMemsetAsync(b->vcode.get(), 0xFF, (size_t)ids, b->stream));
  return true;
}

}  // namespace

void bfs_validate(g500_bfs* b, int64_t root, const int64_t* host_pred,
                  int64_t* te, int64_t* errs, int* ok) {
  g500_graph* g = b->g;
  hipStream_t s = b->stream;
  const int64_t nlocal = g->n;
  const int64_t nglobal = g->max_used + 1;
  if (host_pred) {
    G500_CHECK_HIP(hipMemcpyAsync(b->pred.get(), host_pred, nlocal * sizeof(int64_t),
                                  hipMemcpyHostToDevice, s));
    b->pred_fill_needed = true;  // the next BFS run restores the -1 entries
  } else if (!b->have_result) {
    fail(G500_ERR_STATE, "validate: no BFS result on the device");
  }
  if (!b->vcount.get()) b->vcount.alloc(kCounters, s);
  if (!b->pred_valid.get()) b->pred_valid.alloc((size_t)nlocal, s);
  unsigned long long* cnt = b->vcount.get();
  unsigned long long h[kCounters];
  auto fetch = [&]() {
    G500_CHECK_HIP(hipMemcpyAsync(h, cnt, sizeof(h), hipMemcpyDeviceToHost, s));
    G500_CHECK_HIP(hipStreamSynchronize(s));
  };
  for (int i = 0; i < G500_VERR_NUM; ++i) errs[i] = 0;
  *te = 0;
  *ok = 0;
  G500_CHECK_HIP(hipMemsetAsync(cnt, 0, sizeof(h), s));

  std::shared_ptr<const OrderedEdges> order = held_order(g);
  const bool coded = order && !g->corebfs && code_room(b);  // the first pass makes the codes

  // stage 1-4: ranges, root, self parents, depth map
  hipLaunchKernelGGL(k_v_tree, dim3(grid(nlocal)), dim3(kT), 0, s, b->pred.get(), nlocal,
                     nglobal, root, g->corebfs ? 0 : 1, coded ? b->vcode.get() : nullptr, cnt);
  G500_CHECK_LAUNCH();
  fetch();
  if (h[G500_VERR_RANGE]) {
    errs[G500_VERR_RANGE] = (int64_t)h[G500_VERR_RANGE];
    return;
  }
  if (root < 0 || root >= nlocal) {
    errs[G500_VERR_ROOT] = 1;
    return;
  }
  const int64_t proot = (int64_t)h[kRoot];
  if (pe_parent(proot) != root) {
    errs[G500_VERR_ROOT] = 1;
    return;
  }
  if (h[G500_VERR_SELF_PARENT]) {
    errs[G500_VERR_SELF_PARENT] = (int64_t)h[G500_VERR_SELF_PARENT];
    return;
  }
  if (g->corebfs) {
    hipLaunchKernelGGL(k_v_set_root_depth0, dim3(1), dim3(1), 0, s, b->pred.get(), root);
    G500_CHECK_LAUNCH();
    for (int iter = 0; iter < 0x10000; ++iter) {
      G500_CHECK_HIP(hipMemsetAsync(cnt + kChanged, 0, sizeof(unsigned long long), s));
      hipLaunchKernelGGL(k_v_depth_build, dim3(grid(nlocal)), dim3(kT), 0, s,
                         b->pred.get(), nlocal, root, cnt);
      G500_CHECK_LAUNCH();
      fetch();
      if (!h[kChanged]) break;
    }
  } else if (pe_depth(proot) != 0 || h[G500_VERR_DEPTH_MAP]) {
    errs[G500_VERR_ROOT] = pe_depth(proot) != 0;
    errs[G500_VERR_DEPTH_MAP] = (int64_t)h[G500_VERR_DEPTH_MAP];
    return;
  }

  // stage 5: every input edge, then parent edges
  if (!order && h[kDeep] == 0) order = order_for_pass(g, s);
  const bool tiles = order && (coded || code_room(b));
  if (tiles && !coded) {
    hipLaunchKernelGGL(k_v_tree, dim3(grid(nlocal)), dim3(kT), 0, s, b->pred.get(), nlocal,
                       nglobal, root, 0, b->vcode.get(), cnt);
    G500_CHECK_LAUNCH();
    fetch();
  }
  G500_CHECK_HIP(hipMemsetAsync(b->pred_valid.get(), 0, nlocal, s));
  if (tiles && h[kDeep] == 0) {
    hipLaunchKernelGGL(k_v_tiles, dim3((unsigned)order->n_chunks), dim3(kTileT), 0, s,
                       order->keys.get(), order->chunks.get(), order->part_bits, b->vcode.get(), b->pred.get(), nlocal,
                       g->corebfs ? 0 : 1, b->pred_valid.get(), cnt);
    G500_CHECK_LAUNCH();
  } else if (g->nedges > 0) {
    hipLaunchKernelGGL(k_v_edges, dim3(grid(g->nedges)), dim3(kT), 0, s,
                       g->edges.get(), g->nedges, b->pred.get(), nlocal,
                       b->pred_valid.get(), cnt);
    G500_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(k_v_parent_edges, dim3(grid(nlocal)), dim3(kT), 0, s,
                     b->pred.get(), nlocal, root, b->pred_valid.get(), cnt);
  G500_CHECK_LAUNCH();
  fetch();
  for (int i = 0; i < G500_VERR_NUM; ++i) errs[i] = (int64_t)h[i];
  *te = (int64_t)h[kTE];
  int good = 1;
  for (int i = 0; i < G500_VERR_NUM; ++i)
    if (errs[i]) good = 0;
  *ok = good;
}

}  // namespace g500
