// internal.hpp -- handle types behind the C ABI and the entry points shared
// between the kernel files.
#pragma once

#include <memory>
#include <mutex>
#include <vector>

#include "common.hpp"
#include "primitives.hpp"

namespace g500 {
// The input edges ordered for the validator (order_edges): by the target's
// window of 2^kEdgeWindowBits IDs, then the source's slice of
// 2^kEdgeSliceBits, then the target's part of its window.  64 bits each, from
// the top: window, slice, part (part_bits), the source's place in its slice,
// the target's in its part.  Chunks hold edges of one window and slice.
constexpr int kEdgeWindowBits = 21;
constexpr int kEdgeSliceBits = 16;
constexpr int kEdgePartBits = 11;  // at most
constexpr int64_t kEdgeChunk = 1 << 17;
constexpr int64_t kOrderedEdgesMin = 1 << 20;
constexpr int kOrderedIdBits = 28;
struct EdgeChunk {
  uint64_t first;
  uint32_t count, window, slice, unused;
};
struct OrderedEdges {
  DevBuf<uint64_t> keys;
  DevBuf<EdgeChunk> chunks;
  int64_t n_chunks = 0;
  int part_bits = 0;
};
__host__ __device__ inline uint64_t edge_key(uint32_t s, uint32_t t, int slices_log,
                                             int part_bits) {
  const int low = kEdgeWindowBits - part_bits;
  const uint64_t tile =
      (((uint64_t)(t >> kEdgeWindowBits) << slices_log | s >> kEdgeSliceBits) << part_bits) |
      ((t >> low) & ((1u << part_bits) - 1));
  return tile << (kEdgeSliceBits + low) |
         (uint64_t)(s & ((1u << kEdgeSliceBits) - 1)) << low | (t & ((1u << low) - 1));
}
// the source's place in its slice and the target's in its window
__host__ __device__ inline void edge_places(uint64_t key, int part_bits, uint32_t* s,
                                            uint32_t* t) {
  const int low = kEdgeWindowBits - part_bits;
  *s = (uint32_t)(key >> low) & ((1u << kEdgeSliceBits) - 1);
  *t = (((uint32_t)(key >> (kEdgeSliceBits + low)) & ((1u << part_bits) - 1)) << low) |
       ((uint32_t)key & ((1u << low) - 1));
}
}  // namespace g500

struct g500_graph {
  int device = 0;
  hipStream_t stream = nullptr;

  // input edge list (original IDs), kept resident for validation
  g500::DevBuf<uint2> edges;
  int64_t nedges = 0;
  int64_t capacity = 0;  // edges the buffer holds (appended graphs)
  uint64_t id_or = 0;    // OR of every input ID appended so far
  int id_bits = 0;  // every input ID < 2^id_bits
  bool symmetric_input = false;  // edges already hold both directions

  // construction results (all CSR arrays indexed by relabelled "new" ID)
  bool constructed = false;
  int corebfs = 0;
  int log_n = 0;       // estimated SCALE
  int64_t n = 0;       // 2^log_n
  int64_t n_c = 0;     // vertices with >= 1 CSR edge (new IDs [0, n_c))
  int64_t m = 0;       // deduplicated directed edges
  int64_t m_sym = 0;   // symmetric edges before dedupe
  int64_t max_used = 0;
  int64_t max_deg = 0;
  g500::DevBuf<int64_t> row_off;    // n_c + 1
  g500::DevBuf<uint32_t> col;       // m
  g500::DevBuf<uint2> first;        // n_c: first (highest-degree) neighbour: new ID, original ID
  g500::DevBuf<uint64_t> multi;     // n_c bits: the row has more than one entry
  g500::DevBuf<uint32_t> deg_new;   // n   (symmetric degree incl. duplicates)
  g500::DevBuf<uint32_t> new2orig;  // n
  g500::DevBuf<uint32_t> orig2new;  // n

  // bit v: original ID v has a CSR edge (host copy, lazily made for has_edge,
  // root selection and each run's root)
  std::vector<uint64_t> h_edge_bits;

  // CoreBFS (corebfs != 0): forest parents by original ID (kNoParent = none
  // or reset as unreachable) and the bitmap of vertices that were given a
  // parent while pruning (has_edge counts them, mpi/bfs.hpp:167-170)
  g500::DevBuf<uint32_t> tree_parent;     // n
  g500::DevBuf<uint64_t> has_parent;      // n/64 words
  std::vector<uint32_t> h_tree_parent;    // host copy for the per-root walk
  std::vector<uint64_t> h_has_parent;
  bool core_reset_done = false;           // reset_unreachable applied
  int64_t core_vertices = 0, tree_vertices = 0, removed_parents = 0;
  int64_t hd_root = -1;                   // highest-degree core vertex

  // the input edges once more, in the validator's order (made by the second
  // validation of a graph large enough, given up where the device runs out of
  // memory, else null); all under order_mu: engines of one graph may validate
  // at the same time
  mutable std::mutex order_mu;
  int64_t edge_passes = 0;  // validations that came to the edges before there was an order
  bool order_tried = false;
  std::shared_ptr<const g500::OrderedEdges> ordered;

  g500::ScanWorkspace scan_ws;
  g500::RadixWorkspace radix_ws;

  // engines (plain and batched) created on this graph and not yet destroyed:
  // they hold pointers into it, so the graph may only be freed after them
  int live_engines = 0;

  int64_t device_bytes() const;
  ~g500_graph();
};

namespace g500 {

// gen.hip
void generate_edges(g500_graph* g, int scale, int edgefactor, uint64_t seed1,
                    uint64_t seed2);

// construct.hip
enum class DegreeMode {
  kBothEnds,       // both endpoints of every edge that is no loop
  kSourceNoLoops,  // the source of every edge that is no loop
  kSourceRuns,     // the source of every edge; there are no loops, and the edges of a source
                   // stand together
  kSourceEnd       // the source of every edge, if below nv
};
// CSR of `edges` into g, counted as `mode` says: both directions of each edge
// (kBothEnds) or the one the list holds (force_log_n < 0: estimate the vertex
// space).
void build_csr(g500_graph* g, const uint2* edges, int64_t ne, DegreeMode mode, int force_log_n);
void construct_graph(g500_graph* g, int corebfs);
void ensure_edge_bits(g500_graph* g);
inline bool has_csr_edge(const g500_graph* g, int64_t v) {
  return (g->h_edge_bits[(size_t)(v >> 6)] >> (v & 63)) & 1ull;
}

// csrsort.hip
// deg[v] += edges at v for IDs below nv (every ID counted is, but with kSourceEnd); stats[0] |= the IDs of the edges
// counted, stats[1] += their number
void count_degrees(const uint2* edges, int64_t ne, DegreeMode mode, int64_t nv, uint32_t* deg,
                   unsigned long long* stats, hipStream_t s);
// Buckets in each group of the first of two partition passes, which make at most
// `most` parts each: one to four times as many groups as buckets in each (long
// runs in the second pass), more buckets in each where that would be more groups
// than a pass makes.  1 where one pass makes all the buckets, 0 where two do not.
inline int64_t group_buckets(int64_t buckets, int64_t most) {
  if (buckets <= most) return 1;
  int64_t step = 1;
  while (4 * step * step <= buckets || ceil_div(buckets, step) > most) step *= 2;
  return step <= most ? step : 0;
}

// Sorted rows without repeated entries (g->m, col, row_off) from the edges,
// g's maps and degrees.  False, with nothing kept, where this form cannot sort
// them (an unexpected spread of a long row's targets, or too little memory).
bool build_rows(g500_graph* g, const uint2* edges, int64_t ne, bool symmetric);

// The input edges in the validator's order; null where they are few, their IDs
// too wide or memory is short.
std::shared_ptr<const OrderedEdges> order_edges(const g500_graph* g, hipStream_t s);

// edgeorder.hip: the graph's order, or null
std::shared_ptr<const OrderedEdges> held_order(g500_graph* g);
// The order for a pass over the edges: none for a graph's first pass, made by
// the second.  While one engine makes it, others get none.
std::shared_ptr<const OrderedEdges> order_for_pass(g500_graph* g, hipStream_t s);
// before a graph that may hold an order goes
void forget_ordered_edges(g500_graph* g);

// corebfs.hip
constexpr uint32_t kNoParent = 0xFFFFFFFFu;
// entries allocated past the end of col (aligned 16-byte loads of a row's
// last group may read up to three of them; their values are never used)
constexpr int64_t kColPad = 16;
void corebfs_prune(g500_graph* g);
// reachability reset of the forest after a BFS from hd_root over the core;
// `visited` is that BFS's visited bitmap over core new IDs
void corebfs_reset_unreachable(g500_graph* g, const uint64_t* visited,
                               hipStream_t s);
inline bool has_parent_host(const g500_graph* g, int64_t v) {
  return g->corebfs && (g->h_has_parent[(size_t)(v >> 6)] >> (v & 63)) & 1ull;
}

}  // namespace g500
