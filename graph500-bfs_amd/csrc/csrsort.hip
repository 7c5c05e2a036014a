// csrsort.hip -- vertex degrees and sorted, deduplicated rows from an edge
// list, both by partitioning into LDS-sized pieces.
//
// Degrees.  A vertex's degree is a count of endpoint IDs.  Global atomics ran
// at 24 G/s (and one at a time on a hub: ~12 ns each), 22.8 ms for the 2^29
// endpoints of SCALE 24.  Here the endpoints are first partitioned by their
// upper bits into ranges of 2^16 IDs, only the low 16 bits being stored, and
// each range is then counted in LDS: 2.0 ms at SCALE 24 (0.43 ranges' sizes,
// 0.98 partition, 0.56 counting), near the 1.1 ms its bytes take.  A few ranges
// (up to 2^20 IDs) are counted straight from the edges, each block taking one
// range of one chunk (3 M edges over 2^19 IDs: 0.08 ms, 0.85 with atomics).
//
// Rows.  The keys (new source, new target) of all directed edges, duplicates
// included, are sorted by splitting them into buckets of about kBucketMean
// keys that fit LDS and sorting each bucket there.  Bucket bounds need no
// sampling: the degrees give every row's place in the sorted order, and within
// a row too long for one bucket the targets are taken to be spread as all
// endpoints are, so a bound in the middle of it is the target below which that
// share of all endpoints lies.  Where that holds poorly (long rows without
// repeated edges, say) buckets come out larger than LDS: up to kBigCap keys
// one block sorts them range by range, beyond that (or with a group of buckets
// past its room) the caller sorts with the radix sort.  At SCALE 24 the
// 2^29 keys take 22 ms (radix sort and deduplication: 80): 10.5 for the first
// pass, bound by its random reads of the new IDs, 1.3 + 2.7 for counting and
// moving in the second, 6.8 for the LDS sort, bound by its ballots, 0.9 for the
// last copy.
#include <algorithm>

#include "internal.hpp"

namespace g500 {

namespace {

int bit_length(uint64_t x) { return x ? 64 - __builtin_clzll(x) : 0; }

// ------------------------------------------------------------------ degrees
constexpr int kRangeBits = 16;
constexpr int kRange = 1 << kRangeBits;
constexpr int kDegT = 1024;
// endpoints a thread counts between two barriers: kDegT * 16 increments keep
// a 16-bit counter that held at most 2^15 - 1 below 2^16 (deg_add)
constexpr int kDegBatch = 8;  // edges (two endpoints each)
constexpr int kDegChunk = 1 << 20;  // partitioned endpoints per counting block
constexpr int kMaxDirectRanges = 16;
constexpr int kMaxRanges = 4096;

enum { kBoth = 0, kSource = 1, kSourceAll = 2 };

// Adds one to the 16-bit LDS counter of `id` (relative to the range).  The
// increment that reaches 2^15 moves that amount to global memory, so a
// counter stays below 2^16 as long as fewer than 2^15 increments fall between
// two barriers of the block.
__device__ inline void deg_add(uint32_t* cnt, uint32_t id, uint32_t* __restrict__ deg) {
  const int sh = (id & 1u) * 16;
  const uint32_t old = atomicAdd(&cnt[id >> 1], 1u << sh);
  if (((old >> sh) & 0xFFFFu) == 0x7FFFu) {
    atomicSub(&cnt[id >> 1], 0x8000u << sh);
    atomicAdd(&deg[id], 0x8000u);
  }
}

__device__ inline void deg_flush(const uint32_t* cnt, int ids, uint32_t* __restrict__ deg) {
  for (int i = threadIdx.x; i < ids; i += kDegT) {
    const uint32_t c = (cnt[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu;
    if (c) atomicAdd(&deg[i], c);
  }
}

// stats[0] |= endpoint IDs of non-loop edges, stats[1] += non-loop edges; two
// atomics per block
template <int kThreads>
__device__ inline void edge_stats(uint64_t orv, uint64_t cnt, unsigned long long* stats) {
  __shared__ uint64_t part[2][kThreads / kWave];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    orv |= __shfl_xor(orv, o, kWave);
    cnt += __shfl_xor(cnt, o, kWave);
  }
  if (lane_id() == 0) {
    part[0][threadIdx.x / kWave] = orv;
    part[1][threadIdx.x / kWave] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / kWave; ++w) {
      orv |= part[0][w];
      cnt += part[1][w];
    }
    if (orv) atomicOr(&stats[0], (unsigned long long)orv);
    if (cnt) atomicAdd(&stats[1], (unsigned long long)cnt);
  }
}

// Whether an edge counts, and toward which endpoints.  Only loops may name IDs
// from nv on.
template <int kMode>
__device__ inline bool edge_counts(const uint2& x, int64_t nv) {
  return kMode == kSourceAll ? (int64_t)x.x < nv : x.x != x.y;
}

// Block (chunk, range): counts the endpoints of a chunk of edges that lie in
// one range of 2^16 IDs.
template <int kMode>
__global__ __launch_bounds__(kDegT) void k_deg_direct(const uint2* __restrict__ e, int64_t ne,
                                                     int64_t chunk, int64_t nv,
                                                     uint32_t* __restrict__ deg,
                                                     unsigned long long* stats) {
  __shared__ uint32_t cnt[kRange / 2];
  const uint32_t range = blockIdx.y;
  const int64_t v0 = (int64_t)range << kRangeBits;
  const int ids = (int)(nv - v0 < kRange ? nv - v0 : kRange);
  for (int i = threadIdx.x; i < (ids + 1) / 2; i += kDegT) cnt[i] = 0;
  __syncthreads();
  const int64_t beg = (int64_t)blockIdx.x * chunk;
  const int64_t end = beg + chunk < ne ? beg + chunk : ne;
  uint64_t orv = 0, num = 0;
  for (int64_t i0 = beg; i0 < end; i0 += (int64_t)kDegT * kDegBatch) {
    uint2 x[kDegBatch];
    bool ok[kDegBatch];
#pragma unroll
    for (int k = 0; k < kDegBatch; ++k) {
      const int64_t i = i0 + k * kDegT + threadIdx.x;
      x[k] = i < end ? e[i] : make_uint2(0, 0);
      ok[k] = i < end && edge_counts<kMode>(x[k], nv);
    }
#pragma unroll
    for (int k = 0; k < kDegBatch; ++k) {
      if (!ok[k]) continue;
      if (x[k].x >> kRangeBits == range) deg_add(cnt, x[k].x & (kRange - 1), deg + v0);
      if (kMode == kBoth && x[k].y >> kRangeBits == range)
        deg_add(cnt, x[k].y & (kRange - 1), deg + v0);
      orv |= (uint64_t)(x[k].x | x[k].y);
      ++num;
    }
    __syncthreads();
  }
  deg_flush(cnt, ids, deg + v0);
  if (range == 0) edge_stats<kDegT>(orv, num, stats);
}

// Endpoints per range.
template <int kMode>
__global__ __launch_bounds__(kDegT) void k_deg_ranges(const uint2* __restrict__ e, int64_t ne,
                                                     int64_t nv, int ranges,
                                                     unsigned long long* __restrict__ total,
                                                     unsigned long long* stats) {
  __shared__ uint32_t hist[kMaxRanges];
  for (int i = threadIdx.x; i < ranges; i += kDegT) hist[i] = 0;
  __syncthreads();
  uint64_t orv = 0, num = 0;
  for (int64_t i = (int64_t)blockIdx.x * kDegT + threadIdx.x; i < ne;
       i += (int64_t)gridDim.x * kDegT) {
    const uint2 x = e[i];
    if (!edge_counts<kMode>(x, nv)) continue;
    atomicAdd(&hist[x.x >> kRangeBits], 1u);
    if (kMode == kBoth) atomicAdd(&hist[x.y >> kRangeBits], 1u);
    orv |= (uint64_t)(x.x | x.y);
    ++num;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < ranges; i += kDegT)
    if (hist[i]) atomicAdd(&total[i], (unsigned long long)hist[i]);
  edge_stats<kDegT>(orv, num, stats);
}

// Exclusive scan of one value a thread over a block of kThreads.
template <int kThreads>
__device__ inline uint32_t block_scan(uint32_t v, uint32_t* wsum, uint32_t* total) {
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, kWave);
    if (lane >= o) x += y;
  }
  if (lane == kWave - 1) wsum[wave] = x;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kThreads / kWave; ++w) {
    const uint32_t s = wsum[w];
    off += w < wave ? s : 0u;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return x - v + off;
}

// Partitions the endpoints by range: a tile's endpoints are ordered by range
// in LDS and written as one run per range, at a place reserved with one
// atomic per range and tile.  cursor[r] starts at the range's first slot.
template <int kMode, int kEdges, int kNumRanges>
__global__ __launch_bounds__(kDegT) void k_deg_scatter(const uint2* __restrict__ e, int64_t ne,
                                                      int64_t nv, int ranges,
                                                      unsigned long long* __restrict__ cursor,
                                                      uint16_t* __restrict__ out) {
  constexpr int kPer = kMode == kBoth ? 2 : 1;
  constexpr int kIt = kEdges / kDegT;
  __shared__ uint16_t stage[kEdges * kPer];
  __shared__ uint16_t owner[kEdges * kPer];
  __shared__ uint32_t hist[kNumRanges];
  __shared__ unsigned long long place[kNumRanges];
  __shared__ uint32_t wsum[kDegT / kWave];
  const int t = threadIdx.x;
  for (int i = t; i < ranges; i += kDegT) hist[i] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kEdges;
  uint32_t id[kIt * kPer], rank[kIt * kPer];
  uint32_t use = 0;
#pragma unroll
  for (int k = 0; k < kIt; ++k) {
    const int64_t i = base + k * kDegT + t;
    const uint2 x = i < ne ? e[i] : make_uint2(0, 0);
    const bool ok = i < ne && edge_counts<kMode>(x, nv);
    use |= (uint32_t)ok << k;
    id[k * kPer] = x.x;
    if (kPer == 2) id[k * kPer + 1] = x.y;
  }
#pragma unroll
  for (int k = 0; k < kIt; ++k)
    if ((use >> k) & 1u) {
#pragma unroll
      for (int p = 0; p < kPer; ++p)
        rank[k * kPer + p] = atomicAdd(&hist[id[k * kPer + p] >> kRangeBits], 1u);
    }
  __syncthreads();
  // thread t owns the kOwn ranges from t * kOwn on
  constexpr int kOwn = (kNumRanges + kDegT - 1) / kDegT;
  uint32_t h[kOwn], sum = 0, total;
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const int r = t * kOwn + j;
    h[j] = r < ranges ? hist[r] : 0u;
    sum += h[j];
  }
  uint32_t start = block_scan<kDegT>(sum, wsum, &total);
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const int r = t * kOwn + j;
    if (r < ranges) {
      hist[r] = start;
      if (h[j]) place[r] = atomicAdd(&cursor[r], (unsigned long long)h[j]) - start;
      start += h[j];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kIt; ++k)
    if ((use >> k) & 1u) {
#pragma unroll
      for (int p = 0; p < kPer; ++p) {
        const uint32_t v = id[k * kPer + p], r = v >> kRangeBits;
        const uint32_t pos = hist[r] + rank[k * kPer + p];
        stage[pos] = (uint16_t)v;
        owner[pos] = (uint16_t)r;
      }
    }
  __syncthreads();
  for (uint32_t j = t; j < total; j += kDegT) out[place[owner[j]] + j] = stage[j];
}

// Counts a chunk of partitioned endpoints, range by range (off[r] = first
// slot of range r, off[ranges] = all).
__global__ __launch_bounds__(kDegT) void k_deg_count(const uint16_t* __restrict__ ep,
                                                    const uint64_t* __restrict__ off, int ranges,
                                                    uint32_t* __restrict__ deg) {
  __shared__ uint32_t cnt[kRange / 2];
  const int64_t all = (int64_t)off[ranges];
  const int64_t beg = (int64_t)blockIdx.x * kDegChunk;
  const int64_t end = beg + kDegChunk < all ? beg + kDegChunk : all;
  if (beg >= end) return;
  int lo = 0, hi = ranges;  // last range whose first slot is at or before beg
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if ((int64_t)off[mid] <= beg) lo = mid;
    else hi = mid;
  }
  int64_t pos = beg;
  for (int r = lo; pos < end; ++r) {
    const int64_t rend = (int64_t)off[r + 1] < end ? (int64_t)off[r + 1] : end;
    if (rend <= pos) continue;
    for (int i = threadIdx.x; i < kRange / 2; i += kDegT) cnt[i] = 0;
    __syncthreads();
    uint32_t* d = deg + ((int64_t)r << kRangeBits);
    for (int64_t i0 = pos; i0 < rend; i0 += (int64_t)kDegT * 2 * kDegBatch) {
      uint32_t v[2 * kDegBatch];
#pragma unroll
      for (int k = 0; k < 2 * kDegBatch; ++k) {
        const int64_t i = i0 + k * kDegT + threadIdx.x;
        v[k] = i < rend ? ep[i] : 0xFFFFFFFFu;
      }
#pragma unroll
      for (int k = 0; k < 2 * kDegBatch; ++k)
        if (v[k] != 0xFFFFFFFFu) deg_add(cnt, v[k], d);
      __syncthreads();
    }
    deg_flush(cnt, kRange, d);
    __syncthreads();
    pos = rend;
  }
}

// The general form: any ID space, one atomic per endpoint.
template <int kMode>
__global__ __launch_bounds__(256) void k_deg_atomic(const uint2* __restrict__ e, int64_t ne,
                                                   int64_t nv, uint32_t* __restrict__ deg,
                                                   unsigned long long* stats) {
  uint64_t orv = 0, num = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < ne;
       i += (int64_t)gridDim.x * 256) {
    const uint2 x = e[i];
    if (!edge_counts<kMode>(x, nv)) continue;
    atomicAdd(&deg[x.x], 1u);
    if (kMode == kBoth) atomicAdd(&deg[x.y], 1u);
    orv |= (uint64_t)(x.x | x.y);
    ++num;
  }
  edge_stats<256>(orv, num, stats);
}

// A list without loops in which the edges of a source stand together (the rows
// of a CSR): a source's degree is the place where its run ends less the place
// where it begins, so only the two edges at a change of source touch memory,
// once each (modulo 2^32, in either order).  The partition's counters take
// increments of one address one at a time, which such a list is made of: the
// 1.1 x 10^8 edges of the SCALE-22 core took 2.2 ms there, 0.33 here (2.7 TB/s).
__global__ __launch_bounds__(256) void k_deg_runs(const uint2* __restrict__ e, int64_t ne,
                                                 uint32_t* __restrict__ deg,
                                                 unsigned long long* stats) {
  uint64_t orv = 0, num = 0;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t i0 = (int64_t)blockIdx.x * 256; i0 < ne; i0 += kDegBatch * stride) {
    uint2 x[kDegBatch];
    uint32_t before[kDegBatch];
#pragma unroll
    for (int k = 0; k < kDegBatch; ++k) {
      const int64_t i = i0 + k * stride + threadIdx.x;
      x[k] = i < ne ? e[i] : make_uint2(0, 0);
      before[k] = i > 0 && i < ne ? e[i - 1].x : 0u;  // mostly the lane before's: cached
    }
#pragma unroll
    for (int k = 0; k < kDegBatch; ++k) {
      const int64_t i = i0 + k * stride + threadIdx.x;
      if (i >= ne) break;
      if (i == 0 || before[k] != x[k].x) {
        atomicSub(&deg[x[k].x], (uint32_t)i);
        if (i > 0) atomicAdd(&deg[before[k]], (uint32_t)i);
      }
      if (i == ne - 1) atomicAdd(&deg[x[k].x], (uint32_t)ne);
      orv |= (uint64_t)(x[k].x | x[k].y);
      ++num;
    }
  }
  edge_stats<256>(orv, num, stats);
}

template <int kMode>
void count_mode(const uint2* edges, int64_t ne, int64_t nv, uint32_t* deg,
                unsigned long long* stats, hipStream_t s) {
  constexpr int kPer = kMode == kBoth ? 2 : 1;
  const int64_t ranges = ceil_div(nv, kRange);
  if (ranges <= kMaxDirectRanges && ne >= nv / 16) {
    // a chunk holds as many edges as a range has IDs, so that clearing and
    // flushing the counters costs no more than the counting; beyond 512
    // blocks the chunks grow instead
    const int64_t ids = std::min<int64_t>(nv, kRange);
    const int64_t chunk = std::max<int64_t>({ids, ceil_div(ne * ranges, 512), kDegT});
    hipLaunchKernelGGL(k_deg_direct<kMode>, dim3((unsigned)ceil_div(ne, chunk), (unsigned)ranges),
                       dim3(kDegT), 0, s, edges, ne, chunk, nv, deg, stats);
    G500_CHECK_LAUNCH();
    return;
  }
  // partitioning pays once the ranges hold endpoints enough to be counted in
  // LDS; a sparse list over a large ID space keeps the atomics, and so does
  // one whose endpoints find no room (asked for last)
  IdleReleases released;
  DevBuf<unsigned long long> total;  // per range, then (off) its first slot and a cursor
  DevBuf<uint64_t> off;
  DevBuf<uint16_t> ep;
  ScanWorkspace ws;
  const bool dense = ranges <= kMaxRanges && ne * kPer >= nv;
  if (dense) ws.reserve(ranges);
  if (!dense || !total.try_scratch((size_t)ranges) || !off.try_scratch((size_t)ranges + 1) ||
      !ep.try_scratch((size_t)(ne * kPer))) {
    hipLaunchKernelGGL(k_deg_atomic<kMode>,
                       dim3((unsigned)std::min<int64_t>(ceil_div(ne, 256), 4096)), dim3(256), 0, s,
                       edges, ne, nv, deg, stats);
    G500_CHECK_LAUNCH();
    return;
  }
  G500_CHECK_HIP(hipMemsetAsync(total.get(), 0, ranges * sizeof(unsigned long long), s));
  hipLaunchKernelGGL(k_deg_ranges<kMode>,
                     dim3((unsigned)std::min<int64_t>(ceil_div(ne, kDegT * 8), 1024)), dim3(kDegT),
                     0, s, edges, ne, nv, (int)ranges, total.get(), stats);
  G500_CHECK_LAUNCH();
  exclusive_scan<uint64_t>((const uint64_t*)total.get(), off.get(), ranges, ws, s);
  G500_CHECK_HIP(hipMemcpyAsync(total.get(), off.get(), ranges * sizeof(uint64_t),
                                hipMemcpyDeviceToDevice, s));
  if (ranges <= 1024) {
    constexpr int kEdges = 16384;
    hipLaunchKernelGGL((k_deg_scatter<kMode, kEdges, 1024>), dim3((unsigned)ceil_div(ne, kEdges)),
                       dim3(kDegT), 0, s, edges, ne, nv, (int)ranges, total.get(), ep.get());
  } else {
    constexpr int kEdges = 8192;
    hipLaunchKernelGGL((k_deg_scatter<kMode, kEdges, kMaxRanges>),
                       dim3((unsigned)ceil_div(ne, kEdges)), dim3(kDegT), 0, s, edges, ne, nv,
                       (int)ranges, total.get(), ep.get());
  }
  G500_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_deg_count, dim3((unsigned)ceil_div(ne * kPer, kDegChunk)), dim3(kDegT), 0,
                     s, ep.get(), off.get(), (int)ranges, deg);
  G500_CHECK_LAUNCH();
  G500_CHECK_HIP(hipStreamSynchronize(s));  // the scratch is freed on return
  released.now();
}

// --------------------------------------------------------------------- rows
constexpr int kSortT = 512;
constexpr int kSortWaves = kSortT / kWave;
// Keys the LDS sort holds (40 KB: four blocks on a CU; with 8192 keys and two
// blocks construction took 4-8 % longer at SCALE 18 to 24), keys a bucket is
// laid out for, and the length up to which a row stays in one bucket.
constexpr int kBucketCap = 4096;
constexpr int kBucketMean = 3072;
constexpr int kSplitDegree = 512;
constexpr int kPartItems = 16;
constexpr int kPartTile = kSortT * kPartItems;  // keys partitioned at a time
constexpr int kMaxParts = 2048;                 // buckets of one partition pass

// Lower bounds of the buckets: spl[i] = the key at place i * kBucketMean of
// the sorted order as the degrees foretell it.
__global__ __launch_bounds__(256) void k_splitters(const uint64_t* __restrict__ roff, int64_t n_c,
                                                  uint64_t keys, int64_t buckets, int lg,
                                                  uint64_t* __restrict__ spl) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= buckets) return;
  auto row_at = [&](uint64_t x) {  // last row whose first place is at or before x
    int64_t lo = 0, hi = n_c;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if (roff[mid] <= x) lo = mid;
      else hi = mid;
    }
    return (uint64_t)lo;
  };
  const uint64_t x = (uint64_t)i * kBucketMean;
  const uint64_t v = row_at(x);
  const uint64_t deg = roff[v + 1] - roff[v], rest = x - roff[v];
  uint64_t w = 0;
  if (deg > kSplitDegree && rest > 0)
    w = row_at((uint64_t)((double)rest / (double)deg * (double)keys));
  spl[i] = (v << lg) | w;
}

// The bucket of a key: the last lower bound (LDS, spl[0] below every key) at
// or before it, or where the bounds are the multiples of 2^shift (shift > 0)
// from first << shift on, the key's upper bits.
struct Parts {
  const uint64_t* spl;
  int parts;
  int shift;
  uint64_t first;
};

__device__ inline int part_of(const Parts& p, uint64_t key) {
  if (p.shift > 0) return (int)((key >> p.shift) - p.first);
  const uint64_t* spl = p.spl;
  int lo = 0, hi = p.parts;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (spl[mid] <= key) lo = mid;
    else hi = mid;
  }
  return lo;
}

struct PartLds {
  uint64_t stage[kPartTile];
  uint32_t wsum[kSortWaves];
};

// Keys per bucket of a tile's keys (kPartItems a thread; bit k of `use`: item
// k holds one).
__device__ inline void part_count(const Parts& p, uint32_t* hist, const uint64_t (&key)[kPartItems],
                                  uint32_t use, uint32_t* __restrict__ cnt) {
  for (int i = threadIdx.x; i < p.parts; i += kSortT) hist[i] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPartItems; ++k)
    if ((use >> k) & 1u) atomicAdd(&hist[part_of(p, key[k])], 1u);
  __syncthreads();
  for (int i = threadIdx.x; i < p.parts; i += kSortT)
    if (hist[i]) atomicAdd(&cnt[i], hist[i]);
}

// Moves a tile's keys to their buckets: they are ordered by bucket in LDS and
// written as one run per bucket, at a place reserved with one atomic per bucket
// and tile (cursor[b] = the bucket's next free place).  cap > 0: bucket b may
// only use places below (b + 1) * cap; what does not fit raises *overflow.
// pack_shift: a staged key carries its bucket above this bit (64: no room, the
// bucket is searched for again).
__device__ inline void part_move(PartLds& l, const Parts& p, uint32_t* hist, int64_t* place,
                                 const uint64_t (&key)[kPartItems], uint32_t use,
                                 int pack_shift, unsigned long long* __restrict__ cursor,
                                 int64_t cap, uint64_t* __restrict__ out, uint32_t* overflow) {
  const int t = threadIdx.x, parts = p.parts;
  for (int i = t; i < parts; i += kSortT) hist[i] = 0;
  __syncthreads();
  uint32_t at[kPartItems];  // bucket << 13 | rank in it
#pragma unroll
  for (int k = 0; k < kPartItems; ++k)
    if ((use >> k) & 1u) {
      const uint32_t b = (uint32_t)part_of(p, key[k]);
      at[k] = (b << 13) | atomicAdd(&hist[b], 1u);
    }
  __syncthreads();
  constexpr int kOwn = kMaxParts / kSortT;
  uint32_t h[kOwn], sum = 0, total;
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const int b = t * kOwn + j;
    h[j] = b < parts ? hist[b] : 0u;
    sum += h[j];
  }
  uint32_t start = block_scan<kSortT>(sum, l.wsum, &total);
#pragma unroll
  for (int j = 0; j < kOwn; ++j) {
    const int b = t * kOwn + j;
    if (b < parts) {
      hist[b] = start;
      if (h[j]) {
        const int64_t g = (int64_t)atomicAdd(&cursor[b], (unsigned long long)h[j]);
        if (cap > 0 && g + h[j] > (int64_t)(b + 1) * cap) *overflow = 1;
        place[b] = g - start;
      }
      start += h[j];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPartItems; ++k)
    if ((use >> k) & 1u) {
      const uint32_t b = at[k] >> 13;
      l.stage[hist[b] + (at[k] & 0x1FFFu)] =
          pack_shift < 64 ? key[k] | ((uint64_t)b << pack_shift) : key[k];
    }
  __syncthreads();
  for (uint32_t j = t; j < total; j += kSortT) {
    uint64_t x = l.stage[j];
    int b;
    if (pack_shift < 64) {
      b = (int)(x >> pack_shift);
      x &= (1ull << pack_shift) - 1;
    } else {
      b = part_of(p, x);
    }
    const int64_t q = place[b] + j;
    if (cap == 0 || q < (int64_t)(b + 1) * cap) out[q] = x;
  }
}

// The dynamic LDS of a partition kernel: bounds, places and counters of
// `parts` buckets.
constexpr size_t part_lds(int64_t parts) { return (size_t)parts * 20; }

// What a key is made of: both directions of an edge by new IDs, the one the
// list holds, or the edge itself (loops too) by original IDs as edge_key puts it
// (lg: log2 of the slices; step: the part bits).
enum { kKeyBoth = 0, kKeyOne = 1, kKeyEdge = 2 };

// From the edges: the keys of a tile counted by or moved into the buckets of
// every step-th bound (spl), or of the keys' bits from `shift` on.
template <int kKind, bool kMove>
__global__ __launch_bounds__(kSortT) void k_part_edges(
    const uint2* __restrict__ e, int64_t ne, const uint32_t* __restrict__ o2n, int lg,
    const uint64_t* __restrict__ spl, int64_t step, int parts, int shift, int pack_shift,
    uint32_t* __restrict__ cnt, unsigned long long* __restrict__ cursor, int64_t cap,
    uint64_t* __restrict__ out, uint32_t* overflow) {
  extern __shared__ uint64_t dyn[];
  uint64_t* s = dyn;
  int64_t* place = (int64_t*)(dyn + parts);
  uint32_t* hist = (uint32_t*)(dyn + 2 * parts);
  if (kKind != kKeyEdge)
    for (int i = threadIdx.x; i < parts; i += kSortT) s[i] = spl[(int64_t)i * step];
  const Parts p{s, parts, kKind == kKeyEdge ? shift : 0, 0};
  constexpr int kEdges = kKind == kKeyBoth ? kPartItems / 2 : kPartItems;
  const int64_t base = (int64_t)blockIdx.x * (kEdges * kSortT);
  uint64_t key[kPartItems];
  uint32_t use = 0;
  uint2 x[kEdges];
#pragma unroll
  for (int k = 0; k < kEdges; ++k) {
    const int64_t i = base + k * kSortT + threadIdx.x;
    x[k] = i < ne ? e[i] : make_uint2(0, 0);
  }
#pragma unroll
  for (int k = 0; k < kEdges; ++k) {
    if constexpr (kKind == kKeyEdge) {
      key[k] = edge_key(x[k].x, x[k].y, lg, (int)step);
      use |= (uint32_t)(base + k * kSortT + threadIdx.x < ne) << k;
      continue;
    }
    const bool ok = x[k].x != x[k].y;
    const uint64_t a = ok ? o2n[x[k].x] : 0u, b = ok ? o2n[x[k].y] : 0u;
    if constexpr (kKind == kKeyOne) {
      key[k] = (a << lg) | b;
      use |= (uint32_t)ok << k;
    } else if constexpr (kKind == kKeyBoth) {
      key[2 * k] = (a << lg) | b;
      key[2 * k + 1] = (b << lg) | a;
      use |= (ok ? 3u : 0u) << (2 * k);
    }
  }
  if constexpr (kMove) {
    __shared__ PartLds l;
    part_move(l, p, hist, place, key, use, pack_shift, cursor, cap, out, overflow);
  } else {
    part_count(p, hist, key, use, cnt);
  }
}

// From group blockIdx.y: its keys counted by or moved into its buckets.  The
// group's keys begin at g * in_cap, or with in_cap 0 where the previous
// group's end, and end at in_end[g].
template <bool kMove>
__global__ __launch_bounds__(kSortT) void k_part_keys(
    const uint64_t* __restrict__ in, const unsigned long long* __restrict__ in_end,
    int64_t in_cap, const uint64_t* __restrict__ spl, int64_t buckets, int step, int shift,
    int pack_shift, uint32_t* __restrict__ cnt, unsigned long long* __restrict__ cursor,
    uint64_t* __restrict__ out) {
  extern __shared__ uint64_t dyn[];
  const int64_t g = blockIdx.y;
  int64_t beg, end = (int64_t)in_end[g];
  if (in_cap > 0) {
    beg = g * in_cap;
    end = end < beg + in_cap ? end : beg + in_cap;
  } else {
    beg = g > 0 ? (int64_t)in_end[g - 1] : 0;
  }
  const int64_t base = beg + (int64_t)blockIdx.x * kPartTile;
  if (base >= end) return;
  const int parts = (int)(buckets - g * step < step ? buckets - g * step : step);
  uint64_t* s = dyn;
  int64_t* place = (int64_t*)(dyn + step);
  uint32_t* hist = (uint32_t*)(dyn + 2 * step);
  if (shift == 0)
    for (int i = threadIdx.x; i < parts; i += kSortT) s[i] = spl[g * step + i];
  const Parts p{s, parts, shift, (uint64_t)(g * step)};
  uint64_t key[kPartItems];
  uint32_t use = 0;
#pragma unroll
  for (int k = 0; k < kPartItems; ++k) {
    const int64_t i = base + k * kSortT + threadIdx.x;
    key[k] = i < end ? in[i] : 0;
    use |= (uint32_t)(i < end) << k;
  }
  if constexpr (kMove) {
    __shared__ PartLds l;
    part_move(l, p, hist, place, key, use, pack_shift, cursor + g * step, 0, out, nullptr);
  } else {
    part_count(p, hist, key, use, cnt + g * step);
  }
}

__global__ __launch_bounds__(256) void k_group_places(unsigned long long* __restrict__ cursor,
                                                     int groups, int64_t cap) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i < groups) cursor[i] = (unsigned long long)((int64_t)i * cap);
}

// ---- the LDS sort
constexpr int kSortItems = kBucketCap / kSortT;

struct SortLds {
  uint64_t stage[kBucketCap];
  uint32_t hist[256 * kSortWaves];  // [wave][digit]
  uint32_t wsum[kSortWaves];
  uint64_t wmax[kSortWaves];
};

__device__ inline uint64_t block_max(uint64_t mx, uint64_t* wmax) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t y = __shfl_xor(mx, o, kWave);
    mx = y > mx ? y : mx;
  }
  if (lane_id() == 0) wmax[threadIdx.x / kWave] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) mx = wmax[w] > mx ? wmax[w] : mx;
  __syncthreads();
  return mx;
}

// Sorts the block's n keys (relative to `low`, none above mx) and writes the
// targets of those that differ from their predecessor to out; returns their
// number.  Item k of a lane is key first + 64 k; every thread calls with the
// same items = ceil(n / kSortT).  Least significant digit first, eight bits a
// pass over the bits of mx: a wave owns a run of consecutive keys, the lanes
// with equal digits find one another with eight ballots and count on from the
// wave's own LDS counters, so ranks need no barrier and no atomic; the 2048
// counters (8 waves x 256 digits) are scanned once per pass.
// A row that starts here gets its place, code + index, in rows[]; the first
// key's row may have started earlier, so it takes the minimum.
__device__ inline uint32_t sort_and_write(SortLds& l, uint64_t (&key)[kSortItems], int items,
                                          uint32_t first, uint32_t n, uint64_t mx, uint64_t low,
                                          int lg, uint32_t* __restrict__ out,
                                          unsigned long long code,
                                          unsigned long long* __restrict__ rows) {
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int bits = mx ? 64 - __clzll((long long)mx) : 1;
  for (int shift = 0; shift < bits; shift += 8) {
#pragma unroll
    for (int j = 0; j < 256 * kSortWaves / kSortT; ++j) l.hist[j * kSortT + t] = 0;
    __syncthreads();
    uint32_t rank[kSortItems];
#pragma unroll
    for (int k = 0; k < kSortItems; ++k)
      if (k < items) {
        const bool valid = first + k * kWave < n;
        const uint32_t d = (uint32_t)(key[k] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const bool bit = (d >> b) & 1u;
          const uint64_t bb = __ballot(bit);
          peers &= bit ? bb : ~bb;
        }
        const uint32_t before = (uint32_t)__popcll(peers & lanemask_lt());
        volatile uint32_t* h = &l.hist[wave * 256 + d];
        const uint32_t old = *h;
        rank[k] = old + before;
        if (valid && before == 0) *h = old + (uint32_t)__popcll(peers);
      }
    __syncthreads();
    {  // exclusive scan of the counters by (digit, wave): two threads a digit
      constexpr int kOwn = 256 * kSortWaves / kSortT;
      uint32_t* mine = l.hist + (t & 1) * kOwn * 256 + (t >> 1);
      uint32_t h[kOwn], sum = 0, total;
#pragma unroll
      for (int j = 0; j < kOwn; ++j) {
        h[j] = mine[j * 256];
        sum += h[j];
      }
      uint32_t start = block_scan<kSortT>(sum, l.wsum, &total);
#pragma unroll
      for (int j = 0; j < kOwn; ++j) {
        mine[j * 256] = start;
        start += h[j];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSortItems; ++k)
      if (k < items && first + k * kWave < n)
        l.stage[l.hist[wave * 256 + ((uint32_t)(key[k] >> shift) & 255u)] + rank[k]] = key[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSortItems; ++k)
      if (k < items && first + k * kWave < n) key[k] = l.stage[first + k * kWave];
    __syncthreads();
  }
  uint64_t keep[kSortItems];
  uint32_t kept = 0;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k)
    if (k < items) {
      const uint32_t i = first + k * kWave;
      const uint64_t prev = i > 0 && i < n ? l.stage[i - 1] : ~0ull;
      keep[k] = __ballot(i < n && (i == 0 || key[k] != prev));
      kept += (uint32_t)__popcll(keep[k]);
    }
  if (lane == 0) l.wsum[wave] = kept;
  __syncthreads();
  uint32_t pos = 0, total = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    pos += w < wave ? l.wsum[w] : 0u;
    total += l.wsum[w];
  }
  const uint64_t mask = (1ull << lg) - 1;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k)
    if (k < items) {
      const uint32_t i = first + k * kWave;
      if ((keep[k] >> lane) & 1ull) {
        const uint32_t p = pos + (uint32_t)__popcll(keep[k] & lanemask_lt());
        const uint64_t full = key[k] + low;
        const uint64_t row = full >> lg;
        out[p] = (uint32_t)(full & mask);
        if (i == 0)
          atomicMin(&rows[row], code + p);
        else if (row != (l.stage[i - 1] + low) >> lg)
          rows[row] = code + p;
      }
      pos += (uint32_t)__popcll(keep[k]);
    }
  __syncthreads();
  return total;
}

// One block a bucket (keys [off[f], off[f+1])): its sorted targets without
// repeats go to uniq from off[f] on, their number to ucnt[f].  A bucket larger
// than LDS goes on a list for k_sort_big (big[0] = its length), one past
// kBigCap raises *overflow.
constexpr uint32_t kBigCap = 65536;

__global__ __launch_bounds__(kSortT) void k_sort_buckets(
    const uint64_t* __restrict__ keys, const uint64_t* __restrict__ off,
    const uint64_t* __restrict__ spl, int lg, uint32_t* __restrict__ uniq,
    uint32_t* __restrict__ ucnt, unsigned long long* __restrict__ rows,
    uint32_t* __restrict__ big, uint32_t* overflow) {
  __shared__ SortLds l;
  const int64_t f = blockIdx.x;
  const uint64_t beg = off[f], len = off[f + 1] - beg;
  if (len == 0 || len > (uint64_t)kBucketCap) {
    if (threadIdx.x == 0) {
      ucnt[f] = 0;
      if (len > kBigCap)
        *overflow = 1;
      else if (len)
        big[1 + atomicAdd(&big[0], 1u)] = (uint32_t)f;
    }
    return;
  }
  const uint32_t n = (uint32_t)len;
  const uint64_t low = spl[f];
  const uint64_t* in = keys + beg;
  // the keys are spread evenly over the waves
  const int items = (int)((n + kSortT - 1) / kSortT);
  const uint32_t first = (uint32_t)(threadIdx.x / kWave * items * kWave + lane_id());
  uint64_t key[kSortItems];
  uint64_t mx = 0;
#pragma unroll
  for (int k = 0; k < kSortItems; ++k)
    if (k < items) {
      const uint32_t i = first + k * kWave;
      key[k] = i < n ? in[i] - low : ~0ull;
      if (i < n && key[k] > mx) mx = key[k];
    }
  mx = block_max(mx, l.wmax);
  const uint32_t total = sort_and_write(l, key, items, first, n, mx, low, lg, uniq + beg,
                                        (unsigned long long)f << 32, rows);
  if (threadIdx.x == 0) ucnt[f] = total;
}

// The buckets too large for LDS, one block each: ranges of keys that fit are
// found with a histogram of kBins bins, refined within a bin that does not fit
// by itself, and sorted one after another.  A bin of one key value is that
// value, repeated.
constexpr int kBins = 4096;

__global__ __launch_bounds__(kSortT) void k_sort_big(
    const uint64_t* __restrict__ keys, const uint64_t* __restrict__ off,
    const uint64_t* __restrict__ spl, int lg, uint32_t* __restrict__ uniq,
    uint32_t* __restrict__ ucnt, unsigned long long* __restrict__ rows,
    const uint32_t* __restrict__ big) {
  __shared__ SortLds l;
  __shared__ uint32_t bins[kBins];
  __shared__ uint32_t fit, cum, taken;
  constexpr int kOwn = kBins / kSortT;
  const int t = threadIdx.x;
  for (uint32_t b = blockIdx.x; b < big[0]; b += gridDim.x) {
    const int64_t f = big[1 + b];
    const uint64_t beg = off[f], low = spl[f];
    const uint32_t n = (uint32_t)(off[f + 1] - beg);
    const uint64_t* in = keys + beg;
    uint64_t mx = 0;
    for (uint32_t i = t; i < n; i += kSortT) mx = in[i] - low > mx ? in[i] - low : mx;
    mx = block_max(mx, l.wmax);
    uint32_t written = 0;
    uint64_t lo = 0;  // keys below are done
    bool more = true;
    while (more) {
      int s = (mx - lo ? 64 - __clzll((long long)(mx - lo)) : 0) - 12;
      s = s > 0 ? s : 0;
      for (;;) {
        for (int i = t; i < kBins; i += kSortT) bins[i] = 0;
        if (t == 0) {
          fit = kBins;
          cum = 0;
          taken = 0;
        }
        __syncthreads();
        for (uint32_t i = t; i < n; i += kSortT) {
          const uint64_t k = in[i] - low;
          if (k >= lo && (k - lo) >> s < (uint64_t)kBins) atomicAdd(&bins[(k - lo) >> s], 1u);
        }
        __syncthreads();
        // the leading bins that fit together, and what they hold
        uint32_t h[kOwn], sum = 0, all;
        for (int j = 0; j < kOwn; ++j) {
          h[j] = bins[t * kOwn + j];
          sum += h[j];
        }
        uint32_t at = block_scan<kSortT>(sum, l.wsum, &all);
        for (int j = 0; j < kOwn; ++j) {
          if (at + h[j] > (uint32_t)kBucketCap) {
            atomicMin(&fit, (uint32_t)(t * kOwn + j));
            break;
          }
          at += h[j];
          if (h[j]) atomicMax(&cum, at);
        }
        __syncthreads();
        const uint32_t nb = fit, held = cum;
        if (held > 0) {  // [lo, lo + nb << s) next
          const uint64_t last = lo + (((uint64_t)nb << s) - 1);
          const bool ends = last >= mx || last < lo;
          for (uint32_t i = t; i < n; i += kSortT) {
            const uint64_t k = in[i] - low;
            if (k >= lo && (ends || k <= last)) l.stage[atomicAdd(&taken, 1u)] = k - lo;
          }
          __syncthreads();
          const uint32_t c = taken;
          const int items = (int)((c + kSortT - 1) / kSortT);
          const uint32_t first = (uint32_t)(t / kWave * items * kWave + lane_id());
          uint64_t key[kSortItems];
          uint64_t top = 0;
#pragma unroll
          for (int k = 0; k < kSortItems; ++k)
            if (k < items) {
              const uint32_t i = first + k * kWave;
              key[k] = i < c ? l.stage[i] : ~0ull;
              if (i < c && key[k] > top) top = key[k];
            }
          top = block_max(top, l.wmax);
          written += sort_and_write(l, key, items, first, c, top, low + lo, lg,
                                    uniq + beg + written,
                                    ((unsigned long long)f << 32) + written, rows);
          more = !ends;
          lo = last + 1;
          break;
        }
        lo += (uint64_t)nb << s;  // empty bins, then one that does not fit
        if (s == 0) {
          if (t == 0) {
            const uint64_t full = low + lo;
            uniq[beg + written] = (uint32_t)(full & ((1ull << lg) - 1));
            atomicMin(&rows[full >> lg], ((unsigned long long)f << 32) + written);
          }
          ++written;
          more = lo < mx;
          ++lo;
          __syncthreads();
          break;
        }
        s = s > 12 ? s - 12 : 0;
        __syncthreads();
      }
    }
    if (t == 0) ucnt[f] = written;
    __syncthreads();
  }
}

// The buckets' targets to their final places, one block a bucket.
__global__ __launch_bounds__(256) void k_collect(const uint32_t* __restrict__ uniq,
                                                const uint64_t* __restrict__ off,
                                                const uint32_t* __restrict__ ucnt,
                                                const uint64_t* __restrict__ ubase,
                                                uint32_t* __restrict__ col) {
  const int64_t f = blockIdx.x;
  const uint32_t* in = uniq + off[f];
  const uint32_t n = ucnt[f];
  uint32_t* out = col + ubase[f];
  for (uint32_t i = threadIdx.x; i < n; i += 256) out[i] = in[i];
}

__global__ __launch_bounds__(256) void k_row_offsets(const unsigned long long* __restrict__ rows,
                                                    const uint64_t* __restrict__ ubase,
                                                    int64_t n_c, int64_t m,
                                                    int64_t* __restrict__ row_off) {
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v < n_c)
    row_off[v] = (int64_t)(ubase[rows[v] >> 32] + (rows[v] & 0xFFFFFFFFull));
  else if (v == n_c)
    row_off[v] = m;
}

// out[i] = in[i * step]
__global__ __launch_bounds__(256) void k_every(const uint64_t* __restrict__ in, int64_t step,
                                              int64_t n, uint64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = in[i * step];
}

}  // namespace

void count_degrees(const uint2* edges, int64_t ne, DegreeMode mode, int64_t nv, uint32_t* deg,
                   unsigned long long* stats, hipStream_t s) {
  if (ne <= 0) return;
  switch (mode) {
    case DegreeMode::kBothEnds:
      count_mode<kBoth>(edges, ne, nv, deg, stats, s);
      break;
    case DegreeMode::kSourceNoLoops:
      count_mode<kSource>(edges, ne, nv, deg, stats, s);
      break;
    case DegreeMode::kSourceRuns:
      hipLaunchKernelGGL(k_deg_runs,
                         dim3((unsigned)std::min<int64_t>(ceil_div(ne, 256 * kDegBatch), 4096)),
                         dim3(256), 0, s, edges, ne, deg, stats);
      G500_CHECK_LAUNCH();
      break;
    case DegreeMode::kSourceEnd:
      count_mode<kSourceAll>(edges, ne, nv, deg, stats, s);
      break;
  }
}

// g->col and g->row_off for m entries.  The last entries of col are padding:
// bottom-up scans read aligned 16-byte groups, which may run a few entries past
// the last row.
static void take_rows(g500_graph* g, int64_t m) {
  g->col.alloc_raw((size_t)m + kColPad);
  g->row_off.alloc_raw((size_t)g->n_c + 1);
  G500_CHECK_HIP(hipMemsetAsync(g->col.get() + m, 0, kColPad * sizeof(uint32_t), g->stream));
}

// build_rows; throws NOMEM where something small finds no room.
static bool rows_by_buckets(g500_graph* g, const uint2* edges, int64_t ne, bool symmetric) {
  hipStream_t s = g->stream;
  const int64_t keys = g->m_sym, n_c = g->n_c;
  const int lg = g->log_n;
  if (keys <= 0 || n_c <= 0) return false;
  const int64_t buckets = ceil_div(keys, kBucketMean);
  // one pass up to kMaxParts buckets; above that groups of `step` buckets first
  const int64_t step = group_buckets(buckets, kMaxParts);
  if (step == 0 || lg > 31) return false;
  const int64_t groups = ceil_div(buckets, step);
  const bool two = step > 1;
  const int64_t group_keys = step * kBucketMean;
  const int64_t group_cap = group_keys + group_keys / 8 + kPartTile;
  IdleReleases released;
  DevBuf<uint64_t> roff, spl, part, sorted, off, ubase;
  DevBuf<uint32_t> cnt, ucnt, big, flag, uniq;
  DevBuf<unsigned long long> rows, cursor, gcursor;
  // without room for all this the radix sort still fits
  if ((two && (!part.try_scratch((size_t)(groups * group_cap)) ||
               !gcursor.try_scratch((size_t)groups))) ||
      !sorted.try_scratch((size_t)keys) || (!two && !uniq.try_scratch((size_t)keys)) ||
      !roff.try_scratch((size_t)n_c + 1) || !rows.try_scratch((size_t)n_c) ||
      !spl.try_scratch((size_t)buckets) || !off.try_scratch((size_t)buckets + 1) ||
      !ubase.try_scratch((size_t)buckets + 1) || !cnt.try_scratch((size_t)buckets) ||
      !cursor.try_scratch((size_t)buckets) || !ucnt.try_scratch((size_t)buckets) ||
      !big.try_scratch((size_t)buckets + 1) || !flag.try_scratch(1))
    return false;
  exclusive_scan<uint32_t>(g->deg_new.get(), roff.get(), n_c, g->scan_ws, s);
  hipLaunchKernelGGL(k_splitters, dim3((unsigned)ceil_div(buckets, 256)), dim3(256), 0, s,
                     roff.get(), n_c, (uint64_t)keys, buckets, lg, spl.get());
  G500_CHECK_LAUNCH();
  G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, buckets * sizeof(uint32_t), s));
  G500_CHECK_HIP(hipMemsetAsync(big.get(), 0, sizeof(uint32_t), s));
  G500_CHECK_HIP(hipMemsetAsync(flag.get(), 0, sizeof(uint32_t), s));
  G500_CHECK_HIP(hipMemsetAsync(rows.get(), 0xFF, n_c * sizeof(uint64_t), s));
  const int pack = 2 * lg + bit_length(kMaxParts - 1) <= 64 ? 2 * lg : 64;
  const unsigned tiles = (unsigned)ceil_div(ne, symmetric ? kPartTile : kPartTile / 2);
  auto from_edges = [&](auto kernel, unsigned long long* cur, int64_t cap, uint64_t* out) {
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(kSortT), part_lds(groups), s, edges, ne,
                       g->orig2new.get(), lg, spl.get(), step, (int)groups, 0, pack, cnt.get(), cur,
                       cap, out, flag.get());
    G500_CHECK_LAUNCH();
  };
  auto from_groups = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(group_cap, kPartTile), (unsigned)groups),
                       dim3(kSortT), part_lds(step), s, part.get(), gcursor.get(), group_cap,
                       spl.get(), buckets, (int)step, 0, pack, cnt.get(), cursor.get(),
                       sorted.get());
    G500_CHECK_LAUNCH();
  };
  auto move_edges = symmetric ? k_part_edges<kKeyOne, true> : k_part_edges<kKeyBoth, true>;
  if (two) {
    hipLaunchKernelGGL(k_group_places, dim3((unsigned)ceil_div(groups, 256)), dim3(256), 0, s,
                       gcursor.get(), (int)groups, group_cap);
    G500_CHECK_LAUNCH();
    from_edges(move_edges, gcursor.get(), group_cap, part.get());
    from_groups(k_part_keys<false>);
  } else {
    from_edges(symmetric ? k_part_edges<kKeyOne, false> : k_part_edges<kKeyBoth, false>, nullptr, 0,
               nullptr);
  }
  exclusive_scan<uint32_t>(cnt.get(), off.get(), buckets, g->scan_ws, s);
  G500_CHECK_HIP(hipMemcpyAsync(cursor.get(), off.get(), buckets * sizeof(uint64_t),
                                hipMemcpyDeviceToDevice, s));
  if (two)
    from_groups(k_part_keys<true>);
  else
    from_edges(move_edges, cursor.get(), 0, sorted.get());
  // the first pass's room is free again
  uint32_t* un = two ? (uint32_t*)part.get() : uniq.get();
  hipLaunchKernelGGL(k_sort_buckets, dim3((unsigned)buckets), dim3(kSortT), 0, s, sorted.get(),
                     off.get(), spl.get(), lg, un, ucnt.get(), rows.get(), big.get(), flag.get());
  G500_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_sort_big, dim3((unsigned)std::min<int64_t>(buckets, 512)), dim3(kSortT), 0,
                     s, sorted.get(), off.get(), spl.get(), lg, un, ucnt.get(), rows.get(),
                     big.get());
  G500_CHECK_LAUNCH();
  exclusive_scan<uint32_t>(ucnt.get(), ubase.get(), buckets, g->scan_ws, s);
  uint64_t m = 0;
  uint32_t over = 0;
  G500_CHECK_HIP(hipMemcpyAsync(&m, ubase.get() + buckets, sizeof(m), hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipMemcpyAsync(&over, flag.get(), sizeof(over), hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  if (over) return false;
  take_rows(g, (int64_t)m);
  g->m = (int64_t)m;
  hipLaunchKernelGGL(k_collect, dim3((unsigned)buckets), dim3(256), 0, s, un, off.get(),
                     ucnt.get(), ubase.get(), g->col.get());
  G500_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_row_offsets, dim3((unsigned)ceil_div(n_c + 1, 256)), dim3(256), 0, s,
                     rows.get(), ubase.get(), n_c, g->m, g->row_off.get());
  G500_CHECK_LAUNCH();
  G500_CHECK_HIP(hipStreamSynchronize(s));  // the scratch is freed on return
  released.now();
  return true;
}

bool build_rows(g500_graph* g, const uint2* edges, int64_t ne, bool symmetric) {
  try {
    if (rows_by_buckets(g, edges, ne, symmetric)) return true;
  } catch (const Error& e) {
    if (e.code != G500_ERR_NOMEM) throw;
  }
  g->col.release();
  g->row_off.release();
  return false;
}

std::shared_ptr<const OrderedEdges> order_edges(const g500_graph* g, hipStream_t s) {
  const int64_t ne = g->nedges;
  if (ne < kOrderedEdgesMin || g->id_bits > kOrderedIdBits) return nullptr;
  size_t free_b = 0, total_b = 0;
  G500_CHECK_HIP(hipMemGetInfo(&free_b, &total_b));
  if ((uint64_t)ne * sizeof(uint64_t) > total_b / 16) return nullptr;
  const int wlog = std::max(0, g->id_bits - kEdgeWindowBits);
  const int slog = std::max(0, g->id_bits - kEdgeSliceBits);
  // as many parts of a window as two passes can tell apart
  int pass_log = 0;
  while ((1 << (pass_log + 1)) <= kMaxParts) ++pass_log;
  const int part_bits = std::min(kEdgePartBits, 2 * pass_log - wlog - slog);
  if (part_bits < 0) return nullptr;
  const int tile_shift = kEdgeSliceBits + kEdgeWindowBits - part_bits;
  const int64_t tiles = (int64_t)1 << (wlog + slog + part_bits);
  int step_log = 0;
  if (tiles > kMaxParts)
    while (((int64_t)1 << (2 * step_log)) < tiles) ++step_log;
  const int64_t step = (int64_t)1 << step_log, groups = ceil_div(tiles, step);
  IdleReleases released;
  DevBuf<uint64_t> part, keys, off;
  DevBuf<uint32_t> cnt;
  DevBuf<unsigned long long> cursor;
  if ((step > 1 && !part.try_scratch((size_t)ne)) || !keys.try_scratch((size_t)ne) ||
      !off.try_scratch((size_t)tiles + 1) || !cnt.try_scratch((size_t)tiles) ||
      !cursor.try_scratch((size_t)tiles))
    return nullptr;
  ScanWorkspace ws;
  const unsigned blocks = (unsigned)ceil_div(ne, kPartTile);
  // places of the buckets from their counts
  auto places = [&](int64_t n) {
    exclusive_scan<uint32_t>(cnt.get(), off.get(), n, ws, s);
    G500_CHECK_HIP(hipMemcpyAsync(cursor.get(), off.get(), n * sizeof(uint64_t),
                                  hipMemcpyDeviceToDevice, s));
  };
  auto from_edges = [&](auto kernel, uint64_t* out) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kSortT), part_lds(groups), s, g->edges.get(),
                       ne, (const uint32_t*)nullptr, slog, (const uint64_t*)nullptr,
                       (int64_t)part_bits, (int)groups, tile_shift + step_log, 64, cnt.get(), cursor.get(),
                       (int64_t)0, out, (uint32_t*)nullptr);
    G500_CHECK_LAUNCH();
  };
  G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, groups * sizeof(uint32_t), s));
  from_edges(k_part_edges<kKeyEdge, false>, nullptr);
  places(groups);
  from_edges(k_part_edges<kKeyEdge, true>, step > 1 ? part.get() : keys.get());
  if (step > 1) {
    std::vector<uint32_t> h((size_t)groups);
    DevBuf<unsigned long long> gend;  // the cursors stand at the groups' ends now
    gend.alloc_raw((size_t)groups);
    G500_CHECK_HIP(hipMemcpyAsync(gend.get(), cursor.get(), groups * sizeof(uint64_t),
                                  hipMemcpyDeviceToDevice, s));
    G500_CHECK_HIP(hipMemcpyAsync(h.data(), cnt.get(), groups * sizeof(uint32_t),
                                  hipMemcpyDeviceToHost, s));
    G500_CHECK_HIP(hipStreamSynchronize(s));
    const unsigned most = (unsigned)std::max<int64_t>(
        1, ceil_div((int64_t)*std::max_element(h.begin(), h.end()), kPartTile));
    auto from_groups = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(most, (unsigned)groups), dim3(kSortT), part_lds(step), s,
                         part.get(), gend.get(), (int64_t)0, (const uint64_t*)nullptr, tiles,
                         (int)step, tile_shift, 64, cnt.get(), cursor.get(), keys.get());
      G500_CHECK_LAUNCH();
    };
    G500_CHECK_HIP(hipMemsetAsync(cnt.get(), 0, tiles * sizeof(uint32_t), s));
    from_groups(k_part_keys<false>);
    places(tiles);
    from_groups(k_part_keys<true>);
    G500_CHECK_HIP(hipStreamSynchronize(s));  // gend is freed here
  }
  // chunks of the edges of one window and slice: only where these begin goes to
  // the host (with all 2^22 places of SCALE 24 and up the call took 15.5 ms, now 7.6)
  const int64_t parts = (int64_t)1 << part_bits, runs = tiles >> part_bits;
  std::vector<uint64_t> h((size_t)runs + 1);
  DevBuf<uint64_t> begin;
  begin.alloc_raw(h.size());
  hipLaunchKernelGGL(k_every, dim3((unsigned)ceil_div(runs + 1, 256)), dim3(256), 0, s, off.get(),
                     parts, runs + 1, begin.get());
  G500_CHECK_LAUNCH();
  G500_CHECK_HIP(hipMemcpyAsync(h.data(), begin.get(), h.size() * sizeof(uint64_t),
                                hipMemcpyDeviceToHost, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  std::vector<EdgeChunk> chunks;
  for (uint32_t w = 0; w < 1u << wlog; ++w)
    for (uint32_t c = 0; c < 1u << slog; ++c) {
      const size_t i = ((size_t)w << slog) + c;
      const uint64_t beg = h[i], end = h[i + 1];
      // even pieces
      const uint64_t pieces = (uint64_t)ceil_div((int64_t)(end - beg), kEdgeChunk);
      for (uint64_t k = 0; k < pieces; ++k) {
        const uint64_t a = beg + (end - beg) * k / pieces, e = beg + (end - beg) * (k + 1) / pieces;
        chunks.push_back({a, (uint32_t)(e - a), w, c, 0});
      }
    }
  auto order = std::make_shared<OrderedEdges>();
  order->chunks.alloc_raw(chunks.size());
  G500_CHECK_HIP(hipMemcpyAsync(order->chunks.get(), chunks.data(),
                                chunks.size() * sizeof(EdgeChunk), hipMemcpyHostToDevice, s));
  G500_CHECK_HIP(hipStreamSynchronize(s));
  order->keys.swap(keys);
  order->n_chunks = (int64_t)chunks.size();
  order->part_bits = part_bits;
  released.now();  // the stream was waited for above
  return order;
}

}  // namespace g500
