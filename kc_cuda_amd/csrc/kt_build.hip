// CSR build of large pair lists by two staged splits, on CDNA4.
//
// The second entries (row v, column u) of pairs sorted by u are in no order,
// nor are any of pairs that are not sorted.
// k_part_scatter writes each one straight to its bucket: with thousands of
// buckets per workgroup and thousands of workgroups, the lines being filled
// outgrow the L2 many times over, every 8-byte store becomes a memory
// transaction of its own, and k_bucket_rows' 4-byte stores into a bucket's
// megabytes fare no better (505 M pairs over 50 M vertices: 7.3 and 10.8 ms,
// some 70 bytes of traffic an entry each). Here the entries are split twice
// by up to nine bits of their row's group, low bits first, each time through
// LDS so that a bucket's entries leave in runs, and then a group's few
// thousand slots are put in row order in LDS and written once, in order.
#include <algorithm>

#include "kt_device.h"
#include "kt_kernels.h"

namespace kt {
namespace {

constexpr int kSplitBlock = 512;
constexpr uint32_t kMaxDigits = 512;      // one per thread
constexpr uint32_t kSplitPer = 16;        // entries a thread holds
constexpr uint32_t kSplitStage = kSplitBlock * kSplitPer;  // 64 KB of LDS
constexpr int kRowsBlock = 512;
constexpr uint32_t kRowsPer = 16;
constexpr uint32_t kRowsStage = kRowsBlock * kRowsPer;  // slots of a group put in order in LDS: 32 KB
constexpr uint32_t kMaxGroupRows = kRowsBlock;

// The entries of tile t. First split: a run of the pairs' second entries (v, u)
// or of both of each pair's. Second: a run of the first one's output, cut at
// its bucket bounds (so that a tile holds one low digit and the order within
// it does not matter): start[d] the first entry of bucket d, tiles[d] its
// first tile.
constexpr int kSecondOnes = 0, kBothOnes = 1, kSplitOnce = 2;
template <int kFrom>
struct SplitSrc {
  static constexpr bool kFirst = kFrom != kSplitOnce;
  const uint2* entries;
  uint64_t items, tile;
  uint32_t buckets;  // of the first split
  const uint64_t* start;
  const uint32_t* tiles;
  __device__ __forceinline__ void range(uint32_t t, uint64_t* lo, uint64_t* hi) const {
    if (kFirst) {
      *lo = min(items, uint64_t(t) * tile);
      *hi = min(items, *lo + tile);
      return;
    }
    if (t >= tiles[buckets]) {
      *lo = *hi = 0;
      return;
    }
    uint32_t d0 = 0, d1 = buckets;  // the last bucket whose first tile is at most t
    while (d1 - d0 > 1) {
      const uint32_t mid = (d0 + d1) / 2;
      if (tiles[mid] <= t)
        d0 = mid;
      else
        d1 = mid;
    }
    *lo = start[d0] + uint64_t(t - tiles[d0]) * tile;
    *hi = min(start[d0 + 1], *lo + tile);
  }
  __device__ __forceinline__ uint2 get(uint64_t i) const {
    const uint2 p = entries[kFrom == kBothOnes ? i >> 1 : i];
    const bool turn = kFrom == kSecondOnes || (kFrom == kBothOnes && (i & 1u));
    return turn ? make_uint2(p.y, p.x) : p;
  }
};

// hist[t * digits + d] = tile t's entries of digit d
template <int kFrom>
__global__ __launch_bounds__(kSplitBlock) void k_split_hist(SplitSrc<kFrom> src, uint32_t shift, uint32_t digits,
                                                            uint32_t* hist) {
  __shared__ uint32_t s_cnt[kMaxDigits];
  uint64_t lo, hi;
  src.range(blockIdx.x, &lo, &hi);
  if (threadIdx.x < kMaxDigits) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  constexpr uint32_t kUnroll = 4;
  for (uint64_t i0 = lo; i0 < hi; i0 += kSplitBlock * kUnroll) {  // workgroup-uniform
    uint32_t row[kUnroll];
#pragma unroll
    for (uint32_t k = 0; k < kUnroll; ++k) {
      const uint64_t i = i0 + k * kSplitBlock + threadIdx.x;
      row[k] = i < hi ? src.get(i).x : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < kUnroll; ++k) {
      const uint32_t d = (row[k] >> shift) & (digits - 1);
      const LaneRun r = lane_run(d, i0 + k * kSplitBlock + threadIdx.x < hi);
      if (r.is_head) atomicAdd(&s_cnt[d], r.len);
    }
  }
  __syncthreads();
  if (threadIdx.x < digits) hist[uint64_t(blockIdx.x) * digits + threadIdx.x] = s_cnt[threadIdx.x];
}

// Exclusive scan of one value per thread, kSplitBlock threads.
__device__ __forceinline__ uint32_t digit_scan(uint32_t v) {
  uint32_t total;
  return block_exclusive_scan<kSplitBlock>(v, &total);
}

// Tile t's entries to their digits' places, off_t[t * digits + d] on. 8192
// entries at a time are put in digit order in LDS and written in runs.
template <int kFrom>
__global__ __launch_bounds__(kSplitBlock) void k_split(SplitSrc<kFrom> src, uint32_t shift, uint32_t digits,
                                                       const uint64_t* __restrict__ off_t, uint2* __restrict__ out) {
  __shared__ uint2 s_stage[kSplitStage];
  __shared__ uint32_t s_cnt[kMaxDigits], s_at[kMaxDigits];
  __shared__ uint64_t s_out[kMaxDigits];  // a digit's place in out, less its place in the stage
  const uint32_t tid = threadIdx.x;
  const int lane = lane64();
  uint64_t lo, hi;
  src.range(blockIdx.x, &lo, &hi);
  uint64_t cursor = tid < digits ? off_t[uint64_t(blockIdx.x) * digits + tid] : 0;  // thread d: digit d's
  for (uint64_t i0 = lo; i0 < hi; i0 += kSplitStage) {  // workgroup-uniform
    const uint32_t count = uint32_t(min(uint64_t(kSplitStage), hi - i0));
    if (tid < kMaxDigits) s_cnt[tid] = 0;
    uint2 e[kSplitPer];
    uint32_t rank[kSplitPer];
#pragma unroll
    for (uint32_t k = 0; k < kSplitPer; ++k)
      if (k * kSplitBlock + tid < count) e[k] = src.get(i0 + k * kSplitBlock + tid);
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kSplitPer; ++k) {
      const bool in = k * kSplitBlock + tid < count;
      const uint32_t d = in ? (e[k].x >> shift) & (digits - 1) : 0u;
      const LaneRun r = lane_run(d, in);
      uint32_t at = 0;
      if (r.is_head) at = atomicAdd(&s_cnt[d], r.len);
      rank[k] = __shfl(at, in ? r.head : lane) + uint32_t(lane - r.head);
    }
    __syncthreads();
    const uint32_t mine = tid < kMaxDigits ? s_cnt[tid] : 0u, at = digit_scan(mine);
    if (tid < kMaxDigits) {
      s_at[tid] = at;
      s_out[tid] = cursor - at;
      cursor += mine;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kSplitPer; ++k)
      if (k * kSplitBlock + tid < count) s_stage[s_at[(e[k].x >> shift) & (digits - 1)] + rank[k]] = e[k];
    __syncthreads();
    for (uint32_t i = tid; i < count; i += kSplitBlock) {
      const uint2 x = s_stage[i];
      out[s_out[(x.x >> shift) & (digits - 1)] + i] = x;
    }
    __syncthreads();
  }
}

// The second split's tiles: start[d] = the first split's bucket d, tiles[d] =
// its first tile; one more of both.
__global__ __launch_bounds__(kSplitBlock) void k_split_tiles(const uint64_t* __restrict__ off_b, uint32_t T,
                                                             uint32_t buckets, uint64_t tile, uint64_t* start,
                                                             uint32_t* tiles) {
  const uint32_t d = threadIdx.x;
  const uint64_t lo = off_b[uint64_t(min(d, buckets)) * T], hi = off_b[uint64_t(min(d + 1, buckets)) * T];
  const uint32_t n = uint32_t((hi - lo + tile - 1) / tile), at = digit_scan(n);
  if (d < buckets) {
    start[d] = lo;
    tiles[d] = at;
  }
  if (d + 1 == buckets) {
    start[buckets] = hi;
    tiles[buckets] = at + n;
  }
}

// A group of 2^S rows per workgroup: its second entries are part[beg .. end),
// its first ones fwd[f0[g] .. f0[g + 1]). Ranks within the rows come from one
// LDS counter a row while the entries are read, the columns are put in order
// in LDS and leave as one run (fwd null: part holds all entries). A group with more slots than the stage holds
// (hubs) is counted and placed from memory as k_bucket_rows does.
__global__ __launch_bounds__(kRowsBlock) void k_group_rows(const uint2* __restrict__ part,
                                                           const uint64_t* __restrict__ off_b,
                                                           const uint32_t* __restrict__ tiles, uint32_t T,
                                                           uint32_t low_bits, const uint2* __restrict__ fwd,
                                                           const uint64_t* __restrict__ f0, uint32_t S, uint32_t n,
                                                           uint64_t* off, uint32_t* deg, uint32_t* adj) {
  __shared__ uint32_t s_col[kRowsStage];
  __shared__ uint32_t s_cnt[kMaxGroupRows];
  const uint32_t g = blockIdx.x, tid = threadIdx.x;
  const uint32_t low = g & ((1u << low_bits) - 1u), high = g >> low_bits;
  const uint64_t beg = off_b[uint64_t(high) * T + tiles[low]], end = off_b[uint64_t(high) * T + tiles[low + 1]];
  const uint64_t fb = fwd ? f0[g] : 0, fe = fwd ? f0[g + 1] : 0, base = beg + fb;
  const uint32_t r0 = g << S, nrows = min(1u << S, n - r0);
  const int lane = lane64();
  const uint64_t slots = (end - beg) + (fe - fb);
  const bool staged = slots <= kRowsStage;  // workgroup-uniform
  const uint32_t back = staged ? uint32_t(end - beg) : 0u, all = staged ? uint32_t(slots) : 0u;
  s_cnt[tid] = 0;
  uint2 e[kRowsPer];
  uint32_t rank[kRowsPer];
#pragma unroll
  for (uint32_t k = 0; k < kRowsPer; ++k) {
    const uint32_t i = k * kRowsBlock + tid;
    if (i < all) e[k] = i < back ? part[beg + i] : fwd[fb + (i - back)];
  }
  __syncthreads();
  auto count_all = [&](const uint2* __restrict__ src, uint64_t lo, uint64_t hi) {
    for (uint64_t i0 = lo; i0 < hi; i0 += kRowsBlock) {  // workgroup-uniform
      const bool in = i0 + tid < hi;
      const uint32_t r = in ? src[i0 + tid].x - r0 : 0u;
      const LaneRun run = lane_run(r, in);
      if (run.is_head) atomicAdd(&s_cnt[r], run.len);
    }
  };
  if (staged) {
#pragma unroll
    for (uint32_t k = 0; k < kRowsPer; ++k) {
      if (k * kRowsBlock >= all) break;  // workgroup-uniform
      const bool in = k * kRowsBlock + tid < all;
      const uint32_t r = in ? e[k].x - r0 : 0u;
      const LaneRun run = lane_run(r, in);  // the first entries come in runs of a row
      uint32_t at = 0;
      if (run.is_head) at = atomicAdd(&s_cnt[r], run.len);
      rank[k] = __shfl(at, in ? run.head : lane) + uint32_t(lane - run.head);
    }
  } else {
    count_all(part, beg, end);
    count_all(fwd, fb, fe);
  }
  __syncthreads();
  const uint32_t mine = s_cnt[tid];  // at most 512 rows
  uint32_t total;
  const uint32_t at = block_exclusive_scan<kRowsBlock>(mine, &total);
  if (tid < nrows) {
    off[r0 + tid] = base + at;
    deg[r0 + tid] = mine;
  }
  s_cnt[tid] = at;
  __syncthreads();
  if (staged) {
#pragma unroll
    for (uint32_t k = 0; k < kRowsPer; ++k)
      if (k * kRowsBlock + tid < all) s_col[s_cnt[e[k].x - r0] + rank[k]] = e[k].y;
    __syncthreads();
    for (uint32_t i = tid; i < all; i += kRowsBlock) adj[base + i] = s_col[i];
    return;
  }
  auto place_all = [&](const uint2* __restrict__ src, uint64_t lo, uint64_t hi) {
    for (uint64_t i0 = lo; i0 < hi; i0 += kRowsBlock) {  // workgroup-uniform
      const bool in = i0 + tid < hi;
      const uint2 x = in ? src[i0 + tid] : make_uint2(r0, 0u);
      const LaneRun run = lane_run(x.x - r0, in);
      uint32_t p = 0;
      if (run.is_head) p = atomicAdd(&s_cnt[x.x - r0], run.len);
      p = __shfl(p, in ? run.head : lane);
      if (in) adj[base + p + uint32_t(lane - run.head)] = x.y;
    }
  };
  place_all(part, beg, end);
  place_all(fwd, fb, fe);
}

}  // namespace

// --------------------------------------------------------------- wrappers ---

// Against the bucketed build, random pairs, 20 slots a row (ms, whole build):
// 2^21 pairs 0.121 -> 0.154, 2^22 0.187 -> 0.184, 2^23 0.319 -> 0.244, 2^24
// 0.77 -> 0.40, 2^25 1.55 -> 0.72 (80 slots a row: the same); 505 M pairs 19.0
// -> 10.8 (two counts 1.4, splits 3.2 and 2.5, rows 3.5; 2.7 to 3.5 TB/s). It
// is taken from 2^22 pairs on, shuffled ones too: 2^21 0.158 -> 0.186, 2^22
// 0.288 -> 0.255, 2^23 0.525 -> 0.385, 2^25 2.67 -> 1.43.
// Groups of as many rows, a power of two, as average 6,144 slots or fewer (the
// stage takes 8,192), split by at most nine bits twice, so at most 2^18 of them.
// That holds for every vertex count up to 134 M with up to 400 M pairs; with 505
// M pairs for 70 % of the counts from 5 to 130 M (50 M: 195 k groups; 20, 35, 40
// and 42 M: 273 k to 328 k, which take the bucketed build and its 19 ms), with
// 600 M for 44 %.
bool split_plan(uint32_t n, uint64_t pairs, bool sorted, SplitPlan* p) {
  p->sorted = sorted;
  p->entries = sorted ? pairs : 2 * pairs;
  uint32_t s = 9;  // kMaxGroupRows
  while (s > 0 && double(2 * pairs) / n * double(1u << s) > 6144.0) --s;
  const uint64_t groups = (uint64_t(n) + (1u << s) - 1) >> s;
  uint32_t bits = 2;
  while (bits < 32 && (uint64_t(1) << bits) < groups) ++bits;
  if (bits > 18 || groups < 2) return false;
  p->shift = s;
  p->groups = uint32_t(groups);
  p->low_bits = bits / 2;
  p->high_bits = bits - bits / 2;
  // tiles of whole stages, about 4096 of them
  const uint64_t stages = (p->entries + 4096ull * kSplitStage - 1) / (4096ull * kSplitStage);
  p->tile = kSplitStage * std::max<uint64_t>(2, stages);
  p->tiles1 = uint32_t((p->entries + p->tile - 1) / p->tile);
  p->tiles2 = p->tiles1 + (1u << p->low_bits);
  return true;
}
template <int kFrom>
static SplitSrc<kFrom> split_src(const SplitPlan& p, const uint32_t* from, const uint64_t* start,
                                 const uint32_t* tiles) {
  return SplitSrc<kFrom>{reinterpret_cast<const uint2*>(from), p.entries, p.tile, 1u << p.low_bits, start, tiles};
}
void split_hist(bool first, const SplitPlan& p, const uint32_t* from, const uint64_t* start, const uint32_t* tiles,
                uint32_t* hist, hipStream_t s) {
  const uint32_t lows = 1u << p.low_bits, highs = 1u << p.high_bits;
  if (!first)
    k_split_hist<kSplitOnce><<<p.tiles2, kSplitBlock, 0, s>>>(split_src<kSplitOnce>(p, from, start, tiles),
                                                              p.shift + p.low_bits, highs, hist);
  else if (p.sorted)
    k_split_hist<kSecondOnes><<<p.tiles1, kSplitBlock, 0, s>>>(split_src<kSecondOnes>(p, from, start, tiles), p.shift,
                                                               lows, hist);
  else
    k_split_hist<kBothOnes><<<p.tiles1, kSplitBlock, 0, s>>>(split_src<kBothOnes>(p, from, start, tiles), p.shift,
                                                             lows, hist);
}
void split(bool first, const SplitPlan& p, const uint32_t* from, const uint64_t* start, const uint32_t* tiles,
           const uint64_t* off_t, uint32_t* to, hipStream_t s) {
  auto o = reinterpret_cast<uint2*>(to);
  const uint32_t lows = 1u << p.low_bits, highs = 1u << p.high_bits;
  if (!first)
    k_split<kSplitOnce><<<p.tiles2, kSplitBlock, 0, s>>>(split_src<kSplitOnce>(p, from, start, tiles),
                                                         p.shift + p.low_bits, highs, off_t, o);
  else if (p.sorted)
    k_split<kSecondOnes><<<p.tiles1, kSplitBlock, 0, s>>>(split_src<kSecondOnes>(p, from, start, tiles), p.shift,
                                                          lows, off_t, o);
  else
    k_split<kBothOnes><<<p.tiles1, kSplitBlock, 0, s>>>(split_src<kBothOnes>(p, from, start, tiles), p.shift, lows,
                                                        off_t, o);
}
void split_tiles(const SplitPlan& p, const uint64_t* off_b, uint64_t* start, uint32_t* tiles, hipStream_t s) {
  k_split_tiles<<<1, kSplitBlock, 0, s>>>(off_b, p.tiles1, 1u << p.low_bits, p.tile, start, tiles);
}
void group_rows(const SplitPlan& p, const uint32_t* part, const uint64_t* off_b, const uint32_t* tiles,
                const uint32_t* fwd, const uint64_t* f0, uint32_t n, uint64_t* off, uint32_t* deg, uint32_t* adj,
                hipStream_t s) {
  k_group_rows<<<p.groups, kRowsBlock, 0, s>>>(reinterpret_cast<const uint2*>(part), off_b, tiles, p.tiles2,
                                               p.low_bits, reinterpret_cast<const uint2*>(fwd), f0, p.shift, n, off,
                                               deg, adj);
}

}  // namespace kt
