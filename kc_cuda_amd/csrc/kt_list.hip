// Triangle lists of a sorted-row core.
//
// Removing an edge charges the partners of its triangles (reference:
// src/kc.cu:61-191, 886-1056). Finding those triangles by intersecting the
// edge's rows costs the shorter row's length times a search, again each time;
// on the graphs measured the rows of an edge hold 10 to 25 times more entries
// than it has triangles. So a core whose triangles fit memory lists them once:
// every edge has the pairs of partner edges of its triangles (as many as its
// support), 24 bytes a triangle in all, which the steps of kt_step.hip stream.
#include <algorithm>

#include "kt_device.h"
#include "kt_kernels.h"

namespace kt {
namespace {

// A group of G lanes found triangles of one edge e, at most one a lane (hit),
// with partner edges x and y. They share one atomic of e's cursor: one each
// would queue up on its address (a union of 40 M edges: 27 ms, shared 13).
template <int G>
__device__ __forceinline__ void put_triangles(bool hit, uint32_t e, uint32_t x, uint32_t y, uint32_t* cursor,
                                              uint2* tri) {
  const int lane = lane64();
  const unsigned long long group = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << (lane / G * G);
  const unsigned long long hits = __ballot(hit) & group;
  if (!hit) return;
  const uint32_t ax = atomicAdd(&cursor[x], 1u), ay = atomicAdd(&cursor[y], 1u);
  const int first = __ffsll(hits) - 1;
  uint32_t at = 0;
  if (lane == first) at = atomicAdd(&cursor[e], uint32_t(__popcll(hits)));
  at = __shfl(at, first) + uint32_t(__popcll(hits & ((1ull << lane) - 1ull)));
  tri[at] = make_uint2(x, y);
  tri[ax] = make_uint2(e, y);
  tri[ay] = make_uint2(e, x);
}

// One workgroup per vertex u: out(u) in LDS as a bitmap and a list, the
// out-rows of its neighbours streamed against it by groups of G lanes (the
// support count's enumeration, k_support_bitmap).
template <int G>
__global__ __launch_bounds__(kBlock) void k_tri_fill_bitmap(const uint32_t* __restrict__ off_d,
                                                            const uint32_t* __restrict__ adj_d, uint32_t nc,
                                                            uint32_t words, uint32_t* cursor, uint2* tri) {
  extern __shared__ uint32_t lds[];
  uint32_t* bits = lds;
  uint32_t* list = bits + words;
  const uint32_t tid = threadIdx.x;
  for (uint32_t u = blockIdx.x; u < nc; u += gridDim.x) {
    const uint32_t beg = off_d[u];
    const uint32_t du = off_d[u + 1] - beg;
    if (du < 2) continue;  // block-uniform
    for (uint32_t i = tid; i < du; i += blockDim.x) list[i] = adj_d[beg + i];
    __syncthreads();
    const uint32_t wlo = list[0] >> 5, whi = list[du - 1] >> 5;
    for (uint32_t i = wlo + tid; i <= whi; i += blockDim.x) bits[i] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < du; i += blockDim.x) atomicOr(&bits[list[i] >> 5], 1u << (list[i] & 31));
    __syncthreads();
    const uint32_t wmax = list[du - 1];
    const uint32_t sg = tid / G, lane = tid % G, nsg = blockDim.x / G;
    for (uint32_t i = sg; i + 1 < du; i += nsg) {
      const uint32_t v = list[i];
      const uint32_t vb = off_d[v], ve = off_d[v + 1];
      for (uint32_t j0 = vb; j0 < ve; j0 += G) {
        if (adj_d[j0] > wmax) break;  // rows are sorted: nothing further can hit
        const uint32_t j = j0 + lane;
        uint32_t w = 0;
        bool hit = false;
        if (j < ve) {
          w = adj_d[j];
          hit = w >= list[0] && w <= wmax && ((bits[w >> 5] >> (w & 31)) & 1u);
        }
        put_triangles<G>(hit, beg + i, hit ? beg + lower_bound_u32(list, i + 1, du, w) : 0u, j, cursor, tri);
      }
    }
    __syncthreads();
  }
}

// One group of G lanes per oriented edge, as k_support_edges.
template <int G>
__global__ __launch_bounds__(kBlock) void k_tri_fill_edges(const uint32_t* __restrict__ off_d,
                                                           const uint32_t* __restrict__ adj_d,
                                                           const uint32_t* __restrict__ src, uint32_t mc,
                                                           uint32_t* cursor, uint2* tri) {
  const uint32_t groups = gridDim.x * (blockDim.x / G);
  const uint32_t lane = threadIdx.x % G;
  for (uint32_t e = blockIdx.x * (blockDim.x / G) + threadIdx.x / G; e < mc; e += groups) {
    const uint32_t u = src[e], v = adj_d[e];
    uint32_t ab = e + 1, ae = off_d[u + 1];
    uint32_t bb = off_d[v], be = off_d[v + 1];
    if ((ae - ab) > (be - bb)) {
      uint32_t t = ab; ab = bb; bb = t;
      t = ae; ae = be; be = t;
    }
    for (uint32_t i0 = ab; i0 < ae; i0 += G) {  // group-uniform
      const uint32_t i = i0 + lane;
      uint32_t p = 0;
      bool hit = false;
      if (i < ae) {
        const uint32_t x = adj_d[i];
        p = lower_bound_u32(adj_d, bb, be, x);
        hit = p < be && adj_d[p] == x;
      }
      put_triangles<G>(hit, e, i, p, cursor, tri);
    }
  }
}

// found[0] += the sum of the supports (null: none), found[1] = 1 when a row is
// not strictly ascending above its own vertex, found[2], found[3] = the highest
// support and ~ of the lowest. The count and the fill need not agree on such
// rows (a repeated neighbour is found once by a search, and by each of its
// copies where they are streamed), so entries would miss their lists.
__global__ __launch_bounds__(kBlock) void k_list_size(const uint32_t* __restrict__ sup,
                                                      const uint32_t* __restrict__ src,
                                                      const uint32_t* __restrict__ adj, uint32_t mc,
                                                      unsigned long long* found) {
  __shared__ unsigned long long s_sum[kBlock / kWave];
  __shared__ uint2 s_ends[kBlock / kWave];
  unsigned long long c = 0;
  uint32_t high = 0, low = 0;  // low: ~ the lowest
  bool odd = false;
  for (uint64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < mc; i += gridDim.x * blockDim.x) {
    const uint32_t u = src[i], v = adj[i];
    if (sup) {
      const uint32_t x = sup[i];
      c += x;
      high = max(high, x);
      low = max(low, ~x);
    }
    odd |= v <= u || (i + 1 < mc && src[i + 1] == u && adj[i + 1] <= v);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    c += __shfl_xor(c, o);
    high = max(high, uint32_t(__shfl_xor(high, o)));
    low = max(low, uint32_t(__shfl_xor(low, o)));
  }
  if (lane64() == 0) {
    s_sum[threadIdx.x / kWave] = c;
    s_ends[threadIdx.x / kWave] = make_uint2(high, low);
  }
  if (__syncthreads_or(odd) && threadIdx.x == 0) found[1] = 1;
  if (threadIdx.x == 0 && sup) {
    for (int k = 1; k < kBlock / kWave; ++k) {
      c += s_sum[k];
      high = max(high, s_ends[k].x);
      low = max(low, s_ends[k].y);
    }
    atomicAdd(&found[0], c);
    atomicMax(reinterpret_cast<uint32_t*>(&found[2]), high);
    atomicMax(reinterpret_cast<uint32_t*>(&found[3]), low);
  }
}

}  // namespace

// --------------------------------------------------------------- wrappers ---

void list_size(const int32_t* sup, const uint32_t* src, const uint32_t* adj, uint32_t mc, uint64_t* found,
               hipStream_t s) {
  fill_u64(found, 4, 0, s);
  if (mc)
    k_list_size<<<std::min(grid_for(mc), 1024), kBlock, 0, s>>>(reinterpret_cast<const uint32_t*>(sup), src, adj, mc,
                                                                reinterpret_cast<unsigned long long*>(found));
}

void tri_fill(const uint32_t* off_d, const uint32_t* adj_d, const uint32_t* src, uint32_t nc, uint32_t mc,
              uint32_t max_dout, bool bitmap, int lanes, uint32_t* cursor, uint32_t* tri, hipStream_t s) {
  if (!mc) return;
  uint2* t = reinterpret_cast<uint2*>(tri);
  if (bitmap) {
    const uint32_t words = (nc + 31) / 32;
    const uint32_t lds = 4u * (words + ((max_dout + 63) & ~63u));
    const int grid = int(nc < (1u << 20) ? nc : (1u << 20));
    switch (lanes) {
      case 8: k_tri_fill_bitmap<8><<<grid, kBlock, lds, s>>>(off_d, adj_d, nc, words, cursor, t); break;
      case 16: k_tri_fill_bitmap<16><<<grid, kBlock, lds, s>>>(off_d, adj_d, nc, words, cursor, t); break;
      case 32: k_tri_fill_bitmap<32><<<grid, kBlock, lds, s>>>(off_d, adj_d, nc, words, cursor, t); break;
      default: k_tri_fill_bitmap<64><<<grid, kBlock, lds, s>>>(off_d, adj_d, nc, words, cursor, t); break;
    }
    return;
  }
  const int grid = grid_for(uint64_t(mc) * uint64_t(lanes));
  switch (lanes) {
    case 8: k_tri_fill_edges<8><<<grid, kBlock, 0, s>>>(off_d, adj_d, src, mc, cursor, t); break;
    case 16: k_tri_fill_edges<16><<<grid, kBlock, 0, s>>>(off_d, adj_d, src, mc, cursor, t); break;
    case 32: k_tri_fill_edges<32><<<grid, kBlock, 0, s>>>(off_d, adj_d, src, mc, cursor, t); break;
    default: k_tri_fill_edges<64><<<grid, kBlock, 0, s>>>(off_d, adj_d, src, mc, cursor, t); break;
  }
}

}  // namespace kt
