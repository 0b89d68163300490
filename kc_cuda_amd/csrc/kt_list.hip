// Truss levels of a sorted-row core over triangle lists, on CDNA4.
//
// A level removes, round by round, every edge whose support is below the
// threshold (reference: src/kc.cu:886-1056, 1140-1309), and for each removed
// edge the partners of its triangles lose one. Finding those triangles by
// intersecting the edge's rows costs the shorter row's length times a search,
// again each time; on the graphs measured the rows of an edge hold 10 to 25
// times more entries than it has triangles. So a core whose triangles fit
// memory lists them once: every edge has the pairs of partner edges of its
// triangles (as many as its support), 24 bytes a triangle in all. A round then
// streams its frontier's lists, nothing is recounted (an edge without
// triangles costs nothing to remove) and no row is ever rewritten.
//
// One launch is one step of the search: it walks a round's frontier, or looks
// at the live edges for the next level's. Every workgroup works out from the
// last step's counters what this step does -- the same inputs give all of them
// the same answer -- and the first writes the state for the next. The host
// queues steps in batches and reads the state once per batch.
#include <algorithm>

#include "kt_device.h"
#include "kt_kernels.h"

namespace kt {
namespace {

constexpr int kListGrid = 1024;
constexpr uint32_t kListUnroll = 4;  // list entries a lane has in flight

// --------------------------------------------------------------- the lists --

__device__ __forceinline__ void put_triangle(uint32_t a, uint32_t b, uint32_t c, uint32_t* cursor, uint2* tri) {
  const uint32_t pa = atomicAdd(&cursor[a], 1u), pb = atomicAdd(&cursor[b], 1u), pc = atomicAdd(&cursor[c], 1u);
  tri[pa] = make_uint2(b, c);
  tri[pb] = make_uint2(a, c);
  tri[pc] = make_uint2(a, b);
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
        if (j < ve) {
          const uint32_t w = adj_d[j];
          if (w >= list[0] && w <= wmax && ((bits[w >> 5] >> (w & 31)) & 1u))
            put_triangle(beg + i, beg + lower_bound_u32(list, i + 1, du, w), j, cursor, tri);
        }
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
    for (uint32_t i = ab + lane; i < ae; i += G) {
      const uint32_t x = adj_d[i];
      const uint32_t p = lower_bound_u32(adj_d, bb, be, x);
      if (p < be && adj_d[p] == x) put_triangle(e, i, p, cursor, tri);
    }
  }
}

// --------------------------------------------------------------- the steps --

// What step `it` does, from the state that step it - 1 acted on and what its
// counters say. Counters rotate over three sets: a step reads the last one's,
// adds to its own and clears the next one's.
__device__ __forceinline__ ListState list_next(const ListState& was, const ListCounters& got) {
  ListState s = was;
  const uint32_t c = got.frontier;  // stamped by the last step, not yet walked
  // a level is complete: min = the least support among its edges
  auto record = [&](int32_t thr, uint32_t min) {
    s.level_kmax = min + 2;
    s.level_count = s.alive;
    s.level_floor = thr;
    s.levels += 1;
    if (s.first && s.early_ans && s.alive == s.early_ans && (s.exact_early || min + 2 == s.early_k)) {
      s.level_kmax = s.early_k;
      s.phase = kListDone;
      return true;
    }
    s.first = 0;
    return false;
  };
  auto look = [&](int32_t thr, uint32_t closing) {
    s.phase = kListLook;
    s.thr = thr;
    s.closing = closing;
    s.compact = 2ull * s.alive <= s.live;
  };
  if (was.phase == kListDone) return s;
  if (was.phase == kListEmpty) {
    s.phase = kListDone;
    s.alive = 0;
    return s;
  }
  if (was.phase == kListStart) {
    look(was.thr, 0);
    s.compact = 0;
    return s;
  }
  if (was.phase == kListLook) {
    if (was.compact) {
      s.live = got.live;
      s.buf ^= 1u;
      s.listed = 1;
      s.relists += 1;
    }
    if (got.min == kNone) {  // there are live edges: the last walk left some
      s.err = 1;
      s.phase = kListDone;
      return s;
    }
    // the level below is complete (closing), or the first threshold removes nothing
    if (was.closing && record(was.thr - 1, got.min)) return s;
    if (c == 0) {
      if (!was.closing && record(was.thr, got.min)) return s;
      look(int32_t(got.min) + 1, 0);
      return s;
    }
    s.round += 1;  // the stamp the look gave its frontier
  } else {         // a walk
    if (c == 0) {
      if (s.alive == 0)
        s.phase = kListDone;
      else
        look(was.thr + 1, 1);
      return s;
    }
    s.round += 1;
  }
  s.rounds += 1;
  s.cur ^= 1u;
  // A non-empty level at thr is a (thr + 2)-truss, which has at least
  // (thr + 2)(thr + 1) / 2 edges: with fewer left the level empties at once.
  const int32_t thr = s.thr;
  if (c == s.alive ||
      (thr > 0 && s.alive - c < (unsigned long long)(thr + 2) * (unsigned long long)(thr + 1) / 2)) {
    s.phase = kListEmpty;
    return s;
  }
  s.alive -= c;
  s.phase = kListWalk;
  return s;
}

// The frontier's triangles: a wave takes `per` frontier edges, scans their
// list lengths and deals the concatenated entries out to its lanes; with
// fewer edges than waves, several waves share an edge. Round-synchronous rule:
// a triangle with one frontier edge charges both partners; with two, the
// third edge is charged once -- by the frontier edge of the smaller id; with
// three, nobody. An edge that falls below the threshold is stamped with the
// next round at once (to this round it still counts as live).
__device__ __forceinline__ void list_walk(const ListArgs& a, const ListState& s, const uint32_t* q, uint32_t cnt,
                                          uint32_t* qn, uint32_t* qn_count) {
  __shared__ uint32_t s_e[kBlock], s_beg[kBlock], s_inc[kBlock];
  const int lane = lane64();
  const uint32_t wbase = threadIdx.x & ~uint32_t(kWave - 1);
  const uint32_t nw = gridDim.x * (kBlock / kWave);
  const uint32_t per = min(uint32_t(kWave), (cnt + nw - 1) / nw);
  const uint32_t groups = (cnt + per - 1) / per;
  const uint32_t parts = max(1u, min(uint32_t(kWave), nw / groups));
  const uint32_t items = groups * parts;  // <= nw + cnt
  const uint32_t r = s.round;
  const int32_t thr = s.thr;
  for (uint32_t it = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; it < items; it += nw) {  // wave-uniform
    const uint32_t grp = it / parts, part = it - grp * parts;
    const uint32_t i = grp * per + uint32_t(lane);
    uint32_t e = 0, beg = 0, len = 0;
    if (uint32_t(lane) < per && i < cnt) {
      e = q[i];
      beg = a.tri_off[e];
      // with a support of 0 no triangle of the edge is live
      len = a.sup[e] > 0 ? a.tri_off[e + 1] - beg : 0u;
    }
    uint32_t inc = len;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o);
      if (lane >= o) inc += y;
    }
    const uint32_t total = __shfl(inc, kWave - 1);
    s_e[threadIdx.x] = e;
    s_beg[threadIdx.x] = beg;
    s_inc[threadIdx.x] = inc;
    wave_sync();
    for (uint32_t j0 = part * kWave * kListUnroll; j0 < total; j0 += kWave * kListUnroll * parts) {
      uint32_t me[kListUnroll], xa[kListUnroll], xb[kListUnroll], ma[kListUnroll], mb[kListUnroll];
#pragma unroll
      for (uint32_t k = 0; k < kListUnroll; ++k) {
        const uint32_t j = j0 + k * kWave + uint32_t(lane);
        xa[k] = xb[k] = kNone;
        me[k] = 0;
        if (j < total) {
          uint32_t lo = 0, hi = per - 1;  // owner: first lane whose inclusive length exceeds j
          while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_inc[wbase + mid] > j)
              hi = mid;
            else
              lo = mid + 1;
          }
          const uint32_t before = lo ? s_inc[wbase + lo - 1] : 0u;
          const uint2 t = a.tri[s_beg[wbase + lo] + (j - before)];
          me[k] = s_e[wbase + lo];
          xa[k] = t.x;
          xb[k] = t.y;
        }
      }
#pragma unroll
      for (uint32_t k = 0; k < kListUnroll; ++k) {
        ma[k] = xa[k] != kNone ? a.state[xa[k]] : 0u;
        mb[k] = xb[k] != kNone ? a.state[xb[k]] : 0u;
      }
      int32_t oa[kListUnroll], ob[kListUnroll];  // supports before the decrements
#pragma unroll
      for (uint32_t k = 0; k < kListUnroll; ++k) {
        bool da = false, db = false;
        if (ma[k] >= r && mb[k] >= r) {  // neither partner deleted in an earlier round
          const bool ina = ma[k] == r, inb = mb[k] == r;
          da = !ina && (!inb || me[k] < xb[k]);
          db = !inb && (!ina || me[k] < xa[k]);
        }
        if (!da) xa[k] = kNone;
        if (!db) xb[k] = kNone;
        oa[k] = da ? atomicSub(&a.sup[xa[k]], 1) : 0;
        ob[k] = db ? atomicSub(&a.sup[xb[k]], 1) : 0;
      }
#pragma unroll
      for (uint32_t k = 0; k < kListUnroll; ++k) {
        const bool ca = xa[k] != kNone && oa[k] == thr, cb = xb[k] != kNone && ob[k] == thr;
        if (ca) {
          a.state[xa[k]] = r + 1;
          a.del_thr[xa[k]] = uint32_t(thr);
        }
        if (cb) {
          a.state[xb[k]] = r + 1;
          a.del_thr[xb[k]] = uint32_t(thr);
        }
        wave_append(ca, xa[k], qn, qn_count);
        wave_append(cb, xb[k], qn, qn_count);
      }
    }
    wave_sync();
  }
}

// The live edges below the threshold become the next frontier (stamped), the
// least support among all live edges goes to got->min, and where half of the
// edge list is dead the rest is listed anew.
__device__ __forceinline__ void list_look(const ListArgs& a, const ListState& s, uint32_t* q, ListCounters* mine) {
  __shared__ uint32_t s_base[2];
  __shared__ uint32_t s_min[kBlock / kWave];
  const uint32_t* list = s.listed ? a.live[s.buf] : nullptr;
  uint32_t* next = a.live[s.buf ^ 1u];
  const uint32_t r = s.round + 1;
  const int32_t thr = s.thr;
  constexpr uint32_t kItems = 8, kTile = kBlock * kItems;
  uint32_t best = kNone;
  for (uint32_t t0 = blockIdx.x * kTile; t0 < s.live; t0 += gridDim.x * kTile) {  // block-uniform
    uint32_t e[kItems];
    uint32_t front = 0, keep = 0;
#pragma unroll
    for (uint32_t k = 0; k < kItems; ++k) {
      const uint32_t i = t0 + k * kBlock + threadIdx.x;
      e[k] = i < s.live ? (list ? list[i] : i) : kNone;
    }
#pragma unroll
    for (uint32_t k = 0; k < kItems; ++k)
      if (e[k] != kNone && a.state[e[k]] == kNone) {
        const int32_t x = a.sup[e[k]];
        best = min(best, uint32_t(x));
        if (x < thr)
          front |= 1u << k;
        else
          keep |= 1u << k;
      }
    uint32_t nf, nk = 0;
    uint32_t at = block_exclusive_scan(uint32_t(__popc(front)), &nf), kept = 0;
    if (s.compact) kept = block_exclusive_scan(uint32_t(__popc(keep)), &nk);
    if (threadIdx.x == 0) {
      if (nf) s_base[0] = atomicAdd(&mine->frontier, nf);
      if (nk) s_base[1] = atomicAdd(&mine->live, nk);
    }
    __syncthreads();
    if (nf) at += s_base[0];
    if (nk) kept += s_base[1];
#pragma unroll
    for (uint32_t k = 0; k < kItems; ++k) {
      if ((front >> k) & 1u) {
        a.state[e[k]] = r;
        a.del_thr[e[k]] = uint32_t(thr);
        q[at++] = e[k];
      }
      if (s.compact && ((keep >> k) & 1u)) next[kept++] = e[k];
    }
    __syncthreads();
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = min(best, uint32_t(__shfl_xor(best, o)));
  if (lane64() == 0) s_min[threadIdx.x / kWave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kBlock / kWave; ++k) best = min(best, s_min[k]);
    if (best != kNone) atomicMin(&mine->min, best);
  }
}

// Step `it`. Bound: a chain of seven dependent memory round trips (state,
// counters, queue, list bounds, entries, partner states, decrements) on the
// short rounds that a search is mostly made of.
__global__ __launch_bounds__(kBlock) void k_list_step(ListArgs a, uint32_t it) {
  const ListState was = a.states[it & 1u];
  const ListState s = list_next(was, a.counters[(it + 2) % 3]);
  ListCounters* mine = &a.counters[it % 3];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.states[(it + 1) & 1u] = s;
    ListCounters* clear = &a.counters[(it + 1) % 3];
    clear->frontier = 0;
    clear->live = 0;
    clear->min = kNone;
  }
  if (s.phase == kListWalk) {
    const uint32_t cnt = a.counters[(it + 2) % 3].frontier;
    list_walk(a, s, a.q[s.cur], cnt, a.q[s.cur ^ 1u], &mine->frontier);
  } else if (s.phase == kListLook) {
    list_look(a, s, a.q[s.cur ^ 1u], mine);
  } else if (s.phase == kListEmpty) {  // every edge still live dies at this threshold
    const uint32_t* list = s.listed ? a.live[s.buf] : nullptr;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < s.live; i += gridDim.x * kBlock) {
      const uint32_t e = list ? list[i] : i;
      if (a.state[e] == kNone) {
        a.state[e] = s.round;
        a.del_thr[e] = uint32_t(s.thr);
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_sum_u32(const uint32_t* __restrict__ in, uint32_t n,
                                                    unsigned long long* total) {
  unsigned long long c = 0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) c += in[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (lane64() == 0 && c) atomicAdd(total, c);
}

__global__ void k_list_start(ListArgs a, ListState s) {
  if (threadIdx.x != 0) return;
  a.states[0] = s;
  for (int k = 0; k < 3; ++k) {
    a.counters[k].frontier = 0;
    a.counters[k].live = 0;
    a.counters[k].min = kNone;
  }
}

}  // namespace

// --------------------------------------------------------------- wrappers ---

void sum_u32(const uint32_t* in, uint32_t n, uint64_t* total, hipStream_t s) {
  if (n) k_sum_u32<<<std::min(grid_for(n), 1024), kBlock, 0, s>>>(in, n, reinterpret_cast<unsigned long long*>(total));
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

void list_start(const ListArgs& a, const ListState& first, hipStream_t s) { k_list_start<<<1, kWave, 0, s>>>(a, first); }

void list_steps(const ListArgs& a, uint32_t mc, uint32_t from, uint32_t count, hipStream_t s) {
  const int grid = int(std::max<uint64_t>(1, std::min<uint64_t>((uint64_t(mc) + kBlock - 1) / kBlock, kListGrid)));
  for (uint32_t i = 0; i < count; ++i) k_list_step<<<grid, kBlock, 0, s>>>(a, from + i);
}

}  // namespace kt
