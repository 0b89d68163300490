// Truss levels, one launch per step, on CDNA4.
//
// A level removes, round by round, every edge whose support is below the
// threshold, and the search moves from level to level (reference:
// src/kc.cu:886-1056, 1140-1309). One launch is one step of that: it walks a
// round's frontier, looks at the live edges for the next level's, or drops a
// frontier and counts the rest anew. Every workgroup works out from the last
// step's state and counters what this step does -- the same inputs give all of
// them the same answer -- and the first writes the state for the next, so no
// round waits for the host or for a closing launch. The host queues steps in
// batches and reads the state once per batch.
//
// Two kinds of core are walked: sorted rows through triangle lists
// (kt_list.hip), and dense cores through bit-matrix rows. An edge that falls
// below the threshold is stamped with the next round by whoever takes it
// there; to the round being walked it still counts as live.
#include <hip/hip_ext.h>

#include <algorithm>

#include "kt_device.h"
#include "kt_kernels.h"
#include "kt_tile.h"

namespace kt {
namespace {

// Workgroups a step gets: the most, and the core's edges for each. A core of
// 200 edges is walked 64 edges at a time: by one workgroup in 36 us, by one
// per 32 edges in 9 (256 and 32 edges each, whole solves: 40 vertices 0.61 ->
// 0.51 ms, 200k edges 3.25 -> 3.02 ms with the two round trips less; the same
// from 16 to 64 edges each, and for cores that fill the grid).
constexpr int kStepGrid = 1024;
constexpr uint32_t kGridEdges = 32;
constexpr uint32_t kListUnroll = 4;   // list entries a lane has in flight
constexpr uint32_t kDenseUnroll = 8;  // triangles a lane has in flight (dense walk)
// a dropped frontier of at least 1/32 of the core's edges has the rows rebuilt
constexpr uint32_t kRebuildShare = 32;
constexpr uint32_t kDenseMaxWords = 1024;  // nc <= 65536 on a dense core

// What a step does, from what the last one did and what its counters say.
// Counters rotate over three sets: a step reads the last one's, adds to its
// own and clears the next one's. Queues too: a frontier's own, the one it
// fills, and the last walked one's, whose edges still stand in a dense core's
// rows (pend) until a step clears them.
__device__ __forceinline__ StepState next_step(const StepState& was, const StepCounters& got, const StepRule& rule) {
  StepState s = was;
  const uint32_t c = got.frontier;  // stamped by the last step, not yet walked
  // a level is complete: min = the least support among its edges; true: the
  // search is over (early exit on a first level, or the level budget spent)
  auto record = [&](int32_t thr, uint32_t min) {
    s.level_kmax = min + 2;
    s.level_count = s.alive;
    s.level_floor = thr;
    s.levels += 1;
    if (s.first && s.early_ans && s.alive == s.early_ans && (s.exact_early || min + 2 == s.early_k)) {
      s.level_kmax = s.early_k;
      s.phase = kStepDone;
      return true;
    }
    s.first = 0;
    if (s.max_levels && s.levels >= s.max_levels) {
      s.phase = kStepDone;
      return true;
    }
    return false;
  };
  // the live edges below thr; closing: the level at thr - 1 is complete, and
  // when it is the last one wanted nothing more is collected (peek)
  auto look = [&](int32_t thr, uint32_t closing) {
    s.phase = kStepLook;
    s.thr = thr;
    s.closing = closing;
    s.peek = closing && s.max_levels && s.levels + 1 >= s.max_levels;
    s.compact = rule.relist && 2ull * s.alive <= s.live;
  };
  switch (was.phase) {
    case kStepDone:
    case kStepHost:
      return s;
    case kStepEmpty:
      s.phase = kStepDone;
      s.alive = 0;
      return s;
    case kStepStart:
      look(was.thr, 0);
      return s;
    case kStepResume:
      s.phase = kStepClear;
      return s;
    case kStepClear:
      s.phase = kStepRecount;
      s.pend_cnt = 0;
      return s;
    case kStepLook:
    case kStepRecount:
      s.pend_cnt = 0;
      if (was.phase == kStepLook && was.compact) {
        s.live = got.live;
        s.buf ^= 1u;
        s.listed = 1;
        s.relists += 1;
      }
      if (got.min == kNone) {  // there are live edges: the last walk left some
        s.err = 1;
        s.phase = kStepDone;
        return s;
      }
      if (was.phase == kStepLook && was.closing && record(was.thr - 1, got.min)) return s;
      if (c == 0) {  // nothing below thr (unless closing, its level is complete too)
        if (!(was.phase == kStepLook && was.closing) && record(was.thr, got.min)) return s;
        look(int32_t(got.min) + 1, 0);
        return s;
      }
      break;
    default:  // a walk
      s.pend = was.cur;
      s.pend_cnt = was.cnt;
      if (c == 0) {
        if (s.alive == 0)
          s.phase = kStepDone;
        else
          look(was.thr + 1, 1);
        return s;
      }
  }
  // the next frontier
  s.round += 1;
  s.rounds += 1;
  s.cur = s.cur == 2 ? 0 : s.cur + 1;
  s.cnt = c;
  const int32_t thr = s.thr;
  // A non-empty level at thr is a (thr + 2)-truss, which has at least
  // (thr + 2)(thr + 1) / 2 edges: with fewer left the level empties at once.
  if (c == s.alive ||
      (thr > 0 && s.alive - c < (unsigned long long)(thr + 2) * (unsigned long long)(thr + 1) / 2)) {
    s.phase = kStepEmpty;
    return s;
  }
  s.alive -= c;
  // Dense cores: a walk ANDs each frontier edge's rows and visits about thr
  // triangles at tri_cost, a recount ANDs every live edge's rows (costs in
  // word ANDs; drop_fixed: the two launches it takes).
  const double by_edge = double(s.alive) * double(rule.ws);
  if (rule.dense && double(c) * (double(rule.ws) + rule.tri_cost * double(thr)) >=
                        fmin(by_edge, rule.pair_cost) + rule.drop_fixed) {
    s.recounts += 1;
    s.pairs = by_edge > rule.pair_cost;
    // once three tenths of the edges are gone the host may shrink the matrix
    s.phase = rule.host && 10ull * s.alive <= 7ull * s.host_at ? kStepHost : kStepClear;
    return s;
  }
  s.phase = kStepWalk;
  return s;
}

__device__ __forceinline__ void stamp_dead(const StepArgs& a, uint32_t e, uint32_t round, uint32_t thr) {
  a.state[e] = round;
  a.del_thr[a.orig ? a.orig[e] : e] = thr;
}

// The next frontier's edges found by a workgroup, gathered in LDS and added to
// the queue with one atomic at the end: one per wave that finds some would
// serialise on the queue's counter (5 ns each: a recount of 960 k edges that
// leaves 160 k took 585 us, 35 without its appends).
constexpr uint32_t kOutCap = 1024;
struct Out {
  uint32_t item[kOutCap];
  uint32_t n, base;
};

__device__ __forceinline__ void out_begin(Out& o) {
  if (threadIdx.x == 0) o.n = 0;
  __syncthreads();
}

// A queue's entry for edge e = (u, v): of a sorted-row core the edge, of a
// dense one its ends (16 bits each), which name its rows without a detour
// through the edge's arrays; its id comes from the edge-id matrix while the
// rows are read.
__device__ __forceinline__ uint32_t ends(uint32_t u, uint32_t v) { return u << 16 | v; }

// Edges that fall below thr join the next frontier. Every lane of the wave
// must reach this; what no longer fits in LDS goes to the queue directly.
__device__ __forceinline__ void append_dead(const StepArgs& a, Out& o, bool p, uint32_t e, uint32_t item,
                                            uint32_t round, int32_t thr, uint32_t* qn, uint32_t* qn_count) {
  const unsigned long long mask = __ballot(p);
  if (!mask) return;
  const int lane = lane64(), leader = __ffsll(mask) - 1;
  uint32_t at = 0;
  if (lane == leader) at = atomicAdd(&o.n, uint32_t(__popcll(mask)));
  at = __shfl(at, leader) + uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
  if (p) {
    stamp_dead(a, e, round, uint32_t(thr));
    if (at < kOutCap) o.item[at] = item;
  }
  wave_append(p && at >= kOutCap, item, qn, qn_count);
}

// Every thread of the workgroup, after its last append.
__device__ __forceinline__ void out_end(Out& o, uint32_t* qn, uint32_t* qn_count) {
  __syncthreads();
  const uint32_t n = min(o.n, kOutCap);
  if (threadIdx.x == 0 && n) o.base = atomicAdd(qn_count, n);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < n; i += kBlock) qn[o.base + i] = o.item[i];
}

// Whom a triangle of frontier edge e with partner edges xa, xb charges
// (round-synchronous): with one frontier edge both partners; with two the
// third edge once, by the frontier edge of the smaller id; with three, or
// where an edge died in an earlier round, nobody. ma, mb: the partners'
// stamps, r: the round walked.
__device__ __forceinline__ void charges(uint32_t e, uint32_t xa, uint32_t xb, uint32_t ma, uint32_t mb, uint32_t r,
                                        bool* da, bool* db) {
  *da = *db = false;
  if (ma >= r && mb >= r) {
    const bool ina = ma == r, inb = mb == r;
    *da = !ina && (!inb || e < xb);
    *db = !inb && (!ina || e < xa);
  }
}

// A list core's frontier: a wave takes `per` frontier edges, scans their list
// lengths and deals the concatenated entries out to its lanes; with fewer
// edges than waves, several waves share an edge.
__device__ __forceinline__ void walk_lists(const StepArgs& a, const StepState& s, uint32_t* qn, uint32_t* qn_count) {
  __shared__ uint32_t s_e[kBlock], s_beg[kBlock], s_inc[kBlock];
  __shared__ Out out;
  out_begin(out);
  const uint32_t* q = a.q[s.cur];
  const uint32_t cnt = s.cnt;
  const int lane = lane64();
  const uint32_t wbase = threadIdx.x & ~uint32_t(kWave - 1);
  const uint32_t nw = gridDim.x * (kBlock / kWave);
  const uint32_t per = min(uint32_t(kWave), (cnt + nw - 1) / nw);
  const uint32_t groups = (cnt + per - 1) / per;
  const uint32_t parts = max(1u, min(uint32_t(kWave), nw / groups));
  const uint32_t items = groups * parts;
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
        ma[k] = xa[k] != kNone ? a.state[xa[k]] : 0u;  // 0: before every round
        mb[k] = xb[k] != kNone ? a.state[xb[k]] : 0u;
      }
      int32_t oa[kListUnroll], ob[kListUnroll];  // supports before the decrements
      bool da[kListUnroll], db[kListUnroll];
#pragma unroll
      for (uint32_t k = 0; k < kListUnroll; ++k) {
        charges(me[k], xa[k], xb[k], ma[k], mb[k], r, &da[k], &db[k]);
        oa[k] = da[k] ? atomicSub(&a.sup[xa[k]], 1) : 0;
        ob[k] = db[k] ? atomicSub(&a.sup[xb[k]], 1) : 0;
      }
#pragma unroll
      for (uint32_t k = 0; k < kListUnroll; ++k) {
        append_dead(a, out, da[k] && oa[k] == thr, xa[k], xa[k], r + 1, thr, qn, qn_count);
        append_dead(a, out, db[k] && ob[k] == thr, xb[k], xb[k], r + 1, thr, qn, qn_count);
      }
    }
    wave_sync();
  }
  out_end(out, qn, qn_count);
}

__device__ __forceinline__ void clear_bits(const StepArgs& a, const uint32_t* q, uint32_t cnt) {
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < cnt; i += gridDim.x * kBlock) {
    const uint32_t x = q[i], u = x >> 16, v = x & 0xFFFFu;
    atomicAnd(&a.bits[uint64_t(u) * a.ws + (v >> 6)], ~(1ull << (v & 63)));
    atomicAnd(&a.bits[uint64_t(v) * a.ws + (u >> 6)], ~(1ull << (u & 63)));
  }
}

// Every row anew from the live edges: what clearing many edges' bits one
// atomic at a time would leave (R-MAT-22's pass 2 drops 4.2 M of 6.3 M edges
// first: 3.1 ms of clearing). One workgroup per row, through LDS.
__device__ __forceinline__ void rebuild_rows(const StepArgs& a) {
  __shared__ unsigned long long s_row[kDenseMaxWords];
  for (uint32_t u = blockIdx.x; u < a.nc; u += gridDim.x) {  // workgroup-uniform
    for (uint32_t i = threadIdx.x; i < a.ws; i += kBlock) s_row[i] = 0;
    __syncthreads();
    const uint32_t end = a.off_u[u + 1];
    for (uint32_t j = a.off_u[u] + threadIdx.x; j < end; j += kBlock) {
      const uint32_t w = a.adj_u[j];
      if (a.state[a.eid_u[j]] == kNone) atomicOr(&s_row[w >> 6], 1ull << (w & 63));
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < a.ws; i += kBlock) a.bits[uint64_t(u) * a.ws + i] = s_row[i];
    __syncthreads();
  }
}

// A dense core's frontier: one wave per (frontier edge, chunk of its rows); a
// chunk is 64 words, or 32 or 16 when the frontier is too small to give every
// wave of the grid an item. The common neighbours w of e = (u, v) in the chunk
// are the set bits of bits[u] & bits[v]; their count is scanned across the
// wave and the triangles are dealt out evenly, kDenseUnroll per lane per step,
// whatever words they sit in. The rows may still hold edges that died in the
// last round, which a step clears while the next frontier is walked: the
// partners' stamps tell them apart.
template <bool kEidm>
__device__ __forceinline__ void walk_dense(const StepArgs& a, const StepState& s, uint32_t* qn, uint32_t* qn_count) {
  __shared__ unsigned long long s_t[kBlock];
  __shared__ uint32_t s_inc[kBlock];
  __shared__ Out out;
  out_begin(out);
  const uint32_t* q = a.q[s.cur];
  const uint32_t cnt = s.cnt, ws = a.ws, r = s.round;
  const int32_t thr = s.thr;
  const int lane = lane64();
  const uint32_t wbase = threadIdx.x & ~uint32_t(kWave - 1);
  const uint64_t nw = uint64_t(gridDim.x) * (kBlock / kWave);
  uint32_t cw = kWave;  // words per chunk
  while (cw > 16 && uint64_t(cnt) * ((ws + cw - 1) / cw) < nw) cw >>= 1;
  const uint32_t nch = (ws + cw - 1) / cw;
  const uint64_t items = uint64_t(cnt) * nch;
  const EidOf<kEidm> eid_of{a.eidm, a.bits0, a.pref0, a.off_u, a.eid_u, a.nc, ws};
  for (uint64_t it = uint64_t(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave; it < items; it += nw) {
    const uint32_t qi = uint32_t(it / nch), ch = uint32_t(it - uint64_t(qi) * nch);
    const uint32_t x = q[qi], u = x >> 16, v = x & 0xFFFFu;
    const uint32_t e = eid_of(u, v);
    if (a.stats && ch == 0 && lane == 0) {  // measurement: the edge's merge work, d+(u) + d+(v)
      atomicAdd(&a.stats[0], (unsigned long long)(a.off_d[u + 1] - a.off_d[u] + a.off_d[v + 1] - a.off_d[v]));
      atomicAdd(&a.stats[1], 1ull);
    }
    const uint32_t i = ch * cw + uint32_t(lane);
    unsigned long long t = 0;
    if (uint32_t(lane) < cw && i < ws) t = a.bits[uint64_t(u) * ws + i] & a.bits[uint64_t(v) * ws + i];
    uint32_t inc = uint32_t(__popcll(t));
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o);
      if (lane >= o) inc += y;
    }
    const uint32_t total = __shfl(inc, kWave - 1);
    s_t[threadIdx.x] = t;
    s_inc[threadIdx.x] = inc;
    wave_sync();
    for (uint32_t j0 = 0; j0 < total; j0 += kWave * kDenseUnroll) {
      uint32_t w[kDenseUnroll], xa[kDenseUnroll], xb[kDenseUnroll], ma[kDenseUnroll], mb[kDenseUnroll];
#pragma unroll
      for (uint32_t k = 0; k < kDenseUnroll; ++k) {
        xa[k] = xb[k] = kNone;
        w[k] = 0;
        const uint32_t j = j0 + k * kWave + uint32_t(lane);
        if (j < total) {
          uint32_t lo = 0, hi = kWave - 1;  // owner: first lane whose inclusive count exceeds j
          while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_inc[wbase + mid] > j)
              hi = mid;
            else
              lo = mid + 1;
          }
          const unsigned long long tw = s_t[wbase + lo];
          const uint32_t b = select_bit(tw, j - (s_inc[wbase + lo] - uint32_t(__popcll(tw))));
          w[k] = ((ch * cw + lo) << 6) + b;
          xa[k] = eid_of(u, w[k]);
          xb[k] = eid_of(v, w[k]);
        }
      }
#pragma unroll
      for (uint32_t k = 0; k < kDenseUnroll; ++k) {
        ma[k] = xa[k] != kNone ? a.state[xa[k]] : 0u;
        mb[k] = xb[k] != kNone ? a.state[xb[k]] : 0u;
      }
      int32_t oa[kDenseUnroll], ob[kDenseUnroll];  // supports before the decrements
      bool da[kDenseUnroll], db[kDenseUnroll];
#pragma unroll
      for (uint32_t k = 0; k < kDenseUnroll; ++k) {
        charges(e, xa[k], xb[k], ma[k], mb[k], r, &da[k], &db[k]);
        oa[k] = da[k] ? atomicSub(&a.sup[xa[k]], 1) : 0;
        ob[k] = db[k] ? atomicSub(&a.sup[xb[k]], 1) : 0;
      }
#pragma unroll
      for (uint32_t k = 0; k < kDenseUnroll; ++k) {
        append_dead(a, out, da[k] && oa[k] == thr, xa[k], ends(u, w[k]), r + 1, thr, qn, qn_count);
        append_dead(a, out, db[k] && ob[k] == thr, xb[k], ends(v, w[k]), r + 1, thr, qn, qn_count);
      }
    }
    wave_sync();
  }
  out_end(out, qn, qn_count);
}

// The least support of the workgroup's live edges into got->min.
__device__ __forceinline__ void put_min(uint32_t best, StepCounters* mine) {
  __shared__ uint32_t s_min[kBlock / kWave];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = min(best, uint32_t(__shfl_xor(best, o)));
  if (lane64() == 0) s_min[threadIdx.x / kWave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kBlock / kWave; ++k) best = min(best, s_min[k]);
    if (best != kNone) atomicMin(&mine->min, best);
  }
}

// The live edges below the threshold become the next frontier (none on a
// peek), the least support among all live edges is found, and where half of
// the edge list is dead the rest is listed anew.
template <bool kDense>
__device__ __forceinline__ void look(const StepArgs& a, const StepState& s, uint32_t* qn, StepCounters* mine) {
  __shared__ uint32_t s_base[2];
  const uint32_t* list = s.listed ? a.live[s.buf] : nullptr;
  uint32_t* next = a.live[s.buf ^ 1u];
  const uint32_t r = s.round + 1;
  const int32_t thr = s.peek ? 0 : s.thr;  // no live edge has a support below 0
  // each thread takes two runs of four consecutive edges (16-byte loads) of
  // the whole set, or eight entries of the list, a workgroup apart
  constexpr uint32_t kItems = 8, kTile = kBlock * kItems;
  uint32_t best = kNone;
  for (uint32_t t0 = blockIdx.x * kTile; t0 < s.live; t0 += gridDim.x * kTile) {  // block-uniform
    uint32_t e[kItems], st[kItems];
    int32_t sp[kItems];
    uint32_t front = 0, keep = 0;
    if (!list && t0 + kTile <= s.live) {
      uint4 x[2];
      int4 y[2];
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        const uint32_t i = t0 + (h * kBlock + threadIdx.x) * 4;
        x[h] = *reinterpret_cast<const uint4*>(a.state + i);
        y[h] = *reinterpret_cast<const int4*>(a.sup + i);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) e[4 * h + k] = i + k;
      }
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        st[4 * h] = x[h].x, st[4 * h + 1] = x[h].y, st[4 * h + 2] = x[h].z, st[4 * h + 3] = x[h].w;
        sp[4 * h] = y[h].x, sp[4 * h + 1] = y[h].y, sp[4 * h + 2] = y[h].z, sp[4 * h + 3] = y[h].w;
      }
    } else {
#pragma unroll
      for (uint32_t k = 0; k < kItems; ++k) {
        const uint32_t i = t0 + k * kBlock + threadIdx.x;
        e[k] = i < s.live ? (list ? list[i] : i) : kNone;
      }
#pragma unroll
      for (uint32_t k = 0; k < kItems; ++k) {
        st[k] = e[k] != kNone ? a.state[e[k]] : 0u;
        sp[k] = e[k] != kNone ? a.sup[e[k]] : 0;
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < kItems; ++k)
      if (st[k] == kNone) {
        best = min(best, uint32_t(sp[k]));
        if (sp[k] < thr)
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
        stamp_dead(a, e[k], r, uint32_t(thr));
        qn[at++] = kDense ? ends(a.src[e[k]], a.dst[e[k]]) : e[k];
      }
      if (s.compact && ((keep >> k) & 1u)) next[kept++] = e[k];
    }
    __syncthreads();
  }
  put_min(best, mine);
}

// Exact supports of the live edges of a dense core, popcount(bits[u] &
// bits[v]), after a dropped frontier; those below the threshold become the
// next frontier. A workgroup stages one source row in LDS, its groups of G
// lanes take the row's out-edges.
template <int G>
__device__ __forceinline__ void recount(const StepArgs& a, const StepState& s, uint32_t* qn, StepCounters* mine) {
  __shared__ unsigned long long s_row[kDenseMaxWords];
  __shared__ Out out;
  out_begin(out);
  const uint32_t grp = threadIdx.x / G, ngrp = kBlock / G, lane = threadIdx.x % G;
  const uint32_t ws = a.ws, r = s.round + 1;
  const int32_t thr = s.thr;
  uint32_t best = kNone;
  for (uint32_t u = blockIdx.x; u < a.nc; u += gridDim.x) {  // workgroup-uniform
    const uint32_t e0 = a.off_d[u], e1 = a.off_d[u + 1];
    if (e0 == e1) continue;
    __syncthreads();  // the previous row's readers are done
    const unsigned long long* row = a.bits + uint64_t(u) * ws;
    for (uint32_t i = threadIdx.x; i < ws; i += kBlock) s_row[i] = row[i];
    __syncthreads();
    for (uint32_t b = e0; b < e1; b += ngrp) {  // workgroup-uniform: the appends take whole waves
      const uint32_t e = b + grp;
      const bool live = e < e1 && a.state[e] == kNone;
      uint32_t c = 0;
      if (live) {
        const unsigned long long* o = a.bits + uint64_t(a.dst[e]) * ws;
        for (uint32_t i = lane; i < ws; i += G) c += uint32_t(__popcll(s_row[i] & o[i]));
      }
      c = group_sum<G>(c);
      const bool mine_edge = live && lane == 0;
      if (mine_edge) {
        a.sup[e] = int32_t(c);
        best = min(best, c);
      }
      append_dead(a, out, mine_edge && int32_t(c) < thr, e, ends(u, mine_edge ? a.dst[e] : 0u), r, thr, qn,
                  &mine->frontier);
    }
  }
  out_end(out, qn, &mine->frontier);
  put_min(best, mine);
}

// The same by all pairs of rows on the matrix cores (kt_tile.h), a wave per 32
// x 32 of them. The rows' bits tell the live edges. A core of 3,150 vertices
// with 2 M live edges: 30 us instead of 110 to 135 by edge, so that frontiers
// of a few thousand edges are dropped too (whole solve 74.7 -> 61.9 ms).
constexpr uint32_t kPairRows = 32;
template <bool kEidm>
__device__ __forceinline__ void recount_pairs(const StepArgs& a, const StepState& s, uint32_t* qn,
                                              StepCounters* mine) {
  __shared__ Out out;
  out_begin(out);
  const EidOf<kEidm> eid_of{a.eidm, a.bits0, a.pref0, a.off_u, a.eid_u, a.nc, a.ws};
  const uint32_t nb = (a.nc + kPairRows - 1) / kPairRows, items = tile_items(nb), r = s.round + 1;
  const int32_t thr = s.thr;
  uint32_t best = kNone;
  for (uint32_t t = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; t < items;
       t += gridDim.x * (kBlock / kWave)) {  // wave-uniform
    uint32_t bi, bj;
    if (!tile_of(t, nb, &bi, &bj)) continue;
    Acc4 acc[2][2];
    count_tile<2, 2>(a.bits, a.nc, a.ws, bi * kPairRows, bj * kPairRows, acc);
    tile_edges<2, 2>(a.bits, a.nc, a.ws, bi * kPairRows, bj * kPairRows, acc, eid_of,
                     [&](bool live, uint32_t e, uint32_t u, uint32_t v, uint32_t c) {
                       if (live) {
                         a.sup[e] = int32_t(c);
                         best = min(best, c);
                       }
                       append_dead(a, out, live && int32_t(c) < thr, e, ends(u, v), r, thr, qn, &mine->frontier);
                     });
  }
  out_end(out, qn, &mine->frontier);
  put_min(best, mine);
}

// Step `it`. Bound on the short rounds that a search is mostly made of: a
// chain of dependent memory round trips of about 0.7 us each, past the L2
// (state and counters, queue, rows or list bounds, partner ids or entries,
// stamps, decrements, append), 7 to 9 us in all. One workgroup that walks
// short rounds in a loop, without launches, takes as long for each.
template <bool kDense, bool kEidm, int G>
__global__ __launch_bounds__(kBlock) void k_step(StepArgs a, StepRule rule, uint32_t it) {
  // (loaded together: one round trip)
  const StepState was = a.states[it & 1u];
  const StepCounters got = a.counters[(it + 2) % 3];
  if (was.phase == kStepDone || was.phase == kStepHost) {  // nothing to do
    if (blockIdx.x == 0 && threadIdx.x == 0) a.states[(it + 1) & 1u] = was;
    return;
  }
  const StepState s = next_step(was, got, rule);
  StepCounters* mine = &a.counters[it % 3];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.states[(it + 1) & 1u] = s;
    StepCounters* clear = &a.counters[(it + 1) % 3];
    clear->frontier = 0;
    clear->live = 0;
    clear->min = kNone;
  }
  uint32_t* qn = a.q[s.cur == 2 ? 0 : s.cur + 1];
  // the last walked frontier leaves the rows (a recount finds it gone)
  const bool rebuild = kDense && s.phase == kStepClear && s.cnt >= s.live / kRebuildShare;
  if (kDense && s.pend_cnt && (s.phase == kStepWalk || s.phase == kStepLook || s.phase == kStepClear) && !rebuild)
    clear_bits(a, a.q[s.pend], s.pend_cnt);
  if (s.phase == kStepWalk) {
    if (kDense)
      walk_dense<kEidm>(a, s, qn, &mine->frontier);
    else
      walk_lists(a, s, qn, &mine->frontier);
  } else if (s.phase == kStepLook) {
    look<kDense>(a, s, qn, mine);
  } else if (kDense && s.phase == kStepClear) {
    if (rebuild)
      rebuild_rows(a);
    else
      clear_bits(a, a.q[s.cur], s.cnt);
  } else if (kDense && s.phase == kStepRecount) {
    if (s.pairs)
      recount_pairs<kEidm>(a, s, qn, mine);
    else
      recount<G>(a, s, qn, mine);
  } else if (s.phase == kStepEmpty) {  // every edge still live dies at this threshold
    const uint32_t* list = s.listed ? a.live[s.buf] : nullptr;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < s.live; i += gridDim.x * kBlock) {
      const uint32_t e = list ? list[i] : i;
      if (a.state[e] == kNone) stamp_dead(a, e, s.round, uint32_t(s.thr));
    }
  }
}

__global__ void k_step_start(StepArgs a, StepState s) {
  if (threadIdx.x != 0) return;
  a.states[0] = s;
  for (int k = 0; k < 3; ++k) {
    a.counters[k].frontier = 0;
    a.counters[k].live = 0;
    a.counters[k].min = kNone;
  }
}

template <bool kEidm>
const void* dense_step(uint32_t ws) {
  switch (dense_lanes(ws)) {
    case 8: return reinterpret_cast<const void*>(&k_step<true, kEidm, 8>);
    case 16: return reinterpret_cast<const void*>(&k_step<true, kEidm, 16>);
    case 32: return reinterpret_cast<const void*>(&k_step<true, kEidm, 32>);
    default: return reinterpret_cast<const void*>(&k_step<true, kEidm, 64>);
  }
}

}  // namespace

// --------------------------------------------------------------- wrappers ---

void steps_start(const StepArgs& a, const StepState& first, hipStream_t s) {
  k_step_start<<<1, kWave, 0, s>>>(a, first);
}

void steps_run(const StepArgs& a, const StepRule& rule, uint32_t mc, uint32_t from, uint32_t count, hipStream_t s,
               hipEvent_t* ev) {
  if (rule.dense && a.ws > kDenseMaxWords) fail("dense core: rows longer than the LDS stage");
  const int grid = int(std::max<uint64_t>(1, std::min<uint64_t>((uint64_t(mc) + kGridEdges - 1) / kGridEdges, kStepGrid)));
  const void* fn = !rule.dense ? reinterpret_cast<const void*>(&k_step<false, false, 8>)
                   : a.eidm    ? dense_step<true>(a.ws)
                               : dense_step<false>(a.ws);
  for (uint32_t i = 0; i < count; ++i) {
    StepArgs arg = a;
    StepRule r = rule;
    uint32_t it = from + i;
    void* args[] = {&arg, &r, &it};
    if (ev)
      KT_HIP(hipExtLaunchKernel(fn, dim3(grid), dim3(kBlock), args, 0, s, ev[2 * i], ev[2 * i + 1], 0));
    else
      KT_HIP(hipLaunchKernel(fn, dim3(grid), dim3(kBlock), args, 0, s));
  }
}

}  // namespace kt
