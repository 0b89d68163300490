// Core numbers of a vertex-peel level by local updates on CDNA4.
//
// The reference finds the max core by galloping over thresholds, each peeled
// round by round (src/kc.cu:653-884). A vertex's core number is also the
// fixpoint of e(v) = the largest h such that at least h neighbours have
// e >= h, started from the degrees: every update only lowers e, in any order
// and from any mix of old and new values, and the fixpoint does not depend on
// that order. So a whole level converges in a few dozen launches over the
// whole GPU -- 7 to 70 on the graphs measured, against hundreds of dependent
// peel steps per threshold -- and yields every threshold's core at once.
#include <hip/hip_ext.h>

#include <algorithm>

#include "kt_device.h"
#include "kt_kernels.h"

namespace kt {
namespace {

constexpr uint32_t kCoreLdsBlock = 1024;  // workgroup of the kernels that keep a level's state in LDS
// Levels of one workgroup (34 KB of LDS); 8,192 row slots are 4 k edges.
constexpr uint32_t kCoreSmallN = 4096;
constexpr uint32_t kCoreSmallSlots = 1u << 13;
constexpr uint32_t kLightRegs = 16;   // row entries a lane keeps: a light row has at most 16 * G
constexpr uint32_t kMediumRegs = 64;  // a medium row, taken by one wave, at most 4096
constexpr uint32_t kHeavyRegs = 16;   // and a heavy row, taken by a workgroup of kCoreLdsBlock, 16,384 (kLds)
constexpr uint32_t kHistBins = 1024;  // heavy rows: bins per refinement of the new estimate

// est[v] = deg[v], or 0 (no core of at least `floor` >= 1 holds v) when that
// is below floor or v is not alive; the others are due. Rows of more than
// light_cap entries are listed: counts[0] medium ones, counts[1] heavy ones.
__global__ __launch_bounds__(kBlock) void k_core_est_init(const uint64_t* __restrict__ off,
                                                          const uint32_t* __restrict__ deg,
                                                          const uint32_t* __restrict__ lvl, uint32_t n,
                                                          uint32_t floor, uint32_t light_cap, uint32_t* est,
                                                          uint8_t* due, uint8_t* due_next, uint32_t* medium,
                                                          uint32_t* heavy, uint32_t* counts) {
  const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
  for (uint64_t base = uint64_t(blockIdx.x) * blockDim.x; base < n; base += stride) {  // block-uniform
    const uint64_t v = base + threadIdx.x;
    bool md = false, hv = false;
    if (v < n) {
      const uint32_t d = deg[v];
      const bool in = lvl[v] == kNone && d >= floor;
      const uint64_t len = off[v + 1] - off[v];
      hv = in && len > kMediumRegs * kWave;
      md = in && !hv && len > light_cap;
      est[v] = in ? d : 0u;
      due[v] = in;
      due_next[v] = 0;
    }
    wave_append<uint32_t>(md, uint32_t(v), medium, &counts[0]);
    wave_append<uint32_t>(hv, uint32_t(v), heavy, &counts[1]);
  }
}

// The new estimate of a heavy row by the whole workgroup (NT threads), from
// the row's estimates as read by each(f), which calls f(x) for every entry of
// this thread: counts the entries of at least e, and where they are too few
// narrows the new estimate down with histograms of the estimates in LDS,
// kHistBins bins at a time (one for e <= 1024). Where each() reads the row
// again every time, estimates may have fallen in between; an entry that was
// counted stays counted and one that was not is read at its new value, so the
// result is never below the vertex's core number, and the vertex is due again
// in the next sweep. Returns e when nothing changes; uniform.
template <uint32_t NT, class Each>
__device__ __forceinline__ uint32_t heavy_estimate(uint32_t e, Each each, uint32_t* s_hist, uint32_t* s_word) {
  static_assert(kHistBins % NT == 0, "each thread owns the same number of bins");
  constexpr uint32_t kPer = kHistBins / NT, kWaves = NT / kWave;
  const uint32_t tid = threadIdx.x;
  const int lane = lane64();
  uint32_t c = 0;
  each([&](uint32_t x) { c += x >= e; });
  c = wave_sum(c);
  if (lane == 0) s_word[2 + tid / kWave] = c;
  __syncthreads();
  uint32_t above = 0;  // entries of at least hi
  for (uint32_t k = 0; k < kWaves; ++k) above += s_word[2 + k];
  if (above >= e) {
    __syncthreads();  // s_word is read
    return e;
  }
  uint32_t lo = above, hi = e;  // the answer lies in [lo, hi)
  while (hi - lo > 1) {
    const uint32_t w = (hi - lo + kHistBins - 1) / kHistBins;
    for (uint32_t i = tid; i < kHistBins; i += NT) s_hist[i] = 0;
    __syncthreads();
    each([&](uint32_t x) {
      if (x >= lo && x < hi) atomicAdd(&s_hist[w == 1 ? x - lo : (x - lo) / w], 1u);
    });
    __syncthreads();
    // suffix sums over the bins: thread t owns kPer, from the top down
    const uint32_t top = kHistBins - 1 - tid * kPer;  // its highest bin
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) mine += s_hist[top - k];
    uint32_t inc = mine;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const uint32_t y = __shfl_up(inc, o);
      if (lane >= o) inc += y;
    }
    if (lane == kWave - 1) s_word[2 + tid / kWave] = inc;
    if (tid == 0) {
      s_word[0] = 0;  // 1 + the highest bin whose lower edge is reached
      s_word[1] = 0;  // entries of at least that bin's upper edge
    }
    __syncthreads();
    uint32_t up = above + inc - mine;  // entries of at least the upper edge of `top`
    for (uint32_t k = 0; k < kWaves; ++k)
      if (k < tid / kWave) up += s_word[2 + k];
    uint32_t run = up;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
      const uint32_t i = top - k, edge = lo + i * w;
      run += s_hist[i];  // entries of at least the bin's lower edge
      if (edge < hi && run >= edge) atomicMax(&s_word[0], i + 1);
    }
    __syncthreads();
    const uint32_t pick = s_word[0] ? s_word[0] - 1 : 0u;
    if (pick <= top && pick + kPer > top) {  // the picked bin's owner
      for (uint32_t i = top; i > pick; --i) up += s_hist[i];
      s_word[1] = up;
    }
    __syncthreads();
    above = s_word[1];
    lo = lo + pick * w;
    hi = min(hi, lo + w);
    __syncthreads();
  }
  return lo;
}

// The new estimate of a row of at most R * G entries held by G lanes: x[r] =
// the estimates (0: no entry). Returns e when it stands. Every lane of the
// wave must reach this; regs (wave-uniform): the entries of x in use by any
// lane; gmask: the lanes of this lane's group.
template <uint32_t R>
__device__ __forceinline__ uint32_t row_estimate(const uint32_t (&x)[R], uint32_t e, uint32_t regs,
                                                 unsigned long long gmask) {
  auto count = [&](uint32_t t) {  // row entries of at least t >= 1
    uint32_t c = 0;
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
      if (r < regs) c += uint32_t(__popcll(__ballot(x[r] >= t) & gmask));
    return c;
  };
  // the answer lies in [lo, hi): count(hi) < hi, and count(lo) >= lo since
  // at least count(e) entries are at least e
  const uint32_t ce = count(max(e, 1u));
  uint32_t lo = ce >= e ? e : ce, hi = ce >= e ? e + 1 : e;
  while (__ballot(hi - lo > 1)) {
    const uint32_t mid = lo + (hi - lo) / 2;
    const bool ok = count(max(mid, 1u)) >= mid;
    if (hi - lo > 1) (ok ? lo : hi) = mid;
  }
  return lo;
}

// Sweep it: every due vertex recomputes its estimate from its neighbours'. A
// vertex whose estimate falls from e to h is due in the next sweep (it may
// have read estimates that fell meanwhile), and so is every neighbour that it
// stops supporting: those with an estimate in (h, e]. A sweep in which
// nothing changes leaves the fixpoint. flags[it + 1] = 1 when an estimate
// changed; a sweep after one that changed nothing (flags[it] == 0) returns at
// once. Estimates below floor become 0.
//
// Bound: the gather of the neighbours' estimates. kLds: each workgroup copies
// the level's estimates into LDS as 16-bit words (a level of at most 65,536
// vertices; larger ones, of rows that repeat a neighbour, count as 65,535, and a
// level that ends with such a core is swept again from memory) and gathers there -- a wave's 64
// random words cost a few LDS cycles where the vector cache takes one line a
// cycle -- and sees its own updates at once. Rows of up to 16 * G entries are
// taken by G lanes, rows of up to 4096 by a wave, that keep the estimates in
// registers, so finding the new one costs ballots and no second read; longer
// rows by the workgroup.
template <int G, bool kLds>
__global__ __launch_bounds__(kLds ? kCoreLdsBlock : kBlock) void k_core_est_step(
    const uint64_t* __restrict__ off, const uint32_t* __restrict__ adj, uint32_t n, uint32_t floor, uint32_t* est,
    uint8_t* due, uint8_t* due_next, const uint32_t* __restrict__ medium, const uint32_t* __restrict__ heavy,
    const uint32_t* __restrict__ counts, uint32_t* flags, uint32_t it, unsigned long long* stats) {
  if (flags[it] == 0) return;
  constexpr uint32_t NT = kLds ? kCoreLdsBlock : kBlock;
  __shared__ uint32_t s_hist[kHistBins];
  __shared__ uint32_t s_word[2 + NT / kWave];
  extern __shared__ __align__(16) uint16_t s_est[];
  const uint32_t tid = threadIdx.x;
  if (kLds) {
    // four at a time: est lies on a 16-byte boundary with room for a multiple
    // of four words, s_est too
    auto low = [](uint32_t x) { return min(x, 65535u); };
    for (uint32_t i = tid; i < (n + 3) / 4; i += NT) {
      const uint4 q = reinterpret_cast<const uint4*>(est)[i];
      reinterpret_cast<uint2*>(s_est)[i] = make_uint2(low(q.x) | low(q.y) << 16, low(q.z) | low(q.w) << 16);
    }
    __syncthreads();
  }
  auto get = [&](uint32_t w) -> uint32_t { return kLds ? uint32_t(s_est[w]) : est[w]; };
  // one lane writes a vertex's new estimate
  auto settle = [&](uint32_t v, uint32_t h) {
    est[v] = h;
    if (kLds) s_est[v] = uint16_t(h);
    if (h) due_next[v] = 1;
    flags[it + 1] = 1;
  };
  auto counted = [&](uint64_t slots) {  // measurement: row slots walked, vertices taken
    atomicAdd(&stats[0], (unsigned long long)slots);
    atomicAdd(&stats[1], 1ull);
  };

  const uint32_t hc = counts[1];
  for (uint32_t i = blockIdx.x; i < hc; i += gridDim.x) {  // workgroup-uniform
    const uint32_t v = heavy[i];
    const bool mark = due[v] != 0;
    const uint32_t e = est[v];
    __syncthreads();
    if (!mark) continue;
    if (tid == 0) due[v] = 0;
    if (!e) continue;
    const uint64_t b = off[v];
    const uint64_t len = off[v + 1] - b;
    if (stats && tid == 0) counted(len);
    uint32_t h;
    // a workgroup of kCoreLdsBlock holds rows of up to 16,384 entries in
    // registers; one of kBlock would hold 4,096, which are no heavy rows yet
    bool held = false;
    if constexpr (kLds) held = len <= uint64_t(kHeavyRegs) * NT;
    if (kLds && held) {  // read once
      uint32_t x[kHeavyRegs];
#pragma unroll
      for (uint32_t r = 0; r < kHeavyRegs; ++r) {
        const uint32_t j = r * NT + tid;
        x[r] = j < len ? adj[b + j] : kNone;
      }
#pragma unroll
      for (uint32_t r = 0; r < kHeavyRegs; ++r) x[r] = x[r] != kNone ? get(x[r]) : 0u;
      h = heavy_estimate<NT>(
          e,
          [&](auto f) {
#pragma unroll
            for (uint32_t r = 0; r < kHeavyRegs; ++r)
              if (r * NT < len) f(x[r]);  // no entry: 0, below every bin and e
          },
          s_hist, s_word);
      if (h >= e) continue;
      if (h < floor) h = 0;
#pragma unroll
      for (uint32_t r = 0; r < kHeavyRegs; ++r)
        if (x[r] > h && x[r] <= e) due_next[adj[b + r * NT + tid]] = 1;
    } else {
      h = heavy_estimate<NT>(
          e,
          [&](auto f) {
#pragma unroll 8
            for (uint64_t j = tid; j < len; j += NT) f(get(adj[b + j]));
          },
          s_hist, s_word);
      if (h >= e) continue;
      if (h < floor) h = 0;
#pragma unroll 8
      for (uint64_t j = tid; j < len; j += NT) {
        const uint32_t w = adj[b + j], x = get(w);
        if (x > h && x <= e) due_next[w] = 1;
      }
    }
    if (tid == 0) settle(v, h);
  }

  const uint32_t wid = blockIdx.x * (NT / kWave) + tid / kWave, waves = gridDim.x * (NT / kWave);
  const uint32_t lane = tid & (kWave - 1);
  const uint32_t mc = counts[0];
  for (uint32_t i = wid; i < mc; i += waves) {  // wave-uniform
    const uint32_t v = medium[i];
    if (!due[v]) continue;
    if (lane == 0) due[v] = 0;
    const uint32_t e = est[v];
    if (!e) continue;
    const uint64_t b = off[v];
    const uint32_t len = __builtin_amdgcn_readfirstlane(uint32_t(off[v + 1] - b));
    const uint32_t regs = (len + kWave - 1) / kWave;
    uint32_t x[kMediumRegs];
#pragma unroll
    for (uint32_t r = 0; r < kMediumRegs; ++r) {
      x[r] = kNone;
      if (r < regs) {
        const uint32_t j = r * kWave + lane;
        if (j < len) x[r] = adj[b + j];
      }
    }
#pragma unroll
    for (uint32_t r = 0; r < kMediumRegs; ++r)
      if (r < regs) x[r] = x[r] != kNone ? get(x[r]) : 0u;
    uint32_t h = row_estimate(x, e, regs, ~0ull);
    if (stats && lane == 0) counted(len);
    if (h >= e) continue;
    if (h < floor) h = 0;
    if (lane == 0) settle(v, h);
#pragma unroll
    for (uint32_t r = 0; r < kMediumRegs; ++r)
      if (r < regs && x[r] > h && x[r] <= e) due_next[adj[b + r * kWave + lane]] = 1;
  }

  const uint32_t glane = tid % G;
  const uint32_t groups = gridDim.x * (NT / G);
  const uint32_t shift = lane / G * G;
  const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << shift;
  // wave-uniform trip count: every lane reaches the ballots
  for (uint32_t v0 = wid * (kWave / G); v0 < n; v0 += groups) {
    const uint32_t v = v0 + lane / G;
    uint32_t e = 0, len = 0;
    uint64_t b = 0;
    if (v < n && due[v]) {
      b = off[v];
      const uint64_t l = off[v + 1] - b;
      if (l <= uint64_t(kLightRegs) * G) {  // longer rows: taken above
        if (glane == 0) due[v] = 0;
        e = est[v];
        len = e ? uint32_t(l) : 0u;
      }
    }
    if (!__ballot(e != 0)) continue;
    uint32_t w[kLightRegs], x[kLightRegs];
#pragma unroll
    for (uint32_t r = 0; r < kLightRegs; ++r) {
      const uint32_t j = r * G + glane;
      w[r] = j < len ? adj[b + j] : kNone;
    }
#pragma unroll
    for (uint32_t r = 0; r < kLightRegs; ++r) x[r] = w[r] != kNone ? get(w[r]) : 0u;
    uint32_t h = row_estimate(x, e, kLightRegs, gmask);
    if (stats && e && glane == 0) counted(len);
    if (h < e) {
      if (h < floor) h = 0;
      if (glane == 0) settle(v, h);
#pragma unroll
      for (uint32_t r = 0; r < kLightRegs; ++r)
        if (x[r] > h && x[r] <= e) due_next[w[r]] = 1;
    }
  }
}

// A small level in one launch and one workgroup: rows and estimates in LDS,
// sweeps over every vertex until one changes nothing, then the results (lvl
// as k_core_est_apply writes it, deg of the max core's vertices = their degree
// in it). out[0] = the largest core number, out[1] = 1 when the sweeps
// converged within `cap`; else est and due (every vertex of an estimate) are
// written for k_core_finish. A sweep from LDS takes less than launching one.
template <int G>
__global__ __launch_bounds__(kCoreLdsBlock) void k_core_small(const uint64_t* __restrict__ off,
                                                              const uint32_t* __restrict__ adj, uint32_t n,
                                                              uint32_t floor, uint32_t cap, uint32_t* lvl,
                                                              uint32_t* deg, uint32_t* est, uint8_t* due,
                                                              uint32_t* out, unsigned long long* stats) {
  __shared__ uint16_t s_adj[kCoreSmallSlots];
  __shared__ uint16_t s_off[kCoreSmallN + 1];  // at most kCoreSmallSlots
  __shared__ uint16_t s_e[kCoreSmallN];
  __shared__ uint32_t s_changed, s_top;
  const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1);
  const uint32_t glane = tid % G, shift = lane / G * G;
  const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << shift;
  for (uint32_t v = tid; v <= n; v += kCoreLdsBlock) {
    s_off[v] = uint16_t(off[v]);  // row 0 starts at 0
    if (v < n) {
      const uint32_t d = deg[v];
      s_e[v] = uint16_t(lvl[v] == kNone && d >= floor ? d : 0u);
    }
  }
  const uint32_t slots = uint32_t(off[n]);
  for (uint32_t j = tid; j < slots; j += kCoreLdsBlock) s_adj[j] = uint16_t(adj[j]);
  if (tid == 0) {
    s_top = 0;
    if (stats) {  // measurement: row slots and vertices
      atomicAdd(&stats[0], (unsigned long long)slots);
      atomicAdd(&stats[1], (unsigned long long)n);
    }
  }
  for (uint32_t sweep = 0;; ++sweep) {
    __syncthreads();
    if (tid == 0) s_changed = 0;
    __syncthreads();
    for (uint32_t v0 = tid / kWave * (kWave / G); v0 < n; v0 += kCoreLdsBlock / G) {  // wave-uniform
      const uint32_t v = v0 + lane / G;
      const uint32_t e = v < n ? s_e[v] : 0u;
      if (!__ballot(e != 0)) continue;
      const uint32_t b = e ? s_off[v] : 0u, len = e ? s_off[v + 1] - b : 0u;
      // entries of the row of at least t >= 1, per group
      auto count = [&](uint32_t t) {
        uint32_t c = 0;
        for (uint32_t j = glane; __ballot(j < len); j += G)
          c += uint32_t(__popcll(__ballot(j < len && s_e[s_adj[b + j]] >= t) & gmask));
        return c;
      };
      const uint32_t ce = count(max(e, 1u));
      uint32_t lo = ce >= e ? e : ce, hi = ce >= e ? e + 1 : e;  // as row_estimate
      while (__ballot(hi - lo > 1)) {
        const uint32_t mid = lo + (hi - lo) / 2;
        const bool ok = count(max(mid, 1u)) >= mid;
        if (hi - lo > 1) (ok ? lo : hi) = mid;
      }
      if (lo < e && glane == 0) {
        s_e[v] = uint16_t(lo < floor ? 0u : lo);
        s_changed = 1;
      }
    }
    __syncthreads();
    if (!s_changed) break;
    if (sweep >= cap) {
      for (uint32_t v = tid; v < n; v += kCoreLdsBlock) {
        est[v] = s_e[v];
        due[v] = s_e[v] != 0;
      }
      if (tid == 0) out[0] = out[1] = 0;
      return;
    }
  }
  uint32_t m = 0;
  for (uint32_t v = tid; v < n; v += kCoreLdsBlock) m = max(m, uint32_t(s_e[v]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, uint32_t(__shfl_xor(m, o)));
  if (lane == 0) atomicMax(&s_top, m);
  __syncthreads();
  const uint32_t top = s_top;
  for (uint32_t v = tid; v < n; v += kCoreLdsBlock) {
    const uint32_t e = s_e[v];
    if (top == 0) {
      lvl[v] = floor;
    } else if (e < top) {
      if (lvl[v] == kNone) lvl[v] = e ? e + 1 : floor;
    } else {
      uint32_t c = 0;
      for (uint32_t j = s_off[v]; j < s_off[v + 1]; ++j) c += s_e[s_adj[j]] == top;
      deg[v] = c;
    }
  }
  if (tid == 0) {
    out[0] = top;
    out[1] = 1;
  }
}

// What is left of a level of at most 65,536 vertices whose sweeps make slow
// progress (a core that unravels along paths: each sweep moves the ends by one
// vertex), by one workgroup, estimates and due marks in LDS: a sweep takes a
// list of due vertices, so it costs what they cost and two barriers, not a
// launch; where they are few, one wave runs sweeps on end with no barrier.
//
// From sweep `all` on only vertices of the largest estimate T are taken. Once
// none of them is due, each has T neighbours among them: they are the max core
// (no core is larger than the estimates), and the other estimates are left as
// the upper bounds they are.
//
// out[0] = the largest estimate; out[1] = 1: every estimate is a core number,
// 2: the largest is, 0: not done after `cap` sweeps.
// Bound on a sweep's chain of dependent accesses (row bounds, entries, some ten
// to LDS): 3 us where one vertex is due, as a path's 10 k vertices take 15 ms.
constexpr uint32_t kOneQueue = 4096;  // listed vertices of one sweep (the others wait for a later one)
template <int G>
__global__ __launch_bounds__(kCoreLdsBlock) void k_core_finish(const uint64_t* __restrict__ off,
                                                               const uint32_t* __restrict__ adj, uint32_t n,
                                                               uint32_t floor, uint32_t all, uint32_t cap,
                                                               uint32_t* est, const uint8_t* __restrict__ due,
                                                               uint32_t* out) {
  extern __shared__ __align__(16) uint32_t s_due[];  // marks: listed, or waiting
  __shared__ uint16_t s_q[2][kOneQueue];
  __shared__ uint32_t s_n[2];  // listed (past kOneQueue: waiting)
  __shared__ uint32_t s_top, s_cnt, s_sweep;
  constexpr uint32_t kSolo = 4 * (kWave / G);  // due vertices that one wave takes alone
  const uint32_t words = (n + 31) / 32;
  uint16_t* s_e = reinterpret_cast<uint16_t*>(s_due + words);
  const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
  const uint32_t glane = tid % G, shift = lane / G * G;
  const unsigned long long gmask = (G == 64 ? ~0ull : ((1ull << G) - 1ull)) << shift;
  if (tid == 0) s_n[0] = 0;
  __syncthreads();
  for (uint32_t v0 = wid * kWave; v0 < n; v0 += kCoreLdsBlock) {  // at most kOneQueue are due
    const uint32_t v = v0 + lane;
    if (v < n) s_e[v] = uint16_t(min(est[v], 65535u));
    const unsigned long long mask = __ballot(v < n && due[v] != 0);
    uint32_t at = 0;
    if (lane == 0 && mask) at = atomicAdd(&s_n[0], uint32_t(__popcll(mask)));
    at = __shfl(at, 0) + uint32_t(__popcll(mask & ((1ull << lane) - 1ull)));
    if (((mask >> lane) & 1ull) && at < kOneQueue) s_q[0][at] = uint16_t(v);
    if (lane % 32 == 0 && v < n) s_due[v >> 5] = uint32_t(mask >> lane);
  }
  __syncthreads();

  // the largest estimate and (counted) how many vertices have it
  auto find_top = [&](bool counted) {
    if (tid == 0) s_top = s_cnt = 0;
    __syncthreads();
    uint32_t m = 0;
    for (uint32_t v = tid; v < n; v += kCoreLdsBlock) m = max(m, uint32_t(s_e[v]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, uint32_t(__shfl_xor(m, o)));
    if (lane == 0) atomicMax(&s_top, m);
    __syncthreads();
    m = s_top;
    if (!counted) return m;
    uint32_t c = 0;
    for (uint32_t v = tid; v < n; v += kCoreLdsBlock) c += s_e[v] == m;
    c = wave_sum(c);
    if (lane == 0 && c) atomicAdd(&s_cnt, c);
    __syncthreads();
    return m;
  };
  // list `cur` from the marks, of vertices of estimate `only` (0: any); true
  // when there are marks besides
  constexpr uint32_t kWords = 2;  // due words a thread owns
  auto list_due = [&](uint32_t cur, uint32_t only) {
    uint32_t take[kWords], mine = 0;
    bool other = false;
#pragma unroll
    for (uint32_t h = 0; h < kWords; ++h) {
      const uint32_t w = h * kCoreLdsBlock + tid;
      uint32_t x = w < words ? s_due[w] : 0u;
      if (only)
        for (uint32_t y = x; y; y &= y - 1)
          if (s_e[w * 32 + __ffs(int(y)) - 1] != only) {
            x &= ~(y & (0u - y));
            other = true;
          }
      take[h] = x;
      mine += uint32_t(__popc(x));
    }
    uint32_t total;
    uint32_t at = block_exclusive_scan<kCoreLdsBlock>(mine, &total);
#pragma unroll
    for (uint32_t h = 0; h < kWords; ++h)
      for (uint32_t y = take[h]; y && at < kOneQueue; y &= y - 1, ++at)
        s_q[cur][at] = uint16_t((h * kCoreLdsBlock + tid) * 32 + __ffs(int(y)) - 1);
    if (tid == 0) s_n[cur] = total;
    return __syncthreads_or(other) != 0 || total > kOneQueue;
  };

  uint32_t top = 0;  // not 0: only vertices of this estimate
  // a list's marks go before its sweep reads
  auto unmark = [&](uint32_t cur, uint32_t count, uint32_t first, uint32_t step) {
    for (uint32_t i = first; i < count; i += step) {
      const uint32_t v = s_q[cur][i];
      atomicAnd(&s_due[v >> 5], ~(1u << (v & 31)));
    }
  };
  // a wave's entries of the list, first on and every step; a fall marks and
  // lists vertices for the next sweep
  auto sweep_list = [&](uint32_t cur, uint32_t count, uint32_t first, uint32_t step) {
    auto mark = [&](uint32_t w, bool listed) {
      const uint32_t bit = 1u << (w & 31);
      if (!(atomicOr(&s_due[w >> 5], bit) & bit) && listed) {
        const uint32_t at = atomicAdd(&s_n[cur ^ 1u], 1u);
        if (at < kOneQueue) s_q[cur ^ 1u][at] = uint16_t(w);
      }
    };
    for (uint32_t i0 = first; i0 < count; i0 += step) {  // wave-uniform
      const uint32_t i = i0 + lane / G;
      const uint32_t v = i < count ? s_q[cur][i] : 0u, e = i < count ? s_e[v] : 0u;
      uint64_t b = 0;
      uint32_t len = 0;
      if (e) {
        b = off[v];
        len = uint32_t(off[v + 1] - b);
      }
      auto settle = [&](uint32_t h) {
        s_e[v] = uint16_t(h);
        if (h) mark(v, !top);
        if (top && e == top) atomicSub(&s_cnt, 1u);
      };
      auto supported = [&](uint32_t w, uint32_t x, uint32_t h) {
        if (x > h && x <= e) mark(w, !top || x == top);
      };
      if (!__ballot(len > G)) {  // a lane an entry
        const uint32_t w = glane < len ? adj[b + glane] : kNone;
        const uint32_t x[1] = {w != kNone ? s_e[w] : 0u};
        uint32_t h = row_estimate(x, e, 1, gmask);
        if (h < e) {
          if (h < floor) h = 0;
          if (glane == 0) settle(h);
          if (w != kNone) supported(w, x[0], h);
        }
      } else if (!__ballot(len > kLightRegs * G)) {
        uint32_t w[kLightRegs], x[kLightRegs];
#pragma unroll
        for (uint32_t r = 0; r < kLightRegs; ++r) {
          const uint32_t j = r * G + glane;
          w[r] = j < len ? adj[b + j] : kNone;
        }
#pragma unroll
        for (uint32_t r = 0; r < kLightRegs; ++r) x[r] = w[r] != kNone ? s_e[w[r]] : 0u;
        uint32_t h = row_estimate(x, e, kLightRegs, gmask);
        if (h < e) {
          if (h < floor) h = 0;
          if (glane == 0) settle(h);
#pragma unroll
          for (uint32_t r = 0; r < kLightRegs; ++r)
            if (w[r] != kNone) supported(w[r], x[r], h);
        }
      } else {  // a long row in the wave: read anew for every count
        auto count_row = [&](uint32_t t) {  // entries of the row of at least t >= 1, per group
          uint32_t c = 0;
          for (uint32_t j = glane; __ballot(j < len); j += G)
            c += uint32_t(__popcll(__ballot(j < len && s_e[adj[b + j]] >= t) & gmask));
          return c;
        };
        const uint32_t ce = count_row(max(e, 1u));
        uint32_t lo = ce >= e ? e : ce, hi = ce >= e ? e + 1 : e;  // as row_estimate
        while (__ballot(hi - lo > 1)) {
          const uint32_t mid = lo + (hi - lo) / 2;
          const bool ok = count_row(max(mid, 1u)) >= mid;
          if (hi - lo > 1) (ok ? lo : hi) = mid;
        }
        if (lo < e) {
          const uint32_t h = lo < floor ? 0u : lo;
          if (glane == 0) settle(h);
          for (uint32_t j = glane; j < len; j += G) {
            const uint32_t w = adj[b + j];
            supported(w, s_e[w], h);
          }
        }
      }
    }
  };

  uint32_t cur = 0, done = 0, sweep = 0;
  bool left = s_n[0] > kOneQueue;  // there are marks that are not listed
  while (sweep < cap) {            // (a barrier follows the last writes of s_n and s_cnt)
    if (top ? s_cnt == 0 : sweep >= all && s_n[cur]) {
      __syncthreads();
      top = find_top(true);
      if (top == 0) {
        done = 1;
        break;
      }
      left = list_due(cur, top);
    } else if (s_n[cur] > kOneQueue) {
      left = list_due(cur, top);
    }
    uint32_t count = s_n[cur];
    if (count == 0) {
      if (top || left) left = list_due(cur, top);
      if (s_n[cur]) continue;
      done = top && left ? 2u : 1u;
      break;
    }
    count = min(count, kOneQueue);
    if (count <= kSolo) {
      if (wid == 0) {
        for (;;) {
          if (lane == 0) s_n[cur ^ 1u] = 0;
          unmark(cur, count, lane, kWave);
          wave_sync();
          sweep_list(cur, count, 0, kWave / G);
          wave_sync();
          cur ^= 1u;
          ++sweep;
          count = s_n[cur];
          if (count == 0 || count > kSolo || sweep >= cap || (top ? s_cnt == 0 : sweep >= all)) break;
        }
        if (lane == 0) s_sweep = sweep * 2 + cur;
      }
      __syncthreads();
      sweep = s_sweep / 2;
      cur = s_sweep & 1u;
      __syncthreads();
      continue;
    }
    if (tid == 0) s_n[cur ^ 1u] = 0;
    unmark(cur, count, tid, kCoreLdsBlock);
    __syncthreads();
    sweep_list(cur, count, wid * (kWave / G), kCoreLdsBlock / G);
    __syncthreads();
    cur ^= 1u;
    ++sweep;
  }
  __syncthreads();
  top = find_top(false);
  if (tid == 0) {
    out[0] = top;
    out[1] = done;
  }
  for (uint32_t v = tid; v < n; v += kCoreLdsBlock) est[v] = s_e[v];
}

// Alive vertices (the bitmap) with fewer than k alive neighbours are stamped
// removed at k; *alive += the others. One wave per vertex, which stops
// reading its row once k are found; the bitmap lies in LDS (kLds) or in L2.
template <bool kLds>
__global__ __launch_bounds__(kCoreLdsBlock) void k_core_prune(const uint64_t* __restrict__ off,
                                                              const uint32_t* __restrict__ adj,
                                                              const uint32_t* __restrict__ bits, uint32_t n,
                                                              uint32_t k, uint32_t* __restrict__ lvl,
                                                              uint32_t* alive) {
  extern __shared__ uint32_t s_bits[];
  const uint32_t words = (n + 31) / 32;
  if (kLds) {
    for (uint32_t i = threadIdx.x; i < words; i += kCoreLdsBlock) s_bits[i] = bits[i];
    __syncthreads();
  }
  auto is_alive = [&](uint32_t w) { return ((kLds ? s_bits[w >> 5] : bits[w >> 5]) >> (w & 31)) & 1u; };
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wid = blockIdx.x * (kCoreLdsBlock / kWave) + threadIdx.x / kWave;
  const uint32_t waves = gridDim.x * (kCoreLdsBlock / kWave);
  constexpr uint32_t kUnroll = 4;
  uint32_t kept = 0;
  for (uint32_t v = wid; v < n; v += waves) {  // wave-uniform
    if (!is_alive(v)) continue;
    const uint64_t end = off[v + 1];
    uint32_t c = 0;
    for (uint64_t j0 = off[v]; j0 < end && c < k; j0 += kWave * kUnroll) {
      uint32_t w[kUnroll];
#pragma unroll
      for (uint32_t u = 0; u < kUnroll; ++u) {
        const uint64_t j = j0 + u * kWave + lane;
        w[u] = j < end ? adj[j] : kNone;
      }
#pragma unroll
      for (uint32_t u = 0; u < kUnroll; ++u) c += uint32_t(__popcll(__ballot(w[u] != kNone && is_alive(w[u]))));
    }
    if (c >= k)
      ++kept;
    else if (lane == 0)
      lvl[v] = k;
  }
  if (lane == 0 && kept) atomicAdd(alive, kept);
}

// out[0] = the largest estimate, out[1] = the vertices due (both start at 0).
__global__ __launch_bounds__(kBlock) void k_core_est_max(const uint32_t* __restrict__ est,
                                                         const uint8_t* __restrict__ due, uint32_t n,
                                                         uint32_t* out) {
  uint32_t m = 0, c = 0;
  for (uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < n; v += uint64_t(gridDim.x) * blockDim.x) {
    m = max(m, est[v]);
    c += due[v] != 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, uint32_t(__shfl_xor(m, o)));
  c = wave_sum(c);
  if (lane64() == 0 && m) atomicMax(&out[0], m);
  if (lane64() == 0 && c) atomicAdd(&out[1], c);
}

// Of the vertices alive before, those of the largest core number (*top) stay
// alive, the others carry the lowest threshold that removes them.
__global__ __launch_bounds__(kBlock) void k_core_est_apply(const uint32_t* __restrict__ est, uint32_t n,
                                                           uint32_t floor, const uint32_t* __restrict__ top,
                                                           uint32_t* __restrict__ lvl) {
  const uint32_t t = *top;
  for (uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < n; v += uint64_t(gridDim.x) * blockDim.x) {
    const uint32_t e = est[v];
    if (e < t && lvl[v] == kNone) lvl[v] = e ? e + 1 : floor;
  }
}

__global__ __launch_bounds__(kBlock) void k_core_est_prune(const uint32_t* __restrict__ est, uint32_t n, uint32_t k,
                                                           uint32_t* __restrict__ lvl, uint32_t* removed) {
  uint32_t c = 0;
  for (uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < n; v += uint64_t(gridDim.x) * blockDim.x)
    if (est[v] < k && lvl[v] == kNone) {
      lvl[v] = k;
      ++c;
    }
  c = wave_sum(c);
  if (lane64() == 0 && c) atomicAdd(removed, c);
}

__global__ __launch_bounds__(kBlock) void k_core_clear_removed(const uint32_t* __restrict__ lvl, uint32_t n,
                                                               uint32_t* __restrict__ deg) {
  for (uint64_t v = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < n; v += uint64_t(gridDim.x) * blockDim.x)
    if (lvl[v] != kNone) deg[v] = 0;
}

}  // namespace

// --------------------------------------------------------------- wrappers ---

// Gather from LDS up to this many vertices (16-bit estimates: 128 KB), on
// one workgroup per CU.
constexpr uint32_t kCoreLdsN = 65536;
constexpr int kCoreLdsGrid = 256;

bool core_est_fits_lds(uint32_t n) { return n <= kCoreLdsN; }

void core_est_init(const CoreEst& a, const uint32_t* deg, const uint32_t* lvl, int lanes, hipStream_t s) {
  fill_u32(a.counts, 2, 0, s);
  k_core_est_init<<<std::min(grid_for(a.n), 4096), kBlock, 0, s>>>(a.off, deg, lvl, a.n, a.floor,
                                                                   kLightRegs * uint32_t(lanes), a.est, a.due,
                                                                   a.due_next, a.medium, a.heavy, a.counts);
}

template <bool kLds>
static const void* core_est_kernel(int lanes) {
  switch (lanes) {
    case 8: return reinterpret_cast<const void*>(&k_core_est_step<8, kLds>);
    case 16: return reinterpret_cast<const void*>(&k_core_est_step<16, kLds>);
    case 32: return reinterpret_cast<const void*>(&k_core_est_step<32, kLds>);
    default: return reinterpret_cast<const void*>(&k_core_est_step<64, kLds>);
  }
}

void core_est_steps(CoreEst* a, int lanes, uint32_t count, hipStream_t s, unsigned long long* stats,
                    hipEvent_t* ev) {
  fill_u32(a->flags, 1, 1, s);
  fill_u32(a->flags + 1, count, 0, s);
  const bool lds = a->lds;
  const void* fn = lds ? core_est_kernel<true>(lanes) : core_est_kernel<false>(lanes);
  const int block = lds ? int(kCoreLdsBlock) : kBlock;
  const int grid = std::min(grid_for(uint64_t(a->n) * uint64_t(lanes), block), lds ? kCoreLdsGrid : 4096);
  const size_t bytes = lds ? sizeof(uint16_t) * ((size_t(a->n) + 3) & ~size_t(3)) : 0;
  for (uint32_t it = 0; it < count; ++it) {
    if (it) stats = nullptr;
    void* args[] = {&a->off,    &a->adj,   &a->n,      &a->floor, &a->est, &a->due, &a->due_next,
                    &a->medium, &a->heavy, &a->counts, &a->flags, &it,     &stats};
    if (ev)
      KT_HIP(hipExtLaunchKernel(fn, dim3(grid), dim3(block), args, bytes, s, ev[2 * it], ev[2 * it + 1], 0));
    else
      KT_HIP(hipLaunchKernel(fn, dim3(grid), dim3(block), args, bytes, s));
    std::swap(a->due, a->due_next);
  }
}

constexpr uint32_t kSmallSweeps = 16;     // most small levels take fewer; past them the work is in few vertices
constexpr uint32_t kFinishAll = 64;       // sweeps over all due vertices
constexpr uint32_t kFinishCap = 1u << 16;

bool core_small_fits(uint32_t n, uint64_t slots) { return n <= kCoreSmallN && slots <= kCoreSmallSlots; }
void core_small(const CoreEst& a, uint32_t* lvl, uint32_t* deg, int lanes, uint32_t* out, hipStream_t s,
                unsigned long long* stats, hipEvent_t* ev) {
  const void* fn = lanes == 64   ? reinterpret_cast<const void*>(&k_core_small<64>)
                   : lanes == 32 ? reinterpret_cast<const void*>(&k_core_small<32>)
                   : lanes == 16 ? reinterpret_cast<const void*>(&k_core_small<16>)
                                 : reinterpret_cast<const void*>(&k_core_small<8>);
  CoreEst e = a;
  uint32_t cap = kSmallSweeps;
  void* args[] = {&e.off, &e.adj, &e.n, &e.floor, &cap, &lvl, &deg, &e.est, &e.due, &out, &stats};
  if (ev)
    KT_HIP(hipExtLaunchKernel(fn, dim3(1), dim3(kCoreLdsBlock), args, 0, s, ev[0], ev[1], 0));
  else
    KT_HIP(hipLaunchKernel(fn, dim3(1), dim3(kCoreLdsBlock), args, 0, s));
}

// Up to two rounds of its groups of lanes (256 vertices of short rows): a sweep
// then takes about as long as launching one, 6 us, or half of that
bool core_finish_fits(uint32_t n, uint32_t due, int lanes) {
  return n <= kCoreLdsN && due <= 2 * kCoreLdsBlock / uint32_t(lanes);
}
void core_finish(const CoreEst& e, int lanes, uint32_t* out, hipStream_t s) {
  const size_t bytes = sizeof(uint32_t) * ((e.n + 31) / 32) + sizeof(uint16_t) * size_t(e.n);
  auto launch = [&](auto kernel) {
    kernel<<<1, kCoreLdsBlock, bytes, s>>>(e.off, e.adj, e.n, e.floor, kFinishAll, kFinishCap, e.est, e.due, out);
  };
  switch (lanes) {
    case 8: launch(k_core_finish<8>); break;
    case 16: launch(k_core_finish<16>); break;
    case 32: launch(k_core_finish<32>); break;
    default: launch(k_core_finish<64>); break;
  }
}

void core_prune(const uint64_t* off, const uint32_t* adj, const uint32_t* bits, uint32_t n, uint32_t k, uint32_t* lvl,
                uint32_t* alive, hipStream_t s) {
  if (!n) return;
  const size_t bytes = sizeof(uint32_t) * ((size_t(n) + 31) / 32);
  const int grid = std::min(grid_for(uint64_t(n) * kWave, kCoreLdsBlock), 512);
  if (bytes <= 65536)  // two workgroups per CU
    k_core_prune<true><<<grid, kCoreLdsBlock, bytes, s>>>(off, adj, bits, n, k, lvl, alive);
  else
    k_core_prune<false><<<grid, kCoreLdsBlock, 0, s>>>(off, adj, bits, n, k, lvl, alive);
}

void core_est_max(const CoreEst& a, uint32_t* out, hipStream_t s) {
  fill_u32(out, 2, 0, s);
  k_core_est_max<<<std::min(grid_for(a.n), 1024), kBlock, 0, s>>>(a.est, a.due, a.n, out);
}

void core_est_prune(const uint32_t* est, uint32_t n, uint32_t k, uint32_t* lvl, uint32_t* removed, hipStream_t s) {
  if (n) k_core_est_prune<<<std::min(grid_for(n), 1024), kBlock, 0, s>>>(est, n, k, lvl, removed);
}
void core_clear_removed(const uint32_t* lvl, uint32_t n, uint32_t* deg, hipStream_t s) {
  if (n) k_core_clear_removed<<<std::min(grid_for(n), 4096), kBlock, 0, s>>>(lvl, n, deg);
}
void core_est_apply(const CoreEst& a, const uint32_t* top, uint32_t* lvl, hipStream_t s) {
  k_core_est_apply<<<std::min(grid_for(a.n), 4096), kBlock, 0, s>>>(a.est, a.n, a.floor, top, lvl);
}

}  // namespace kt
