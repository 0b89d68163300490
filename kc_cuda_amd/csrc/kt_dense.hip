// Dense core views built through their bit-matrix rows, on CDNA4.
//
// The reference counts out-degrees, fills and sorts the oriented rows and
// transposes them into undirected rows with edge ids (src/kc.cu:1311-1673).
// On a core dense enough for bit-matrix rows those rows come first, in rank
// order: their set bits are the sorted neighbours, and a popcount prefix tells
// the place of every neighbour in its row, so the oriented and undirected rows
// and the edge ids are read off them without a sort or a transpose.
//
// What bounds it: launches and waits on small cores (7 launches and 2 waits
// where counting, sorting and transposing the rows took 29 and 3), the reads
// of the core's rows in the level (through `to`) and the nc^2 entry edge-id
// matrix on large ones. Measured on whole solves, same process and inputs:
// 40 vertices 0.89 -> 0.73 ms, 16k edges 0.97 -> 0.85 ms, 200k edges 3.07 ->
// 2.86 ms, R-MAT scale 22 (a core of 8.8k vertices) 16.0 -> 14.1 ms. The old
// route is left for sorted-row cores, and for rows that are no simple graph.
#include <algorithm>

#include "kt_device.h"
#include "kt_kernels.h"
#include "kt_tile.h"

namespace kt {
namespace {

constexpr uint32_t kMaxRowWords = 1024;  // nc <= 65536

// Row r (the vertex inv[r] of the level): the ranks of its neighbours in the
// core as bits, exclusive popcount prefixes per word, and its degree and
// out-degree (neighbours of a higher rank). One workgroup per row, its bits in
// LDS.
__global__ __launch_bounds__(kBlock) void k_rank_rows(const uint64_t* __restrict__ off,
                                                      const uint32_t* __restrict__ adj,
                                                      const uint32_t* __restrict__ to,
                                                      const uint32_t* __restrict__ inv, uint32_t nc, uint32_t ws,
                                                      unsigned long long* bits0, unsigned long long* bits,
                                                      uint32_t* pref0, uint32_t* du, uint32_t* dout) {
  __shared__ unsigned long long s_row[kMaxRowWords];
  __shared__ uint32_t s_in;
  constexpr uint32_t kUnroll = 4;
  for (uint32_t r = blockIdx.x; r < nc; r += gridDim.x) {  // workgroup-uniform
    for (uint32_t i = threadIdx.x; i < ws; i += kBlock) s_row[i] = 0;
    __syncthreads();
    const uint32_t v = inv[r];
    const uint64_t end = off[v + 1];
    for (uint64_t j0 = off[v] + threadIdx.x; j0 < end; j0 += kBlock * kUnroll) {
      uint32_t w[kUnroll];
#pragma unroll
      for (uint32_t k = 0; k < kUnroll; ++k) w[k] = j0 + k * kBlock < end ? adj[j0 + k * kBlock] : kNone;
#pragma unroll
      for (uint32_t k = 0; k < kUnroll; ++k) w[k] = w[k] != kNone ? to[w[k]] : kNone;
#pragma unroll
      for (uint32_t k = 0; k < kUnroll; ++k)
        if (w[k] != kNone) atomicOr(&s_row[w[k] >> 6], 1ull << (w[k] & 63));
    }
    __syncthreads();
    uint32_t carry = 0;
    for (uint32_t c0 = 0; c0 < ws; c0 += kBlock) {
      const uint32_t i = c0 + threadIdx.x;
      const unsigned long long x = i < ws ? s_row[i] : 0ull;
      uint32_t total;
      const uint32_t before = carry + block_exclusive_scan(uint32_t(__popcll(x)), &total);
      if (i < ws) {
        const uint64_t at = uint64_t(r) * ws + i;
        bits0[at] = x;
        bits[at] = x;
        pref0[at] = before;
        if (i == r >> 6) s_in = before + uint32_t(__popcll(x & ((1ull << (r & 63)) - 1ull)));
      }
      carry += total;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      du[r] = carry;
      dout[r] = carry - s_in;
    }
  }
}

// Exclusive sums of dout and du (off_d and off_u, nc + 1 entries) by one
// workgroup, and ebase[r] = off_d[r] less r's neighbours of a lower rank: the
// neighbour at place k of row r has the edge id ebase[r] + k. *simple
// = 1 when the bits stand for all of the rows' `slots` slots and
// as many lie above the diagonal as below; else the view is left without edges.
constexpr uint32_t kScanBlock = 1024;
__global__ __launch_bounds__(kScanBlock) void k_rank_scan(const uint32_t* __restrict__ du,
                                                          const uint32_t* __restrict__ dout, uint32_t nc,
                                                          uint64_t slots, uint32_t* off_d, uint32_t* off_u,
                                                          uint32_t* ebase, uint32_t* simple) {
  __shared__ uint2 s_w[kScanBlock / kWave];
  __shared__ uint2 s_total;
  const uint32_t tid = threadIdx.x;
  const int lane = lane64();
  // thread t owns a run of rows
  const uint32_t per = (nc + kScanBlock - 1) / kScanBlock;
  const uint32_t r0 = min(nc, tid * per), r1 = min(nc, r0 + per);
  uint32_t a = 0, b = 0;
  for (uint32_t r = r0; r < r1; ++r) {
    a += dout[r];
    b += du[r];
  }
  uint32_t ia = a, ib = b;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t ya = __shfl_up(ia, o), yb = __shfl_up(ib, o);
    if (lane >= o) {
      ia += ya;
      ib += yb;
    }
  }
  if (lane == kWave - 1) s_w[tid / kWave] = make_uint2(ia, ib);
  __syncthreads();
  uint32_t xa = ia - a, xb = ib - b;
  for (uint32_t k = 0; k < tid / kWave; ++k) {
    xa += s_w[k].x;
    xb += s_w[k].y;
  }
  if (tid == kScanBlock - 1) s_total = make_uint2(xa + a, xb + b);
  __syncthreads();
  const bool ok = s_total.y == slots && 2ull * s_total.x == slots;
  for (uint32_t r = r0; r < r1; ++r) {
    const uint32_t d = dout[r], u = du[r];
    off_d[r] = ok ? xa : 0u;
    off_u[r] = ok ? xb : 0u;
    ebase[r] = xa - (u - d);
    xa += d;
    xb += u;
  }
  if (tid == kScanBlock - 1) {
    off_d[nc] = ok ? xa : 0u;
    off_u[nc] = ok ? xb : 0u;
    *simple = ok ? 1u : 0u;
  }
}

// The rows' entries: undirected (neighbour, edge id), oriented (neighbour,
// source), the edge-id matrix (null: none) and fresh peel state; *simple = 0
// when a bit below the diagonal has no mirror (as many lie above, so then all
// have one). One wave per
// row and run of words, a word's 64 bits on the wave's lanes, so every array
// is written in order.
constexpr uint32_t kFillWords = 16;
__global__ __launch_bounds__(kBlock) void k_rank_fill(const unsigned long long* __restrict__ bits0,
                                                      const uint32_t* __restrict__ pref0,
                                                      const uint32_t* __restrict__ off_u,
                                                      const uint32_t* __restrict__ ebase, uint32_t nc, uint32_t ws,
                                                      uint32_t* adj_u, uint32_t* eid_u, uint32_t* adj_d,
                                                      uint32_t* src, uint32_t* orig, uint32_t* state,
                                                      uint32_t* del_thr, uint32_t* eidm, uint32_t* simple) {
  const uint32_t lane = uint32_t(lane64());
  const unsigned long long below = (1ull << lane) - 1ull;
  const uint32_t runs = (ws + kFillWords - 1) / kFillWords;
  const uint64_t items = uint64_t(nc) * runs, waves = uint64_t(gridDim.x) * (kBlock / kWave);
  if (off_u[nc] == 0) return;  // no edges, or not a simple graph
  for (uint64_t it = uint64_t(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave; it < items; it += waves) {
    const uint32_t r = uint32_t(it / runs), i0 = uint32_t(it - uint64_t(r) * runs) * kFillWords;
    const uint32_t i1 = min(ws, i0 + kFillWords);
    const uint32_t ub = off_u[r], eb = ebase[r];
    const unsigned long long rbelow = (1ull << (r & 63)) - 1ull;
    for (uint32_t i = i0; i < i1; ++i) {  // wave-uniform
      const uint64_t at = uint64_t(r) * ws + i;
      const unsigned long long x = bits0[at];
      if (!((x >> lane) & 1ull)) continue;
      const uint32_t w = i * 64 + lane, k = pref0[at] + uint32_t(__popcll(x & below));
      uint32_t e;
      if (w > r) {
        e = eb + k;
        adj_d[e] = w;
        src[e] = r;
        orig[e] = e;
        state[e] = kNone;
        del_thr[e] = kNone;
      } else {  // the edge of w's row
        const uint64_t q = uint64_t(w) * ws + (r >> 6);
        if (!((bits0[q] >> (r & 63)) & 1ull)) {  // rows from lines need not mirror each other
          *simple = 0;
          continue;
        }
        e = ebase[w] + pref0[q] + uint32_t(__popcll(bits0[q] & rbelow));
      }
      adj_u[ub + k] = w;
      eid_u[ub + k] = e;
      if (eidm) eidm[uint64_t(r) * nc + w] = e;
    }
  }
}

// Every edge's support through the matrix cores (kt_tile.h): 2 x 2 waves of 64
// x 64 pairs per workgroup. Bound on the rows' reads: a block of pairs reads
// 256 rows, so blocks go to the dies (workgroups in turn) in squares of side x
// side, which share their rows in a die's L2.
constexpr uint32_t kTileRows = 128;
template <bool kEidm>
__global__ __launch_bounds__(kBlock) void k_dense_count(const unsigned long long* __restrict__ bits,
                                                        EidOf<kEidm> eid_of, uint32_t nb, uint32_t side,
                                                        int32_t* sup) {
  constexpr uint32_t kDies = 8;
  const uint32_t ns = (nb + side - 1) / side, cells = side * side;
  const uint32_t q = blockIdx.x / kDies, sq = q / cells * kDies + blockIdx.x % kDies, in = q % cells;
  uint32_t si, sj;
  if (sq >= tile_items(ns) || !tile_of(sq, ns, &si, &sj)) return;
  const uint32_t bi = si * side + in / side, bj = sj * side + in % side;
  if (bi > bj || bj >= nb) return;
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t u0 = bi * kTileRows + wave / 2 * 64, v0 = bj * kTileRows + wave % 2 * 64;
  if (u0 > v0 || v0 >= eid_of.nc) return;
  Acc4 acc[4][4];
  count_tile<4, 4>(bits, eid_of.nc, eid_of.ws, u0, v0, acc);
  tile_edges<4, 4>(bits, eid_of.nc, eid_of.ws, u0, v0, acc, eid_of,
                   [&](bool live, uint32_t e, uint32_t, uint32_t, uint32_t c) {
                     if (live) sup[e] = int32_t(c);
                   });
}

// *out = the longest of the rows (starts at 0)
__global__ __launch_bounds__(kBlock) void k_max_row(const uint32_t* __restrict__ off, uint32_t rows, uint32_t* out) {
  uint32_t m = 0;
  for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x)
    m = max(m, off[r + 1] - off[r]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, uint32_t(__shfl_xor(m, o)));
  if (lane64() == 0 && m) atomicMax(out, m);
}

}  // namespace

// --------------------------------------------------------------- wrappers ---

void rank_rows(const uint64_t* off, const uint32_t* adj, const uint32_t* to, const uint32_t* inv, uint32_t nc,
               uint32_t ws, uint64_t* bits0, uint64_t* bits, uint32_t* pref0, uint32_t* du, uint32_t* dout,
               hipStream_t s) {
  if (ws > kMaxRowWords) fail("dense core: rows longer than the LDS stage");
  if (nc)
    k_rank_rows<<<std::min<uint32_t>(nc, 16384), kBlock, 0, s>>>(
        off, adj, to, inv, nc, ws, reinterpret_cast<unsigned long long*>(bits0),
        reinterpret_cast<unsigned long long*>(bits), pref0, du, dout);
}
void rank_scan(const uint32_t* du, const uint32_t* dout, uint32_t nc, uint64_t slots, uint32_t* off_d,
               uint32_t* off_u, uint32_t* ebase, uint32_t* simple, hipStream_t s) {
  k_rank_scan<<<1, kScanBlock, 0, s>>>(du, dout, nc, slots, off_d, off_u, ebase, simple);
}
void rank_fill(const uint64_t* bits0, const uint32_t* pref0, const uint32_t* off_u, const uint32_t* ebase, uint32_t nc,
               uint32_t ws, uint32_t* adj_u, uint32_t* eid_u, uint32_t* adj_d, uint32_t* src, uint32_t* orig,
               uint32_t* state, uint32_t* del_thr, uint32_t* eidm, uint32_t* simple, hipStream_t s) {
  const uint64_t waves = uint64_t(nc) * ((ws + kFillWords - 1) / kFillWords);
  if (nc)
    k_rank_fill<<<std::min(grid_for(waves * kWave), 8192), kBlock, 0, s>>>(
        reinterpret_cast<const unsigned long long*>(bits0), pref0, off_u, ebase, nc, ws, adj_u, eid_u, adj_d, src,
        orig, state, del_thr, eidm, simple);
}
// Measured (vertices, edges; by edge -> by pairs): 1,268, 483 k: 20 -> 23 us;
// 1,535, 912 k: 37 -> 23; 2,867, 878 k: 39 -> 34; 3,150, 3.05 M: 136 -> 39;
// 4,048, 945 k: 59 -> 61; 5,701, 2.35 M: 170 -> 112; 9,109, 6.25 M: 645 -> 331;
// 14,697, 15.8 M: 2,530 -> 1,020. By edge about 10^6 word ANDs a us, by pairs
// 12 * 10^6 plus some 15 us.
double dense_pair_cost(uint32_t nc, uint32_t ws) { return double(nc) * nc / 24.0 * ws; }
bool dense_by_pairs(uint32_t nc, uint32_t mc, uint32_t ws) {
  return double(mc) * ws > 15e6 + dense_pair_cost(nc, ws);
}
void dense_count(const uint64_t* bits, const uint32_t* pref0, const uint32_t* off_u, const uint32_t* eid_u,
                 const uint32_t* eidm, uint32_t nc, uint32_t ws, int32_t* sup, hipStream_t s) {
  if (!nc) return;
  auto b = reinterpret_cast<const unsigned long long*>(bits);
  const uint32_t nb = (nc + kTileRows - 1) / kTileRows;
  // squares once the rows outgrow a die's L2 (4 MB)
  const uint32_t side = uint64_t(nc) * ws * 8 > (4u << 20) ? 8u : 1u;
  const uint32_t squares = (tile_items((nb + side - 1) / side) + 7) / 8 * 8;
  const uint32_t grid = squares * side * side;
  if (eidm)
    k_dense_count<true><<<grid, kBlock, 0, s>>>(b, EidOf<true>{eidm, b, pref0, off_u, eid_u, nc, ws}, nb, side, sup);
  else
    k_dense_count<false><<<grid, kBlock, 0, s>>>(b, EidOf<false>{eidm, b, pref0, off_u, eid_u, nc, ws}, nb, side, sup);
}
void max_row(const uint32_t* off, uint32_t rows, uint32_t* out, hipStream_t s) {
  fill_u32(out, 1, 0, s);
  if (rows) k_max_row<<<std::min(grid_for(rows), 1024), kBlock, 0, s>>>(off, rows, out);
}

}  // namespace kt
