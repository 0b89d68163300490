// Common-neighbour counts of a dense core's bit-matrix rows on the matrix
// cores: count(u, v) = popcount(bits[u] & bits[v]) for all pairs of a tile of
// rows, as a product of 0/1 matrices.
//
// A row's bits become 4-bit floats in registers: the bits j, j + 4, j + 8, ...
// of a 32-bit word, shifted down and masked, are eight of them (e2m1 0b0001 =
// 0.5, doubled by the operand's block scale), so a word costs seven VALU
// operations and one v_mfma_scale_f32_16x16x128_f8f6f4 takes 128 bits of 16 x
// 16 pairs in 16 cycles: 64 AND-popcounts of 64-bit words a cycle and SIMD,
// where the VALU does 4. Products are 0 or 1 and sums at most 65536: exact in
// the fp32 accumulators. The order of a row's bits along the product does not
// matter as long as both operands use the same.
#pragma once

#include "kt_device.h"

namespace kt {

typedef int Fp4x32 __attribute__((ext_vector_type(8)));  // 4-bit operand: the lower four words
typedef float Acc4 __attribute__((ext_vector_type(4)));
// a 16-byte load from a row that starts on 8 bytes
typedef uint32_t Quad8 __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ Fp4x32 bits_to_fp4(uint32_t x) {
  Fp4x32 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = int((x >> j) & 0x11111111u);
  r[4] = r[5] = r[6] = r[7] = 0;
  return r;
}

// acc[i][j] (lane l, element k) = count(u0 + 16 i + (l / 16) 4 + k,
// v0 + 16 j + l % 16) by one wave. Rows past nc stand for row nc - 1: their
// counts are not to be used. Lane l loads 16 bytes of row l % 16 of each
// operand: words 2 (l / 16) and the next of every 8.
template <int MI, int NI>
__device__ __forceinline__ void count_tile(const unsigned long long* __restrict__ bits, uint32_t nc, uint32_t ws,
                                           uint32_t u0, uint32_t v0, Acc4 (&acc)[MI][NI]) {
  constexpr int kScale = 128;  // 2^1: 0.5 -> 1
  const uint32_t lane = uint32_t(lane64()), row = lane & 15u, g = lane >> 4;
  const unsigned long long* p[MI + NI];
#pragma unroll
  for (int i = 0; i < MI; ++i) p[i] = bits + uint64_t(min(u0 + 16 * i + row, nc - 1)) * ws + 2 * g;
#pragma unroll
  for (int j = 0; j < NI; ++j) p[MI + j] = bits + uint64_t(min(v0 + 16 * j + row, nc - 1)) * ws + 2 * g;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = Acc4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const Quad8 (&x)[MI + NI]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      Fp4x32 a[MI], b[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) a[i] = bits_to_fp4(x[i][s]);
#pragma unroll
      for (int j = 0; j < NI; ++j) b[j] = bits_to_fp4(x[MI + j][s]);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i], b[j], acc[i][j], 4, 4, 0, kScale, 0, kScale);
    }
  };
  const uint32_t full = ws / 8;  // whole chunks of 8 words
  Quad8 x[MI + NI], y[MI + NI];
  if (full) {
#pragma unroll
    for (int i = 0; i < MI + NI; ++i) x[i] = *reinterpret_cast<const Quad8*>(p[i]);
  }
  for (uint32_t c = 0; c < full; ++c) {  // the next chunk's loads are in flight over this one's products
    if (c + 1 < full) {
#pragma unroll
      for (int i = 0; i < MI + NI; ++i) y[i] = *reinterpret_cast<const Quad8*>(p[i] + 8 * (c + 1));
    }
    multiply(x);
#pragma unroll
    for (int i = 0; i < MI + NI; ++i) x[i] = y[i];
  }
  if (full * 8 < ws) {  // the rest of the rows, word by word
    const uint32_t w = full * 8 + 2 * g;
#pragma unroll
    for (int i = 0; i < MI + NI; ++i) {
      const unsigned long long lo = w < ws ? p[i][8 * full] : 0ull, hi = w + 1 < ws ? p[i][8 * full + 1] : 0ull;
      x[i] = Quad8{uint32_t(lo), uint32_t(lo >> 32), uint32_t(hi), uint32_t(hi >> 32)};
    }
    multiply(x);
  }
}

// The id of edge (x, w) of a dense core: from the edge-id matrix, or from the
// place of w in x's row.
template <bool kEidm>
struct EidOf {
  const uint32_t* eidm;
  const unsigned long long* bits0;
  const uint32_t *pref0, *off_u, *eid_u;
  uint32_t nc, ws;
  __device__ __forceinline__ uint32_t operator()(uint32_t x, uint32_t w) const {
    if (kEidm) return eidm[uint64_t(x) * nc + w];
    const uint64_t at = uint64_t(x) * ws + (w >> 6);
    const unsigned long long below = bits0[at] & ((1ull << (w & 63)) - 1ull);
    return eid_u[off_u[x] + pref0[at] + uint32_t(__popcll(below))];
  }
};

// Tiles (bi <= bj) of the upper triangle of nb x nb, rows i and nb - 1 - i
// folded into one of nb + 1 tiles: item t of tile_items(nb); false: none.
__host__ __device__ __forceinline__ uint32_t tile_items(uint32_t nb) { return (nb + 1) / 2 * (nb + 1); }
__host__ __device__ __forceinline__ bool tile_of(uint32_t t, uint32_t nb, uint32_t* bi, uint32_t* bj) {
  const uint32_t r = t / (nb + 1), c = t - r * (nb + 1);
  if (c < nb - r) {
    *bi = r;
    *bj = r + c;
    return true;
  }
  *bi = nb - 1 - r;
  *bj = *bi + (c - (nb - r));
  return *bi != r;  // the middle row of an odd nb has no partner
}

// The live edges among a tile's pairs: found(live, edge, u, v, count) by all
// lanes of the wave, 4 MI NI times; each edge once (u < v).
template <int MI, int NI, typename E, typename F>
__device__ __forceinline__ void tile_edges(const unsigned long long* __restrict__ bits, uint32_t nc, uint32_t ws,
                                           uint32_t u0, uint32_t v0, const Acc4 (&acc)[MI][NI], E&& eid_of,
                                           F&& found) {
  static_assert(64 % (16 * NI) == 0, "a tile's columns must lie in one word");
  const uint32_t lane = uint32_t(lane64()), g = lane >> 4, col = lane & 15u;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    uint32_t live = 0, e[4][NI];
    unsigned long long word[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t u = u0 + 16 * i + 4 * g + k;
      word[k] = u < nc ? bits[uint64_t(u) * ws + (v0 >> 6)] : 0ull;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const uint32_t u = u0 + 16 * i + 4 * g + k, v = v0 + 16 * j + col;
        e[k][j] = kNone;
        if (u < v && ((word[k] >> (v & 63u)) & 1ull)) {
          live |= 1u << (k * NI + j);
          e[k][j] = eid_of(u, v);
        }
      }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < NI; ++j)
        found((live >> (k * NI + j)) & 1u, e[k][j], u0 + 16 * i + 4 * g + k, v0 + 16 * j + col,
              uint32_t(acc[i][j][k]));
  }
}

}  // namespace kt
