// Life-like automata over many generations with the cells packed one bit
// each: the steady steps of a Life iteration on 1-byte cells (Moore(1), 2-D,
// Wrap / Remove / Reflect).
//
// An iteration packs its grid once (life_pack_kernel), advances it in packed
// form (lifep_kernel, many generations per launch) and unpacks it once
// (life_unpack_kernel).  The packed rows live in the first bytes of the
// iteration's own two buffers, row by row inside the cells of that row, so
// no workspace is needed: both buffers are rewritten in full by the two
// single steps that end every iteration.
//
// lifep_kernel: a lane holds one 32-cell word of K consecutive rows in
// registers, a wave 64 words (2 rim words and 62 words of results) and a
// workgroup 16 waves stacked along the rows.  Per generation each wave hands
// its first and last row to its neighbours through LDS (two buffers, one
// barrier) and computes its interior rows before it waits.  The tile's outer
// rows and the rim words lose one row / one bit per generation, so a launch
// of `gens` generations stores the tile without `gens` rows on each side,
// and gens <= 32 keeps all 62 words exact.
//
// Why this split: a generation of Conway's rule costs 14 full-rate VALU
// operations per 32 cells (2 lane moves, 2 funnel shifts and 10 v_bitop3),
// against 12 per 16 cells for windows that carry their own rim bits, and a
// tile of 16 K rows recomputes only 2 gens rows where a wave marching alone
// down a chunk of 32 rows recomputed 2 gens of every 32 + 2 gens.  Packed
// rows move 1/8 of the bytes, so memory no longer bounds it.
//
// Cells outside the array follow the reference's getneighbor
// (src/array.jl:129-179) in every generation: Wrap and Reflect load rows and
// rim bits at their wrapped / mirrored coordinates, whose evolution is the
// wrapped / mirrored cells' (Wrap is a translation, and the Life count does
// not depend on order); Remove holds outside rows and bits at padval after
// every generation.
#pragma once

#include "lifeb_kernel.hpp"

namespace sth {

// Packed row y of a buffer: 4-byte words from the first 4-byte boundary of
// the row, in one of four slots by row: consecutive rows of a pitch of 2^k
// bytes would otherwise start on the same memory channel and use 1/8 of
// them.  n0 >= kLifepMinN0 leaves room for the slots inside every row.
constexpr int kLifepMinN0 = 64;
constexpr int kLifepWaves = 16;   // waves of a workgroup
constexpr int kLifepOut = 62;     // words of results per wave
constexpr int kLifepMaxGens = 32; // a rim word's bits

struct LifepParams {
  char* src;  // logical cell (0, 0)
  char* dst;
  int64_t s1, d1;  // row pitch in bytes
  int32_t n0, n1;
  int32_t words;   // packed words per row
  int32_t gens;    // generations of this launch
  int32_t tiles_x, tiles_y;
  uint32_t pad;    // 0 or ~0: the padval's bit
  uint32_t birth, survive;  // neighbour counts 0..8
};

__host__ __device__ __forceinline__ int32_t lifep_words(int64_t n0) { return static_cast<int32_t>((n0 + 31) >> 5); }

__device__ __forceinline__ uint32_t* lifep_row(char* base, int64_t pitch, int32_t y, int32_t words) {
  const uint64_t a = (reinterpret_cast<uint64_t>(base + static_cast<int64_t>(y) * pitch) + 3) & ~uint64_t(3);
  return reinterpret_cast<uint32_t*>(a) + (y & 3) * words;
}

// 32 bits of a packed row from bit `p` >= 0 on (bits past the last word: any).
__device__ __forceinline__ uint32_t lifep_bits(const uint32_t* row, int32_t p, int32_t words) {
  const int32_t i = p >> 5;
  const int32_t i0 = i < words ? i : words - 1, i1 = i + 1 < words ? i + 1 : words - 1;
  return __builtin_amdgcn_alignbit(row[i1], row[i0], p & 31);
}

// Horizontal 3-sum of a row's words across the wave: s + 2 c = left + own + right.
__device__ __forceinline__ void lifep_hsum(uint32_t w, uint32_t& s, uint32_t& c) {
  const uint32_t l = __builtin_amdgcn_alignbit(w, lane_shift<-1>(w), 31);
  const uint32_t r = __builtin_amdgcn_alignbit(lane_shift<1>(w), w, 1);
  s = bop3<kA3 ^ kB3 ^ kC3>(l, w, r);
  c = bop3<(kA3 & kB3) | (kA3 & kC3) | (kB3 & kC3)>(l, w, r);
}

// Any birth / survive rule on the 3 x 3 sum S = 0..9 including the centre: a
// tree of selects on the sum's bits over the ten outcomes (a dead cell of
// sum S has S neighbours, a live one S - 1).
__device__ __forceinline__ uint32_t lifep_rule(uint32_t sa, uint32_t ca, uint32_t sb, uint32_t cb, uint32_t sc,
                                               uint32_t cc, uint32_t alive, uint32_t birth, uint32_t survive) {
  constexpr uint32_t kMaj = (kA3 & kB3) | (kA3 & kC3) | (kB3 & kC3), kXor = kA3 ^ kB3 ^ kC3;
  constexpr uint32_t kMux = (kA3 & kB3) | (~kA3 & kC3);  // a ? b : c
  const uint32_t b0 = bop3<kXor>(sa, sb, sc), c1 = bop3<kMaj>(sa, sb, sc);
  const uint32_t u0 = bop3<kXor>(ca, cb, cc), u1 = bop3<kMaj>(ca, cb, cc);
  const uint32_t b1 = c1 ^ u0, k = c1 & u0, b2 = u1 ^ k, b3 = u1 & k;
  uint32_t leaf[10];
#pragma unroll
  for (int S = 0; S < 10; ++S) {
    const uint32_t bm = S < 9 ? 0u - ((birth >> S) & 1u) : 0u;
    const uint32_t sm = S > 0 ? 0u - ((survive >> (S > 0 ? S - 1 : 0)) & 1u) : 0u;
    leaf[S] = bop3<kMux>(alive, sm, bm);
  }
  const uint32_t m01 = bop3<kMux>(b0, leaf[1], leaf[0]), m23 = bop3<kMux>(b0, leaf[3], leaf[2]);
  const uint32_t m45 = bop3<kMux>(b0, leaf[5], leaf[4]), m67 = bop3<kMux>(b0, leaf[7], leaf[6]);
  const uint32_t m89 = bop3<kMux>(b0, leaf[9], leaf[8]);
  const uint32_t lo = bop3<kMux>(b1, m23, m01), hi = bop3<kMux>(b1, m67, m45);
  return bop3<kMux>(b3, m89, bop3<kMux>(b2, hi, lo));
}

template <int K, bool CONWAY, int BC>
__global__ __launch_bounds__(kLifepWaves * 64) void lifep_kernel(LifepParams p) {
  constexpr bool REMOVE = BC == STH_REMOVE, REFLECT = BC == STH_REFLECT;
  __shared__ uint32_t edge[2][kLifepWaves][2][64];  // first and last row of every wave, two generations
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int tile = xcd_block_id(static_cast<int>(blockIdx.x), p.tiles_x * p.tiles_y, 1);
  const int strip = tile % p.tiles_x;
  const int32_t n0 = p.n0, n1 = p.n1, words = p.words, gens = p.gens;
  // rows of the tile: gens rim rows, the results, gens rim rows
  const int32_t y0 = (tile / p.tiles_x) * (kLifepWaves * K - 2 * gens) - gens + wave * K;
  const int32_t wi = strip * kLifepOut - 1 + lane;  // this lane's word
  const int32_t c = wi * 32;                        // its first column
  // waves with a word that is not wholly inside the row (uniform)
  const bool xedge = strip == 0 || (strip * kLifepOut + 63) * 32 > n0;

  // ---- load
  uint32_t w[K];
  uint32_t keep = 0xffffffffu;  // bits of columns inside the row
  {
    if (c < 0 || c >= n0) keep = 0u;
    else if (c + 32 > n0) keep = (1u << (n0 - c)) - 1u;
    // edge words: own bits from bit pa (masked), the rest from bit pb on,
    // moved up by q (Wrap) or reversed (Reflect)
    int32_t pa = 0, pb = 0, q = 0;
    if constexpr (!REMOVE) {
      pa = keep ? c : 0;
      if (c < 0) {
        pb = REFLECT ? 1 : n0 - 32;
      } else if (c < n0) {
        q = REFLECT ? 0 : (n0 - c) & 31;
        pb = REFLECT ? 2 * n0 - 33 - c : 0;
      } else {
        pb = REFLECT ? 2 * n0 - 33 - c : c - n0;
      }
      if (pb < 0 || pb > n0) pb = 0;  // words too far out to reach a result
    } else {
      pa = keep ? c : 0;
    }
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const int32_t y = y0 + r;
      const int32_t ym = REMOVE ? (y < 0 ? 0 : (y >= n1 ? n1 - 1 : y)) : lifeb_map_row(y, n1, REFLECT);
      const uint32_t* row = lifep_row(p.src, p.s1, ym, words);
      if (!xedge) {
        w[r] = row[wi];
      } else {
        const uint32_t own = row[pa >> 5];
        uint32_t far = p.pad;
        if constexpr (!REMOVE) {
          far = lifep_bits(row, pb, words);
          far = REFLECT ? __builtin_bitreverse32(far) : far << q;
        }
        w[r] = (own & keep) | (far & ~keep);
      }
      if constexpr (REMOVE) {
        if (y < 0 || y >= n1) w[r] = p.pad;
      }
    }
  }
  // Remove: waves with outside rows or bits reset them every generation
  const bool reset = REMOVE && (xedge || y0 < 0 || y0 + K > n1);

  // ---- generations
  edge[0][wave][0][lane] = w[0];
  edge[0][wave][1][lane] = w[K - 1];
  for (int g = 0; g < gens; ++g) {
    uint32_t hs[K], hc[K];
#pragma unroll
    for (int r = 0; r < K; ++r) lifep_hsum(w[r], hs[r], hc[r]);
    auto next = [&](uint32_t sa, uint32_t ca, int r, uint32_t sc, uint32_t cc) -> uint32_t {
      uint32_t v;
      if constexpr (CONWAY) v = conway_bits(sa, ca, hs[r], hc[r], sc, cc, w[r]);
      else v = lifep_rule(sa, ca, hs[r], hc[r], sc, cc, w[r], p.birth, p.survive);
      if constexpr (REMOVE) {
        if (reset) {
          const int32_t y = y0 + r;
          v = bop3<(kA3 & kB3) | (~kB3 & kC3)>(v, keep, p.pad);
          if (y < 0 || y >= n1) v = p.pad;
        }
      }
      return v;
    };
    uint32_t v[K];
#pragma unroll
    for (int r = 1; r + 1 < K; ++r) v[r] = next(hs[r - 1], hc[r - 1], r, hs[r + 1], hc[r + 1]);
    // the neighbours' rows of this generation (the outermost waves': any)
    __syncthreads();
    const int b = g & 1;
    uint32_t ts, tc, bs, bc;
    lifep_hsum(edge[b][wave > 0 ? wave - 1 : 0][1][lane], ts, tc);
    lifep_hsum(edge[b][wave < kLifepWaves - 1 ? wave + 1 : wave][0][lane], bs, bc);
    if constexpr (K == 1) {
      v[0] = next(ts, tc, 0, bs, bc);
    } else {
      v[0] = next(ts, tc, 0, hs[1], hc[1]);
      v[K - 1] = next(hs[K - 2], hc[K - 2], K - 1, bs, bc);
    }
#pragma unroll
    for (int r = 0; r < K; ++r) w[r] = v[r];
    edge[b ^ 1][wave][0][lane] = w[0];
    edge[b ^ 1][wave][1][lane] = w[K - 1];
  }

  // ---- store
  if (lane >= 1 && lane <= kLifepOut && wi < words) {
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const int32_t l = wave * K + r, y = y0 + r;  // y >= 0 for every result row
      if (l >= gens && l < kLifepWaves * K - gens && y < n1) lifep_row(p.dst, p.d1, y, words)[wi] = w[r];
    }
  }
}

// ------------------------------------------------------------ host side

// Rows per wave and generations per launch for an n0 x n1 grid: the pair
// with the least time per generation by a model in cycles of one SIMD -- a
// tile's 4 waves per SIMD take 4 cycles per operation and row, every tile a
// CU runs adds to that, a generation's exchange costs about 350 and a launch
// (its start, loads and stores) about 6000.
struct LifepShape {
  int32_t k, gens, tiles_x, tiles_y;
};
constexpr int kLifepRows[] = {1, 2, 3, 4, 6, 8, 10, 12, 14, 16};

inline void lifep_grid(int64_t n0, int64_t n1, int k, int gens, int32_t* tx, int32_t* ty) {
  *tx = static_cast<int32_t>((lifep_words(n0) + kLifepOut - 1) / kLifepOut);
  const int64_t rows = kLifepWaves * k - 2 * gens;
  *ty = static_cast<int32_t>((n1 + rows - 1) / rows);
}

inline LifepShape lifep_shape(int64_t n0, int64_t n1, bool conway, int cus) {
  LifepShape best{};
  double least = 0;
  const double ops = conway ? 14 : 38;
  for (int k : kLifepRows)
    for (int g = 2; g <= kLifepMaxGens && kLifepWaves * k - 2 * g >= 1; ++g) {
      LifepShape s{k, g, 0, 0};
      lifep_grid(n0, n1, k, g, &s.tiles_x, &s.tiles_y);
      const int64_t tiles = static_cast<int64_t>(s.tiles_x) * s.tiles_y;
      const double rounds = static_cast<double>((tiles + cus - 1) / cus);
      const double t = 6000.0 / g + 350.0 + rounds * (kLifepWaves / 4) * 4.0 * k * ops;
      if (!best.k || t < least) {
        best = s;
        least = t;
      }
    }
  return best;
}

using LifepFn = void (*)(const LifepParams&, hipStream_t);
// The launcher for K rows per wave, and the two conversions (life_packed.hip).
LifepFn lifep_launcher(int k, bool conway, int bc);
void launch_life_pack(LifepParams p, hipStream_t s);
void launch_life_unpack(LifepParams p, hipStream_t s);

}  // namespace sth
