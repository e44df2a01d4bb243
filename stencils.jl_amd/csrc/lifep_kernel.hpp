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
// registers.  `lpr` = 64, 32 or 16 lanes stand side by side (two of them rim
// words, the others results) and the 64 / lpr groups of a wave one above the
// other; a workgroup stacks 16 waves.  Per generation each group hands its
// first and last row to its neighbours through LDS (two buffers, one
// barrier); interior rows are computed before the wait.  The tile's outer
// rows and the rim words lose one row / one bit per generation, so a launch
// of `gens` generations stores the tile without `gens` rows on each side,
// and gens <= 32 keeps the other words exact.
//
// Why this split: a generation of Conway's rule costs 15 full-rate VALU
// operations per 32 cells (2 lane moves, 2 funnel shifts, 10 v_bitop3 and the
// share of the exchanged rows), against 12 per 16 cells for windows that
// carry their own rim bits, and a tile recomputes only its rim where a wave
// marching alone down a chunk of 32 rows recomputed 2 gens of every
// 32 + 2 gens.  Groups of 32 or 16 lanes make the tile squarer (less rim) and
// fit more widths.  Packed rows move 1/8 of the bytes; the kernel is bound by
// VALU issue, and by the load and store of the tile, which do not overlap.
//
// Cells outside the array follow the reference's getneighbor
// (src/array.jl:129-179) in every generation: Wrap and Reflect load rows and
// rim bits at their wrapped / mirrored coordinates, whose evolution is the
// wrapped / mirrored cells' (Wrap is a translation, and the Life count does
// not depend on order); Remove holds outside rows and bits at padval after
// every generation.
#pragma once

#include "lifeb_kernel.hpp"
#include "lifep_shape.hpp"

namespace sth {

// Packed row y of a buffer: 4-byte words in the cells of row y / 4, which
// holds four packed rows one after another from its first 4-byte boundary
// on.  n0 >= kLifepMinN0 leaves room for them.
constexpr int kLifepMinN0 = 64;

struct LifepParams {
  char* src;  // logical cell (0, 0)
  char* dst;
  int64_t s1, d1;  // row pitch in bytes
  int32_t n0, n1;
  int32_t words;   // packed words per row
  int32_t gens;    // generations of this launch
  int32_t lpr_shift;  // log2 of the lanes side by side
  int32_t tiles_x, tiles_y;
  uint32_t pad;    // 0 or ~0: the padval's bit
  uint32_t birth, survive;  // neighbour counts 0..8
};

__device__ __forceinline__ uint32_t* lifep_row(char* base, int64_t pitch, int32_t y, int32_t words) {
  const uint64_t a = (reinterpret_cast<uint64_t>(base + static_cast<int64_t>(y >> 2) * pitch) + 3) & ~uint64_t(3);
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
  __shared__ uint32_t edge[2][kLifepWaves * 2 * 64];  // first and last row of every group, two generations
  const int lpr = 1 << p.lpr_shift, groups = kLifepWaves << (6 - p.lpr_shift);
  const int col = static_cast<int>(threadIdx.x) & (lpr - 1);
  const int group = static_cast<int>(threadIdx.x) >> p.lpr_shift;
  const int tile = xcd_block_id(static_cast<int>(blockIdx.x), p.tiles_x * p.tiles_y, 1);
  const int strip = tile % p.tiles_x;
  const int32_t n0 = p.n0, n1 = p.n1, words = p.words, gens = p.gens;
  // rows of the tile: gens rim rows, the results, gens rim rows
  const int32_t t0 = (tile / p.tiles_x) * (groups * K - 2 * gens) - gens;
  const int32_t y0 = t0 + group * K;             // this lane's first row
  const int32_t wi = strip * (lpr - 2) - 1 + col;  // its word
  const int32_t c = wi * 32;                     // the word's first column
  // tiles with a word that is not wholly inside the row, or a row outside
  const bool xedge = strip == 0 || (strip * (lpr - 2) + lpr - 1) * 32 > n0;
  const bool yedge = t0 < 0 || t0 + groups * K > n1;

  // ---- load: every load of the lane's rows is issued before the first use
  uint32_t w[K];
  uint32_t keep = 0xffffffffu;  // bits of columns inside the row
  if (c < 0 || c >= n0) keep = 0u;
  else if (c + 32 > n0) keep = (1u << (n0 - c)) - 1u;
  {
    const uint32_t* row[K];
#pragma unroll
    for (int r = 0; r < K; ++r) {
      int32_t ym = y0 + r;
      if (yedge) ym = REMOVE ? (ym < 0 ? 0 : (ym >= n1 ? n1 - 1 : ym)) : lifeb_map_row(ym, n1, REFLECT);
      row[r] = lifep_row(p.src, p.s1, ym, words);
    }
    if (!xedge) {
#pragma unroll
      for (int r = 0; r < K; ++r) w[r] = row[r][wi];
    } else {
      // own bits (masked); the rest from bit pb on, moved up by q (Wrap) or
      // reversed (Reflect), or padval
      const int32_t io = keep ? wi : 0;
      int32_t pb = 0, q = 0;
      uint32_t lo[K], hi[K];
      if constexpr (!REMOVE) {
        if (c < 0) {
          pb = REFLECT ? 1 : n0 - 32;
        } else if (c < n0) {
          q = REFLECT ? 0 : (n0 - c) & 31;
          pb = REFLECT ? 2 * n0 - 33 - c : 0;
        } else {
          pb = REFLECT ? 2 * n0 - 33 - c : c - n0;
        }
        if (pb < 0 || pb > n0) pb = 0;  // words too far out to reach a result
        const int32_t i = pb >> 5, i0 = i < words ? i : words - 1, i1 = i + 1 < words ? i + 1 : words - 1;
#pragma unroll
        for (int r = 0; r < K; ++r) {
          lo[r] = row[r][i0];
          hi[r] = row[r][i1];
        }
      }
#pragma unroll
      for (int r = 0; r < K; ++r) w[r] = row[r][io];
#pragma unroll
      for (int r = 0; r < K; ++r) {
        uint32_t far = p.pad;
        if constexpr (!REMOVE) {
          far = __builtin_amdgcn_alignbit(hi[r], lo[r], pb & 31);
          far = REFLECT ? __builtin_bitreverse32(far) : far << q;
        }
        w[r] = (w[r] & keep) | (far & ~keep);
      }
    }
  }
  // Remove: tiles with outside rows or bits set them to padval, now and after
  // every generation
  const bool reset = REMOVE && (xedge || yedge);
  auto held = [&](uint32_t v, int r) -> uint32_t {
    const uint32_t k = y0 + r < 0 || y0 + r >= n1 ? 0u : keep;
    return bop3<(kA3 & kB3) | (~kB3 & kC3)>(v, k, p.pad);
  };
  if (reset) {
#pragma unroll
    for (int r = 0; r < K; ++r) w[r] = held(w[r], r);
  }

  // ---- generations
  uint32_t* const mine = &edge[0][(group * 2) * lpr + col];  // first row; last row lpr further
  const uint32_t* const above = group > 0 ? mine - lpr : mine;
  const uint32_t* const below = group < groups - 1 ? mine + 2 * lpr : mine;
  constexpr int kBuf = kLifepWaves * 2 * 64;
  mine[0] = w[0];
  mine[lpr] = w[K - 1];
  for (int g = 0; g < gens; ++g) {
    uint32_t hs[K], hc[K];
#pragma unroll
    for (int r = 0; r < K; ++r) lifep_hsum(w[r], hs[r], hc[r]);
    auto next = [&](uint32_t sa, uint32_t ca, int r, uint32_t sc, uint32_t cc) -> uint32_t {
      if constexpr (CONWAY) return conway_bits(sa, ca, hs[r], hc[r], sc, cc, w[r]);
      else return lifep_rule(sa, ca, hs[r], hc[r], sc, cc, w[r], p.birth, p.survive);
    };
    uint32_t v[K];
#pragma unroll
    for (int r = 1; r + 1 < K; ++r) v[r] = next(hs[r - 1], hc[r - 1], r, hs[r + 1], hc[r + 1]);
    // the neighbours' rows of this generation (the outermost groups': any)
    __syncthreads();
    const int b = (g & 1) * kBuf;
    uint32_t ts, tc, bs, bc;
    lifep_hsum(above[b], ts, tc);
    lifep_hsum(below[b], bs, bc);
    if constexpr (K == 1) {
      v[0] = next(ts, tc, 0, bs, bc);
    } else {
      v[0] = next(ts, tc, 0, hs[1], hc[1]);
      v[K - 1] = next(hs[K - 2], hc[K - 2], K - 1, bs, bc);
    }
    if (reset) {
#pragma unroll
      for (int r = 0; r < K; ++r) v[r] = held(v[r], r);
    }
#pragma unroll
    for (int r = 0; r < K; ++r) w[r] = v[r];
    mine[kBuf - b] = w[0];
    mine[kBuf - b + lpr] = w[K - 1];
  }

  // ---- store
  if (col >= 1 && col <= lpr - 2 && wi < words) {
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const int32_t l = group * K + r, y = y0 + r;  // y >= 0 for every result row
      if (l >= gens && l < groups * K - gens && y < n1) lifep_row(p.dst, p.d1, y, words)[wi] = w[r];
    }
  }
}

// ------------------------------------------------------------ host side

using LifepFn = void (*)(const LifepParams&, hipStream_t);
// The launcher for K rows per wave, and the two conversions (life_packed.hip).
LifepFn lifep_launcher(int k, bool conway, int bc);
void launch_life_pack(LifepParams p, hipStream_t s);
void launch_life_unpack(LifepParams p, hipStream_t s);

}  // namespace sth
