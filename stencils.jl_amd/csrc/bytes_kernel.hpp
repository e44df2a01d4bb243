// Maximum / minimum over a stencil of one-byte integers (UInt8, Int8):
// runtime-compiled for a call's offsets, one plane of a 2-D or 3-D array.
//
// The largest or smallest of a set of whole numbers does not depend on the
// order in which they are compared, so the fold is factored: each source row
// is reduced along dim 1 once per distinct set of columns the stencil has in
// a row (runs of columns by doubling), and an output combines its rows'
// results.  5 x 5 without the centre: about 8 operations per two cells
// instead of 23 per cell.
//
// Work split: as the streaming kernel (a lane owns 16 cells of KY rows, a
// wave 2^lpr_shift lanes of a row), with two cells per register: pair i holds
// cells i and i + 8 of the lane's 16 in its 16-bit halves, so a step along
// dim 1 is another register and no shift, and v_pk_max_u16 / v_pk_min_u16
// compare two cells.  A lane's 16 cells are one load, the cells on either
// side one word each, also at a row's ends.  The last lanes of a row start at n0 - 16: no
// load straddles the end, and the cells two lanes share are written twice
// with one value.
//
// Bound by the loads and stores (2 bytes per cell): Moore(2) maximum of
// 8192^2 UInt8 31 us, 4.4 TB/s, with eight rows per lane, 33 with four (88 us
// in the streaming kernel; 38 us with single-byte loads for the cells beside a
// row's ends).
#pragma once

#include "stream_kernel.hpp"

namespace sth {

constexpr int kBytesV = 16;       // cells per lane along dim 1
constexpr int kBytesMinN0 = 32;  // fewest cells of a row: the last lane's left neighbours are inside it

using PairU16 = uint16_t __attribute__((ext_vector_type(2)));

template <int OPK>
__device__ __forceinline__ PairU16 pair_ext(PairU16 a, PairU16 b) {
  if constexpr (OPK == OP_MAX) return __builtin_elementwise_max(a, b);
  else return __builtin_elementwise_min(a, b);
}

// The extreme of N consecutive pairs.  The same sub-runs recur at the
// neighbouring positions and in the other row sets, where the compiler
// finds them computed.
template <int OPK, int N>
__device__ __forceinline__ PairU16 pair_run(const PairU16* q) {
  if constexpr (N == 1) return q[0];
  else if constexpr (N == 2) return pair_ext<OPK>(q[0], q[1]);
  else if constexpr (N == 3) return pair_ext<OPK>(pair_run<OPK, 2>(q), q[2]);
  else if constexpr (N == 4) return pair_ext<OPK>(pair_run<OPK, 2>(q), pair_run<OPK, 2>(q + 2));
  else return pair_ext<OPK>(pair_run<OPK, 4>(q), pair_run<OPK, N - 4>(q + 4));
}

// The extreme of the pairs q[b] whose bit b is set in MASK.
template <int OPK, uint32_t MASK>
__device__ __forceinline__ PairU16 pair_set(const PairU16* q) {
  constexpr int first = __builtin_ctz(MASK);
  constexpr int run = __builtin_ctz(~(MASK >> first));
  constexpr uint32_t rest = MASK & ~(((1u << run) - 1u) << first);
  const PairU16 r = pair_run<OPK, run>(q + first);
  if constexpr (rest == 0) return r;
  else return pair_ext<OPK>(r, pair_set<OPK, rest>(q));
}

// The columns of the stencil's row dy: bit RX + dx.
template <class Sh>
constexpr uint32_t row_columns(int dy) {
  uint32_t m = 0;
  for (int k = 0; k < Sh::L; ++k)
    if (Sh::off[k][1] == dy) m |= 1u << (Sh::RX + Sh::off[k][0]);
  return m;
}

// Source row IY - RY of a lane's rows into the results of output rows J, J + 1, ...
template <int OPK, class Sh, int KY, int IY, int J>
__device__ __forceinline__ void bytes_row(const PairU16* q, PairU16 (&acc)[KY][8], bool (&any)[KY]) {
  if constexpr (J < KY) {
    constexpr int dy = IY - Sh::RY - J;
    if constexpr (dy >= -Sh::RY && dy <= Sh::RY) {
      constexpr uint32_t mask = row_columns<Sh>(dy);
      if constexpr (mask != 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const PairU16 h = pair_set<OPK, mask>(q + i);
          acc[J][i] = any[J] ? pair_ext<OPK>(acc[J][i], h) : h;
        }
        any[J] = true;
      }
    }
    bytes_row<OPK, Sh, KY, IY, J + 1>(q, acc, any);
  }
}

template <int OPK, class Sh, int KY, int IY>
__device__ __forceinline__ void bytes_rows(const uint32_t (&w)[KY + 2 * Sh::RY][6], PairU16 (&acc)[KY][8],
                                           bool (&any)[KY]) {
  if constexpr (IY < KY + 2 * Sh::RY) {
    // pair i of cells i and i + 8 from words i / 4 and i / 4 + 2 (word 0 is the one on the left)
    PairU16 q[8 + 2 * Sh::RX];
#pragma unroll
    for (int k = 0; k < 8 + 2 * Sh::RX; ++k) {
      const int c = k - Sh::RX + 4;
      const uint32_t sel = 0x0c040c00u + 0x00010001u * static_cast<uint32_t>(c & 3);
      q[k] = __builtin_bit_cast(PairU16, __builtin_amdgcn_perm(w[IY][c / 4 + 2], w[IY][c / 4], sel));
    }
    bytes_row<OPK, Sh, KY, IY, 0>(q, acc, any);
    bytes_rows<OPK, Sh, KY, IY + 1>(w, acc, any);
  }
}

template <typename S, int OPK, class Sh, int KY>
__global__ __launch_bounds__(256) void bytes_kernel(MapParams p) {
  static_assert(sizeof(S) == 1 && (OPK == OP_MAX || OPK == OP_MIN), "extremes of one-byte integers");
  static_assert(Sh::RX <= 3 && Sh::RZ == 0, "the columns beside a lane's cells are one word; one plane");
  constexpr int RX = Sh::RX, RY = Sh::RY, V = kBytesV, NY = KY + 2 * RY;
  const int nblocks = p.tiles_x * p.tiles_y * p.tiles_z;
  const int bid = xcd_block_id(static_cast<int>(blockIdx.x), nblocks, p.xcd_remap);
  const int bx = bid % p.tiles_x;
  const int byz = bid / p.tiles_x;
  const int64_t z0 = byz / p.tiles_y;
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);

  const int64_t n0 = p.src.n0, n1 = p.src.n1;
  const int lsh = p.lpr_shift, LPR = 1 << lsh, RPW = 64 >> lsh;
  const int64_t wy0 = (static_cast<int64_t>(byz % p.tiles_y) * 4 + wave) * KY * RPW;
  if (wy0 >= n1) return;  // uniform: the wave has no rows (no barrier follows)
  const int64_t y0 = wy0 + static_cast<int64_t>(lane >> lsh) * KY;
  const int64_t wx0 = static_cast<int64_t>(bx) * LPR * V;
  const int64_t xl = wx0 + static_cast<int64_t>(lane & (LPR - 1)) * V;
  const int64_t x0 = xl < n0 - V ? xl : n0 - V;  // n0 >= kBytesMinN0 (host)
  const bool halo = p.read_halo != 0;
  const int64_t h0 = halo ? p.src.h0 : 0, h1 = halo ? p.src.h1 : 0;
  const uint8_t* __restrict__ sbase = reinterpret_cast<const uint8_t*>(p.src.base) + z0 * p.src.s2;
  const int64_t s1 = p.src.s1;
  const bool rows_direct = wy0 - RY >= -h1 && wy0 + RPW * KY - 1 + RY < n1 + h1;
  const bool x_direct = wx0 - 4 >= -h0 && wx0 + LPR * V + 4 <= n0 + h0;
  const uint32_t pv = static_cast<uint32_t>(p.padval & 0xffu) * 0x01010101u;

  uint32_t w[NY][6];  // the word left of the lane's cells, their four, the word on the right
  if (rows_direct && x_direct) {
#pragma unroll
    for (int iy = 0; iy < NY; ++iy) {
      const uint8_t* row = sbase + (y0 - RY + iy) * s1 + x0;
      __builtin_memcpy(&w[iy][1], row, 16);
      if constexpr (RX > 0) {
        __builtin_memcpy(&w[iy][0], row - 4, 4);
        __builtin_memcpy(&w[iy][5], row + 16, 4);
      }
    }
  } else {
    // Per lane: where the words holding the RX cells on either side start,
    // and the bytes of (padval, word) that go where the fast path has them.
    // A lane's neighbours are inside the array (or the halo), or all outside,
    // where they are RX cells in a row elsewhere, forwards (Wrap) or backwards
    // (Reflect); only a row end less than RX cells past a lane's last cell
    // mixes both, and there the word is put together byte by byte.
    constexpr uint32_t kSame = 0x03020100u, kBack = 0x00010203u, kPad = 0x07060504u;
    constexpr uint32_t kUp = RX == 1 ? 0x000c0c0cu : (RX == 2 ? 0x01000c0cu : 0x0201000cu);
    constexpr uint32_t kDown = RX == 1 ? 0x0c0c0c03u : (RX == 2 ? 0x0c0c0302u : 0x0c030201u);
    int64_t xl4 = x0 - RX, xr4 = x0 + V + RX - 4;
    uint32_t sel_l = kUp, sel_r = kDown;
    if (xl4 < -h0) {
      xl4 = p.bc == STH_WRAP ? n0 - 4 : (p.bc == STH_REMOVE ? 0 : 1);
      sel_l = p.bc == STH_WRAP ? kSame : (p.bc == STH_REMOVE ? kPad : kBack);
    }
    const bool mixed = x0 + V < n0 + h0 && x0 + V + RX > n0 + h0;
    if (x0 + V + RX > n0 + h0) {
      xr4 = p.bc == STH_WRAP ? 0 : (p.bc == STH_REMOVE ? 0 : n0 - 5);
      sel_r = p.bc == STH_WRAP ? kSame : (p.bc == STH_REMOVE ? kPad : kBack);
    }
    const bool any_mixed = RX > 1 && __any(mixed);
    int32_t xm[RX + 1];
    bool xpad[RX + 1];
#pragma unroll
    for (int i = 0; i < RX; ++i) {
      xpad[i] = false;
      xm[i] = static_cast<int32_t>(resolve_row(x0 + V + i, n0, h0, RX, halo, p.bc, xpad[i]));
    }
#pragma unroll
    for (int iy = 0; iy < NY; ++iy) {
      bool pad = false;
      const int64_t ym = resolve_row(y0 - RY + iy, n1, h1, RY, halo, p.bc, pad);
      const uint8_t* row = sbase + ym * s1;
      __builtin_memcpy(&w[iy][1], row + x0, 16);
      w[iy][0] = w[iy][5] = 0;
      if constexpr (RX > 0) {
        uint32_t l, r;
        __builtin_memcpy(&l, row + xl4, 4);
        __builtin_memcpy(&r, row + xr4, 4);
        w[iy][0] = __builtin_amdgcn_perm(pv, l, sel_l);
        w[iy][5] = __builtin_amdgcn_perm(pv, r, sel_r);
        if (any_mixed) {
          w[iy][5] = 0;
#pragma unroll
          for (int i = 0; i < RX; ++i)
            w[iy][5] |= (xpad[i] ? pv & 0xffu : static_cast<uint32_t>(row[xm[i]])) << (8 * i);
        }
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) w[iy][k] = pad ? pv : w[iy][k];
    }
  }
  // signed cells compare as unsigned ones with their top bit flipped
  constexpr uint32_t kFlip = Elem<S>::is_signed ? 0x80808080u : 0u;
  if constexpr (kFlip != 0) {
#pragma unroll
    for (int iy = 0; iy < NY; ++iy)
#pragma unroll
      for (int k = 0; k < 6; ++k) w[iy][k] ^= kFlip;
  }
  PairU16 acc[KY][8];
  bool any[KY];
#pragma unroll
  for (int j = 0; j < KY; ++j) any[j] = false;
  bytes_rows<OPK, Sh, KY, 0>(w, acc, any);

  uint8_t* __restrict__ dbase = reinterpret_cast<uint8_t*>(p.dst.base) + z0 * p.dst.s2;
#pragma unroll
  for (int j = 0; j < KY; ++j) {
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint32_t a[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = __builtin_bit_cast(uint32_t, acc[j][4 * k + i]);
      const uint32_t lo = __builtin_amdgcn_perm(a[1], a[0], 0x06020400u);  // cells 0, 1, 8, 9
      const uint32_t hi = __builtin_amdgcn_perm(a[3], a[2], 0x06020400u);
      o[k] = __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ kFlip;
      o[k + 2] = __builtin_amdgcn_perm(hi, lo, 0x07060302u) ^ kFlip;
    }
    if (y0 + j < n1 && xl < n0) __builtin_memcpy(dbase + (y0 + j) * p.dst.s1 + x0, o, 16);
  }
}

}  // namespace sth
