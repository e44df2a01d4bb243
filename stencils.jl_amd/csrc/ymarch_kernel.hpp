// Up to G steps of a 2-D radius-1 stencil update per launch (temporal blocking)
// for the steady steps of an iteration: generation t + G from generation t,
// the generations between held in registers.
//
// Every wave works alone (no LDS, no barriers).  Each lane holds one 16-byte
// vector of V cells of a row.  The kYmOut lanes RL .. RL + 55 own the output
// columns X0 .. X0 + 56 V - 1, the RL = ceil(G / V) lanes on either side are
// rims, the rest idle along.
// The wave marches down a chunk of rows: generation-t rows are loaded
// kYmAhead rows ahead into a register queue of raw vectors (nothing touches a
// vector before its row is due, so the compiler waits for that row only),
// and as soon as row i of generation t is there, row i - k of generation
// t + k is computed from rows i - k - 1 .. i - k + 1 of generation t + k - 1
// for k = 1 .. G, each generation keeping three rows in registers.  Row
// i - G of generation t + G is stored.  A launch of fewer generations
// (p.gens < G) lets its first G - gens stages pass rows on unchanged.
// Neighbours along x come from the lane's own vector and, at its ends, from
// the adjacent lanes (DPP wave shifts); along y from the queues.  Chunks
// overlap by G rows on each side.
//
// What bounds it: vector operations and their latency (the bytes of 4096^2
// f32, 8 steps per launch, take 3 us per step).  100 steps of f32 heat on
// 4096^2: 1675 us with two steps per launch, 636 us with eight.  Where the rims
// are most of what eight (six, four) steps compute, the host launches the
// kernel built for two (march_cost.hpp).
//
// Exactness: every value uses the shared fold expressions in offset order,
// every generation is rounded to the storage type as a store would round it,
// Wrap outside cells are translations of inside ones (src/array.jl:167-179)
// and Remove outside cells read padval in every generation
// (src/array.jl:133-135).  Under Reflect the cells of the generations between
// that lie next to the array are replaced by the cells they mirror
// (src/array.jl:154-166) before the next generation reads them.
#pragma once

#include <type_traits>

#include "march_tiles.hpp"
#include "stream_kernel.hpp"
#include "tile_kernel.hpp"
#include "zmarch2_kernel.hpp"

namespace sth {

template <typename Raw>
constexpr int ymarch_v() {
  return 16 / static_cast<int>(sizeof(Raw));
}

// Most steps per launch for a type and a stencil length.  More steps move
// fewer bytes per step but keep more rows in registers and recompute more
// rim: measured per step on 16384^2 (Wrap), f32 Laplacian (L = 4) with 2 / 4 /
// 6 / 8: 207 / 106 / 75 / 60 us; f32 sum of 9 with 4 / 6: 107 / 78 us; bf16
// Laplacian with 2 / 4 / 6: 134 / 86 / 95 us (eight cells per vector: six
// steps need every register).
template <typename Raw>
constexpr int ymarch_gens(int L) {
  return sizeof(Raw) == 2 ? 4 : (L <= 4 ? 8 : 6);
}

// One fold over the stencil at element i of a lane's vector: row slots q0
// (dy = -1), q1, q2; lm / rp are the element left of element 0 and right of
// element V-1 (from the neighbouring lanes) for each row slot.
template <typename S, int OPK, class Sh, int V, int I, class P>
__device__ __forceinline__ void ym_fold_terms(typename AccOf<S, OPK>::type& acc, uint32_t& cnt,
                                              const typename Staged<S>::type (&q0)[V],
                                              const typename Staged<S>::type (&q1)[V],
                                              const typename Staged<S>::type (&q2)[V],
                                              const typename Staged<S>::type (&lm)[3],
                                              const typename Staged<S>::type (&rp)[3], int i, const P& p) {
  if constexpr (I < Sh::L) {
    constexpr int dx = Sh::off[I][0], dy = Sh::off[I][1];
    const auto& q = dy < 0 ? q0 : (dy == 0 ? q1 : q2);
    const int k = i + dx;
    const auto v = k < 0 ? lm[dy + 1] : (k >= V ? rp[dy + 1] : q[k < 0 ? 0 : (k >= V ? V - 1 : k)]);
    fold_step<S, OPK>(acc, cnt, I, v, p);
    ym_fold_terms<S, OPK, Sh, V, I + 1>(acc, cnt, q0, q1, q2, lm, rp, i, p);
  }
}

// c ? x : y on values that stay values: a select between two elements of one
// register array would otherwise become a load through a selected address,
// for which the compiler moves the array to LDS.
template <typename Val>
__device__ __forceinline__ Val select_val(bool c, Val x, Val y) {
  STH_OPAQUE(x);
  STH_OPAQUE(y);
  return c ? x : y;
}

// element `k` of q for the one bit k set in `bits` (bits is a run-time mask)
template <int V, typename Val>
__device__ __forceinline__ Val pick(const Val (&q)[V], uint32_t bits) {
  Val r = q[0];
#pragma unroll
  for (int k = 1; k < V; ++k) r = select_val(((bits >> k) & 1u) != 0, q[k], r);
  return r;
}

template <typename S, int OPK, class Sh, int G, int BC>
__global__ __launch_bounds__(256) void ymarch_kernel(MapParams p) {
  constexpr bool REMOVE = BC == STH_REMOVE, REFLECT = BC == STH_REFLECT;
  using Raw = typename Elem<S>::raw;
  using Val = typename Staged<S>::type;
  using A = typename AccOf<S, OPK>::type;
  using O = typename OutOf<S, OPK>::type;
  using ORaw = typename Elem<O>::raw;
  constexpr int V = ymarch_v<Raw>();
  constexpr int RL = (G + V - 1) / V;  // rim lanes on each side
  static_assert(sizeof(ORaw) == sizeof(Raw), "iterations keep the element type");
  static_assert(Sh::RX <= 1 && Sh::RY <= 1 && Sh::RZ == 0, "2-D radius-1 stencils only");
  static_assert(2 * RL + kYmOut <= 64, "the rims fit beside the output lanes");

  const int lane = static_cast<int>(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int nblocks = p.tiles_x * p.tiles_y;
  const int bid = xcd_block_id(static_cast<int>(blockIdx.x), nblocks, p.xcd_remap);
  const int bx = bid % p.tiles_x;
  const int by = bid / p.tiles_x;

  const int32_t n0 = static_cast<int32_t>(p.src.n0), n1 = static_cast<int32_t>(p.src.n1);
  // four waves of a block take four consecutive row chunks
  const int32_t rc = p.tiles_z;  // rows per chunk
  const int32_t yb = (by * 4 + wave) * rc;
  const int32_t ye = yb + rc < n1 ? yb + rc : n1;
  if (yb >= ye) return;  // uniform: the wave has no rows
  const int32_t gens = p.gens;      // generations of this launch, 1 .. G
  const int idle = G - gens;        // stages that pass rows on
  const YmTiles tiles = ymarch_tiles(n0, p.tiles_x, V, RL);
  const bool whole = n0 % V == 0 || tiles.spread;  // every vector lies wholly inside or outside the row (uniform)
  const int32_t X0 = tiles.first(bx, V);            // first output column
  const Val pv = stage<S>(raw_from_bits<Raw>(p.padval));
  constexpr int64_t es = sizeof(Raw);

  // 32-bit byte offsets (the host checks the extent), loads always inside
  // the array, stores of lanes and cells that own no result dropped by the
  // buffer range check (offset 2^31 is past the destination's extent)
  const __amdgpu_buffer_rsrc_t src = buf_rsrc(p.src.base, 0xffffffffu);
  const int64_t dext = ((p.dst.n1 - 1) * p.dst.s1 + p.dst.n0) * es;
  const __amdgpu_buffer_rsrc_t dst = buf_rsrc(p.dst.base, static_cast<uint32_t>(dext));
  constexpr uint32_t kDrop = 0x80000000u;

  // mapped coordinate of c; cells beyond the G-cell rim feed no stored
  // result and are clamped into it first (n >= kYmMinCells > G, or n > G = 2
  // rows, checked on the host, so every mapped rim cell lies inside the array)
  auto map_c = [&](int32_t c, int32_t n) -> int32_t {
    c = c < -G ? -G : (c > n + G - 1 ? n + G - 1 : c);
    if (c < 0) return REMOVE ? 0 : (REFLECT ? -c : c + n);
    if (c >= n) return REMOVE ? 0 : (REFLECT ? 2 * n - 2 - c : c - n);
    return c;
  };
  // this lane's columns: x0 .. x0 + V - 1
  const int32_t x0 = X0 + V * (lane - RL);
  // whole vectors: one load from column sx on (Reflect: mirrored vectors are
  // reversed after the load)
  const bool vout = x0 < 0 || x0 >= n0;
  uint32_t sxb;
  {
    int32_t sx = x0;
    if (x0 < 0) sx = REMOVE ? 0 : (REFLECT ? 1 - V - x0 : x0 + n0);
    else if (x0 >= n0) sx = REMOVE ? 0 : (REFLECT ? 2 * n0 - 1 - V - x0 : x0 - n0);
    sx = sx < 0 ? 0 : (sx > n0 - V ? n0 - V : sx);  // lanes beyond the rims: any vector
    sxb = static_cast<uint32_t>(sx) * static_cast<uint32_t>(es);
  }
  // otherwise cell by cell where a vector is not wholly inside
  const bool x_direct = x0 >= 0 && x0 + V <= n0;
  uint32_t xb[V];
  bool xout[V];
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int32_t x = x0 + i;
    xout[i] = x < 0 || x >= n0;
    xb[i] = static_cast<uint32_t>(map_c(x, n0)) * static_cast<uint32_t>(es);
  }
  const bool store_lane = lane >= RL && lane < RL + kYmOut;
  uint32_t xs[V];  // store offsets; kDrop where the lane owns no result
#pragma unroll
  for (int i = 0; i < V; ++i)
    xs[i] = store_lane && x0 + i < n0 ? static_cast<uint32_t>(x0 + i) * static_cast<uint32_t>(es) : kDrop;
  const bool store_vec = !store_lane || x0 + V <= n0;  // (a rim lane's whole vector is dropped)

  constexpr int P = kYmAhead;     // and the unroll
  static_assert(P % 3 == 0, "the unroll is a multiple of both rings");
  RawVec<Raw, V> raw[P];          // loaded rows: row i in slot i % P (i = 0 is yb - gens)
  Val h[G][3][V];                 // generation t + k, row i - k in slot i % 3, k = 0 .. G - 1
  Val he[G][3][2];                // the cells left of element 0 / right of element V - 1
#pragma unroll
  for (int k = 0; k < G; ++k)
#pragma unroll
    for (int s = 0; s < 3; ++s) {
#pragma unroll
      for (int i = 0; i < V; ++i) h[k][s][i] = Val(0);
      he[k][s][0] = he[k][s][1] = Val(0);
    }

  // The row loop has three bodies: kPlain (no lane or row leaves the array, or
  // Wrap with whole vectors), kEdge (whole vectors, with the Remove and Reflect
  // fix-ups) and kAny (vectors that straddle an edge, idle stages).
  constexpr int kPlain = 0, kEdge = 1, kAny = 2;
  auto load_row = [&](auto body, int i, RawVec<Raw, V>& r) {
    const uint32_t yoff = static_cast<uint32_t>(static_cast<int64_t>(map_c(yb - gens + i, n1)) * p.src.s1 * es);
    if (decltype(body)::value != kAny || whole) {
      r = buf_load<RawVec<Raw, V>>(src, sxb, yoff);
    } else if (x_direct) {
      r = buf_load<RawVec<Raw, V>>(src, xb[0], yoff);
    } else {
#pragma unroll
      for (int k = 0; k < V; ++k) r.e[k] = buf_load<Raw>(src, xb[k], yoff);
    }
  };
  const bool reversed = REFLECT && whole && vout;
  // lanes outside the row, or all of them on a row outside: a lane mask, so
  // that the selects on it stay selects
  const uint64_t vout_mask = __builtin_amdgcn_ballot_w64(vout);
  auto cells_out = [&](bool yout) -> bool {
    const uint64_t m = yout ? ~uint64_t(0) : vout_mask;
#if __has_builtin(__builtin_amdgcn_inverse_ballot_w64)
    return __builtin_amdgcn_inverse_ballot_w64(m);
#else  // the runtime compiler that comes with PyTorch
    return ((m >> lane) & 1u) != 0;
#endif
  };
  auto stage_row = [&](auto body, int i, const RawVec<Raw, V>& m, Val (&r)[V]) {
    constexpr int B = decltype(body)::value;
    const int32_t y = yb - gens + i;
    const bool yout = y < 0 || y >= n1;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      Raw v = m.e[k];
      if constexpr (B != kPlain && REFLECT) v = select_val(reversed, m.e[V - 1 - k], m.e[k]);
      // a copy, not a rename: the loaded registers are free for the next load,
      // which would otherwise be copied (and waited for) at the loop's end
      r[k] = stage<S>(copy_here(v));
      if constexpr (B == kEdge && REMOVE) r[k] = cells_out(yout) ? pv : r[k];
      if constexpr (B == kAny && REMOVE) r[k] = yout || xout[k] ? pv : r[k];
    }
  };
  // neighbours of a row's end elements from the adjacent lanes
  auto edges = [&](const Val (&r)[V], Val (&e)[2]) {
    e[0] = lane_shift<-1>(r[V - 1]);
    e[1] = lane_shift<1>(r[0]);
  };
  // Reflect: a generation's cells just outside the array, x = -1 and x = n0,
  // take the values of the cells they mirror, x = 1 and x = n0 - 2 -- the
  // reference reads those cells there, and a fold over the mirrored
  // neighbourhood would sum in the reverse order.
  // The lanes and elements concerned are fixed per wave, so the fix-up is
  // selects on per-lane masks, with no branch in the row loop.
  const int32_t pr = n0 - (X0 - RL * V);  // x = n0 in this wave's cells (uniform)
  const bool rim_in = pr >= 0 && pr < 64 * V;
  const int32_t pr_c = rim_in ? pr : 2;  // any in-range position when unused
  const int rim_lane = pr_c / V, rim_elem = pr_c % V;
  const int mir_lane = (pr_c - 2) / V, mir_elem = (pr_c - 2) % V;  // x = n0 - 2
  const bool left_fix = X0 == 0 && lane == RL - 1;
  const bool right_fix = rim_in && lane == rim_lane;
  const bool from_prev = mir_lane != rim_lane;
  // Element choices as bit masks the compiler cannot see through: a runtime
  // element index would make it index the register arrays, which it then
  // moves to LDS.
  uint32_t mir_bits = 1u << mir_elem;
  uint32_t rim_bits = right_fix ? 1u << rim_elem : 0u;
  STH_OPAQUE(mir_bits);
  STH_OPAQUE(rim_bits);
  const bool rim_first = REFLECT && x0 == n0;  // whole vectors: x = n0 is a lane's first cell
  auto reflect_columns = [&](auto body, Val (&r)[V]) {
    if (decltype(body)::value == kEdge || whole) {
      const Val right = lane_shift<1>(r[1]), left = lane_shift<-1>(r[V - 2]);
      r[V - 1] = select_val(left_fix, right, r[V - 1]);
      r[0] = select_val(rim_first, left, r[0]);
      return;
    }
    const Val from_right = lane_shift<1>(r[1]);  // lane l: lane l+1's element 1 (x = 1 for the last left rim lane)
    const Val same = pick<V>(r, mir_bits);
    const Val prev = lane_shift<-1>(same);  // lane l: lane l-1's element mir_elem
    const Val mirrored = from_prev ? prev : same;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      if (k == V - 1) r[k] = left_fix ? from_right : r[k];
      r[k] = ((rim_bits >> k) & 1u) ? mirrored : r[k];
    }
  };

  const bool x_edge = X0 < RL * V || X0 + (64 - RL) * V > n0;
  const bool y_edge = BC != STH_WRAP && (yb < gens || ye + gens > n1);
  auto march = [&](auto body) {
    constexpr int B = decltype(body)::value;
    const int nrow = (ye - yb) + 2 * gens;    // generation-t rows yb - gens .. ye + gens - 1
    const int nit = (ye - yb) + gens + G;     // until row ye - 1 leaves the last stage
#pragma unroll
    for (int i = 0; i < P; ++i) {
      load_row(body, i < nrow ? i : nrow - 1, raw[i]);
      __builtin_amdgcn_sched_barrier(0);  // in row order, as the loop waits for them
    }
    for (int i0 = 0; i0 < nit; i0 += P) {
#pragma unroll
      for (int u = 0; u < P; ++u) {
        // (no exit inside the unrolled rows: the copies it would take at the
        // loop's end wait for every load; rows past ye are dropped.  And no
        // motion between rows: the scheduler would sink the loads.)
        __builtin_amdgcn_sched_barrier(0);
        const int i = i0 + u;
        // row i is due; row i + P (past the chunk: its last row) into its slot
        stage_row(body, i, raw[u], h[0][u % 3]);
        __builtin_amdgcn_sched_barrier(0);
        load_row(body, i + P < nrow ? i + P : nrow - 1, raw[u]);
        edges(h[0][u % 3], he[0][u % 3]);
        // stage k: row yb - gens + i - k, one generation on (k > idle) or as it is
#pragma unroll
        for (int k = 1; k <= G; ++k) {
          // slots of rows j - 1, j, j + 1 (j = i - k) of generation k - 1
          const int a = (u + 1) % 3, b = (u + 2) % 3, c = u % 3;
          auto& r0 = h[k - 1][a];
          const auto& r1 = h[k - 1][b];
          auto& r2 = h[k - 1][c];
          auto& f0 = he[k - 1][a];
          const auto& f1 = he[k - 1][b];
          auto& f2 = he[k - 1][c];
          if (B == kAny && k < G && k <= idle) {
            auto& n = h[k < G ? k : 0][u % 3];
#pragma unroll
            for (int e = 0; e < V; ++e) n[e] = r1[e];
            he[k < G ? k : 0][u % 3][0] = f1[0];
            he[k < G ? k : 0][u % 3][1] = f1[1];
            continue;
          }
          const int32_t y = yb - gens + i - k;
          // Reflect: rows y = -1 and y = n1 of the generations between are
          // rows 1 and n1 - 2 (generation t's are loaded mirrored)
          if (B != kPlain && REFLECT && k > 1) {
            if (y == 0) {
#pragma unroll
              for (int e = 0; e < V; ++e) r0[e] = r2[e];
              f0[0] = f2[0];
              f0[1] = f2[1];
            }
            if (y == n1 - 1) {
#pragma unroll
              for (int e = 0; e < V; ++e) r2[e] = r0[e];
              f2[0] = f0[0];
              f2[1] = f0[1];
            }
          }
          const Val lm[3] = {f0[0], f1[0], f2[0]};
          const Val rp[3] = {f0[1], f1[1], f2[1]};
          RawVec<ORaw, V> out;
#pragma unroll
          for (int e = 0; e < V; ++e) {
            A acc = A(0);
            uint32_t cnt = 0;
            ym_fold_terms<S, OPK, Sh, V, 0>(acc, cnt, r0, r1, r2, lm, rp, e, p);
            out.e[e] = narrow<O>(fold_finish<S, OPK>(acc, cnt, r1[e], Sh::L, p));
          }
          if (k < G) {
            auto& n = h[k < G ? k : 0][u % 3];
#pragma unroll
            for (int e = 0; e < V; ++e) n[e] = stage<S>(out.e[e]);
            if constexpr (B != kPlain && REMOVE) {
              const bool yout = y < 0 || y >= n1;
#pragma unroll
              for (int e = 0; e < V; ++e) n[e] = (B == kEdge ? cells_out(yout) : yout || xout[e]) ? pv : n[e];
            }
            if constexpr (B != kPlain && REFLECT) reflect_columns(body, n);
            edges(n, he[k < G ? k : 0][u % 3]);
          } else {
            // rows before the chunk (the first gens + G steps) and after it are dropped
            const bool st = i >= gens + G && y < ye;
            const uint32_t yoff = st ? static_cast<uint32_t>(static_cast<int64_t>(y) * p.dst.s1 * es) : 0u;
            if (B != kAny || whole || store_vec) {
              buf_store<RawVec<ORaw, V>, kStoreNT>(out, dst, st ? xs[0] : kDrop, yoff);
            } else {
#pragma unroll
              for (int e = 0; e < V; ++e) buf_store<ORaw, kStoreNT>(out.e[e], dst, st ? xs[e] : kDrop, yoff);
            }
          }
        }
      }
    }
  };
  if (idle > 0 || (x_edge && !whole))
    march(std::integral_constant<int, kAny>{});
  else if (BC != STH_WRAP && (x_edge || y_edge))
    march(std::integral_constant<int, kEdge>{});
  else
    march(std::integral_constant<int, kPlain>{});
}

template <typename S, int OPK, class Sh, int G>
void launch_ymarch(const MapParams& p, hipStream_t s) {
  const unsigned nb = static_cast<unsigned>(p.tiles_x) * p.tiles_y;
  if (p.bc == STH_REMOVE)
    hipLaunchKernelGGL((ymarch_kernel<S, OPK, Sh, G, STH_REMOVE>), dim3(nb), dim3(256), 0, s, p);
  else if (p.bc == STH_REFLECT)
    hipLaunchKernelGGL((ymarch_kernel<S, OPK, Sh, G, STH_REFLECT>), dim3(nb), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((ymarch_kernel<S, OPK, Sh, G, STH_WRAP>), dim3(nb), dim3(256), 0, s, p);
}

}  // namespace sth
