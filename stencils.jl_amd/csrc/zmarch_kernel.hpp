// Up to G steps of a 3-D star stencil (VonNeumann(1, 3)) per launch for the
// steady steps of an iteration: generation t + G from generation t, the
// generations between held in registers.
//
// A workgroup of kZmWaves waves owns 64 columns (one per lane) by
// kZmWaves R rows (R per wave) and marches through a chunk of z planes.
// Generation-t planes are loaded kZmAhead planes ahead; as soon as plane i of
// generation t is there, plane i - k of generation t + k is computed from
// planes i - k - 1 .. i - k + 1 of generation t + k - 1 for k = 1 .. G, each
// generation keeping three planes of R rows per lane in registers.  Plane
// i - G of generation t + G is stored: the inner (64 - 2 G) x (rows - 2 G)
// cells, the rest is rim.  Neighbours along z are in the lane's own planes,
// along x in the adjacent lanes (DPP wave shifts), along y in the lane's own
// rows or, for a wave's first and last row, in the wave beside it, which
// leaves its first and last rows in LDS: those of a plane computed in one
// step of the march are read in the next, so one barrier per step and two
// buffers are enough.  Chunks overlap by G planes on each side.  A launch of
// fewer generations (p.gens < G) lets its first G - gens stages pass planes on.
//
// What bounds it: vector operations (9 per cell and step for the Laplacian,
// twice that with the rims and overlaps of 256^3).  Two steps per launch and
// waves that work alone (zmarch2_kernel) are bound by memory.  100 steps of
// f32 heat on 256^3: 1730 us with zmarch2_kernel, 1160 us with this one.
//
// Exactness: every value uses the shared fold expressions in offset order and
// every generation is rounded to the storage type as a store would round it.
// Under Wrap outside cells are translations of inside ones (src/array.jl:167-179).
// Under Remove and Reflect no outside cell is kept: a cell at the array's edge
// takes padval (src/array.jl:133-135) or the cell on its other side, which is
// the one the reference's mirrored index reads (src/array.jl:154-166).
#pragma once

#include <type_traits>

#include "march_tiles.hpp"
#include "zmarch2_kernel.hpp"

namespace sth {

constexpr int kZmAhead = 3;  // planes loaded ahead

// Offsets along one axis at a time, one cell: what the kernel's exchange covers.
template <class Sh>
constexpr bool is_star3() {
  for (int k = 0; k < Sh::L; ++k) {
    int s = 0;
    for (int d = 0; d < 3; ++d) s += Sh::off[k][d] < 0 ? -Sh::off[k][d] : Sh::off[k][d];
    if (s > 1) return false;
  }
  return true;
}

// The seven values a star stencil reads.
template <typename Val>
struct Star {
  Val c, xm, xp, ym, yp, zm, zp;
};

template <typename S, int OPK, class Sh, int I, class P>
__device__ __forceinline__ void star_fold(typename AccOf<S, OPK>::type& acc, uint32_t& cnt,
                                          const Star<typename Staged<S>::type>& v, const P& p) {
  if constexpr (I < Sh::L) {
    constexpr int dx = Sh::off[I][0], dy = Sh::off[I][1], dz = Sh::off[I][2];
    fold_step<S, OPK>(acc, cnt, I,
                      dx < 0 ? v.xm : dx > 0 ? v.xp : dy < 0 ? v.ym : dy > 0 ? v.yp : dz < 0 ? v.zm : dz > 0 ? v.zp : v.c,
                      p);
    star_fold<S, OPK, Sh, I + 1>(acc, cnt, v, p);
  }
}

template <typename S, int OPK, class Sh, int BC>
__global__ __launch_bounds__(64 * kZmWaves) void zmarch_kernel(MapParams p) {
  using Raw = typename Elem<S>::raw;
  using Val = typename Staged<S>::type;
  using A = typename AccOf<S, OPK>::type;
  using O = typename OutOf<S, OPK>::type;
  constexpr int G = kZmGens, R = kZmRows, NW = kZmWaves;
  static_assert(is_star3<Sh>(), "star stencils of reach 1");
  static_assert(sizeof(Val) == 4 && sizeof(typename Elem<O>::raw) == sizeof(Raw), "4-byte values");
  constexpr uint32_t es = sizeof(Raw);

  // first and last row of every wave, per generation, of the last step's planes
  __shared__ Val border[2][G][NW][2][64];

  const int lane = static_cast<int>(threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int nblocks = p.tiles_x * p.tiles_y * p.tiles_z;
  const int bid = xcd_block_id(static_cast<int>(blockIdx.x), nblocks, p.xcd_remap);
  const int bx = bid % p.tiles_x;
  const int bt = bid / p.tiles_x;
  const int by = bt % p.tiles_y;
  const int bz = bt / p.tiles_y;
  const int32_t n0 = static_cast<int32_t>(p.src.n0), n1 = static_cast<int32_t>(p.src.n1),
                n2 = static_cast<int32_t>(p.src.n2);
  const int32_t zc = (n2 + p.tiles_z - 1) / p.tiles_z;
  const int32_t zb = bz * zc;
  const int32_t ze = zb + zc < n2 ? zb + zc : n2;
  if (zb >= ze) return;  // the whole workgroup: no barrier is missed
  const int32_t gens = p.gens;  // generations of this launch, 1 .. G
  const int idle = G - gens;
  const int32_t x = bx * kZmOutX - G + lane;
  const int32_t Y0 = by * kZmOutY - G + wave * R;  // the wave's first row
  const Val pv = stage<S>(raw_from_bits<Raw>(p.padval));

  // 32-bit byte offsets (the host checks the extent); loads stay inside the
  // array, stores of lanes that own no result are dropped by the range check
  const __amdgpu_buffer_rsrc_t src = buf_rsrc(p.src.base, 0xffffffffu);
  const int64_t dext = ((p.dst.n2 - 1) * p.dst.s2 + (p.dst.n1 - 1) * p.dst.s1 + p.dst.n0) * es;
  const __amdgpu_buffer_rsrc_t dst = buf_rsrc(p.dst.base, static_cast<uint32_t>(dext));
  // Wrap: the mapped coordinate (n >= kZmMinCells > G: one wrap; beyond the rim
  // clamped into it); else any cell inside
  auto map_c = [&](int32_t c, int32_t n) -> int32_t {
    if (BC == STH_WRAP) {
      c = c < -G ? -G : (c > n + G - 1 ? n + G - 1 : c);
      return c < 0 ? c + n : (c >= n ? c - n : c);
    }
    return c < 0 ? 0 : (c >= n ? n - 1 : c);
  };
  const uint32_t xb = static_cast<uint32_t>(map_c(x, n0)) * es;
  const bool store_lane = lane >= G && lane < 64 - G && x < n0;
  const uint32_t xbo = store_lane ? static_cast<uint32_t>(x) * es : 0x80000000u;
  uint32_t yload[R];  // uniform
#pragma unroll
  for (int r = 0; r < R; ++r)
    yload[r] = static_cast<uint32_t>(static_cast<int64_t>(map_c(Y0 + r, n1)) * p.src.s1) * es;
  // the rows this wave stores: r0 .. r1 - 1
  const int32_t ylo = by * kZmOutY, yhi = ylo + kZmOutY < n1 ? ylo + kZmOutY : n1;

  Raw raw[kZmAhead][R];  // loaded planes: plane i in slot i % kZmAhead (i = 0 is zb - gens)
  Val h[G][3][R];        // generation t + k, plane i - k in slot i % 3
#pragma unroll
  for (int k = 0; k < G; ++k)
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int r = 0; r < R; ++r) h[k][s][r] = Val(0);

  const int nplane = (ze - zb) + 2 * gens;  // generation-t planes zb - gens .. ze + gens - 1
  const int nit = (ze - zb) + gens + G;
  auto load_plane = [&](int i, Raw (&q)[R]) {
    const int j = i < nplane ? i : nplane - 1;
    const uint32_t zoff = static_cast<uint32_t>(static_cast<int64_t>(map_c(zb - gens + j, n2)) * p.src.s2) * es;
#pragma unroll
    for (int r = 0; r < R; ++r) q[r] = buf_load<Raw>(src, xb, zoff + yload[r]);
  };
  const int up = wave > 0 ? wave - 1 : 0, down = wave < NW - 1 ? wave + 1 : NW - 1;  // (rim rows at the ends)
  // the array's edges in this wave: x = -1 is lane G - 1 of the first tile and
  // y = -1 row G - 1 of its first wave; x = n0 any lane, y = n1 - 1 any row
  const bool left = bx == 0, top = by == 0 && wave == 0;
  const bool at_end = x == n0, right = n0 - (bx * kZmOutX - G) < 64;
  const int rh = n1 - 1 - Y0;
  const bool bottom = rh >= 0 && rh < R;
  static_assert(G + 1 < R && G + 1 < 16, "the cells mirrored at the first edges are in the same wave and DPP row");
  // lanes 0 .. 3 take the values of lanes 2 .. 5 (x = -1 that of x = 1)
  auto mirror_left = [](Val v) -> Val {
    const int w = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(Val, __builtin_amdgcn_update_dpp(w, w, 0x102 /* row_shl:2 */, 0x1, 0x1, false));
  };

  // Bodies of the march: kPlain (Wrap, or no cell of the workgroup sees the
  // array's edge), kEdge, kAny (also idle stages).
  constexpr int kPlain = 0, kEdge = 1, kAny = 2;
  auto march = [&](auto body) {
    constexpr int B = decltype(body)::value;
    constexpr bool EDGE = B != kPlain && BC != STH_WRAP;
#pragma unroll
    for (int i = 0; i < kZmAhead; ++i) load_plane(i, raw[i]);
    for (int i0 = 0; i0 < nit; i0 += 6) {
#pragma unroll
      for (int u = 0; u < 6; ++u) {
        // (steps past the end compute planes that are not stored: every wave
        // meets every barrier)
        const int i = i0 + u;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; ++r) h[0][u % 3][r] = stage<S>(copy_here(raw[u % kZmAhead][r]));
        __builtin_amdgcn_sched_barrier(0);
        load_plane(i + kZmAhead, raw[u % kZmAhead]);
        // the rows beside this wave's, of the planes that the last step made
        const int rd = (u + 1) & 1, wr = u & 1;
        Val above[G], below[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
          above[k] = border[rd][k][up][1][lane];
          below[k] = border[rd][k][down][0][lane];
        }
        border[wr][0][wave][0][lane] = h[0][u % 3][0];
        border[wr][0][wave][1][lane] = h[0][u % 3][R - 1];
        // stage k: plane z = zb - gens + i - k
#pragma unroll
        for (int k = 1; k <= G; ++k) {
          auto& q0 = h[k - 1][(u + 1) % 3];
          auto& q1 = h[k - 1][(u + 2) % 3];
          auto& q2 = h[k - 1][u % 3];
          const int32_t z = zb - gens + i - k;
          if constexpr (EDGE) {
            // The cells outside that this plane's edge cells read take padval,
            // or the value of the cell on the edge cell's other side; each
            // branch is uniform and skipped by waves away from that edge.
            constexpr bool REM = BC == STH_REMOVE;
            if (z == 0) {
#pragma unroll
              for (int r = 0; r < R; ++r) q0[r] = REM ? pv : q2[r];
            }
            if (z == n2 - 1) {
#pragma unroll
              for (int r = 0; r < R; ++r) q2[r] = REM ? pv : q0[r];
            }
            if (top) q1[G - 1] = REM ? pv : q1[G + 1];
            if (bottom) {
#pragma unroll
              for (int r = 0; r < R; ++r) {
                const Val m = REM ? pv : (r > 0 ? q1[r > 0 ? r - 1 : 0] : above[k - 1]);
                if (r < R - 1) q1[r < R - 1 ? r + 1 : 0] = r == rh ? m : q1[r < R - 1 ? r + 1 : 0];
                else below[k - 1] = r == rh ? m : below[k - 1];
              }
            }
            if (left) {
#pragma unroll
              for (int r = 0; r < R; ++r) q1[r] = REM ? (lane < G ? pv : q1[r]) : mirror_left(q1[r]);
            }
            if (right) {
#pragma unroll
              for (int r = 0; r < R; ++r) {
                const Val m = REM ? pv : lane_shift<-1>(lane_shift<-1>(q1[r]));
                q1[r] = at_end ? m : q1[r];
              }
            }
          }
          auto cell = [&](int r) {
            const int32_t y = Y0 + r;
            Star<Val> v;
            v.c = q1[r];
            v.xm = lane_shift<-1>(q1[r]);
            v.xp = lane_shift<1>(q1[r]);
            v.ym = r > 0 ? q1[r > 0 ? r - 1 : 0] : above[k - 1];
            v.yp = r < R - 1 ? q1[r < R - 1 ? r + 1 : 0] : below[k - 1];
            v.zm = q0[r];
            v.zp = q2[r];
            A acc = A(0);
            uint32_t cnt = 0;
            star_fold<S, OPK, Sh, 0>(acc, cnt, v, p);
            return narrow<O>(fold_finish<S, OPK>(acc, cnt, v.c, Sh::L, p));
          };
          if (k < G) {
            const bool pass = B == kAny && k <= idle;
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const auto res = cell(r);
              h[k < G ? k : 0][u % 3][r] = B == kAny && pass ? q1[r] : stage<S>(res);
            }
          } else if (i >= gens + G && z < ze) {
            // (one branch for the plane, the rows that are not stored dropped:
            // a shift from another lane joins the sum it feeds only within a block)
            const uint32_t zst = static_cast<uint32_t>(static_cast<int64_t>(z) * p.dst.s2) * es;
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const int32_t y = Y0 + r;
              const bool own = y >= ylo && y < yhi;
              const auto res = cell(r);
              buf_store<Raw>(res, dst, own ? xbo : 0x80000000u,
                             own ? zst + static_cast<uint32_t>(static_cast<int64_t>(y) * p.dst.s1) * es : 0u);
            }
          }
          if (k < G) {
            border[wr][k < G ? k : 0][wave][0][lane] = h[k < G ? k : 0][u % 3][0];
            border[wr][k < G ? k : 0][wave][1][lane] = h[k < G ? k : 0][u % 3][R - 1];
          }
        }
        __syncthreads();
      }
    }
  };
  const int32_t X0 = bx * kZmOutX - G, YB = by * kZmOutY - G;
  const bool edge = BC != STH_WRAP && (X0 <= 0 || X0 + 64 >= n0 || YB <= 0 || YB + NW * R >= n1 || zb <= gens ||
                                       ze + gens >= n2);
  if (Y0 >= n1 + G) {  // rows that feed no result: only the barriers
    for (int i = 0; i < (nit + 5) / 6 * 6; ++i) __syncthreads();
    return;
  }
  if (idle > 0) march(std::integral_constant<int, kAny>{});
  else if (edge) march(std::integral_constant<int, kEdge>{});
  else march(std::integral_constant<int, kPlain>{});
}

template <typename S, int OPK, class Sh>
void launch_zmarch(const MapParams& p, hipStream_t s) {
  const unsigned nb = static_cast<unsigned>(p.tiles_x) * p.tiles_y * p.tiles_z;
  if (p.bc == STH_REMOVE)
    hipLaunchKernelGGL((zmarch_kernel<S, OPK, Sh, STH_REMOVE>), dim3(nb), dim3(64 * kZmWaves), 0, s, p);
  else if (p.bc == STH_REFLECT)
    hipLaunchKernelGGL((zmarch_kernel<S, OPK, Sh, STH_REFLECT>), dim3(nb), dim3(64 * kZmWaves), 0, s, p);
  else
    hipLaunchKernelGGL((zmarch_kernel<S, OPK, Sh, STH_WRAP>), dim3(nb), dim3(64 * kZmWaves), 0, s, p);
}

}  // namespace sth
