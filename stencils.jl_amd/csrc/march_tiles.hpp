// How the marching kernels cut an array into tiles: plain C++ (constexpr, so
// that device code may call it too), with no HIP in it.
#pragma once

#include <stdint.h>

namespace sth {

// Output lanes per wave of ymarch_kernel: 56 lanes of 16 bytes make each row
// segment a whole number of 128-byte lines (62 lanes measured 7% slower on
// 16384^2 f32 from partial-line writes), and leave up to four rim lanes on
// each side.
constexpr int kYmOut = 56;

// The column tiles of ymarch_kernel: `tiles` of 56 vectors of `v` cells over
// a row of n0 >= 1 cells, with `rim` vectors beside each.
struct YmTiles {
  int step, rest;  // spread tiles start step or step + 1 (the first `rest` of them) cells apart
  bool spread;     // tiles end at the row's end, not at whole multiples of their width

  // First column of tile b.  (The remainder goes to the first steps one cell
  // each: two tiles are never further apart than a tile is wide.)
  constexpr int first(int b, int v) const {
    return spread ? b * step + (b < rest ? b : rest) : b * kYmOut * v;
  }
};

// Tiles of a row that is no whole number of vectors are spread evenly with the
// last one ending at the row's end, so that no lane's vector straddles either
// edge (cells of two tiles are computed and stored twice, with the same
// values), unless the first two are closer than a rim.
constexpr YmTiles ymarch_tiles(int n0, int tiles, int v, int rim) {
  const int slack = n0 - kYmOut * v;  // the last tile's first column
  const int step = tiles > 1 ? slack / (tiles - 1) : 0;
  return YmTiles{step, tiles > 1 ? slack - step * (tiles - 1) : 0, n0 % v != 0 && step >= rim * v};
}

// Fewest steps per launch that ymarch_kernel is built for.
constexpr int kYmShortGens = 2;

// Fewest cells per axis: more than the rims and a vector.
constexpr int kYmMinCells = 16;

// Rows loaded ahead of the row consumed: two workgroups per CU (the
// registers' limit) need six.  4096^2 f32, 8 generations: 6.9 us per step with
// three rows ahead, 5.3 with six.
constexpr int kYmAhead = 6;

// The name of ymarch_kernel built for `gens` steps per launch.
constexpr const char* ymarch_name(int gens) {
  return gens == 8 ? "ymarch/8" : gens == 6 ? "ymarch/6" : gens == 4 ? "ymarch/4" : "ymarch/2";
}

struct YmGrid {
  int64_t tx, ty, rows;  // column tiles, groups of four row chunks, rows per chunk
};

// Grid of ymarch_kernel for an n0 x n1 array: 56 V-column tiles x groups of
// four row chunks; the chunk length travels in tiles_z.  A wave's time is
// rows + 2 G row steps, each about w + 1/4 of a wave's issue time on a CU
// that holds w workgroups (and no less than 1.6 of it alone, where latency
// shows), so one or two workgroups per CU, or a few rounds of two, are
// compared: 4096^2 f32, 8 generations: one per CU 64 us, two 48 us, three
// 50 us; a partial second round costs a whole one.
constexpr YmGrid ymarch_grid(int64_t n0, int64_t n1, int v, int gens, int64_t cus) {
  const int64_t gx = (n0 + kYmOut * v - 1) / (kYmOut * v);
  if (gens == kYmShortGens) {  // bound by memory: as many waves as fill every SIMD several times over
    const int64_t chunks = (32 * cus + gx - 1) / gx;
    int64_t rc = (n1 + chunks - 1) / chunks;
    if (rc < 14) rc = 14;
    rc = (rc + 2 * gens + kYmAhead - 1) / kYmAhead * kYmAhead - 2 * gens;
    return YmGrid{gx, (n1 + 4 * rc - 1) / (4 * rc), rc};
  }
  int64_t best_rc = n1;
  double least = 0;
  for (int c = 0; c < 6; ++c) {  // one workgroup per CU, then 1 .. 5 rounds of two
    const int64_t blocks = c == 0 ? cus : 2 * cus * c;
    const int64_t g = blocks / gx > 0 ? blocks / gx : 1;
    // row steps come in whole unrolled groups
    const int64_t steps = ((n1 + 4 * g - 1) / (4 * g) + 2 * gens + kYmAhead - 1) / kYmAhead * kYmAhead;
    const int64_t rc = steps - 2 * gens;
    const int64_t total = gx * ((n1 + 4 * rc - 1) / (4 * rc));
    const double rounds = static_cast<double>((total + 2 * cus - 1) / (2 * cus));
    const double t = static_cast<double>(steps) * (total <= cus ? 1.6 : 2.25 * rounds);
    if (c == 0 || t < least) {
      least = t;
      best_rc = rc;
    }
  }
  return YmGrid{gx, (n1 + 4 * best_rc - 1) / (4 * best_rc), best_rc};
}

constexpr int kZmGens = 4;   // most steps per launch of zmarch_kernel
constexpr int kZmWaves = 8;  // two per SIMD: a wave takes up to 256 registers
constexpr int kZmRows = 8;   // rows per wave
constexpr int kZmOutX = 64 - 2 * kZmGens;
constexpr int kZmOutY = kZmWaves * kZmRows - 2 * kZmGens;
constexpr int kZmMinCells = 16;  // fewest cells per axis: more than the rims

// Plane steps of a workgroup of zmarch_kernel that owns zc planes: they and
// 2 G of overlap, in whole unrolled groups of six.
constexpr int64_t zmarch_steps(int64_t zc) { return (zc + 2 * kZmGens + 5) / 6 * 6; }

struct ZmGrid {
  int64_t tx, ty, tz;  // tiles along dims 1 and 2, chunks of planes
  int64_t time;        // its rounds of workgroups times their plane steps
};

// Grid of zmarch_kernel for an n0 x n1 x n2 array on `cus` compute units (a
// workgroup fills one): the fewest z chunks of those that make whole rounds
// shortest.  For each number of rounds, the chunks that fill them give the
// fewest plane steps, and the fewest chunks of as many steps are taken; more
// rounds end the search once what the planes and the overlaps take at least
// is past the best.  (A walk over every chunk count took 7 ms of host time at
// n2 = 10^6, this one 0.1 us.)
constexpr ZmGrid zmarch_grid(int64_t n0, int64_t n1, int64_t n2, int64_t cus) {
  const int64_t gx = (n0 + kZmOutX - 1) / kZmOutX, gy = (n1 + kZmOutY - 1) / kZmOutY, g = gx * gy;
  ZmGrid best{gx, gy, 1, (g + cus - 1) / cus * zmarch_steps(n2)};
  for (int64_t rounds = (g + cus - 1) / cus; rounds * 2 * kZmGens + g * n2 / cus < best.time; ++rounds) {
    const int64_t fill = rounds * cus / g, most = fill < n2 ? fill : n2;
    const int64_t steps = zmarch_steps((n2 + most - 1) / most), zc = steps - 2 * kZmGens;
    const int64_t chunks = (n2 + zc - 1) / zc;
    const int64_t time = (g * chunks + cus - 1) / cus * steps;
    if (time < best.time) best = ZmGrid{gx, gy, chunks, time};
    if (most == n2) break;
  }
  return best;
}

}  // namespace sth
