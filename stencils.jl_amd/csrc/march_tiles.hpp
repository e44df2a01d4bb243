// How the marching kernels cut an array into tiles: plain C++ (constexpr, so
// that device code may call it too), with no HIP in it.
#pragma once

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

}  // namespace sth
