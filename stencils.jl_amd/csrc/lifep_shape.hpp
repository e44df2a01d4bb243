// Tiles of the packed Life kernel (lifep_kernel.hpp): plain C++, with no HIP in it.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

namespace sth {

constexpr int kLifepWaves = 16;   // waves of a workgroup
constexpr int kLifepMaxGens = 32; // a rim word's bits

constexpr int32_t lifep_words(int64_t n0) { return static_cast<int32_t>((n0 + 31) >> 5); }

// Rows per lane, generations per launch and lanes side by side for an
// n0 x n1 grid: those with the least time per generation by a model fitted to measured launches
// (in microseconds, 64 lanes side by side; 8192^2: K = 12, G = 1 / 8 / 15 take 9.4 / 16.7 / 23.6,
// K = 6, G = 7 takes 14.5; 4096^2: K = 6, G = 16 / 23 take 14.8 / 19.0;
// 1501 x 1333: K = 1, G = 4 takes 3.9, K = 3, G = 8 / 16 take 6.4 / 9.3).  A
// launch costs 2.7 and 0.7 per MB of packed grid (its loads and stores are
// not overlapped with generations); a generation costs 0.083 per row of a
// wave and tile a CU holds, and at least its exchange, 0.25 + 0.05 K.
struct LifepShape {
  int32_t k, gens, lpr_shift;
};
constexpr int kLifepRows[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 14, 16};

inline void lifep_grid(int64_t n0, int64_t n1, int k, int gens, int lpr_shift, int32_t* tx, int32_t* ty) {
  const int out = (1 << lpr_shift) - 2;
  *tx = static_cast<int32_t>((lifep_words(n0) + out - 1) / out);
  const int64_t rows = (kLifepWaves << (6 - lpr_shift)) * k - 2 * gens;
  *ty = static_cast<int32_t>((n1 + rows - 1) / rows);
}

inline LifepShape lifep_search(int64_t n0, int64_t n1, bool conway, int cus) {
  LifepShape best{};
  double least = 0;
  const double work = conway ? 1.0 : 2.6;  // operations per word against Conway's 15
  const double fixed = 2.7 + 0.7e-6 * (static_cast<double>(n0) * static_cast<double>(n1) / 8.0);
  for (int sh = 4; sh <= 6; ++sh)
    for (int k : kLifepRows)
      for (int g = 2; g <= kLifepMaxGens && (kLifepWaves << (6 - sh)) * k - 2 * g >= 1; ++g) {
        int32_t tx, ty;
        lifep_grid(n0, n1, k, g, sh, &tx, &ty);
        const int64_t tiles = static_cast<int64_t>(tx) * ty;
        const double per_cu = static_cast<double>((tiles + cus - 1) / cus);
        const double t = fixed / g + std::max(0.25 + 0.05 * k * work, 0.08 + per_cu * 0.083 * k * work);
        if (!best.k || t < least) {
          best = LifepShape{k, g, sh};
          least = t;
        }
      }
  return best;
}

// lifep_search, remembered: some 1300 shapes take it 12 us, which a call of a
// few generations would wait for before its first launch.  The shapes depend
// on these four numbers alone; past kLifepShapes of them all are forgotten.
constexpr size_t kLifepShapes = 1024;
inline LifepShape lifep_shape(int64_t n0, int64_t n1, bool conway, int cus) {
  static std::mutex m;
  static std::map<std::tuple<int64_t, int64_t, bool, int>, LifepShape> known;
  const auto key = std::make_tuple(n0, n1, conway, cus);
  {
    std::lock_guard<std::mutex> lk(m);
    const auto it = known.find(key);
    if (it != known.end()) return it->second;
  }
  const LifepShape s = lifep_search(n0, n1, conway, cus);
  std::lock_guard<std::mutex> lk(m);
  if (known.size() >= kLifepShapes) known.clear();
  known.emplace(key, s);
  return s;
}

}  // namespace sth
