// Packed Life iterations (lifep_kernel.hpp): the byte <-> bit conversions, and
// the instances and launchers of the generation kernel.
#include "lifep_kernel.hpp"

namespace sth {

namespace {

// 16 bytes, any value -> 16 bits (bit i: byte i is nonzero).
__device__ __forceinline__ uint32_t pack16_any(const uint4 v) {
  uint4 n;
  n.x = norm01(v.x);
  n.y = norm01(v.y);
  n.z = norm01(v.z);
  n.w = norm01(v.w);
  return pack16(n);
}

// 16 bytes at any address: one load or store instruction (the target runs
// global accesses in unaligned mode).
__device__ __forceinline__ uint4 load16(const uint8_t* p) {
  uint4 v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}

// Packs a grid of bytes (any value; nonzero is alive), one word per lane.
// The last word of a row reads the row's last 32 cells.  Four rows per
// thread keep eight loads in flight.
constexpr int kLifeIoRows = 4;
__global__ __launch_bounds__(256) void life_pack_kernel(LifepParams p) {
  const int32_t n0 = p.n0, n1 = p.n1, words = p.words;
  const int bx = static_cast<int>(blockIdx.x) % p.tiles_x, by = static_cast<int>(blockIdx.x) / p.tiles_x;
  const int32_t wi = bx * 256 + static_cast<int>(threadIdx.x);
  if (wi >= words) return;
  const int32_t x = wi * 32 + 32 <= n0 ? wi * 32 : n0 - 32;
  const int up = wi * 32 - x;  // cells of the load before the word
  uint4 lo[kLifeIoRows], hi[kLifeIoRows];
#pragma unroll
  for (int j = 0; j < kLifeIoRows; ++j) {
    const int32_t y = by * kLifeIoRows + j < n1 ? by * kLifeIoRows + j : n1 - 1;
    const uint8_t* row = reinterpret_cast<const uint8_t*>(p.src) + static_cast<int64_t>(y) * p.s1 + x;
    lo[j] = load16(row);
    hi[j] = load16(row + 16);
  }
#pragma unroll
  for (int j = 0; j < kLifeIoRows; ++j) {
    const int32_t y = by * kLifeIoRows + j;
    if (y < n1) lifep_row(p.dst, p.d1, y, words)[wi] = (pack16_any(lo[j]) | (pack16_any(hi[j]) << 16)) >> up;
  }
}

// Unpacks a grid, 16 cells per lane; the last lane of a row writes the row's
// last 16 cells (some of them a second time, with the same values).
__global__ __launch_bounds__(256) void life_unpack_kernel(LifepParams p) {
  const int32_t n0 = p.n0, n1 = p.n1, words = p.words;
  const int bx = static_cast<int>(blockIdx.x) % p.tiles_x, by = static_cast<int>(blockIdx.x) / p.tiles_x;
  int32_t x = (bx * 256 + static_cast<int>(threadIdx.x)) * 16;
  if (x >= n0) return;
  if (x + 16 > n0) x = n0 - 16;
  uint32_t v[kLifeIoRows];
#pragma unroll
  for (int k = 0; k < kLifeIoRows; ++k) {
    const int32_t y = by * kLifeIoRows + k < n1 ? by * kLifeIoRows + k : n1 - 1;
    v[k] = lifep_bits(lifep_row(p.src, p.s1, y, words), x, words);
  }
#pragma unroll
  for (int k = 0; k < kLifeIoRows; ++k) {
    const int32_t y = by * kLifeIoRows + k;
    const uint4 cells = unpack16(v[k] << 8);
    if (y < n1) __builtin_memcpy(p.dst + static_cast<int64_t>(y) * p.d1 + x, &cells, sizeof cells);
  }
}

template <int K, bool CONWAY, int BC>
void launch_lifep(const LifepParams& p, hipStream_t s) {
  hipLaunchKernelGGL((lifep_kernel<K, CONWAY, BC>), dim3(static_cast<unsigned>(p.tiles_x) * p.tiles_y),
                     dim3(kLifepWaves * 64), 0, s, p);
}

template <int K>
LifepFn pick(bool conway, int bc) {
  if (bc == STH_REMOVE) return conway ? &launch_lifep<K, true, STH_REMOVE> : &launch_lifep<K, false, STH_REMOVE>;
  if (bc == STH_REFLECT) return conway ? &launch_lifep<K, true, STH_REFLECT> : &launch_lifep<K, false, STH_REFLECT>;
  return conway ? &launch_lifep<K, true, STH_WRAP> : &launch_lifep<K, false, STH_WRAP>;
}

}  // namespace

LifepFn lifep_launcher(int k, bool conway, int bc) {
  switch (k) {
    case 1: return pick<1>(conway, bc);
    case 2: return pick<2>(conway, bc);
    case 3: return pick<3>(conway, bc);
    case 4: return pick<4>(conway, bc);
    case 5: return pick<5>(conway, bc);
    case 6: return pick<6>(conway, bc);
    case 7: return pick<7>(conway, bc);
    case 8: return pick<8>(conway, bc);
    case 9: return pick<9>(conway, bc);
    case 10: return pick<10>(conway, bc);
    case 11: return pick<11>(conway, bc);
    case 12: return pick<12>(conway, bc);
    case 14: return pick<14>(conway, bc);
    default: return pick<16>(conway, bc);
  }
}

void launch_life_pack(LifepParams p, hipStream_t s) {
  p.tiles_x = (p.words + 255) / 256;
  p.tiles_y = (p.n1 + kLifeIoRows - 1) / kLifeIoRows;
  hipLaunchKernelGGL(life_pack_kernel, dim3(static_cast<unsigned>(p.tiles_x) * p.tiles_y), dim3(256), 0, s, p);
}

void launch_life_unpack(LifepParams p, hipStream_t s) {
  p.tiles_x = (p.n0 + 16 * 256 - 1) / (16 * 256);
  p.tiles_y = (p.n1 + kLifeIoRows - 1) / kLifeIoRows;
  hipLaunchKernelGGL(life_unpack_kernel, dim3(static_cast<unsigned>(p.tiles_x) * p.tiles_y), dim3(256), 0, s, p);
}

}  // namespace sth
