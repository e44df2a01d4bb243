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

// Packs a grid of bytes (any value; nonzero is alive): one word per lane,
// from aligned 16-byte loads where they lie inside the row, byte by byte at
// the row's ends.  Four rows per thread keep enough loads in flight.
constexpr int kLifeIoRows = 4;
__global__ __launch_bounds__(256) void life_pack_kernel(LifepParams p) {
  const int32_t n0 = p.n0, n1 = p.n1, words = p.words;
  const int bx = static_cast<int>(blockIdx.x) % p.tiles_x, by = static_cast<int>(blockIdx.x) / p.tiles_x;
  const int32_t wi = bx * 256 + static_cast<int>(threadIdx.x);
  if (wi >= words) return;
  const int32_t x = wi * 32;
#pragma unroll
  for (int j = 0; j < kLifeIoRows; ++j) {
    const int32_t y = by * kLifeIoRows + j;
    if (y >= n1) break;
    const uint8_t* row = reinterpret_cast<const uint8_t*>(p.src) + static_cast<int64_t>(y) * p.s1;
    const int mis = static_cast<int>(reinterpret_cast<uint64_t>(row) & 15);  // uniform
    uint32_t out = 0;
    if (x >= mis && x - mis + (mis ? 48 : 32) <= n0) {
      const uint4* a = reinterpret_cast<const uint4*>(row + x - mis);
      const uint32_t lo = pack16_any(a[0]) | (pack16_any(a[1]) << 16);
      out = mis ? __builtin_amdgcn_alignbit(pack16_any(a[2]), lo, mis) : lo;
    } else {
      for (int i = 0; i < 32; ++i)
        if (x + i < n0 && row[x + i]) out |= 1u << i;
    }
    lifep_row(p.dst, p.d1, y, words)[wi] = out;
  }
}

// Unpacks a grid: 16 cells per lane, stored as one aligned 16-byte vector
// where it lies inside the row, byte by byte at the row's ends.
__global__ __launch_bounds__(256) void life_unpack_kernel(LifepParams p) {
  const int32_t n0 = p.n0, n1 = p.n1, words = p.words;
  const int bx = static_cast<int>(blockIdx.x) % p.tiles_x, by = static_cast<int>(blockIdx.x) / p.tiles_x;
  const int32_t j = bx * 256 + static_cast<int>(threadIdx.x);
#pragma unroll
  for (int k = 0; k < kLifeIoRows; ++k) {
    const int32_t y = by * kLifeIoRows + k;
    if (y >= n1) break;
    uint8_t* row = reinterpret_cast<uint8_t*>(p.dst) + static_cast<int64_t>(y) * p.d1;
    const int mis = static_cast<int>(reinterpret_cast<uint64_t>(row) & 15);  // uniform
    const int32_t x = 16 * j - mis;
    if (x >= n0) continue;
    const uint32_t* bits = lifep_row(p.src, p.s1, y, words);
    const uint32_t v = x >= 0 ? lifep_bits(bits, x, words) : bits[0] << -x;
    if (x >= 0 && x + 16 <= n0) {
      *reinterpret_cast<uint4*>(row + x) = unpack16(v << 8);
    } else {
      for (int i = 0; i < 16; ++i)
        if (x + i >= 0 && x + i < n0) row[x + i] = static_cast<uint8_t>((v >> i) & 1u);
    }
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
    case 6: return pick<6>(conway, bc);
    case 8: return pick<8>(conway, bc);
    case 10: return pick<10>(conway, bc);
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
  // 16-cell groups of a row whose first cell may sit at the end of one
  p.tiles_x = (p.n0 + 15 + 16 * 256 - 1) / (16 * 256);
  p.tiles_y = (p.n1 + kLifeIoRows - 1) / kLifeIoRows;
  hipLaunchKernelGGL(life_unpack_kernel, dim3(static_cast<unsigned>(p.tiles_x) * p.tiles_y), dim3(256), 0, s, p);
}

}  // namespace sth
