// Batched gather: many independent mapstencil calls of mixed sizes, shapes
// and reductions in one launch.
//
// The host flattens the tiles of every job into one index space (job j owns
// tiles [tile_begin_j, tile_begin_{j+1})) and launches one workgroup per
// strip of `tiles_per_block` consecutive tiles; the hardware dispatcher hands
// strips to CUs as they free up, so cheap and expensive jobs balance without
// atomics or barriers (a single device-wide atomic tile counter measured much
// slower: same-address atomics serialise in L2).  A workgroup finds its first
// job in the job table and walks forward.  Each tile runs the streaming body
// of the job's (shape, op) variant.  A batch of one variant, and 3-D ones,
// run a kernel that holds this variant alone; 2-D jobs of several variants
// run one kernel that holds them all and branches per tile (uniformly): a
// launch per variant lasts as long as its slowest workgroup, with most of the
// chip idle behind it, and costs the host a launch each.
// Results are bit-identical to one sth_map call per job (same fold
// expressions per cell).
#pragma once

#include "stream_kernel.hpp"

namespace sth {

struct BatchJob {
  DevArr src;
  DevArr dst;
  int32_t bc;
  int32_t read_halo;
  uint64_t padval;
  OpParams op;
  int32_t variant;  // case of the generated dispatch switch
  int32_t tiles_x, tiles_y, tiles_z;
  int32_t lpr_shift;   // streaming body: log2 of the lanes per row
  int32_t pad_;
  int64_t tile_begin;  // first tile of this job in the flattened index space
};

struct BatchParams {
  const BatchJob* jobs;
  int32_t njobs;
  int32_t tiles_per_block;
  int64_t total_tiles;
};

// `Dispatch::run(job, bx, by, bz, lane, wave)` runs the streaming body of the
// kernel's variant; it is generated per (storage type, shape, op) and
// force-inlined into the kernel, which makes no calls.
template <typename S, class Dispatch>
__device__ __forceinline__ void batch_run(const BatchParams& bp, const BatchJob* __restrict__ jobs, int64_t b) {
  // `jobs` is read-only and aliases nothing the kernel writes, so its fields
  // stay in scalar registers instead of being reloaded after every store.
  const int lane = static_cast<int>(threadIdx.x) & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  int64_t t = b * bp.tiles_per_block;
  const int64_t tend = t + bp.tiles_per_block < bp.total_tiles ? t + bp.tiles_per_block : bp.total_tiles;
  if (t >= tend) return;
  // The last job whose first tile is <= t: every lane looks at one job (at
  // one range of jobs first, when they are many), one or two loads in a row
  // where a binary search takes one per halving.
  int j = 0;
  if (bp.njobs > 64) {
    const int step = (bp.njobs + 63) / 64;
    const int i = lane * step;
    const uint64_t m = __builtin_amdgcn_ballot_w64(i < bp.njobs && jobs[i < bp.njobs ? i : 0].tile_begin <= t);
    j = (63 - __builtin_clzll(m)) * step;  // job 0 starts at tile 0: m has a bit
  }
  for (bool more = true; more;) {
    const int i = j + lane;
    const uint64_t m = __builtin_amdgcn_ballot_w64(i < bp.njobs && jobs[i < bp.njobs ? i : 0].tile_begin <= t);
    const int last = 63 - __builtin_clzll(m);
    j += last;
    more = last == 63;  // (ends: the jobs do)
  }
  j = __builtin_amdgcn_readfirstlane(j);
  for (; t < tend; ++t) {
    while (j + 1 < bp.njobs && jobs[j + 1].tile_begin <= t) ++j;
    const BatchJob job = jobs[j];  // a register copy for the tile
    // a job's own tile count fits in 32 bits (checked on the host)
    const uint32_t local = static_cast<uint32_t>(t - job.tile_begin);
    const uint32_t tx = static_cast<uint32_t>(job.tiles_x), ty = static_cast<uint32_t>(job.tiles_y);
    const int bx = static_cast<int>(local % tx);
    const uint32_t byz = local / tx;
    const int by = static_cast<int>(byz % ty);
    const int bz = static_cast<int>(byz / ty);
    Dispatch::run(job, bx, by, bz, lane, wave);
  }
}

template <typename S, class Dispatch>
__global__ __launch_bounds__(256) void batch_kernel(BatchParams bp, const BatchJob* __restrict__ jobs) {
  batch_run<S, Dispatch>(bp, jobs, xcd_block_id(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x), 1));
}

// Every 2-D variant in one kernel.  Blocks go to the XCDs round robin: of
// each 8 kBatchChunk consecutive strips an XCD takes kBatchChunk neighbours,
// which share halo rows in its L2, and every XCD gets a share of each job
// (one contiguous range per XCD would leave the long stencils to a few).
// (60 f32 arrays of 64^2 .. 2048^2, 296 MB: 94 us with chunks of 16, 97 with
// 4, 99 with 64; one launch per variant 150 us.)  Four waves per SIMD: 85 us
// against 94 with the three that the longest stencils' registers leave;
// 8-byte types would spill at four.
constexpr int kBatchChunk = 16;
template <typename S, class Dispatch>
__global__ __launch_bounds__(256, sizeof(typename Elem<S>::raw) == 8 ? 3 : 4) void batch_all_kernel(BatchParams bp, const BatchJob* __restrict__ jobs) {
  int64_t b = blockIdx.x;
  constexpr int kSpan = 8 * kBatchChunk;
  const int64_t span = b / kSpan * kSpan;
  if (span + kSpan <= static_cast<int64_t>(gridDim.x)) {
    const int r = static_cast<int>(b - span);
    b = span + (r & 7) * kBatchChunk + (r >> 3);
  }
  batch_run<S, Dispatch>(bp, jobs, b);
}

using BatchLaunchFn = void (*)(const BatchParams&, unsigned blocks, hipStream_t);

struct BatchVariant {
  int dtype;
  int op;
  int L;
  int ndim;
  const int8_t* offs;
  int variant;
  int sv, sky;  // streaming tile: 64*sv cells x 4*sky rows
  int klass;    // the batched kernel that runs this variant (one per variant)
};

constexpr int kBatchAll = 0;  // klass of the kernel that runs every 2-D variant (0 is no variant)

struct BatchKernelEntry {
  int dtype;
  int klass;
  BatchLaunchFn fn;
  int ndim;  // stencil dims
};

std::vector<BatchVariant>& batch_variants();
std::vector<BatchKernelEntry>& batch_kernels();

template <typename S, class Dispatch>
void launch_batch(const BatchParams& bp, unsigned blocks, hipStream_t s) {
  hipLaunchKernelGGL((batch_kernel<S, Dispatch>), dim3(blocks), dim3(256), 0, s, bp, bp.jobs);
}

template <typename S, class Dispatch>
void launch_batch_all(const BatchParams& bp, unsigned blocks, hipStream_t s) {
  hipLaunchKernelGGL((batch_all_kernel<S, Dispatch>), dim3(blocks), dim3(256), 0, s, bp, bp.jobs);
}

}  // namespace sth
