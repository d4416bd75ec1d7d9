// The tile-list kernel of batches whose grooms are of several launch classes
// or wide forms: every one that a point count gets in a launch that fills the
// chip, in one kernel; a span names its own.  Built once for each use of the
// caches (-DFTL_CACHE=<FtlCache>).
//
// A kernel per class, side by side, has to be forked and joined (the second
// starts 8 us after the first, the join and the next frame's first kernel
// follow 20 us after the last), and the last waves of each run on a chip that
// empties; here the launch's tiles are one list, the costliest first.  Us a
// frame as kernels per class and as this one (8 iterations, 300 to 150,000
// strands a groom):
//   16 grooms of 4 to 20 points in wind 70.6, 34.5;  23 of 12 to 64 92.9, 54.3
//   5 of 16 and 32 in wind 92.4, 73.7;               27 of 8 to 64 84.8, 52.0
//   25 of 8 to 64 275, 240;                          26 of 12 to 64 in wind 322, 297
//   32 of 8 to 64, every groom moving, 497, 460
// (The kernels per class then were branches of a graph.  As launches forked
// from the caller's stream, over 1,462 drawn mixes, those small enough for
// FTL_WIDE_ALL either way among them: 0.97 to 4.3 times this one, 1.7 in the mean.)
// The small classes run at the large ones' four waves per SIMD here, also where
// one fills most of the batch: 1M strands of 4 points, whose own kernel runs
// eight, beside 3,000 of 8 took 65.1 us by class and 49.8 here, in wind 67.0 and
// 61.5, at 2 iterations in wind 62.5 and 59.8.  A batch of one class keeps its own
// kernel, as does one with grooms whose lanes were set or whose class the tables
// pick from outside FTL_DEFAULT_CLASSES.
#include "ftl_launch.h"
#include "ftl_wide.h"

#ifndef FTL_CACHE
#error "build with -DFTL_CACHE=<0, 1 or 2>"
#endif

namespace {

using namespace ftl_wide_impl;

#define FTL_PASTE2(a, b) a##b
#define FTL_PASTE(a, b) FTL_PASTE2(a, b)

constexpr FtlCache kCache = (FtlCache)FTL_CACHE;

// The stage of any of them.
constexpr size_t stage_bytes() {
  size_t n = sizeof(float4) * wide_stage(8);
#define FTL_TS(id, M, G, GU) n = n > sizeof(ftl_tile_impl::TileLds<M, G, GU>) ? n : sizeof(ftl_tile_impl::TileLds<M, G, GU>);
  FTL_DEFAULT_CLASSES(FTL_TS)
#undef FTL_TS
  return n;
}

// Four waves per SIMD, as the largest of its classes runs.
__global__ __launch_bounds__(FTL_WAVE) __attribute__((amdgpu_waves_per_eu(4, 8)))
void ftl_tiles_all_kernel(const FtlStep* __restrict__ grooms, const FtlSpan* __restrict__ spans, int nspans) {
  __shared__ __attribute__((aligned(16))) char sh[stage_bytes()];
  const int t = (int)blockIdx.x;
  const int s = span_of(spans, nspans, t);
  const int gi = __builtin_amdgcn_readfirstlane(spans[s].groom);
  const int tile = t - __builtin_amdgcn_readfirstlane(spans[s].tile0);
  switch (__builtin_amdgcn_readfirstlane(spans[s].cls)) {
#define FTL_TC(id, M, G, GU)                                                          \
  case id:                                                                            \
    ftl_tile_impl::ftl_tile<M, G, GU, kCache, ftl_tile_impl::kWindAny>(               \
        grooms[gi], tile * (FTL_WAVE / G), *(ftl_tile_impl::TileLds<M, G, GU>*)sh);   \
    break;
    FTL_DEFAULT_CLASSES(FTL_TC)
#undef FTL_TC
#define FTL_TW(M, G)                                                                      \
  case ftl_wide_id(M, G):                                                                 \
    ftl_wide_tile<M, G, kCache>(grooms[gi], tile * (FTL_WAVE / G), (float4*)sh);          \
    break;
    FTL_DEFAULT_FORMS(FTL_TW)
#undef FTL_TW
  }
}

}  // namespace

hipError_t FTL_PASTE(ftl_launch_tiles_all_, FTL_CACHE)(const FtlStep* grooms, const FtlSpan* spans, int nspans,
                                                      int ntiles, hipStream_t stream) {
  hipLaunchKernelGGL(ftl_tiles_all_kernel, dim3(ntiles), dim3(FTL_WAVE), 0, stream, grooms, spans, nspans);
  return hipGetLastError();
}
