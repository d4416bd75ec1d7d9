// Kernels of the wide forms (ftl_wide.h) with FTL_WIDE_LANES lanes per strand
// (one translation unit per lane count): the plain step of one groom, and, of
// the forms of launches that fill the chip, the tile-list kernel of batched
// frames.  FTL_WIDE_LANES = 0: the tile-list
// kernel that holds every form, for batches small enough to be one launch.
#include <hip/hip_ext.h>

#include "ftl_launch.h"
#include "ftl_wide.h"

#ifndef FTL_WIDE_LANES
#error "build with -DFTL_WIDE_LANES=<lanes per strand, or 0>"
#endif

namespace {

using namespace ftl_wide_impl;

#define FTL_PASTE2(a, b) a##b
#define FTL_PASTE(a, b) FTL_PASTE2(a, b)

#if FTL_WIDE_LANES > 0

template <int M, int G, FtlCache CP>
__global__ __launch_bounds__(FTL_WAVE) void ftl_wide_kernel(FtlStep arg) {
  (void)arg;
#if defined(__HIP_DEVICE_COMPILE__)
  const FtlStep& A = *(const FtlStep*)__builtin_amdgcn_kernarg_segment_ptr();
#else
  const FtlStep& A = arg;
#endif
  __shared__ float4 sh[wide_stage(M)];
  ftl_wide_tile<M, G, CP>(A, blockIdx.x * (FTL_WAVE / G), sh);
}

#if FTL_WIDE_LANES != 16
template <int M, int G, FtlCache CP>
__global__ __launch_bounds__(FTL_WAVE) void ftl_wide_tiles_kernel(const FtlStep* __restrict__ grooms,
                                                                  const FtlSpan* __restrict__ spans, int nspans) {
  __shared__ float4 sh[wide_stage(M)];
  const int t = (int)blockIdx.x;
  const int s = span_of(spans, nspans, t);
  const int gi = __builtin_amdgcn_readfirstlane(spans[s].groom);
  const int s0 = (t - __builtin_amdgcn_readfirstlane(spans[s].tile0)) * (FTL_WAVE / G);
  ftl_wide_tile<M, G, CP>(grooms[gi], s0, sh);
}
#endif

#define FTL_LEVEL FTL_PASTE(FTL_LEVEL_FORMS_, FTL_WIDE_LANES)
#define FTL_DEFAULT FTL_PASTE(FTL_DEFAULT_FORMS_, FTL_WIDE_LANES)

}  // namespace

hipError_t FTL_PASTE(ftl_launch_wide_, FTL_WIDE_LANES)(int m, const FtlStep& A, hipStream_t stream, hipEvent_t start,
                                                       hipEvent_t stop, FtlCache cp) {
  constexpr int spt = FTL_WAVE / FTL_WIDE_LANES;
  const dim3 grid((A.nstrands + spt - 1) / spt), block(FTL_WAVE);
  switch (m) {
#define FTL_WL(M, G)                                                                                      \
  case M:                                                                                                 \
    FTL_WITH_CACHE(cp, hipExtLaunchKernelGGL((ftl_wide_kernel<M, G, CP>), grid, block, 0, stream, start, stop, 0, A)) \
    return hipGetLastError();
    FTL_DEFAULT(FTL_WL)
#undef FTL_WL
#define FTL_WL(M, G)                                                                                                \
  case M:                                                                                                          \
    hipExtLaunchKernelGGL((ftl_wide_kernel<M, G, kCacheThrough>), grid, block, 0, stream, start, stop, 0, A);      \
    return hipGetLastError();
    FTL_LEVEL(FTL_WL)
#undef FTL_WL
  }
  return hipErrorInvalidValue;
}

#if FTL_WIDE_LANES != 16
hipError_t FTL_PASTE(ftl_launch_wide_tiles_, FTL_WIDE_LANES)(int m, const FtlStep* grooms, const FtlSpan* spans,
                                                             int nspans, int ntiles, hipStream_t stream, FtlCache cp) {
  const dim3 grid(ntiles), block(FTL_WAVE);
  switch (m) {
#define FTL_WT(M, G)                                                                                              \
  case M:                                                                                                         \
    FTL_WITH_CACHE(cp, hipLaunchKernelGGL((ftl_wide_tiles_kernel<M, G, CP>), grid, block, 0, stream, grooms, spans, nspans)) \
    return hipGetLastError();
    FTL_DEFAULT(FTL_WT)
#undef FTL_WT
  }
  return hipErrorInvalidValue;
}
#endif

#else  // every form in one kernel

// A batch whose waves all fit the chip at once (ftl_wide_level) is one launch
// of this kernel, whatever the point counts of its grooms: a span names its
// form.  The kernel carries the registers of its largest form, which costs
// such a batch nothing.  (Class kernels side by side, forked and joined in the
// graph, start 8 to 20 us apart: 24 grooms of 300 to 5,000 strands with 4 to
// 20 points in wind took 70 us a frame as four class kernels of 11 to 35 us.)
__global__ __launch_bounds__(FTL_WAVE) void ftl_wide_all_kernel(const FtlStep* __restrict__ grooms,
                                                                const FtlSpan* __restrict__ spans, int nspans) {
  __shared__ float4 sh[wide_stage(8)];
  const int t = (int)blockIdx.x;
  const int s = span_of(spans, nspans, t);
  const int gi = __builtin_amdgcn_readfirstlane(spans[s].groom);
  const int tile = t - __builtin_amdgcn_readfirstlane(spans[s].tile0);
  switch (__builtin_amdgcn_readfirstlane(spans[s].cls)) {
#define FTL_WA(M, G)                                                              \
  case ftl_wide_id(M, G):                                                         \
    ftl_wide_tile<M, G, kCacheThrough>(grooms[gi], tile * (FTL_WAVE / G), sh);    \
    break;
    FTL_LEVEL_FORMS_4(FTL_WA) FTL_DEFAULT_FORMS_4(FTL_WA) FTL_LEVEL_FORMS_8(FTL_WA) FTL_DEFAULT_FORMS_8(FTL_WA)
    FTL_LEVEL_FORMS_16(FTL_WA)
#undef FTL_WA
  }
}

}  // namespace

hipError_t ftl_launch_wide_all(const FtlStep* grooms, const FtlSpan* spans, int nspans, int ntiles,
                               hipStream_t stream) {
  hipLaunchKernelGGL(ftl_wide_all_kernel, dim3(ntiles), dim3(FTL_WAVE), 0, stream, grooms, spans, nspans);
  return hipGetLastError();
}

#endif
