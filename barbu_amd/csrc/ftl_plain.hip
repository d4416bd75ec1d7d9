// Plain (one groom) FTL step kernels for one launch class, selected at build
// time with -DFTL_CLASS_ID=<id>: one wave64 workgroup per tile of strands, or,
// for launches with wind, workgroups of four tiles sharing an LDS copy of the
// wind lattice; and the tile-list kernel of batched frames.  Each kernel comes
// in three forms, by how its loads and stores use the caches (ftl_cache_for).
#include <hip/hip_ext.h>

#include "ftl_classes.h"
#include "ftl_launch.h"
#include "ftl_tile.h"

#ifndef FTL_CLASS_ID
#error "build with -DFTL_CLASS_ID=<launch class>"
#endif
#ifndef FTL_WIND_LDS
#define FTL_WIND_LDS 1
#endif

namespace {

template <int ID>
struct ClassOf;
#define FTL_CO(id, M_, G_, GU_, W_, CH_)         \
  template <>                                \
  struct ClassOf<id> {                       \
    static constexpr int M = M_, G = G_, W = W_; \
    static constexpr bool GU = GU_;          \
  };
FTL_CLASSES(FTL_CO)
#undef FTL_CO

using CL = ClassOf<FTL_CLASS_ID>;

// Occupancy target of the class (waves per SIMD the register allocator aims at).
#ifdef FTL_WPE_OVERRIDE
constexpr int kWavesPerEu = FTL_WPE_OVERRIDE;
#else
constexpr int kWavesPerEu = CL::W;
#endif
// Load-phase prefetch depth: one row for the forms that target six or more
// waves per SIMD (their register budget), FTL_LOAD_AHEAD for the others.
constexpr int kLoadAhead = kWavesPerEu >= 6 ? 1 : FTL_LOAD_AHEAD;

// With wind: four tiles (waves) per workgroup share one LDS copy of the wind
// lattice, so the load phase's gathers are LDS reads (their waits are
// independent of the HBM row loads in flight) instead of global gathers.
// Wave w of workgroup b steps tile 4b + w.  The copy is the half lattice (each
// node's first float4, 8 KB): four stages plus it make 40 KB, so the four
// workgroups of a CU at four waves per SIMD fit its 160 KB.  (Eight-tile
// workgroups with the whole lattice also fit, but a workgroup holds its LDS
// until its slowest tile ends.)  Used by the classes that run at most four
// waves per SIMD.
#ifndef FTL_WIND_WAVES
#define FTL_WIND_WAVES 4
#endif
constexpr int kWindWaves = FTL_WIND_WAVES;
// eight-wave groups copy the whole lattice, four-wave groups its half lattice
constexpr int kWindHalf = kWindWaves == 4;
constexpr int kLatticeF4 = (kWindHalf ? 1 : 2) * FTL_WIND_GRID * FTL_WIND_GRID * FTL_WIND_GRID;
constexpr size_t kWindGroupLds =
    kWindWaves * sizeof(ftl_tile_impl::TileLds<CL::M, CL::G, CL::GU>) + kLatticeF4 * sizeof(float4);
// workgroups per CU at the class's occupancy target (4 waves per SIMD for the
// classes that reach it)
constexpr int kWindGroupsPerCu = (kWavesPerEu == 2 ? 8 : 16) / kWindWaves;
constexpr bool kWindLds = (kWavesPerEu == 4 || kWavesPerEu == 2) && kWindGroupsPerCu * kWindGroupLds <= 160 * 1024;

// How the class uses the caches.  A lane of a guarded class of 8 or 16 points
// holds a strand that is no whole lines, and stores part of a line at a time:
// written through or streamed, the parts do not merge in the L2 (us a step,
// default against ftl_cache_for's choice: 33 MB of 7 points at 2 iterations 14.3,
// 19.2, with wind 18.6, 23.7; 134 MB with wind 76.6, 88.8; 440 MB 222, 340; 440 MB
// of 11 points 296, 576).
constexpr FtlCache class_cache(FtlCache cp) {
  return CL::GU && CL::G == 1 && CL::M > 4 && CL::M <= 16 ? kCacheDefault : cp;
}

// A class with the LDS form never runs its plain kernel with wind.
constexpr int kPlainWind = kWindLds && FTL_WIND_LDS ? ftl_tile_impl::kWindOff : ftl_tile_impl::kWindAny;

template <FtlCache CP>
__global__ __launch_bounds__(FTL_WAVE) __attribute__((amdgpu_waves_per_eu(kWavesPerEu, 8)))
void ftl_plain_kernel(FtlStep arg) {
  (void)arg;
  // The descriptor is read in place from the kernel-argument segment (scalar
  // loads, runtime-indexed collider array) instead of through a private copy
  // of the by-value argument.
#if defined(__HIP_DEVICE_COMPILE__)
  const FtlStep& A = *(const FtlStep*)__builtin_amdgcn_kernarg_segment_ptr();
#else
  const FtlStep& A = arg;
#endif
  __shared__ ftl_tile_impl::TileLds<CL::M, CL::G, CL::GU> sh;
  ftl_tile_impl::ftl_tile<CL::M, CL::G, CL::GU, CP, kPlainWind, kLoadAhead>(
      A, blockIdx.x * (FTL_WAVE / CL::G), sh);
}

template <FtlCache CP>
__global__ __launch_bounds__(FTL_WAVE * kWindWaves) __attribute__((amdgpu_waves_per_eu(kWavesPerEu, 8)))
void ftl_plain_wind_kernel(FtlStep arg) {
  (void)arg;
#if defined(__HIP_DEVICE_COMPILE__)
  const FtlStep& A = *(const FtlStep*)__builtin_amdgcn_kernarg_segment_ptr();
#else
  const FtlStep& A = arg;
#endif
  // (a one-element placeholder for the classes that do not use this form)
  __shared__ float4 lattice[kWindLds ? kLatticeF4 : 1];
  __shared__ ftl_tile_impl::TileLds<CL::M, CL::G, CL::GU> sh[kWindLds ? kWindWaves : 1];
  if constexpr (kWindLds) {
    for (int i = (int)threadIdx.x; i < kLatticeF4; i += FTL_WAVE * kWindWaves)
      lattice[i] = A.wind[kWindHalf ? 2 * i : i];
    __syncthreads();
    constexpr int spt = FTL_WAVE / CL::G;
    const int ntiles = (A.nstrands + spt - 1) / spt;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / FTL_WAVE);
    const int t = (int)blockIdx.x * kWindWaves + w;
    if (t < ntiles)
      ftl_tile_impl::ftl_tile<CL::M, CL::G, CL::GU, CP, ftl_tile_impl::kWindOn, kLoadAhead, kWindHalf ? 2 : 1>(
          A, t * spt, sh[w], lattice);
  }
}

}  // namespace

#define FTL_PASTE2(a, b) a##b
#define FTL_PASTE(a, b) FTL_PASTE2(a, b)

// start / stop (may be null): events that take the kernel's own start and end
// timestamps (hipExtLaunchKernelGGL), for per-launch timing.
hipError_t FTL_PASTE(ftl_launch_plain_, FTL_CLASS_ID)(const FtlStep& A, hipStream_t stream, hipEvent_t start,
                                                      hipEvent_t stop, FtlCache cp) {
  constexpr int spt = FTL_WAVE / CL::G;
  const int nblocks = (A.nstrands + spt - 1) / spt;
  if (nblocks <= 0) return hipSuccess;
  if (kWindLds && FTL_WIND_LDS && A.wind_grid) {
    const dim3 grid((nblocks + kWindWaves - 1) / kWindWaves), block(FTL_WAVE * kWindWaves);
    FTL_WITH_CACHE(cp, hipExtLaunchKernelGGL(ftl_plain_wind_kernel<class_cache(CP)>, grid, block, 0, stream, start, stop, 0, A))
    return hipGetLastError();
  }
  FTL_WITH_CACHE(cp, hipExtLaunchKernelGGL(ftl_plain_kernel<class_cache(CP)>, dim3(nblocks), dim3(FTL_WAVE), 0, stream, start, stop, 0, A))
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Tile-list form of the same class for batched frames: workgroup b steps the
// tiles b, b + grid, b + 2 grid, ... of the 64-lane tiles of any grooms of
// this class, each groom a span of consecutive tiles; a workgroup finds its
// tile's groom by a search over the spans' first tiles.  With grid = number of tiles (the batched default)
// each workgroup takes one tile and the hardware dispatcher balances the
// load; a smaller grid makes the workgroups persistent.  (A shared atomic
// work counter was measured 2-5x slower: every claim contends on one address
// across the eight XCDs.)

namespace {

template <FtlCache CP>
__global__ __launch_bounds__(FTL_WAVE) __attribute__((amdgpu_waves_per_eu(kWavesPerEu, 8)))
void ftl_tiles_kernel(const FtlStep* __restrict__ grooms, const FtlSpan* __restrict__ spans, int nspans,
                      int ntiles) {
  __shared__ ftl_tile_impl::TileLds<CL::M, CL::G, CL::GU> sh;
  constexpr int spt = FTL_WAVE / CL::G;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int lo = ftl_tile_impl::span_of(spans, nspans, t);
    const int gi = __builtin_amdgcn_readfirstlane(spans[lo].groom);
    const int s0 = (t - __builtin_amdgcn_readfirstlane(spans[lo].tile0)) * spt;
    ftl_tile_impl::ftl_tile<CL::M, CL::G, CL::GU, CP, ftl_tile_impl::kWindAny, kLoadAhead>(grooms[gi], s0, sh);
  }
}

}  // namespace

hipError_t FTL_PASTE(ftl_launch_tiles_, FTL_CLASS_ID)(const FtlStep* grooms, const FtlSpan* spans, int nspans,
                                                      int ntiles, int grid, hipStream_t stream, FtlCache cp) {
  if (ntiles <= 0 || nspans <= 0) return hipSuccess;
  FTL_WITH_CACHE(cp, hipLaunchKernelGGL(ftl_tiles_kernel<class_cache(CP)>, dim3(grid), dim3(FTL_WAVE), 0, stream, grooms, spans, nspans,
                                        ntiles))
  return hipGetLastError();
}

int FTL_PASTE(ftl_tiles_occ_, FTL_CLASS_ID)() {
  int blocks = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, ftl_tiles_kernel<kCacheDefault>, FTL_WAVE, 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return blocks;
}
