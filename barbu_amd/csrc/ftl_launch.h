// Host-side entry points of the kernels (ftl_plain.hip, ftl_misc.hip), used by the C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include "ftl_classes.h"
#include "ftl_device.h"

// Launch classes: (points per lane M, lanes per strand G, guarded).
int ftl_num_classes();
int ftl_class_m(int cls);
int ftl_class_g(int cls);
int ftl_class_guarded(int cls);

// How a launch that steps state_bytes (positions and velocities, read and
// rewritten in place) uses the caches.  By the size of that state against the
// 256 MB Infinity Cache, in us per step, one groom stepped over and over:
//   up to 144 MB through: its lines do not wait dirty in the XCDs' L2s for the
//     end of the kernel to write them out (against default: 32 MB of 16 points
//     29.2 -> 27.2 and 31.6 -> 29.9 with wind, 134 MB of 4 points 53.0 -> 50.0
//     and 58.0 -> 56.2, 102 MB of 64 points 58.2 -> 56.4);
//   up to 384 MB default: part of the state is still cached when the next step
//     reads it, which both of the others lose (268 MB of 32 points with wind
//     111.5, through 113.3, stream 120; 201 MB 105.2 -> 106.7 with through
//     where three grooms take turns);
//   above it stream: none of it would still be cached, so neither loads nor
//     stores keep their lines (1 GB of 32 points: default 435, stores alone
//     405, with the loads 391; 922 MB of 24 points, three grooms in turn, 347
//     -> 323).  The launch classes' loads stay cached with wind (405 against
//     413) and where lines are shared (ftl_tile); the wide forms' do not (-1 to
//     +1.5%, and a test of the wind ahead of their loads costs as much).
// The guarded classes of 5 to 16 points on one lane use the default at every
// size (ftl_plain.hip).
FtlCache ftl_cache_for(size_t state_bytes);
#define FTL_WITH_CACHE(cp, ...)                                                      \
  switch (cp) {                                                                      \
    case kCacheThrough: { constexpr FtlCache CP = kCacheThrough; __VA_ARGS__; break; } \
    case kCacheStream: { constexpr FtlCache CP = kCacheStream; __VA_ARGS__; break; }   \
    default: { constexpr FtlCache CP = kCacheDefault; __VA_ARGS__; break; }            \
  }
// start / stop: optional events bracketing the kernel itself (timing).
hipError_t ftl_launch_plain(int cls, const FtlStep& A, hipStream_t stream, hipEvent_t start = nullptr,
                            hipEvent_t stop = nullptr);
// Wide forms (ftl_wide.h).  The level of a launch over n grooms (16, 8 or 4:
// the lanes per strand its long strands take), or 0 when it fills the chip.
int ftl_wide_level(int ncu, const int* nstrands, const int* npoints, int n);
// The form of a groom in a launch of that level; at level 0, the form of the
// point counts no exact launch class holds, or -1 (a launch class is faster).
// plain: in a plain step, with its use of the caches and whether it has wind.
int ftl_wide_form(int level, int npoints, bool plain = false, FtlCache cp = kCacheDefault, bool wind = false);
// The plain step of one groom by a wide form.
hipError_t ftl_launch_wide(int form, const FtlStep& A, hipStream_t stream, hipEvent_t start = nullptr,
                           hipEvent_t stop = nullptr);
// Whether FTL_TILES_ALL holds a launch class or wide form.
bool ftl_in_tiles_all(int cls);
// Tile-list kernel of one class over the ntiles tiles of spans[0..nspans)
// (every groom of that class, in tile order): workgroup b steps tiles b,
// b + grid, ...  cls may be a wide form (ftl_wide_id), FTL_WIDE_ALL or FTL_TILES_ALL, one
// workgroup per tile.
hipError_t ftl_launch_tiles(int cls, const FtlStep* grooms, const FtlSpan* spans, int nspans, int ntiles, int grid,
                            hipStream_t stream, FtlCache cp);
// Resident tile-list workgroups per CU for a class.
int ftl_tiles_blocks_per_cu(int cls);
// Skinning of mesh vertices (and normals when nout is not null): mode 0 dual
// quaternions (2 float4 per bone), mode 1 linear blending (3 float4 rows per
// bone, joint 0xff = identity).
hipError_t ftl_launch_skin(int mode, int nverts, const float4* bones, const int4* joints, const float4* weights,
                           const float4* rest, const float4* nrest, float4* out, float4* nout, hipStream_t stream);
// Per strand of a skinned groom: the root on its bound triangle and, when
// normals is not null, the unit normal there.
hipError_t ftl_launch_root_frames(int nstrands, const int4* bind, const int4* tris, const float4* verts,
                                  const float4* normals, float4* roots, float4* nout, hipStream_t stream);
// Copies bytes (a multiple of 16) from pinned, coherent host memory to the
// device with a kernel on `stream`.
hipError_t ftl_launch_upload(const void* host_src, void* dst, size_t bytes, hipStream_t stream);
hipError_t ftl_launch_copy(const void* src, void* dst, size_t n16, int ncu, hipStream_t stream);
