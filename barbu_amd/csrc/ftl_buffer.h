// Bounded 16-byte loads and stores through raw buffers, with their cache hints.
#pragma once

#include "ftl_classes.h"
#include "ftl_device.h"

namespace ftl_dev {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t BufferRsrc;

// Raw buffer of `bytes` from p: dword offsets at or past its end load 0 and
// store nothing.  A workgroup's rows go through one whose end is the
// workgroup's, so a partial one needs no clamp and no store mask, and a row's
// address is the lane's first plus a constant.
__device__ __forceinline__ BufferRsrc buffer_of(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00027000);
}
template <bool STREAM>
__device__ __forceinline__ float4 buffer_load4(BufferRsrc r, unsigned byte) {
  const f4v t = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte, 0, STREAM ? 2 : 0));
  return make_float4(t.x, t.y, t.z, t.w);
}
// The cache bits of the instruction: sc1 (16) writes through the XCD's L2, nt
// (2) marks the line as not to be kept.
template <FtlCache CP>
__device__ __forceinline__ void buffer_store4(BufferRsrc r, unsigned byte, float4 v) {
  constexpr int bits = CP == kCacheThrough ? 16 : CP == kCacheStream ? 2 : 0;
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, f4v{v.x, v.y, v.z, v.w}), r, (int)byte, 0, bits);
}

}  // namespace ftl_dev
