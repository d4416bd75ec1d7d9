// Tile function of the wide forms: G = 2 to 16 lanes per strand, few points per
// lane (M <= 8), any point count N <= G * M.
//
// The step of a strand is a serial chain of (K + lanes - 1) * M point updates
// (the lane pipeline of ftl_tile.h), about 17 dependent vector instructions
// each.  A launch too small to fill the chip is bound by that chain and by the
// round trips of its loads, not by throughput, so these forms trade vector
// work (lanes idle while the pipeline fills and drains) for a shorter chain:
// 16 points take 23 updates on 16 lanes, 72 on 2.  All of a tile's rows are
// loaded at once.
//
// Differences from ftl_tile.h: a tile's strands are one contiguous run of
// float4s, read and written row by row whatever the point count (no slot is
// padded), through buffer descriptors whose bounds are the tile's (lanes past
// its end read zeros and store nothing); a lane finds its points in the LDS
// stage by element, and the strand's last lane is (N - 1) / M, so one form
// takes every point count up to G * M.  With M = 1 there is no stage: a lane
// loads and stores its own element.
#pragma once

#include "ftl_tile.h"

namespace ftl_wide_impl {

using namespace ftl_tile_impl;

// Stage slot of element e: permuted within its block of 8 so that lanes that
// read at a stride of 2, 4 or 8 elements fall on different banks.
__device__ __forceinline__ int element_slot(int e) { return e ^ ((e >> 3) & 7); }

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
// Sum over the G lanes of a strand, in every lane (quad permutes, then mirrors
// of the half row and the row).
template <int G>
__device__ __forceinline__ float lanes_sum(float x) {
  x += dpp<0xB1>(x);
  if (G >= 4) x += dpp<0x4E>(x);
  if (G >= 8) x += dpp<0x141>(x);
  if (G >= 16) x += dpp<0x140>(x);
  return x;
}
// The next lane's value (row_shl:1; used by lanes whose next lane is of the
// same strand).
__device__ __forceinline__ float3 from_next_lane(float3 x) { return f3(dpp<0x101>(x.x), dpp<0x101>(x.y), dpp<0x101>(x.z)); }

// Float4s of a form's LDS stage.
constexpr int wide_stage(int m) { return m > 1 ? FTL_WAVE * m : 1; }

template <int M, int G, FtlCache CP>
__device__ __forceinline__ void ftl_wide_tile(const FtlStep& A, int strand0, float4* stage) {
  constexpr int SPT = FTL_WAVE / G;
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & (FTL_WAVE - 1);
  const int g = lane % G, ls = lane / G;
  const int N = A.npoints;
  const int nst = min(SPT, A.nstrands - strand0);
  const bool valid = ls < nst;
  const int nl = min(max(N - g * M, 0), M);  // points on this lane
  const int last = (N - 1) / M;              // the lane of a strand's last point
  const size_t at = (size_t)strand0 * N;
  const unsigned bytes = (unsigned)(nst * N) * 16u;
  const BufferRsrc bpos = buffer_of(A.pos + at, bytes), bvel = buffer_of(A.vel + at, bytes);
  // Row i holds element 64 i + lane; with M = 1 a lane's row is its own point
  // (lanes without one address past the end).
  const unsigned own = M > 1 ? 16u * lane : (g < N ? 16u * (ls * N + g) : 0x80000000u);

  float4 x[M], v[M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    x[i] = buffer_load4<CP == kCacheStream>(bpos, own + 1024u * i);
    v[i] = buffer_load4<CP == kCacheStream>(bvel, own + 1024u * i);
  }
  // The strand's root, on every lane (the collider cull needs it there).
  float3 x0, p0;
  {
    const float4 r = buffer_load4<false>(bpos, 16u * (unsigned)(ls * N));
    x0 = f3(r.x, r.y, r.z);
    const float3 src = A.rmode == kRootModel ? x0 : root_source(A, strand0 + min(ls, nst - 1));
    p0 = A.model_ident ? src : transform(A, src);
  }
  const float3 u0 = sub3(p0, x0);

  const float dt = A.dt, dt2 = A.dt2;
  const float3 F0 = f3(A.force[0], A.force[1], A.force[2]);
  const bool wind = A.wind_grid != 0;
  WindArgs W;
  W.T = (GlobalFloat4*)pin_p(A.wind);
  W.freq = A.wind_freq;
  W.off[0] = A.wind_off[0];
  W.off[1] = A.wind_off[1];
  W.off[2] = A.wind_off[2];
  float3 p[M];
  LenRegs<M> l;
#pragma unroll
  for (int i = 0; i < M; ++i) {
    float3 F = F0;
    if (wind) {
      const float3 w = wind_blend(wind_fetch(W, f3(x[i].x, x[i].y, x[i].z)));
      F = f3(F0.x + w.x, F0.y + w.y, F0.z + w.z);
    }
    const float3 pr = f3(__builtin_fmaf(dt2, F.x, __builtin_fmaf(dt, v[i].x, x[i].x)),
                         __builtin_fmaf(dt2, F.y, __builtin_fmaf(dt, v[i].y, x[i].y)),
                         __builtin_fmaf(dt2, F.z, __builtin_fmaf(dt, v[i].z, x[i].z)));
    if constexpr (M > 1) {
      stage[element_slot(FTL_WAVE * i + lane)] = make_float4(pr.x, pr.y, pr.z, x[i].w);
    } else {
      p[0] = pr;
      l.set(0, x[0].w);
    }
  }
  // Element of the lane's point j in the tile (slots past the strand's last
  // point read that point).
  auto element = [&](int j) { return ls * N + min(g * M + j, N - 1); };
  if constexpr (M > 1) {
    tile_sync();
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const float4 t = stage[element_slot(element(j))];
      p[j] = f3(t.x, t.y, t.z);
      l.set(j, t.w);
    }
    tile_sync();
  }
  const bool root = g == 0;
  p[0] = sel3(root, p0, p[0]);
  // The sweeps use sigma * l.  The position store needs l itself: kept where
  // the registers are there, else read again from the step's input.
  const bool unit_sigma = A.sigma == 1.0f;
  constexpr bool kKeepLen = M <= 4;
  float wl[M];
#pragma unroll
  for (int j = 0; j < M; ++j) wl[j] = kKeepLen ? l.get(j) : 0.0f;
  if (!unit_sigma) {
    const float sg = A.sigma;
#pragma unroll
    for (int j = 0; j < M; ++j) l.set(j, sg * l.get(j));
  }

  unsigned reach;
  {
    float L = 0.0f;
#pragma unroll
    for (int j = 0; j < M; ++j)
      if (j < nl) L += fabsf(l.get(j));
    L = lanes_sum<G>(L);
    const unsigned mine = valid ? reachable_colliders(A, p0, L) : 0u;
    unsigned any = 0u;
#pragma unroll
    for (int k = 0; k < FTL_NCOL; ++k)
      if (__ballot((mine >> k) & 1u) != 0ull) any |= 1u << k;
    reach = __builtin_amdgcn_readfirstlane(any);
  }
  int cm;  // colliders the tile meets
  const Spheres S = load_spheres(A, reach, cm);
  const VelArgs V = vel_args(A);

  const int K = A.iterations;
  float3 q[M];
  float3 lead = p0;
  for (int t = 0; t < K - 1; ++t)
    sweep_pipe<M, G, true, false, 0, M>(S, p, l, lead, g, t >= g, false, nullptr, q, cm);
  for (int t = K - 1; t < K + last; ++t) {
    const int it = t - g;
    sweep_pipe<M, G, true, true, 0, M>(S, p, l, lead, g, it >= 0 && it < K, it == K - 1, nullptr, q, cm);
  }

  // Settle (as in ftl_tile): velocities from the last iteration's corrections,
  // then its collisions.
  const float4* __restrict__ pp = A.pos + at + (size_t)(valid ? ls : 0) * N;
  const int tip = g == last ? nl - 1 : -1;
  const float3 c0 = sub3(p[0], q[0]);
  const float3 cn = from_next_lane(c0);
  bool bad = false;
  float3 c = c0;
  float4 out[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const float3 mine = c;
    c = m + 1 < M ? sub3(p[m + 1 < M ? m + 1 : m], q[m + 1 < M ? m + 1 : m]) : cn;
    float3 u = mul3(c, V.delta);
    if (m == 0) u = sel3(root, u0, u);
    u = sel3(tip == m, mine, u);
    if (m > 0 || !root) collide<true>(S, p[m], u, cm);
    const float3 w = out_velocity(V, pp, min(g * M + m, N - 1), p[m], u);
    out[m] = make_float4(w.x, w.y, w.z, 0.0f);
    if (m == nl - 1)
      bad = !(isfinite(p[m].x) && isfinite(p[m].y) && isfinite(p[m].z) && isfinite(w.x) && isfinite(w.y) &&
              isfinite(w.z));
  }
  // Stores: velocities, then positions (DFTL and the rest lengths of a scaled
  // step read the input positions: all of it before the first position store).
  if constexpr (!kKeepLen) {
#pragma unroll
    for (int j = 0; j < M; ++j) wl[j] = unit_sigma ? l.get(j) : pp[min(g * M + j, N - 1)].w;
  }
  auto store_rows = [&](BufferRsrc b) {
    if constexpr (M > 1) {
#pragma unroll
      for (int j = 0; j < M; ++j)
        if (j < nl) stage[element_slot(ls * N + g * M + j)] = out[j];
      tile_sync();
#pragma unroll
      for (int i = 0; i < M; ++i) buffer_store4<CP>(b, own + 1024u * i, stage[element_slot(FTL_WAVE * i + lane)]);
      tile_sync();
    } else {
      buffer_store4<CP>(b, own, out[0]);
    }
  };
  store_rows(bvel);
#pragma unroll
  for (int j = 0; j < M; ++j) out[j] = make_float4(p[j].x, p[j].y, p[j].z, wl[j]);
  store_rows(bpos);
  bad = bad && valid;
  const unsigned long long b = __ballot(bad);
  if (b != 0ull && lane == (int)(__ffsll((long long)b) - 1))
    __hip_atomic_store(A.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace ftl_wide_impl
