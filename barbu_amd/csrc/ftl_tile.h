// Tile function of the FTL step kernels (included by the per-class kernel
// translation units).
//
// Semantics: src/shaders/hair/01_simulation/cs_simulation.glsl (tcoppex/barbu)
//   predict / root          :179-193
//   SatisfyConstraints      :155-161 (K x {DistanceConstraint; CollisionConstraint})
//   DistanceConstraint      :93-127  (serial FTL sweep + damped velocity shift)
//   CollideSphere           :129-147
//   Eq. 9 / VelocityControl :79-84, :200-204 (DFTL mode)
//
// Mapping (the reference runs one 4-lane workgroup per strand with a serial
// sweep on lane 0, :88-127):
//   * A tile is one wave64.  Each strand is owned by G consecutive lanes
//     (G = 1, 2 or 4); lane g holds control points [g*M, g*M + M) in VGPRs for
//     the whole step (M = npoints / G).
//   * Load: the tile's strands are contiguous in HBM; they are read in chunks of
//     C points per lane with fully coalesced float4 loads, integrated (predict /
//     root) in that layout, and transposed through an XOR-swizzled LDS buffer.
//   * Constraints: each lane sweeps its own points.  With G > 1 the lanes of a
//     strand form a pipeline across iterations: lane g runs iteration t - g at
//     time step t and takes its leader point (lane g-1's last point, before
//     collisions) through a cross-lane shuffle.  K iterations take K + G - 1
//     time steps.
//   * Only the last iteration's velocity reaches the output (every iteration
//     overwrites u_i for i >= 1 before reading it), so velocity work, the
//     damped shift and the reflections are done in the last iteration only.
//     With G > 1 the lanes of a strand reach it at different time steps; each
//     then parks its points' positions before the sweep, skips its collisions,
//     and all lanes form their velocities and collide together after the
//     pipeline drains (settle).
//   * Store: the inverse of the load, through the same LDS buffer, so every
//     global store writes whole 128-byte lines.  Velocities leave chunk by
//     chunk (G = 1: during the last sweep; G > 1: as they settle), positions
//     after them.
//   * In place: a tile owns its strands, so no second buffer and no copy-back.

#pragma once

#include <type_traits>

#include "ftl_buffer.h"
#include "ftl_classes.h"
#include "ftl_device.h"
#ifndef FTL_NO_DFTL
#define FTL_NO_DFTL 0
#endif
// Rows of the load phase whose loads are in flight ahead of the row being
// integrated (default of the forms with at most four waves per SIMD).
#ifndef FTL_LOAD_AHEAD
#define FTL_LOAD_AHEAD 3
#endif

using namespace ftl_dev;

namespace ftl_tile_impl {

enum { kVelShipped = 0, kVelDftl = 1 };
enum { kRootModel = 0, kRootRest = 1, kRootSkinned = 2 };

template <int M, int G, bool GUARD>
struct Tile {
  static constexpr int C = ftl_chunk_of(M, G, GUARD);  // points per lane per load/store chunk
  static constexpr int SPT = FTL_WAVE / G;   // strands per tile
};

// Points of a lane that a pipelined form parks in LDS for the settle pass
// (their positions before the last iteration's sweep, three floats each): the
// first chunk, in the load/store stage, which is idle between the load and the
// stores.  The others wait in registers.  Forms with at most 8 points per lane
// park all of theirs in registers: their budget holds them.  The 24-point form
// parks two chunks (at its three waves per SIMD the LDS has room for them, and
// its registers do not: 14 spilled with one).
template <int M, int G, bool GUARD>
constexpr int kParkLds = M <= 8 ? 0 : (M == 24 ? 2 : 1) * Tile<M, G, GUARD>::C;

// Component c of chunk point j of a lane, in the stage seen as floats (parked
// positions, then the chunk's velocities): 24 columns of 65 floats, so that
// neither a wave's own accesses (lane by lane) nor the flush's (8 points of 8
// lanes) fall on one bank.
__device__ __forceinline__ int park_slot(int j, int c, int lane) { return (3 * j + c) * (FTL_WAVE + 1) + lane; }

// LDS slot of (owner lane r, point j of the chunk): XOR swizzle, conflict-free
// for both the per-lane and the coalesced access order.
template <int C>
__device__ __forceinline__ int slot(int r, int j) {
  return r * C + (j ^ (r & (C - 1)));
}

// Rest lengths of the lane's points.  With one lane per strand they live in
// LDS (point-major, so a wave's reads are conflict-free), leaving the VGPRs to
// the positions; the pipelined forms keep them in registers.
template <int M>
struct LenRegs {
  float v[M];
  __device__ __forceinline__ float get(int j) const { return v[j]; }
  __device__ __forceinline__ void set(int j, float x) { v[j] = x; }
};
struct LenLds {
  float* base;  // lane's column: element j at base[j * FTL_WAVE]
  __device__ __forceinline__ float get(int j) const { return base[j * FTL_WAVE]; }
  __device__ __forceinline__ void set(int j, float x) { base[j * FTL_WAVE] = x; }
};

// Parameters of the final iteration's velocities, read once per tile into
// scalar registers (reloading them point by point costs a scalar-memory wait
// each).
struct VelArgs {
  int dftl;  // DFTL Eq. 9 instead of the shipped correction
  float inv_dt, maxv, maxv2, delta;
};

__device__ __forceinline__ VelArgs vel_args(const FtlStep& A) {
  VelArgs V;
  V.dftl = pin_i(!FTL_NO_DFTL && A.vmode == kVelDftl);
  V.inv_dt = pin_s(A.inv_dt);
  V.maxv = pin_s(A.maxv);
  V.maxv2 = pin_s(A.maxv2);
  V.delta = pin_s(A.delta);
  return V;
}

// Stored velocity of a final point: the damped, reflected correction u as
// shipped, or DFTL Eq. 9 with VelocityControl (:79-84, :201-204).  In DFTL
// mode x is re-read from memory, where the point's position is still the
// step's input (positions are written after all velocities).
__device__ __forceinline__ float3 out_velocity(const VelArgs& V, const float4* __restrict__ pp, int j, float3 p,
                                               float3 u) {
  if (FTL_NO_DFTL || !V.dftl) return u;
  const float4 x = pp[j];
  float3 v = f3(((p.x - x.x) - u.x) * V.inv_dt, ((p.y - x.y) - u.y) * V.inv_dt, ((p.z - x.z) - u.z) * V.inv_dt);
  const float dp = dot3(v, v);
  if (dp > V.maxv2) v = mul3(v, V.maxv * rsqrt_c(dp));
  return v;
}

// Root source of strand s for the rest and skinned root modes (the model
// mode's source is the root's own input position).
__device__ __forceinline__ float3 root_source(const FtlStep& A, int s) {
  if (A.rmode == kRootRest) {
    const float4 r = A.roots[s];
    return f3(r.x, r.y, r.z);
  }
  const int4 b = A.bind[s];
  const int4 t = A.tris[b.x];
  const float w1 = __int_as_float(b.y), w2 = __int_as_float(b.z);
  const float w0 = (1.0f - w1) - w2;
  const float4 a = A.skinned[t.x], bb = A.skinned[t.y], c = A.skinned[t.z];
  return f3(__builtin_fmaf(w2, c.x, __builtin_fmaf(w1, bb.x, w0 * a.x)),
            __builtin_fmaf(w2, c.y, __builtin_fmaf(w1, bb.y, w0 * a.y)),
            __builtin_fmaf(w2, c.z, __builtin_fmaf(w1, bb.z, w0 * a.z)));
}

// Orders the tile's LDS stage accesses across the lanes of its wave.  A tile
// is one wave and only that wave touches its stage, so no workgroup barrier
// is needed (several tiles may share a workgroup): LDS instructions of one
// wave execute in issue order, and the fences keep the compiler from moving
// stage accesses across this point.
__device__ __forceinline__ void tile_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Byte offset, within the tile, of the lane's point in row 0 of chunk c (row k
// is RS * N points further).  Row k of a chunk holds, in lane ln, point ln % C
// of the chunk of owner lane r = k * (64 / C) + ln / C.  64 / C is a multiple
// of G and of C, so from row to row only the strand moves, by RS = 64 / C / G,
// and the stage slot by 64.  GUARD: points past the strand read its last one
// (CLAMP) or address past the tile, which stores nothing.
template <int M, int G, bool GUARD, bool CLAMP>
__device__ __forceinline__ unsigned row_offset(int N, int c, int lane) {
  constexpr int C = Tile<M, G, GUARD>::C;
  static_assert((FTL_WAVE / C) % G == 0 && (FTL_WAVE / C) % C == 0, "rows of a chunk hold whole strands");
  const int r0 = lane / C, j = lane % C;
  int cp = (r0 % G) * M + c * C + j;
  if (GUARD && CLAMP) cp = min(cp, N - 1);
  const unsigned off = 16u * (unsigned)((r0 / G) * N + cp);
  return GUARD && !CLAMP && cp >= N ? 0x80000000u : off;
}

// Rows of a flush read from the stage together: all eight at once would need
// 32 registers beside the strand's.
#ifndef FTL_FLUSH_ROWS
#define FTL_FLUSH_ROWS 2
#endif
constexpr int kFlushRows = FTL_FLUSH_ROWS;

// Writes chunk c of the tile (C points per lane, staged in LDS) to dst in the
// coalesced order of the load.  Called by the whole wave.
template <int M, int G, bool GUARD, FtlCache CP>
__device__ __forceinline__ void flush_chunk(BufferRsrc dst, int N, int c, const float4* __restrict__ stage, int lane) {
  constexpr int C = Tile<M, G, GUARD>::C;
  constexpr int RS = FTL_WAVE / C / G;
  // Recomputed here (opaque lane): keeping the load phase's addresses alive
  // until the stores would cost registers for the whole step.
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const unsigned off = row_offset<M, G, GUARD, false>(N, c, ln);
  const float4* __restrict__ t0 = stage + slot<C>(ln / C, ln % C);
  tile_sync();
#pragma unroll
  for (int k = 0; k < C; ++k) {
    buffer_store4<CP>(dst, off + 16u * (unsigned)(k * RS * N), t0[k * FTL_WAVE]);
    if (k % kFlushRows == kFlushRows - 1) __builtin_amdgcn_sched_barrier(0);
  }
  tile_sync();
}

// The same for velocities, staged as three floats per point (park_slot).
template <int M, int G, bool GUARD, FtlCache CP>
__device__ __forceinline__ void flush_velocities(BufferRsrc dst, int N, int c, const float* stage, int lane) {
  constexpr int C = Tile<M, G, GUARD>::C;
  constexpr int RS = FTL_WAVE / C / G;
  int ln = lane;
  asm volatile("" : "+v"(ln));
  const unsigned off = row_offset<M, G, GUARD, false>(N, c, ln);
  const float* t0 = stage + park_slot(ln % C, 0, ln / C);
  tile_sync();
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const float* t = t0 + k * (FTL_WAVE / C);
    buffer_store4<CP>(dst, off + 16u * (unsigned)(k * RS * N),
                      make_float4(t[0], t[FTL_WAVE + 1], t[2 * (FTL_WAVE + 1)], 0.0f));
    if (k % kFlushRows == kFlushRows - 1) __builtin_amdgcn_sched_barrier(0);
  }
  tile_sync();
}

// Collisions of a sweep's points (not its last iteration), after all of the
// sweep's constraints: a constraint reads its leader before the leader's
// collision, so the collisions may follow the whole sweep.  Colliders outside,
// points inside: each collider's centre and squared radius are copied to
// vector registers once per sweep, since a vector instruction with a scalar
// operand issues at half the rate of one with vector operands only when
// several waves share a SIMD.  Each point still meets the colliders in order
// with the same operations.  Point j takes part when on && j < jend && (j > 0
// || on0).
//
// Lanes of more than four points take them in pairs: where strands lie against
// a collider, every point of the wave is hit by some lane, and a hit is a serial
// chain of 15 instructions.  A pair's chains run side by side on all lanes,
// and only the three that write a point run under its hits' mask (kernel us
// point by point and in pairs: 262k x 32, one collider 110.9, 107.5, two in
// wind 131.0, 128.5; 50k x 64 at 16 iterations 84.0, 81.8).  Shorter lanes do
// not: there the launch runs eight waves to a SIMD, which cover the chain
// (1M x 4 59.0, 61.0), or one, where the longer code counts (4k x 16 9.1, 9.8).
template <int M>
__device__ __forceinline__ void collide_sweep(const Spheres& S, float3 (&p)[M], bool on, bool on0, int jend,
                                              int n) {
  constexpr bool kPairs = M > 4 && M % 2 == 0;
  if (kPairs && !on) return;
#pragma unroll
  for (int k = 0; k < FTL_NCOL; ++k) {
    if (!more_colliders(n, k)) break;
    float cx = S.c[k][0], cy = S.c[k][1], cz = S.c[k][2], r2 = S.r2[k];
    // (with one or two points the copies cost more than they save)
    if constexpr (M > 2) asm volatile("" : "+v"(cx), "+v"(cy), "+v"(cz), "+v"(r2));
    const float3 c = f3(cx, cy, cz);
    if constexpr (kPairs) {
#pragma unroll
      for (int j = 0; j < M; j += 2) {
        // (a guarded lane's slots past the strand's last point: 100k points of 5,
        // 11 and 20 a strand on one lane 15.1, 26.5, 51.0 us with them, 14.2, 25.0,
        // 48.1 without)
        if (j >= jend) continue;
        float3 w[2];
        float d[2];
        unsigned long long hit[2];  // the lanes whose point is hit
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          w[i] = sub3(p[j + i], c);
          d[i] = dot3(w[i], w[i]);
          hit[i] = __ballot(d[i] < r2 && (j + i > 0 || on0) && j + i < jend);
        }
        if ((hit[0] | hit[1]) == 0) continue;
#pragma unroll
        for (int i = 0; i < 2; ++i) w[i] = mul3(w[i], rsqrt_c(d[i]));
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float3& q = p[j + i];
          unsigned long long lanes;
          asm("s_and_saveexec_b64 %[s], %[h]\n\t"
              "v_fma_f32 %[x], %[r], %[wx], %[cx]\n\t"
              "v_fma_f32 %[y], %[r], %[wy], %[cy]\n\t"
              "v_fma_f32 %[z], %[r], %[wz], %[cz]\n\t"
              "s_mov_b64 exec, %[s]"
              : [x] "+v"(q.x), [y] "+v"(q.y), [z] "+v"(q.z), [s] "=&s"(lanes)
              : [h] "s"(hit[i]), [r] "s"(S.r[k]), [wx] "v"(w[i].x), [wy] "v"(w[i].y), [wz] "v"(w[i].z), [cx] "v"(cx),
                [cy] "v"(cy), [cz] "v"(cz)
              : "scc");
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < M; ++j) {
        if (j >= jend) continue;
        const float3 w = sub3(p[j], c);
        const float dp = dot3(w, w);
        if (on && (j > 0 || on0) && dp < r2) {
          const float is = rsqrt_c(dp);
          p[j] = fma3(S.r[k], mul3(w, is), c);
        }
      }
    }
  }
}

// Points 1 .. M - 1 of a lane, each led by the one before it.  The points are
// updated in their own registers under the lane mask (a select would be three
// vector instructions with a scalar mask operand); a point's leader is the
// previous point before that point's collision.  len(j): sigma * rest length.
template <int M, typename Len>
__device__ __forceinline__ void sweep_points(float3 (&p)[M], Len len) {
#pragma unroll
  for (int j = 1; j < M; j += 3) {
    if (j + 2 < M) {
      ftl_points3(p[j], p[j + 1], p[j + 2], p[j - 1], len(j), len(j + 1), len(j + 2));
    } else {
      ftl_point(p[j], p[j - 1], len(j));
      if (j + 1 < M) ftl_point(p[j + 1], p[j], len(j + 1));
    }
  }
}

// One sweep of DistanceConstraint over this lane's points (G == 1), followed
// by the collisions of its points.  FINAL: last iteration, which
// also forms the velocities, stages them and flushes every completed chunk;
// the lane's last point is left to the caller (its velocity is the raw
// correction and its collision comes after the sweep).
template <int M, bool GUARD, bool FINAL, FtlCache CP>
__device__ __forceinline__ void sweep(const FtlStep& A, const VelArgs& V, const Spheres& S, float3 (&p)[M],
                                      const LenLds& l, int nl,
                                      const float4* __restrict__ pp, float3& clast,
                                      float4* __restrict__ stage, BufferRsrc bvel, int N, int lane, int cm) {
  constexpr int C = Tile<M, 1, GUARD>::C;
  // Opaque per sweep: keeps the compiler from hoisting sigma * l[j] out of the
  // iteration loop into M extra registers (one multiply per point instead).
  float sg = A.sigma;
  asm volatile("" : "+v"(sg));
  const float dl = V.delta;
  if (!FINAL) {
    sweep_points<M>(p, [&](int j) { return sg * l.get(j); });
    // Collisions of points 1 .. last (the root never collides; with GUARD the
    // slots past the last point are not collided at all).
    collide_sweep<M>(S, p, true, false, GUARD ? nl : M, cm);
    return;
  }
#pragma unroll
  for (int j = 1; j < M; ++j) {
    // GUARD: slots j >= nl hold copies of the last point; they are swept like
    // the others (finite, never stored) so the loop keeps a fixed shape.
    // The leader p[j-1] has not been collided yet: its collision follows.
    const float3 q = p[j];
    ftl_point(p[j], p[j - 1], sg * l.get(j));
    const float3 pn = p[j];
    const float3 c = sub3(pn, q);
    if (!GUARD || j < nl) {
      // Point m = j-1 is final: u = delta * c_j.  The root keeps its own,
      // p0 - x0 (:192), formed here from x0, which is still in memory.
      const int m = j - 1;
      float3 pm = p[m];
      float3 u = mul3(c, dl);
      if (m == 0) {
        const float4 x0 = pp[0];
        u = sub3(pm, f3(x0.x, x0.y, x0.z));
      } else {
        collide<true>(S, pm, u, cm);
      }
      p[m] = pm;
      const float3 v = out_velocity(V, pp, m, pm, u);
      stage[slot<C>(lane, m % C)] = make_float4(v.x, v.y, v.z, 0.0f);
      if (m % C == C - 1) flush_chunk<M, 1, GUARD, CP>(bvel, N, m / C, stage, lane);
    }
    if (GUARD ? (j == nl - 1) : (j == M - 1)) clast = c;
  }
}

// The value of the previous lane of the same row of 16 lanes (DPP row_shr:1,
// one vector instruction; the first lane of a row reads 0).  The lanes of a
// strand (G = 2 or 4) never straddle a row, so lane g > 0 of a strand reads
// lane g - 1, and lane 0 of a strand, which never uses the value, reads
// another strand's lane or 0.
__device__ __forceinline__ float from_prev_lane(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x111, 0xf, 0xf, true));
}

// One time step of the lane pipeline (G > 1): every lane runs the same code;
// `active` lanes perform iteration t - g.  PARK: some lane may be in its last
// iteration (the last G time steps): those lanes (`fin`) keep their points'
// positions before the sweep (PL of them in LDS, the others in q) and leave
// their collisions to the settle pass.  lead: the previous lane's last point
// of the same iteration, before its collision; the next step's is fetched
// here, between the sweep and the collisions.
// GUARD: the last lane of a strand may hold fewer than M points; the slots
// after its last one hold copies of the last input point, which are swept
// (finite, never stored).
template <int M, int G, bool GUARD, bool PARK, int PL, int NQ>
__device__ __forceinline__ void sweep_pipe(const Spheres& S, float3 (&p)[M], const LenRegs<M>& l, float3& lead, int g,
                                           bool active, bool fin, float* park, float3 (&q)[NQ],
                                           int cm) {
  if (PARK && fin) {
#pragma unroll
    for (int j = 0; j < M; ++j) {
      if (j < PL) {
        park[park_slot(j, 0, 0)] = p[j].x;
        park[park_slot(j, 1, 0)] = p[j].y;
        park[park_slot(j, 2, 0)] = p[j].z;
      } else {
        q[j - PL] = p[j];
      }
    }
  }
  if (active) {
    if (g != 0) ftl_point(p[0], lead, l.get(0));  // (lane 0's slot 0 is the root)
    sweep_points<M>(p, [&](int j) { return l.get(j); });  // l holds sigma * rest length
  }
  // (An inactive lane's value is read only by the next lane while that lane is
  // inactive too: fill and drain shift by one step per lane.)
  lead = f3(from_prev_lane(p[M - 1].x), from_prev_lane(p[M - 1].y), from_prev_lane(p[M - 1].z));
  // Every point collides after the whole sweep (the root of lane 0 excepted).
  collide_sweep<M>(S, p, PARK ? active && !fin : active, g != 0, M, cm);
}

// Shared memory of one tile: the load/store stage, and the rest lengths of
// the forms with one lane per strand (an empty base for the others, so a
// pipelined tile takes exactly its stage).
template <int M, bool ON>
struct TileLens {
  float lens[FTL_WAVE * M];
};
template <int M>
struct TileLens<M, false> {};

template <int M, int G, bool GUARD>
struct TileLds : TileLens<M, G == 1> {
  static constexpr int kStage = FTL_WAVE * Tile<M, G, GUARD>::C;
  static constexpr int kPark = (3 * kParkLds<M, G, GUARD> * (FTL_WAVE + 1) + 3) / 4;
  float4 stage[G > 1 && kPark > kStage ? kPark : kStage];
};

// PD: rows of the load phase whose loads are in flight ahead of the row being
// integrated (each costs 7 VGPRs; the forms with a high occupancy target use 1).
// LW: where the wind gathers read the groom's wind lattice: 0 global memory,
// 1 wl = the whole lattice copied to LDS by the workgroup, 2 wl = its half
// lattice (first float4 of each node) in LDS.
// WIND: whether the launch has wind, where the kernel knows.
enum { kWindOff = 0, kWindOn = 1, kWindAny = 2 };
template <int M, int G, bool GUARD, FtlCache CP, int WIND, int PD_ = FTL_LOAD_AHEAD, int LW = 0>
__device__ __forceinline__ void ftl_tile(const FtlStep& A, int strand0, TileLds<M, G, GUARD>& sh,
                                         const float4* wl = nullptr) {
  float4* __restrict__ stage = sh.stage;
  constexpr int C = Tile<M, G, GUARD>::C;
  // Opaque: in the tile-list kernel (a workgroup may step several tiles)
  // nothing lane-derived is hoisted out of the tile loop (it would stay live, in registers, across every tile).
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & (FTL_WAVE - 1);
  const int g = (G == 1) ? 0 : (lane % G);
  const int N = GUARD ? A.npoints : M * G;
  // points held by this lane: with G > 1 and GUARD the strand's last lane
  // holds N - (G - 1) * M of its M slots (the guarded pipelined classes take
  // (G - 1) * M < N <= G * M)
  const int nl = GUARD ? (G == 1 ? A.npoints : min(max(A.npoints - g * M, 0), M)) : M;
  const int nstr = A.nstrands;
  const int strand = strand0 + lane / G;
  const bool valid = strand < nstr;
  const int slast = nstr - 1;

  float3 p[M];
  using Len = typename std::conditional<G == 1, LenLds, LenRegs<M>>::type;
  Len l;
  if constexpr (G == 1) l.base = sh.lens + lane;

  // ---- load + integrate, through LDS ------------------------------------
  // Row i of the tile is point i % C of chunk i / C of every owner lane, read
  // in the coalesced order (64 consecutive float4 per instruction).  Loads run
  // PD rows ahead of the row being integrated, and a row's wind gathers are
  // issued before the loads of row i + PD: loads return in issue order, so
  // waiting for the gathers never waits for HBM.  (Lanes past a partial tile
  // read zeros, and what they compute is never stored.)
  const float dt = pin_s(A.dt), dt2 = pin_s(A.dt2);
  const float3 F0 = f3(pin_s(A.force[0]), pin_s(A.force[1]), pin_s(A.force[2]));
  WindArgs W;
  W.T = (GlobalFloat4*)pin_p(A.wind);
  W.freq = pin_s(A.wind_freq);
  W.off[0] = pin_s(A.wind_off[0]);
  W.off[1] = pin_s(A.wind_off[1]);
  W.off[2] = pin_s(A.wind_off[2]);
  // The root source of the lane's strand, fetched first so that its latency
  // overlaps the row loads.  The root's row slot carries its input position
  // through the transpose; the root is formed from both after it.
  const bool owns_root = (G == 1 || g == 0);
  float3 rsrc = f3(0.f, 0.f, 0.f);
  if (owns_root && A.rmode != kRootModel) rsrc = root_source(A, min(strand, slast));
  __builtin_amdgcn_sched_barrier(0);

  const size_t at = (size_t)strand0 * N;
  const unsigned bytes = 16u * (unsigned)(min(Tile<M, G, GUARD>::SPT, nstr - strand0) * N);
  const BufferRsrc bpos = buffer_of(A.pos + at, bytes), bvel = buffer_of(A.vel + at, bytes);
  float3 u0 = f3(0.f, 0.f, 0.f);
  // With and without wind are two copies of the phase, so that neither tests
  // it row by row.
  auto load_phase = [&](auto wind_on) {
    constexpr bool wind = decltype(wind_on)::value;
    // (The compiler otherwise joins what the copies have in common at their
    // heads and keeps it alive through both: the 8-point forms of one lane took
    // 92 to 96 VGPRs, or spilled, against 79 to 90.  Us a step of one lane a
    // strand, joined and apart: 524k strands of 8 points 67.7, 66.2 with wind,
    // 58.0, 52.7 without; 600k of 7 90.4, 88.8 with wind, 73.3, 70.0 without.)
    if constexpr (wind)
      asm volatile("; with wind" ::: "memory");
    else
      asm volatile("; without wind" ::: "memory");
    constexpr int RS = FTL_WAVE / C / G;
    // Streaming loads (ftl_cache_for) keep no line, so a line that two rows read
    // comes twice: not for strands that are no whole lines, nor for the 4-point
    // form, which they slow as well.  (Us a step above 384 MB, with and without
    // them: 546 MB of 4 points 246, 215; of 7, one lane, 477, 304; of 20, two
    // lanes, 389, 274; of 31, two lanes, 440 MB 466, 324; but of 40 and 48 on one
    // lane they gain 4 to 15%.)
    constexpr bool kStream = CP == kCacheStream && !wind && (GUARD ? M >= 48 : M * G > 4);
    // (the global gathers' taps leave the registers for two rows)
    constexpr int PD = wind && LW == 0 && PD_ > 2 ? 2 : PD_ < M ? PD_ : M;
    float4 xr[PD + 1], vr[PD + 1];
    const int r0 = lane / C;
    float4* const row_slot = stage + slot<C>(r0, lane % C);
    const bool root_row = r0 % G == 0 && lane % C == 0;  // in the rows of chunk 0
    const unsigned off0 = row_offset<M, G, GUARD, true>(N, 0, lane);
    auto load_row = [&](int i) {
      const unsigned first = GUARD ? row_offset<M, G, GUARD, true>(N, i / C, lane) : off0 + 16u * (i / C * C);
      const unsigned off = first + 16u * (unsigned)(i % C * RS * N);
      xr[i % (PD + 1)] = buffer_load4<kStream>(bpos, off);
      vr[i % (PD + 1)] = buffer_load4<kStream>(bvel, off);
    };
#pragma unroll
    for (int i = 0; i < PD; ++i) load_row(i);
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const int c = i / C;
      const float4 x = xr[i % (PD + 1)], v = vr[i % (PD + 1)];
      WindTaps wt;
      if constexpr (wind) {
        if constexpr (LW == 2)
          wt = wind_fetch_half(wl, W, f3(x.x, x.y, x.z));
        else if constexpr (LW == 1)
          wt = wind_fetch_from(wl, W, f3(x.x, x.y, x.z));
        else
          wt = wind_fetch(W, f3(x.x, x.y, x.z));
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i + PD < M) load_row(i + PD);
      __builtin_amdgcn_sched_barrier(0);
      float3 F = F0;
      if constexpr (wind) {
        const float3 w = wind_blend(wt);
        F = f3(F0.x + w.x, F0.y + w.y, F0.z + w.z);
      }
      float3 pr = f3(__builtin_fmaf(dt2, F.x, __builtin_fmaf(dt, v.x, x.x)),
                     __builtin_fmaf(dt2, F.y, __builtin_fmaf(dt, v.y, x.y)),
                     __builtin_fmaf(dt2, F.z, __builtin_fmaf(dt, v.z, x.z)));
      if (c == 0 && root_row) pr = f3(x.x, x.y, x.z);
      row_slot[i % C * FTL_WAVE] = make_float4(pr.x, pr.y, pr.z, x.w);
      __builtin_amdgcn_sched_barrier(0);
      if (i % C == C - 1) {
        tile_sync();
#pragma unroll
        for (int k = 0; k < C; ++k) {
          const float4 t = stage[slot<C>(lane, k)];
          p[c * C + k] = f3(t.x, t.y, t.z);
          // The copy takes the length out of the read's four registers, which the
          // allocator otherwise keeps together: 126 -> 109 VGPRs at M = 16, and
          // with that four waves per SIMD instead of two (50k strands of 64
          // points with wind 86.6 -> 84.8 us, 262k of 32 133.1 -> 131.7 us).
          float len = t.w;
          if constexpr (G > 1) asm volatile("v_mov_b32 %0, %1" : "=v"(len) : "v"(t.w));
          l.set(c * C + k, len);
        }
        tile_sync();
        if (c == 0 && owns_root) {
          // root: p0 = M * source (:190-193); the pipelined forms keep u0 = p0 - x0
          const float3 x0 = p[0];
          const float3 src = A.rmode == kRootModel ? x0 : rsrc;
          p[0] = A.model_ident ? src : transform(A, src);
          if (G > 1) u0 = sub3(p[0], x0);
        }
      }
    }
  };
  if (WIND == kWindOn || (WIND == kWindAny && A.wind_grid))
    load_phase(std::true_type{});
  else
    load_phase(std::false_type{});

  // ---- rest lengths scaled once per tile (pipelined forms) ---------------
  // Every sweep uses sigma * l[j]: formed here once, the same product each
  // iteration formed before.  With sigma == 1 it is l[j] itself; otherwise
  // the position store re-reads the rest lengths from the step's input.  (The
  // one-lane forms keep their lengths in LDS and multiply per point: the
  // store's re-read costs them registers they do not have.)
  const bool unit_sigma = G == 1 || A.sigma == 1.0f;
  if (!unit_sigma) {
    const float sg = A.sigma;
#pragma unroll
    for (int j = 0; j < M; ++j) l.set(j, sg * l.get(j));
  }

  // ---- colliders the wave can reach this step ----------------------------
  unsigned reach;
  {
    float L = 0.0f;
#pragma unroll
    for (int j = 0; j < M; ++j)
      // |sigma * l|: a negative length scale or rest length still places a
      // point that far from its leader.
      if (j >= (G == 1 ? 1 : 0) && (!GUARD || j < nl)) L += fabsf(G == 1 ? A.sigma * l.get(j) : l.get(j));
    float3 root = p[0];
    if (G > 1) {
      // strand total and root, from the lanes of the strand
      for (int o = 1; o < G; o <<= 1) L += __shfl_xor(L, o, G);
      root = f3(__shfl(root.x, 0, G), __shfl(root.y, 0, G), __shfl(root.z, 0, G));
    }
    const unsigned mine = valid ? reachable_colliders(A, root, L) : 0u;
    unsigned any = 0u;
#pragma unroll
    for (int k = 0; k < FTL_NCOL; ++k)
      if (__ballot((mine >> k) & 1u) != 0ull) any |= 1u << k;
    reach = __builtin_amdgcn_readfirstlane(any);
  }
  int cm;  // colliders the tile meets
  const Spheres S = load_spheres(A, reach, cm);
  const VelArgs V = vel_args(A);

  // ---- constraints ------------------------------------------------------
  // Lane's own points, for the DFTL re-read of x (never stored through).
  const float4* __restrict__ pp = A.pos + (size_t)(valid ? strand : 0) * N + (size_t)g * M;
  const int K = A.iterations;
  bool bad = false;
  if constexpr (G == 1) {
    float3 clast = f3(0.f, 0.f, 0.f);
    float3 u;
    for (int it = 0; it < K - 1; ++it)
      sweep<M, GUARD, false, CP>(A, V, S, p, l, nl, pp, clast, stage, bvel, N, lane, cm);
    sweep<M, GUARD, true, CP>(A, V, S, p, l, nl, pp, clast, stage, bvel, N, lane, cm);
    // The last point: velocity = raw correction, collisions deferred to here.
    u = clast;
#pragma unroll
    for (int j = 1; j < M; ++j) {
      if (GUARD ? (j == nl - 1) : (j == M - 1)) {
        float3 pm = p[j];
        collide<true>(S, pm, u, cm);
        p[j] = pm;
        const float3 v = out_velocity(V, pp, j, pm, u);
        bad = !(isfinite(pm.x) && isfinite(pm.y) && isfinite(pm.z) && isfinite(v.x) && isfinite(v.y) &&
                isfinite(v.z));
        stage[slot<C>(lane, j % C)] = make_float4(v.x, v.y, v.z, 0.0f);
        flush_chunk<M, G, GUARD, CP>(bvel, N, j / C, stage, lane);
      }
    }
  } else {
    static_assert(16 % G == 0, "a strand's lanes lie in one row of 16 lanes");
    constexpr int PL = kParkLds<M, G, GUARD>;
    constexpr int NQ = M - PL;
    float* const park = (float*)stage + lane;
    float3 q[NQ];  // every lane fills it in its last iteration
    // No lane is in its last iteration before time step K - 1.  (lane 0 of a
    // strand never reads its lead: its slot 0 is the root)
    float3 lead = p[0];
    for (int t = 0; t < K - 1; ++t)
      sweep_pipe<M, G, GUARD, false, PL, NQ>(S, p, l, lead, g, t >= g, false, park, q, cm);
    for (int t = K - 1; t < K + G - 1; ++t) {
      const int it = t - g;
      sweep_pipe<M, G, GUARD, true, PL, NQ>(S, p, l, lead, g, it >= 0 && it < K, it == K - 1, park, q, cm);
    }
    // Settle: the last iteration's corrections c_j = p_j - parked p_j give the
    // velocities u_j = delta * c_(j+1) (the next lane's first for a lane's last
    // point; the strand's last point keeps its own, the root p0 - x0), then the
    // iteration's collisions push the points and reflect the velocities.  Once
    // per lane: done inside the pipeline's last G steps, this work ran in every
    // one of them for one lane group in G (about 16 vector instructions per
    // point and step).  The long forms are bound by vector issue: 50,021 x 64
    // at 16 iterations 95.0 -> 87.7 us, 60,013 x 20 with wind 42.8 -> 40.1, a
    // frame of 32 uneven grooms 540 -> 525, 262,144 x 32 with wind 137.1 -> 135.1.
    auto parked = [&](int j) -> float3 {
      return j < PL ? f3(park[park_slot(j, 0, 0)], park[park_slot(j, 1, 0)], park[park_slot(j, 2, 0)])
                    : q[j < PL ? 0 : j - PL];
    };
    const float3 c0 = sub3(p[0], parked(0));
    const float3 cn = f3(__shfl_down(c0.x, 1, G), __shfl_down(c0.y, 1, G), __shfl_down(c0.z, 1, G));
    const int tip = g == G - 1 ? nl - 1 : -1;  // slot of the strand's last point on its lane
    const bool root = g == 0;
    float dl = V.delta;
    asm volatile("" : "+v"(dl));
    float3 c = c0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float3 own = c;
      c = m + 1 < M ? sub3(p[m + 1 < M ? m + 1 : m], parked(m + 1 < M ? m + 1 : m)) : cn;
      float3 u = mul3(c, dl);
      if (m == 0) u = sel3(root, u0, u);
      if (GUARD || m == M - 1) u = sel3(tip == m, own, u);
      if (m > 0 || !root) collide<true>(S, p[m], u, cm);
      // GUARD: slots past the strand's last point read its first point
      // instead, and the result is dropped
      const float3 v = out_velocity(V, pp, GUARD && m >= nl ? 0 : m, p[m], u);
      // (the point's own parked words, no longer needed)
      park[park_slot(m % C, 0, 0)] = v.x;
      park[park_slot(m % C, 1, 0)] = v.y;
      park[park_slot(m % C, 2, 0)] = v.z;
      if (GUARD ? m == nl - 1 : m == M - 1)
        bad = !(isfinite(p[m].x) && isfinite(p[m].y) && isfinite(p[m].z) && isfinite(v.x) && isfinite(v.y) &&
                isfinite(v.z));
      if (m % C == C - 1) flush_velocities<M, G, GUARD, CP>(bvel, N, m / C, (float*)stage, lane);
    }
  }
  // positions, after every velocity (DFTL reads the step's input positions);
  // the stage addresses are formed anew (opaque lane): kept from the load
  // phase they would hold eight registers through the sweeps
  int sl = lane;
  asm volatile("" : "+v"(sl));
#pragma unroll
  for (int c = 0; c < M / C; ++c) {
    if (GUARD && G == 1 && c * C >= nl) continue;
    float w[C];
    if (unit_sigma) {
#pragma unroll
      for (int j = 0; j < C; ++j) w[j] = l.get(c * C + j);
    } else {
      // the unscaled rest lengths, from the input (positions are written
      // below); a guarded lane's slots past the strand read its last point
#pragma unroll
      for (int j = 0; j < C; ++j) w[j] = pp[GUARD ? min(c * C + j, nl - 1) : c * C + j].w;
    }
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const float3 q = p[c * C + j];
      stage[slot<C>(sl, j)] = make_float4(q.x, q.y, q.z, w[j]);
    }
    flush_chunk<M, G, GUARD, CP>(bpos, N, c, stage, lane);
  }
  bad = bad && valid;
  const unsigned long long b = __ballot(bad);
  // A plain (system-scope) store of 1, not a read-modify-write: the word may
  // live in pinned host memory (the serving loop's per-request flags), and
  // every writer stores the same value.
  if (b != 0ull && lane == (int)(__ffsll((long long)b) - 1))
    __hip_atomic_store(A.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The span of tile t of a launch: the last whose first tile is at or before t
// (spans[0].tile0 == 0).  The wave's lanes read 64 first tiles at a time, so a
// search over n spans makes log64(n) dependent loads (a scalar binary search
// makes log2(n), each a round trip at the head of the tile).
__device__ __forceinline__ int span_of(const FtlSpan* __restrict__ spans, int nspans, int t) {
  const int lane = (int)threadIdx.x & (FTL_WAVE - 1);
  int lo = 0, n = nspans;
  for (;;) {
    const int stride = (n + FTL_WAVE - 1) / FTL_WAVE;
    const int i = lane * stride;
    const bool before = i < n && spans[lo + min(i, n - 1)].tile0 <= t;
    const int k = max((int)__builtin_popcountll(__ballot(before)) - 1, 0);
    lo += k * stride;
    if (stride == 1) return lo;
    n = min(stride, n - k * stride);
  }
}

}  // namespace ftl_tile_impl
