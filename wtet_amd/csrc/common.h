// Shared layout, encodings and small helpers for the triangulation kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "predicates.h"

namespace wtet {

constexpr uint32_t kInvalid = 0xFFFFFFFFu;
constexpr uint64_t kVoteNone = 0xFFFFFFFFFFFFFFFFull;

// A slot's queue tag (Mesh::tqueue): the last flip iteration in which the tet,
// as an entry of the list, proposed a flip (or, with kWaits, was left to a
// later one).  Its own thread then appends it to the next list, won or lost,
// so that a list takes each tet once with no atomic, and the tag stands for
// the proposal's vote for the tet itself.  kListed | i while it waits in the
// list that iteration i begins with, over an insertion round; kFreed for a
// slot that a 3-2 flip freed (its record then holds kInvalid as first vertex
// and a live neighbour to go on to).
constexpr uint32_t kWaits = 0x40000000u;
constexpr uint32_t kListed = 0x80000000u;
constexpr uint32_t kFreed = 0xFFFFFFFFu;

// Face f of a tet is the face opposite vertex f.  kFace[f] lists its three
// vertex positions ordered so that (face..., v_f) is an even permutation of
// (v0, v1, v2, v3): for a tet with raw orient3d < 0, orient3d(face, v_f) < 0.
WT_HD int face_vi(int f, int k) {
  // {1,3,2}, {0,2,3}, {0,3,1}, {0,1,2}
  const uint32_t packed = (1u | 3u << 2 | 2u << 4) | (0u | 2u << 2 | 3u << 4) << 6 |
                          (0u | 3u << 2 | 1u << 4) << 12 | (0u | 1u << 2 | 2u << 4) << 18;
  return (int)((packed >> (6 * f + 2 * k)) & 3u);
}

// adjacency: (tet << 2) | face, kInvalid when none
WT_HD uint32_t enc_opp(uint32_t t, uint32_t f) { return (t << 2) | f; }
WT_HD uint32_t opp_tet(uint32_t e) { return e >> 2; }
WT_HD uint32_t opp_face(uint32_t e) { return e & 3u; }

// Component i (0..3, chosen at run time) of a quad, by selects on i's bits and
// on single components.  Not as a chain of tests of i: the compiler makes a
// switch of such a chain, a tree of branches with the exec mask saved and
// restored at each (k_flip_decide_exec: 114 branches in 1,640 instructions, 23
// in 882 with selects; 100k points 3.07 -> 2.70 ms, 1M 7.11 -> 6.81 ms).
template <typename T>
WT_HD T pick4(int i, T a, T b, T c, T d) {
  const bool odd = (i & 1) != 0, hi = (i & 2) != 0;
  const T ab = odd ? b : a, cd = odd ? d : c;
  return hi ? cd : ab;
}
WT_HD uint32_t get4(const uint4& v, int i) { return pick4(i, v.x, v.y, v.z, v.w); }
WT_HD void set4(uint4& v, int i, uint32_t x) {
  v.x = i == 0 ? x : v.x;
  v.y = i == 1 ? x : v.y;
  v.z = i == 2 ? x : v.z;
  v.w = i == 3 ? x : v.w;
}
// the component that equals x (one does)
WT_HD int find4(const uint4& v, uint32_t x) {
  const int hi = (v.z == x) | (v.w == x), odd = (v.y == x) | (v.w == x);
  return 2 * hi + odd;
}

// Points: xyz in f32, w holds the SoS rank (original input id) as bits.
WT_HD uint32_t pt_rank(const float4& p) { return f32_bits(p.w); }

// ---------------------------------------------------------------------------
// atomics (device instructions; plain host builtins for host-side callers)
// ---------------------------------------------------------------------------
WT_HD uint64_t at_min_u64(uint64_t* p, uint64_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return atomicMin((unsigned long long*)p, (unsigned long long)v);
#else
  return __atomic_fetch_min(p, v, __ATOMIC_RELAXED);
#endif
}
WT_HD uint32_t at_add_u32(uint32_t* p, uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return atomicAdd(p, v);
#else
  return __atomic_fetch_add(p, v, __ATOMIC_RELAXED);
#endif
}

// the same at workgroup scope, for data that one workgroup owns while it
// runs: performed in the XCD's L2, not at the memory side
WT_HD void wg_min_u64(uint64_t* p, uint64_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  (void)__hip_atomic_fetch_min((unsigned long long*)p, (unsigned long long)v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
#else
  (void)__atomic_fetch_min(p, v, __ATOMIC_RELAXED);
#endif
}

// Append to a list with one atomic per wavefront: the active lanes that call
// this together get consecutive slots.
WT_HD uint32_t append_slot(uint32_t* counter) {
#if defined(__HIP_DEVICE_COMPILE__)
  uint64_t mask = __ballot(1);
  int lane = __lane_id();
  int leader = __ffsll((unsigned long long)mask) - 1;
  uint32_t rank = __popcll(mask & ((1ull << lane) - 1ull));
  uint32_t base = 0;
  if (lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(mask));
  base = __shfl(base, leader);
  return base + rank;
#else
  return __atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED);
#endif
}

// 32-bit mixing hash (lowbias32) used to vary walk face order
WT_HD uint32_t hash32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

}  // namespace wtet
