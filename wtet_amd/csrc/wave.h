// Device helpers that work on a whole wavefront, for the kernels of kernels.hip.
#pragma once

#include "ops.h"
#include "prep.h"

namespace wtet {

// Adds this thread's local counters to the global u64 counters (one atomic
// per counter per wavefront).  Must be reached by every lane of the wave.
__device__ __forceinline__ void flush_stats(const PredStats& ls, uint64_t* st) {
  if (!st) return;
  unsigned long long* g = reinterpret_cast<unsigned long long*>(st);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    uint32_t v = ls.c[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if (__lane_id() == 0 && v) atomicAdd(g + k, (unsigned long long)v);
  }
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
  uint32_t lo = __shfl_xor((uint32_t)v, m), hi = __shfl_xor((uint32_t)(v >> 32), m);
  return ((uint64_t)hi << 32) | lo;
}

// The votes of one wave (lane's point i, valid below U).  Lanes voting for
// the same tet as the wave's first pending lane combine their keys with a
// wave min first (a few passes), so early rounds -- when most points still
// share a few tets -- issue one atomic per wave instead of one per point;
// the remaining lanes vote directly.
template <class MS>
__device__ __forceinline__ void vote_wave(const MS& M, const uint32_t* uvert, const uint32_t* utet,
                                          uint32_t i, uint32_t U) {
  uint64_t key = kVoteNone;
  uint32_t t = 0;
  if (i < U) {
    t = utet[i];
    key = vote_key(M, uvert, utet, i);
  }
  bool pending = key != kVoteNone;
  for (int pass = 0; pass < 4; ++pass) {
    uint64_t act = __ballot(pending);
    if (!act) break;
    int leader = __ffsll((unsigned long long)act) - 1;
    uint32_t lt = __shfl(t, leader);
    bool mine = pending && t == lt;
    uint64_t k = mine ? key : kVoteNone;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      uint64_t o = shfl_xor_u64(k, off);
      k = o < k ? o : k;
    }
    if (__lane_id() == leader) at_min_u64(&TVOTE(M, lt), k);
    if (mine) pending = false;
  }
  if (pending) at_min_u64(&TVOTE(M, t), key);
}

// sorted position j of cloud c: kept unless it is a redundant duplicate;
// the uninserted list holds (vertex j + 4c, start super tet 5c)
__device__ __forceinline__ bool keep_point(const float4* pts, const uint64_t* keys, uint32_t n,
                                           const Clouds& K, uint32_t j, uint32_t* c,
                                           uint32_t* capped) {
  if (j >= n) return false;
  *c = cloud_of_key(K, keys[j]);
  return !redundant_dup(pts + 4u * *c, keys, n, j, capped);
}

// The full check of list entry j's face f, four lanes per tet, one per face
// (f = this lane's index modulo 4; a tet's lanes are consecutive in the
// wave and all take part): each lane runs its face's staged insphere and,
// where the face's apex lies inside, the three orient3d that classify the
// flip; the lowest face that proposes is the tet's proposal, as a loop over
// the faces would choose it.  A tet's faces
// then reach the exact and SoS stages together rather than one after another
// in divergent passes.
template <class MS>
__device__ __forceinline__ void flip_check_faces(const MS& M, const uint32_t* act, uint4* prop, uint32_t j,
                                                 int f, uint32_t it, PredStats* st) {
  const uint32_t t = act[j];
  const uint32_t info = INFO(M, t);
  const uint4 tv = TV(M, t);
  const uint4 tov = TOV(M, t);
  const bool live = (info & kAlive) && tv.x != M.inf && tv.y != M.inf && tv.z != M.inf && tv.w != M.inf;
  bool qual = false;
  uint32_t kind = 0u, bad = 0u, third = kInvalid;
  if (live) {
    float P[4][3], Q[4][3];
    uint32_t R[4], RQ[4];
    for (int q = 0; q < 4; ++q) load_pt(M, get4(tv, q), P[q], &R[q]);
    for (int q = 0; q < 4; ++q) load_pt(M, get4(tov, q), Q[q], &RQ[q]);
    qual = flip_face_full(M, t, tov, P, R, Q, RQ, f, st, &kind, &bad, &third);
  }
  const uint64_t qb = __ballot(qual);
  const uint32_t g0 = __lane_id() & ~3u;
  const uint32_t grp = (uint32_t)(qb >> g0) & 0xFu;
  const uint32_t cf = grp ? (uint32_t)__builtin_ctz(grp) : 0u;
  const uint32_t pk = (uint32_t)f | kind << 2 | bad << 3;
  const uint32_t pk_c = (uint32_t)__shfl((int)pk, (int)(g0 + cf));
  const uint32_t third_c = (uint32_t)__shfl((int)third, (int)(g0 + cf));
  if (f == 0) {
    // each entry is in the list once and only its lanes touch its info
    INFO(M, t) = info & ~kQueued;
    if (grp) prop[j] = flip_propose(M, t, cf, (pk_c >> 2) & 1u, pk_c >> 3, third_c, it);
    else prop[j].x = kInvalid;
  }
}

}  // namespace wtet
