// Device helpers that work on a whole wavefront, and the flip iteration of one
// workgroup.
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

// The smallest of the wave's values, by lane shifts within the vector unit: rows
// of 16 lanes (row_shr 1, 2, 4, 8), then row to row (row_bcast 15, 31) into lane
// 63.  Every lane of the wave calls it.
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
#define WT_MIN_STEP(ctrl, rows) v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, ctrl, rows, 0xF, false))
  WT_MIN_STEP(0x111, 0xF);
  WT_MIN_STEP(0x112, 0xF);
  WT_MIN_STEP(0x114, 0xF);
  WT_MIN_STEP(0x118, 0xF);
  WT_MIN_STEP(0x142, 0xA);
  WT_MIN_STEP(0x143, 0xC);
#undef WT_MIN_STEP
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The votes of one wave (lane's point i, valid below U; a higher lane's point is
// a later one).  The lanes that vote for the tet of the wave's first pending lane
// elect one vote: the smallest upper word of their keys, and the lowest lane that
// has it, since the lower word is the point.  After kVotePasses such tets the
// remaining lanes vote directly.  The atomics bound the vote (27 G/s on random
// lines): with 4 passes, each a minimum of whole keys through LDS shuffles, 53.2 us
// a launch at 1M points, 9.9 at 100k, 5.6 on a sphere of 50k, 74.1 for 2,048
// clouds; now 48.2, 8.3, 5.4 and 61.5 (16 passes: 46.9, 9.6, 6.7, 55.7).
constexpr int kVotePasses = 8;
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
  const uint32_t hi = (uint32_t)(key >> 32);
  for (int pass = 0; pass < kVotePasses; ++pass) {
    const uint64_t act = __ballot(pending);
    if (!act) break;
    const uint32_t lt = (uint32_t)__builtin_amdgcn_readlane((int)t, __ffsll((unsigned long long)act) - 1);
    const bool mine = pending && t == lt;
    const uint32_t least = wave_min_u32(mine ? hi : 0xFFFFFFFFu);
    const uint64_t have = __ballot(mine && hi == least);
    if (__lane_id() == __ffsll((unsigned long long)have) - 1) mesh_min(M, &TVOTE(M, lt), key);
    if (mine) pending = false;
  }
  if (pending) mesh_min(M, &TVOTE(M, t), key);
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

// The tests of the three edges of every lane's face (inside: the lane has
// one), spread over the wave's active lanes (lanes 0..n-1): job j is edge j % 3
// of the (j / 3)th such lane.  Each lane gets its bits: edge k has the segment
// a-o beyond it.  One after another on the lanes that have a face, the three
// tests kept most of the wave idle for three times as long: 16 tets rarely
// have more than 21 such faces.
template <class MS>
__device__ __forceinline__ uint32_t face_edges_wave(const MS& M, bool inside, const FaceEdges& E, PredStats* st) {
  const uint64_t mask = __ballot(inside);
  const uint32_t n = (uint32_t)__popcll(__ballot(1)), lane = __lane_id();
  const uint32_t jobs = 3u * (uint32_t)__popcll(mask);
  const uint32_t mine = 3u * (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
  uint32_t beyond = 0u;
  for (uint32_t b = 0; b < jobs; b += n) {
    const uint32_t j = b + lane, k = j % 3u;
    // the lane of the job's face: the (j / 3)th set bit of the mask
    uint32_t want = j < jobs ? j / 3u : 0u, src = 0u;
#pragma unroll
    for (uint32_t w = 32u; w > 0u; w >>= 1) {
      const uint32_t low = (uint32_t)__popcll(mask >> src & ((1ull << w) - 1ull));
      if (want >= low) {
        want -= low;
        src += w;
      }
    }
    FaceEdges F;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      F.a[q] = __shfl(E.a[q], (int)src);
      F.o[q] = __shfl(E.o[q], (int)src);
#pragma unroll
      for (int i = 0; i < 3; ++i) F.v[i][q] = __shfl(E.v[i][q], (int)src);
      F.rv[q] = (uint32_t)__shfl((int)E.rv[q], (int)src);
    }
    F.ra = (uint32_t)__shfl((int)E.ra, (int)src);
    F.ro = (uint32_t)__shfl((int)E.ro, (int)src);
    bool out = false;
    if (j < jobs) {
      float X[3], Y[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        X[q] = k == 0u ? F.v[0][q] : (k == 1u ? F.v[1][q] : F.v[2][q]);
        Y[q] = k == 0u ? F.v[1][q] : (k == 1u ? F.v[2][q] : F.v[0][q]);
      }
      const uint32_t rx = k == 0u ? F.rv[0] : (k == 1u ? F.rv[1] : F.rv[2]);
      const uint32_t ry = k == 0u ? F.rv[1] : (k == 1u ? F.rv[2] : F.rv[0]);
      out = o3s<false>(M, X, Y, F.a, F.o, rx, ry, F.ra, F.ro, st) > 0;
    }
    const uint64_t res = __ballot(out);
#pragma unroll
    for (uint32_t q = 0; q < 3u; ++q) {
      const uint32_t d = mine + q - b;  // wraps below b
      if (d < n) beyond |= (uint32_t)(res >> d & 1u) << q;
    }
  }
  return beyond;
}

// The full check of list entry j's face f, four lanes per tet, one per face
// (f = this lane's index modulo 4; a tet's lanes are consecutive in the
// wave and all take part; the wave's active lanes are its first): each lane
// runs its face's staged insphere, the wave the edge tests of the faces whose
// apex lies inside; the lowest face that proposes is the tet's proposal, as a
// loop over the faces would choose it.  A tet's faces
// then reach the exact and SoS stages together rather than one after another
// in divergent passes.
template <class MS>
__device__ __forceinline__ void flip_check_faces(const MS& M, const uint32_t* act, uint4* prop, uint32_t j,
                                                 int f, uint32_t it, PredStats* st) {
  const uint32_t t = act[j];
  const uint4 tv = TV(M, t);
  const uint4 tov = TOV(M, t);
  const bool live = tv.x != kInvalid && tv.x != M.inf && tv.y != M.inf && tv.z != M.inf && tv.w != M.inf;
  bool inside = false, qual = false;
  FaceEdges E = {};
  if (live) {
    float P[4][3], Q[4][3];
    uint32_t R[4], RQ[4];
    for (int q = 0; q < 4; ++q) load_pt(M, get4(tv, q), P[q], &R[q]);
    for (int q = 0; q < 4; ++q) load_pt(M, get4(tov, q), Q[q], &RQ[q]);
    inside = flip_face_inside(M, tov, P, R, Q, RQ, f, st, &E);
  }
  uint32_t kind = 0u, bad = 0u, third = kInvalid;
  const uint32_t beyond = face_edges_wave(M, inside, E, st);
  if (inside) qual = flip_face_kind(M, t, tov, f, beyond, &kind, &bad, &third);
  const uint64_t qb = __ballot(qual);
  const uint32_t g0 = __lane_id() & ~3u;
  const uint32_t grp = (uint32_t)(qb >> g0) & 0xFu;
  const uint32_t cf = grp ? (uint32_t)__builtin_ctz(grp) : 0u;
  const uint32_t pk = (uint32_t)f | kind << 2 | bad << 3;
  const uint32_t pk_c = (uint32_t)__shfl((int)pk, (int)(g0 + cf));
  const uint32_t third_c = (uint32_t)__shfl((int)third, (int)(g0 + cf));
  if (f == 0) {
    if (grp) prop[j] = flip_propose(M, t, cf, opp_tet(*opp_word(M, t, cf)), (pk_c >> 2) & 1u, pk_c >> 3, third_c, it);
    else prop[j].x = kInvalid;
  }
}

// The full walk of point i, four lanes per point, one per face (f = this
// lane's index modulo 4; a point's lanes are consecutive in the wave and all
// take part): the steps of walk_to_t, whose four exact face tests run side by
// side instead of one after another.  A walk is a chain of those tests, so
// a wave waits for one per step, not four (19 walks of 10,000 uniform points
// in exact mode: 160 -> 43 us each).  go_on: the lean walk stopped in utet[i],
// where its filter could not decide; starting over from the point's old tet, the
// walks of a 48^3 lattice took 69 us a launch, 57 going on.
template <class MS>
__device__ __forceinline__ void relocate_faces(const MS& M, const uint32_t* uvert, uint32_t* utet, uint32_t i, int f,
                                               uint32_t it0, bool go_on, PredStats* st) {
  uint32_t t = utet[i];
  if (!go_on && !walk_start(M, it0, &t)) return;
  float Q[3];
  uint32_t rq;
  load_pt(M, uvert[i], Q, &rq);
  const uint32_t seed = walk_seed(i), g0 = __lane_id() & ~3u;
  bool there = false;
  for (uint32_t step = 0; step < kWalkLimit && !there; ++step) {
    const uint4 tv = TV(M, t);
    const uint4 to = TN(M, t);
    const uint32_t r0 = hash32(seed + step * 0x9E3779B9u) & 3u;
    float A[3], B[3], C[3];
    uint32_t ra, rb, rc;
    load_pt(M, get4(tv, face_vi(f, 0)), A, &ra);
    load_pt(M, get4(tv, face_vi(f, 1)), B, &rb);
    load_pt(M, get4(tv, face_vi(f, 2)), C, &rc);
    const bool beyond = o3s<false>(M, A, B, C, Q, ra, rb, rc, rq, st) < 0;
    const uint32_t m = (uint32_t)(__ballot(beyond) >> g0) & 0xFu;
    const uint32_t rot = ((m >> r0) | (m << (4u - r0))) & 0xFu;
    there = m == 0u;
    if (!there) t = opp_tet(get4(to, (int)(((uint32_t)ctz32(rot) + r0) & 3u)));
  }
  if (f == 0) {
    if (!there) at_add_u32(&M.ctr[C_WALK_FAIL], 1u);
    utet[i] = t;
  }
}

// ---------------------------------------------------------------------------
// A flip iteration in one workgroup: barriers in place of launches, counters
// in LDS, atomics at workgroup scope.
// ---------------------------------------------------------------------------
struct WgCounters {
  uint32_t act_next;  // length of the next active list
  uint32_t slots;     // next free tet slot
  uint32_t flips;     // flips of this iteration
  uint32_t slow;      // entries deferred to the full predicates
};

__device__ __forceinline__ uint32_t lds_add(uint32_t* counter, uint32_t v) {
  return __hip_atomic_fetch_add(counter, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// the active lanes that call this together get consecutive entries of an LDS
// counter
__device__ __forceinline__ uint32_t lds_slot(uint32_t* counter) {
  const uint64_t mask = __ballot(1);
  const int lane = __lane_id(), leader = __ffsll((unsigned long long)mask) - 1;
  uint32_t base = 0;
  if (lane == leader) base = lds_add(counter, (uint32_t)__popcll(mask));
  return __shfl(base, leader) + __popcll(mask & ((1ull << lane) - 1ull));
}

// The full predicates on the entries list[0..n) (null: 0..n-1), out of line:
// their registers and stack stay out of the phases that run for every entry.
template <class MS, int BS>
__device__ __noinline__ void wg_slow_check(MS M, const uint32_t* act, uint4* prop, const uint32_t* list, uint32_t n,
                                           uint32_t it, uint64_t* st) {
  PredStats ls = {};
  for (uint32_t k = threadIdx.x; k < 4u * n; k += BS)
    flip_check_faces(M, act, prop, list ? list[k >> 2] : k >> 2, (int)(k & 3u), it, &ls);
  flush_stats(ls, st);
}

// The full point split (walk: relocation) of the points list[0..n) (null:
// 0..n-1), out of line for the same reason.  a: the round (walk: the flip
// iterations before it).
template <class MS, int BS>
__device__ __noinline__ void wg_slow_points(MS M, const uint32_t* uvert, uint32_t* utet, const uint32_t* list,
                                            uint32_t n, uint32_t a, bool walk, uint64_t* st) {
  PredStats ls = {};
  if (walk) {
    for (uint32_t k = threadIdx.x; k < 4u * n; k += BS)
      relocate_faces(M, uvert, utet, list ? list[k >> 2] : k >> 2, (int)(k & 3u), a, list != nullptr, &ls);
  } else {
    for (uint32_t k = threadIdx.x; k < n; k += BS) (void)split_points_body_t<false>(M, uvert, utet, list ? list[k] : k, a, &ls);
  }
  flush_stats(ls, st);
}

// exclusive rank of `flag` within the workgroup of BS threads, *total its
// count; every thread calls it; w: BS / 64 words of LDS
template <int BS>
__device__ __forceinline__ uint32_t wg_rank(bool flag, uint32_t* total, uint32_t* w) {
  const uint64_t m = __ballot(flag);
  const uint32_t wave = threadIdx.x >> 6;
  if (__lane_id() == 0) w[wave] = __popcll(m);
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (uint32_t k = 0; k < BS / 64; ++k) {
    off += k < wave ? w[k] : 0u;
    tot += w[k];
  }
  __syncthreads();
  *total = tot;
  return off + __popcll(m & ((1ull << __lane_id()) - 1ull));
}

// Checks, decides and executes the A entries of act (tag it); the entries of
// the next iteration go to next.  Every thread of the workgroup of BS threads
// calls it.  On return c.act_next, c.slots, c.flips and c.slow hold the
// results and every thread may read them; c.slots counts on from its value
// before the call.  prop, slow_t: A entries of scratch; out: four per flip
// (at most half as many as the mesh has tets).
template <class MS, int BS>
__device__ __forceinline__ void wg_flip_iteration(const MS& M, WgCounters& c, const uint32_t* act, uint32_t* next,
                                                  uint4* prop, uint32_t* slow_t, uint4* out, uint32_t A,
                                                  uint32_t it, uint64_t* st) {
  const uint32_t tid = threadIdx.x;
  const uint64_t lt = (1ull << __lane_id()) - 1ull;
  const bool filtered = M.mode == PRED_FILTERED;
  if (tid == 0) {
    c.act_next = 0u;
    c.flips = 0u;
    c.slow = 0u;
  }
  __syncthreads();
  uint32_t ns = A;
  if (filtered) {
    PredStats ls = {};
    for (uint32_t j = tid; j < A; j += BS)
      if (flip_check_lean(M, act[j], prop, j, it, &ls)) slow_t[lds_slot(&c.slow)] = j;
    flush_stats(ls, st);
    __syncthreads();
    ns = c.slow;
  }
  if (ns) {
    wg_slow_check<MS, BS>(M, act, prop, filtered ? slow_t : nullptr, ns, it, st);
    __syncthreads();
  }
  // a wave claims its flips, fresh slots and queue entries with one LDS
  // atomic of three lanes
  for (uint32_t b = 0; b < A; b += BS) {
    const uint32_t j = b + tid;
    uint4 pr = make_uint4(kInvalid, 0u, 0u, 0u);
    if (j < A) pr = prop[j];
    uint32_t qid[2], nq, nslot;
    FlipTets F;
    const bool win = flip_decide_load(M, pr, it, qid, &nq, &nslot, F);
    const uint32_t nqa = nq + nslot;
    const uint64_t bw = __ballot(win), bs = __ballot(nslot), q0 = __ballot(nqa & 1u), q1 = __ballot(nqa & 2u);
    const uint32_t l = __lane_id();
    uint32_t* p = l == 0u ? &c.flips : (l == 1u ? &c.slots : &c.act_next);
    const uint32_t v = l == 0u ? __popcll(bw) : (l == 1u ? __popcll(bs) : __popcll(q0) + 2u * __popcll(q1));
    uint32_t claim = 0u;
    if (l < 3u && v) claim = lds_add(p, v);
    const uint32_t cf = __shfl(claim, 0) + __popcll(bw & lt);
    const uint32_t cs = __shfl(claim, 1) + __popcll(bs & lt);
    const uint32_t cq = __shfl(claim, 2) + __popcll(q0 & lt) + 2u * __popcll(q1 & lt);
    if (nq > 0u) next[cq] = qid[0];
    if (nq > 1u) next[cq + 1u] = qid[1];
    if (win) {
      if (nslot) next[cq + nq] = cs;
      flip_exec_loaded(M, pr, F, it, nslot ? cs : kInvalid, &out[4 * (size_t)cf]);
    }
  }
  __syncthreads();
  const uint32_t nf = c.flips;
  for (uint32_t k = tid; k < nf; k += BS) flip_update_body(M, out, k, it);
  __syncthreads();
}

}  // namespace wtet
