// Per-element bodies of the insertion/flip round kernels.
//
// One call handles one element (an uninserted point, a winning tet, an
// active tet, an executed flip).  The __global__ wrappers live in
// kernels.hip.  The algorithm follows the reference's phase-1 loop
// (src/phase1.rs:16-1431): vote -> 1-to-4 split -> point split -> flip
// iterations (check, vote, flip, adjacency update) -> point relocation,
// re-designed around device-resident lists instead of full-array scans.
#pragma once

#include "common.h"

namespace wtet {

// device-side counters (Mesh::ctr)
enum Ctr : int {
  // read by every thread of the flip kernels, written between kernels: the
  // first line.  Counters that take atomics at volume sit 1 KB or more apart,
  // away from it and from each other.
  C_IT = 0,         // flip iterations before this batch (fvote keys, stamps, queue tags)
  C_PAR = 1,        // which of the two active lists the batch begins with
  C_STOP = 2,       // set when an iteration could overflow the tet slots
  C_ROUND = 3,      // insertion round (split records)
  C_CAP = 4,        // tet slot capacity
  C_PEAKA = 5,      // longest active list seen
  C_TETS_IT = 6,    // C_TETS when the batch of iterations began
  C_SLOW_SUM = 7,   // tets deferred by the lean flip check, summed over iterations
  C_SLOW_LAST = 8,  // tets deferred in the last iteration
  C_WALK_FAIL = 9,  // relocation walks that hit the step limit
  C_WIN = 10,       // insertions this round
  C_ALIVE = 11,     // alive tets (output compaction)
  C_BADTET = 12,    // points found in a tet touching infinity (must stay 0)
  C_NPTS = 13,      // points to insert (input minus exact duplicates)
  C_DUPSCAN = 14,   // duplicate scans that hit their length cap
  C_IT0 = 16,       // flip iterations before this round
  C_CHECK_SUM = 20, // list entries checked in launched iterations, summed (wraps)
  C_RUN_PICKS = 17, // of k_rounds_small: rounds it picked,
  C_RUN_SUMU = 18,  // the points they chose from,
  C_RUN_DONE = 19,  // whether the last round is over,
  C_RUN_CROWDED = 21,  // and whether its last round left too many to the full predicates (SmallRun::list_full)
  C_SURV = 15,      // uninserted points (the pick's winners leave at the split)
  C_TETS = 256,     // next free tet slot (the winners' at the split)
  C_LIST = 512,     // length of the active list between batches of iterations
  C_SLOW_P = 768,   // points deferred by the lean point split
  C_SLOW_R = 1024,  // points deferred by the lean relocation
  C_SLOW_T = 1280,  // tets deferred by the lean audit
  C_VIOL = 1536,    // non-Delaunay faces found by the audit
  C_FAILREC = 1537, // recorded violation entries
  C_HEAD = 1792,    // the counters the host reads
  // one slot per iteration of a batch, a 128-byte line apart, and a zero
  // slot after the last: list length, executed flips, deferred tets, and
  // whether the iteration ran
  C_ITA = C_HEAD,
  C_ITF = C_ITA + 65 * 32,
  C_ITS = C_ITF + 65 * 32,
  C_ITR = C_ITS + 65 * 32,
  C_COUNT = C_ITR + 65 * 32
};
constexpr int kMaxBatch = 64;  // flip iterations in a batch

// per-call sums over flip iterations (u64, device)
enum IterSum : int {
  S_CHECKED = 0,        // tets checked
  S_FLIPS = 1,          // flips executed
  S_ITERS = 2,          // iterations
  S_FLIPS23 = 3,        // 2-3 flips (the rest are 3-2)
  S_SMALL_CHECKED = 4,  // of S_CHECKED: in one-workgroup kernels
  S_SMALL_FLIPS = 5,    // of S_FLIPS: in one-workgroup kernels
  S_COUNT = 8
};

// Adjacency of a tet slot in one 32-byte record: per face f, w[2f] = the
// neighbour across it ((tet << 2) | face) and w[2f + 1] = that neighbour's
// vertex opposite the face.  The flip check reads its own slot only, and
// the adjacency update rewrites a face with one 8-byte store.
struct __attribute__((aligned(32))) AdjRec {
  uint4 lo;  // faces 0, 1
  uint4 hi;  // faces 2, 3
};

// One tet slot's record, a 64-byte half line: everything about it that plain
// stores write and that the kernels read at random.  What atomics write (the
// votes) is in arrays of its own: atomics complete at the memory side, and a
// plain store beside them would leave the line dirty in an XCD's L2.  Measured against an array per field (the check then read
// three lines of a tet, a flip wrote three of each new tet): see
// k_flip_decide_exec.
struct __attribute__((aligned(64))) TetRec {
  AdjRec adj;      // neighbours and the vertices across the faces
  uint4 v;         // vertex ids; x = kInvalid when a 3-2 flip freed the slot
  uint2 split;     // (round, first new slot) for a tet split this round
  uint32_t point;  // the point inserted into a tet split this round; in a freed
                   // slot a live neighbour
  uint32_t stamp;  // tag of the last flip iteration that took the tet apart
};

// Where the faces of a tet destroyed by a flip went: for each external face
// f, w[2f] = (new tet << 2) | face and w[2f + 1] = the new tet's vertex
// opposite it (one 8-byte load per face in flip_update_body).
struct __attribute__((aligned(32))) FlipMsg {
  uint4 lo;  // faces 0, 1
  uint4 hi;  // faces 2, 3
};

// message of a destroyed tet: new neighbour pointers e (kInvalid where
// unused), all opposite the vertex v
WT_HD void set_msg(FlipMsg* m, uint4 e, uint32_t v) {
  m->lo = make_uint4(e.x, v, e.y, v);
  m->hi = make_uint4(e.z, v, e.w, v);
}

static_assert(sizeof(AdjRec) == 32, "adjacency record layout");
static_assert(sizeof(TetRec) == 64, "half a line per slot");
static_assert(sizeof(FlipMsg) == 32, "flip message layout");

struct Mesh {
  const float4* pts;  // n + 5 points (n real, 4 super, 1 infinity)
  TetRec* rec;
  FlipMsg* tmsg;     // per slot destroyed by a flip this iteration
  uint32_t* tqueue;  // queue tag (kListed, kFreed)
  uint64_t* tvote;   // insertion vote (min key)
  uint64_t* fvote;   // flip vote (min key, iteration-tagged)
  uint32_t* ctr;     // Ctr counters
  uint32_t inf;      // id of the infinity vertex
  int mode;          // PredMode
};

WT_HD uint4& TV(const Mesh& M, uint32_t t) { return M.rec[t].v; }
WT_HD AdjRec& ADJ(const Mesh& M, uint32_t t) { return M.rec[t].adj; }
WT_HD uint2& TSPLIT(const Mesh& M, uint32_t t) { return M.rec[t].split; }
WT_HD uint32_t& TPOINT(const Mesh& M, uint32_t t) { return M.rec[t].point; }
WT_HD uint32_t& TFWD(const Mesh& M, uint32_t t) { return M.rec[t].point; }
WT_HD uint32_t& FSTAMP(const Mesh& M, uint32_t t) { return M.rec[t].stamp; }
WT_HD FlipMsg& TMSG(const Mesh& M, uint32_t t) { return M.tmsg[t]; }
WT_HD uint32_t& TQUEUE(const Mesh& M, uint32_t t) { return M.tqueue[t]; }
WT_HD uint64_t& TVOTE(const Mesh& M, uint32_t t) { return M.tvote[t]; }
WT_HD uint64_t& FVOTE(const Mesh& M, uint32_t t) { return M.fvote[t]; }
WT_HD bool slot_alive(const Mesh& M, uint32_t t) { return M.tqueue[t] != kFreed; }

// The same mesh while one workgroup alone changes it: its atomics need the
// workgroup's scope only and complete in the XCD's L2 instead of at the
// memory side.
struct WgMesh : Mesh {};

// atomics at the scope the mesh is shared at
WT_HD void mesh_min(const Mesh&, uint64_t* p, uint64_t v) { at_min_u64(p, v); }
WT_HD void mesh_min(const WgMesh&, uint64_t* p, uint64_t v) { wg_min_u64(p, v); }

template <class MS>
WT_HD uint4 TN(const MS& M, uint32_t t) {
  uint4 a = ADJ(M, t).lo, b = ADJ(M, t).hi;
  return make_uint4(a.x, a.z, b.x, b.z);
}
template <class MS>
WT_HD uint4 TOV(const MS& M, uint32_t t) {
  uint4 a = ADJ(M, t).lo, b = ADJ(M, t).hi;
  return make_uint4(a.y, a.w, b.y, b.w);
}
// both halves of slot t's record: neighbours n and opposite vertices ov
template <class MS>
WT_HD void set_adj(const MS& M, uint32_t t, uint4 n, uint4 ov) {
  ADJ(M, t).lo = make_uint4(n.x, ov.x, n.y, ov.y);
  ADJ(M, t).hi = make_uint4(n.z, ov.z, n.w, ov.w);
}
template <class MS>
WT_HD void load_pt(const MS& M, uint32_t v, float* out, uint32_t* rank) {
  float4 p = M.pts[v];
  out[0] = p.x;
  out[1] = p.y;
  out[2] = p.z;
  *rank = pt_rank(p);
}

// Predicates of the lean (FAST) and full bodies.  FAST runs the FP32 filter
// alone and returns 2 when it cannot decide; the body then stops with no
// side effect and reports the element as deferred, and a second kernel
// runs the full staged predicates on the deferred elements only.
template <bool FAST, class MS>
WT_HD int o3s(const MS& M, const float* a, const float* b, const float* c, const float* d,
              uint32_t ra, uint32_t rb, uint32_t rc, uint32_t rd, PredStats* st) {
  if (FAST) return orient3d_sos_fast(a, b, c, d, st);
  return orient3d_sos(a, b, c, d, ra, rb, rc, rd, M.mode, st);
}

template <bool FAST, class MS>
WT_HD int o4s(const MS& M, const float* a, const float* b, const float* c, const float* d,
              const float* e, uint32_t ra, uint32_t rb, uint32_t rc, uint32_t rd, uint32_t re,
              PredStats* st) {
  if (FAST) return orient4d_fast(a, b, c, d, e, st);
  return orient4d(a, b, c, d, e, ra, rb, rc, rd, re, M.mode, st);
}

template <class MS>
WT_HD uint32_t* opp_word(const MS& M, uint32_t t, uint32_t f) {
  return reinterpret_cast<uint32_t*>(&ADJ(M, t)) + 2 * f;
}

// face f of slot t: neighbour pointer and opposite vertex in one store
template <class MS>
WT_HD void set_face(const MS& M, uint32_t t, uint32_t f, uint32_t n, uint32_t ov) {
  reinterpret_cast<uint2*>(&ADJ(M, t))[f] = make_uint2(n, ov);
}

// ---------------------------------------------------------------------------
// vote: each uninserted point bids for its tet; the key prefers the point
// deepest inside the circumsphere (equivalently nearest the circumcentre:
// -insphere = 6|vol|(r^2 - d^2) for a raw-negative tet), ties to the
// lowest list position.  src/shaders/vote.wgsl:89-281 (two passes there).
// ---------------------------------------------------------------------------
// returns kVoteNone when the point must not vote
template <class MS>
WT_HD uint64_t vote_key(const MS& M, const uint32_t* uvert, const uint32_t* utet, uint32_t i) {
  // The key is computed before the infinity test (every id, infinity
  // included, is a loadable point), so that the point's own id and
  // coordinates load beside its tet's vertices: two round trips.
  uint32_t t = utet[i], q = uvert[i];
  uint4 tv = TV(M, t);
  float a[3], b[3], c[3], d[3], p[3];
  uint32_t r;
  load_pt(M, q, p, &r);
  load_pt(M, tv.x, a, &r);
  load_pt(M, tv.y, b, &r);
  load_pt(M, tv.z, c, &r);
  load_pt(M, tv.w, d, &r);
  double det = insphere_eval<double>(a, b, c, d, p).det;
  double val = -det;
  if (!(val > 0.0)) val = 0.0;
  float fv = (float)val;
  uint64_t key = ((uint64_t)(0xFFFFFFFFu - f32_bits(fv)) << 32) | i;
  bool bad = tv.x == M.inf || tv.y == M.inf || tv.z == M.inf || tv.w == M.inf;
  if (bad) at_add_u32(&M.ctr[C_BADTET], 1u);
  return bad ? kVoteNone : key;
}

// Point i is inserted this round when it holds its tet's vote and no tet
// within `ring` face-steps holds a smaller key.  Inserting only into
// non-adjacent tets keeps the stars of simultaneous insertions apart, which
// is what leaves concurrent flipping unable to finish (faces that are
// neither 2-3 nor 3-2 flippable); the deferred points win a later round.
// Reads votes only, so every thread sees the same decision.
template <class MS>
WT_HD bool is_winner(const MS& M, const uint32_t* utet, uint32_t i, int ring) {
  uint32_t t = utet[i];
  uint64_t kt = TVOTE(M, t);
  if ((uint32_t)(kt & 0xFFFFFFFFull) != i) return false;
  if (ring <= 0) return true;
  const uint4 to = TN(M, t);
  // the four votes in one round trip
  bool win = true;
  for (int f = 0; f < 4; ++f) win &= TVOTE(M, opp_tet(get4(to, f))) >= kt;
  if (!win || ring <= 1) return win;
  for (int f = 0; f < 4; ++f) {
    const uint4 no = TN(M, opp_tet(get4(to, f)));
    for (int g = 0; g < 4; ++g) {
      const uint32_t n2 = opp_tet(get4(no, g));
      win &= n2 == t || TVOTE(M, n2) >= kt;
    }
  }
  return win;
}

// ---------------------------------------------------------------------------
// 1-to-4 split of tet t at point p (src/shaders/split.wgsl:104-327).
// Child j replaces vertex j by p, so it keeps t's orientation and holds
// t's face j.  Child 0 reuses slot t, children 1..3 use base..base+2.
// ---------------------------------------------------------------------------
WT_HD uint32_t child_slot(uint32_t t, uint32_t base, uint32_t j) {
  return j == 0 ? t : base + j - 1;
}

// c[0..3] receives the children's slots; returns which of them join the
// active list of iteration `it` (bit j for child j; slot t only if the list
// does not hold it yet: the pick marked what it does).
// The neighbours' split records are loaded before any store: this kernel
// writes those of fresh slots only, never a neighbour's.
template <class MS>
WT_HD uint32_t split_body(const MS& M, const uint2* wlist, uint32_t k, uint32_t round, uint32_t it,
                          uint32_t c[4]) {
  uint32_t t = wlist[k].x, p = wlist[k].y;
  uint32_t base = TSPLIT(M, t).y;
  const uint32_t tag = TQUEUE(M, t);
  uint4 tv = TV(M, t);
  uint4 to = TN(M, t);
  uint4 tov = TOV(M, t);
  c[0] = t, c[1] = base, c[2] = base + 1, c[3] = base + 2;
  uint2 ns[4];
  uint32_t np[4];
  for (int j = 0; j < 4; ++j) {
    uint32_t nt = opp_tet(get4(to, j));
    ns[j] = TSPLIT(M, nt);
    np[j] = TPOINT(M, nt);  // read for every neighbour, used where it splits
  }
  for (int j = 0; j < 4; ++j) {
    uint4 nv = tv;
    set4(nv, j, p);
    // child i (i != j) keeps t's vertex j opposite their shared face
    uint4 no, nov;
    for (int i = 0; i < 4; ++i)
      if (i != j) {
        set4(no, i, enc_opp(c[i], (uint32_t)j));
        set4(nov, i, get4(tv, j));
      }
    uint32_t e = get4(to, j);
    uint32_t nt = opp_tet(e), nf = opp_face(e);
    if (ns[j].x == round) {
      // the neighbour splits too: its child nf holds its point opposite
      set4(no, j, enc_opp(child_slot(nt, ns[j].y, nf), nf));
      set4(nov, j, np[j]);
    } else {
      set4(no, j, e);
      set4(nov, j, get4(tov, j));
      set_face(M, nt, nf, enc_opp(c[j], (uint32_t)j), p);
    }
    TV(M, c[j]) = nv;
    set_adj(M, c[j], no, nov);
    TVOTE(M, c[j]) = kVoteNone;
    if (j > 0) {  // fresh slot: initialise every per-slot field
      TQUEUE(M, c[j]) = 0u;
      FVOTE(M, c[j]) = kVoteNone;
      TSPLIT(M, c[j]) = make_uint2(0u, 0u);
      FSTAMP(M, c[j]) = 0u;
    }
  }
  return tag == (kListed | it) ? 0xEu : 0xFu;
}

// ---------------------------------------------------------------------------
// move an uninserted point of a split tet into its child
// (src/shaders/split_points.wgsl:222-335): three orient3d_sos tests.
// ---------------------------------------------------------------------------
template <bool FAST, class MS>
WT_HD bool split_points_body_t(const MS& M, const uint32_t* uvert, uint32_t* utet, uint32_t i,
                               uint32_t round, PredStats* st) {
  uint32_t t = utet[i];
  uint32_t q = uvert[i];
  uint2 sp = TSPLIT(M, t);
  if (sp.x != round) return false;
  uint32_t base = sp.y;
  uint4 c0 = TV(M, t);      // (p, v1, v2, v3)
  uint32_t v0 = TV(M, base).x;  // child 1 = (v0, p, v2, v3)
  uint32_t p = c0.x, v1 = c0.y, v2 = c0.z, v3 = c0.w;
  // the six points in one round trip
  float Pp[3], P0[3], P1[3], P2[3], P3[3], Q[3];
  uint32_t rp, r0, r1, r2, r3, rq;
  load_pt(M, p, Pp, &rp);
  load_pt(M, v0, P0, &r0);
  load_pt(M, v1, P1, &r1);
  load_pt(M, v2, P2, &r2);
  load_pt(M, v3, P3, &r3);
  load_pt(M, q, Q, &rq);
  // children 0 | 1 across plane (p, v2, v3): +1 -> v0's side -> not child 0
  int sa = o3s<FAST>(M, Pp, P3, P2, Q, rp, r3, r2, rq, st);
  if (sa == 2) return true;
  int a = sa > 0 ? 1 : 0;
  // children 2 | 3 across plane (v0, p, v1): +1 -> v2's side -> not child 2
  int sb = o3s<FAST>(M, P0, Pp, P1, Q, r0, rp, r1, rq, st);
  if (sb == 2) return true;
  int b = sb > 0 ? 3 : 2;
  // decide between a and b on their shared face: face b of (v0, v1, v2, v3)
  // with vertex a replaced by p -- (w0, v3, w1) for b = 2, (w0, w1, v2) for
  // b = 3, where w0 = a ? v0 : p and w1 = a ? p : v1 (chosen by value)
  float X[3], Y[3], Z[3];
  for (int k = 0; k < 3; ++k) {
    float w0 = a ? P0[k] : Pp[k], w1 = a ? Pp[k] : P1[k];
    X[k] = w0;
    Y[k] = b == 2 ? P3[k] : w1;
    Z[k] = b == 2 ? w1 : P2[k];
  }
  uint32_t rw0 = a ? r0 : rp, rw1 = a ? rp : r1;
  int s = o3s<FAST>(M, X, Y, Z, Q, rw0, b == 2 ? r3 : rw1, b == 2 ? rw1 : r2, rq, st);
  if (s == 2) return true;
  int child = s > 0 ? a : b;
  utet[i] = child_slot(t, base, (uint32_t)child);
  return false;
}

// ---------------------------------------------------------------------------
// flip proposals (src/shaders/check_delaunay_{fast,exact}.wgsl, flip votes
// src/shaders/mark_rejected_flips.wgsl:61-178)
// proposal: x = t, y = face | kind << 2 | edge << 3, z = neighbour, w = third tet
// kind 0: 2-3 flip, 1: 3-2 flip around edge (edge = rotation of the face triple)
// ---------------------------------------------------------------------------
WT_HD uint64_t flip_key(uint32_t it, uint32_t t) {
  return ((uint64_t)(0xFFFFFFFFu - it) << 32) | t;
}

// xyz of point k (0..3, chosen at run time) of a tet's four, by selects
WT_HD void pick_xyz(const float (*P)[3], int k, float* out) {
  for (int c = 0; c < 3; ++c) out[c] = pick4(k, P[0][c], P[1][c], P[2][c], P[3][c]);
}

// The proposal of tet t across face f (its kind, offending edge and third
// tet as flip_check_lean finds them, nt the neighbour): votes for the other tets it involves;
// its tag is the vote for its own.  A vote is an atomic minimum on a random
// line, 27 G/s on this card, a tag a store, 89 G/s.
template <class MS>
WT_HD uint4 flip_propose(const MS& M, uint32_t t, uint32_t f, uint32_t nt, uint32_t kind, uint32_t bad, uint32_t third,
                         uint32_t it) {
  uint64_t key = flip_key(it, t);
  TQUEUE(M, t) = it;
  mesh_min(M, &FVOTE(M, nt), key);
  if (kind == 1u) mesh_min(M, &FVOTE(M, third), key);
  return make_uint4(t, f | kind << 2 | bad << 3, nt, third);
}

// The insphere filters take one of the tet's vertices as origin: a real point
// (coordinates in [0, 1]; a super vertex has |x| >= 100), from which every
// difference is as short as the tet allows.  origin_of: which of the four;
// swap_origin exchanges it with P[0] (and back), which flips the determinant's
// sign.
WT_HD bool near_coord(float x) { return x >= -2.0f && x <= 2.0f; }
WT_HD int origin_of(const float (*P)[3]) {
  int k = near_coord(P[2][0]) ? 2 : 3;
  k = near_coord(P[1][0]) ? 1 : k;
  return near_coord(P[0][0]) ? 0 : k;
}
WT_HD void swap_origin(float (*P)[3], int k) {
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float v = P[0][c];
    P[0][c] = pick4(k, P[0][c], P[1][c], P[2][c], P[3][c]);
    P[1][c] = k == 1 ? v : P[1][c];
    P[2][c] = k == 2 ? v : P[2][c];
    P[3][c] = k == 3 ? v : P[3][c];
  }
}

// What the filters say about one face whose apex o lies inside the
// circumsphere: kFaceNo (no flip), kFaceFlip (*kind, *bad set; *pthird is the
// tet's vertex opposite the third tet of a 3-2 flip) or kFaceUndecided.
enum FaceCheck : int { kFaceNo = 0, kFaceFlip = 1, kFaceUndecided = 2 };
WT_HD int face_classify(const float* x, const float* y, const float* z, const float* a, const float* o,
                        const int* pos, const uint4& tov, uint32_t ov, uint32_t* kind, uint32_t* bad,
                        int* pthird, PredStats* st) {
  // differences are taken from o, or, where o is a super vertex, from a:
  // exchanging the two negates every determinant
  const bool far = !near_coord(o[0]);
  float p[3], q[3];
  for (int k = 0; k < 3; ++k) p[k] = far ? o[k] : a[k], q[k] = far ? a[k] : o[k];
  int s[3];
  orient3d_edges_f32(x, y, z, p, q, s);
  if (far)
    for (int k = 0; k < 3; ++k) s[k] = s[k] == 2 ? 2 : -s[k];
  if (s[0] == 2 || s[1] == 2 || s[2] == 2) return kFaceUndecided;
  for (int k = 0; k < 3; ++k) stat_inc(st, 0);
  // edge k: the line a-o should pass on the face side (raw sign > 0)
  int nbad = (s[0] < 0) + (s[1] < 0) + (s[2] < 0);
  int b = s[0] < 0 ? 0 : (s[1] < 0 ? 1 : 2);
  *kind = nbad == 1 ? 1u : 0u;
  *bad = nbad == 1 ? (uint32_t)b : 0u;
  *pthird = b == 0 ? pos[2] : (b == 1 ? pos[0] : pos[1]);
  if (nbad == 0) return kFaceFlip;
  // 3-2 needs the edge to have degree 3: the tet across t's face opposite the
  // third vertex must have o as its apex
  return nbad == 1 && get4(tov, *pthird) == ov ? kFaceFlip : kFaceNo;
}

// Lean check of list entry j, tet t, one thread per tet: FP32 filters, and the FP64
// filter for the faces whose insphere they leave.  The first face (in order)
// that can flip is proposed; true (with no vote cast) when a
// face before it is undecided, and the entry needs the full predicates.
template <class MS>
WT_HD bool flip_check_lean(const MS& M, uint32_t t, uint4* prop, uint32_t j, uint32_t it, PredStats* st) {
  // Two memory round trips: the slot's record (vertices and opposite
  // vertices), then all eight points (the point array includes the infinity
  // vertex, so every id is loadable).
  uint4 tv = TV(M, t);
  uint4 to = TN(M, t);
  uint4 tov = TOV(M, t);
  prop[j].x = kInvalid;
  if (tv.x == kInvalid) return false;  // freed since it was queued
  if (tv.x == M.inf || tv.y == M.inf || tv.z == M.inf || tv.w == M.inf) return false;
  float P[4][3], Q[4][3];
  uint32_t r;
  for (int k = 0; k < 4; ++k) load_pt(M, get4(tv, k), P[k], &r);
  for (int k = 0; k < 4; ++k) load_pt(M, get4(tov, k), Q[k], &r);
  // bit f: the apex across face f lies inside, or the filters cannot tell
  uint32_t in = 0u, und = 0u;
  const int org = origin_of(P);
  if (org) swap_origin(P, org);
  const int inside = org ? 1 : -1;
  {
    const InsphereTet<float> q = insphere_tet<float>(P[0], P[1], P[2], P[3]);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      if (get4(tov, f) == M.inf) continue;
      int s = insphere_query_f32(q, P[0], Q[f]);
      if (s == 2) und |= 1u << f;
      else stat_inc(st, 4);
      if (s == inside) in |= 1u << f;
    }
  }
  if (und) {
    const InsphereTet<double> q = insphere_tet<double>(P[0], P[1], P[2], P[3]);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      if (!((und >> f) & 1u)) continue;
      int s = insphere_query_f64(q, P[0], Q[f]);
      if (s == 2) continue;
      stat_inc(st, 5);
      und &= ~(1u << f);
      if (s == inside) in |= 1u << f;
    }
  }
  if (org) swap_origin(P, org);
  // the faces left, in order: most lanes have at most one or two
  uint32_t todo = in | und;
  while (todo) {
    const int f = ctz32(todo);
    if ((und >> f) & 1u) return true;
    todo &= todo - 1u;
    float A[3], O[3], X[3], Y[3], Z[3];
    const int pos[3] = {face_vi(f, 0), face_vi(f, 1), face_vi(f, 2)};
    pick_xyz(P, f, A);
    pick_xyz(Q, f, O);
    pick_xyz(P, pos[0], X);
    pick_xyz(P, pos[1], Y);
    pick_xyz(P, pos[2], Z);
    uint32_t kind, bad;
    int pthird;
    const int v = face_classify(X, Y, Z, A, O, pos, tov, get4(tov, f), &kind, &bad, &pthird, st);
    if (v == kFaceUndecided) return true;
    if (v == kFaceNo) continue;
    const uint32_t third = kind ? opp_tet(get4(to, pthird)) : kInvalid;
    prop[j] = flip_propose(M, t, (uint32_t)f, opp_tet(get4(to, f)), kind, bad, third, it);
    return false;
  }
  return false;
}

// point k (0..3, chosen at run time) of a tet's four: selects instead of an
// indexed local array, which would live in scratch memory
WT_HD void pick_pt(const float (*P)[3], const uint32_t* R, int k, float* out, uint32_t* r) {
  pick_xyz(P, k, out);
  *r = pick4(k, R[0], R[1], R[2], R[3]);
}

// A face whose apex o across it is tested: its three vertices v, the tet's
// vertex a opposite it, and o, with their ranks.
struct FaceEdges {
  float v[3][3], a[3], o[3];
  uint32_t rv[3], ra, ro;
};

// The apex across face f of a tet lies inside its circumsphere (full
// predicates).  P, R: the tet's points and ranks; Q, RQ: the vertices across
// its faces.
template <class MS>
WT_HD bool flip_face_inside(const MS& M, const uint4& tov, const float (*P)[3], const uint32_t* R,
                            const float (*Q)[3], const uint32_t* RQ, int f, PredStats* st, FaceEdges* E) {
  if (get4(tov, f) == M.inf) return false;
  pick_pt(Q, RQ, f, E->o, &E->ro);
  pick_pt(P, R, f, E->a, &E->ra);
  for (int k = 0; k < 3; ++k) pick_pt(P, R, face_vi(f, k), E->v[k], &E->rv[k]);
  return o4s<false>(M, P[0], P[1], P[2], P[3], E->o, R[0], R[1], R[2], R[3], E->ro, st) <= 0;
}

// The flip of face f whose apex lies inside, from bits k: the segment a-o
// passes beyond edge (v[k], v[k + 1]).  False when no flip fits.  kind (1:
// 3-2), the offending edge and the third tet (3-2)
template <class MS>
WT_HD bool flip_face_kind(const MS& M, uint32_t t, const uint4& tov, int f, uint32_t beyond, uint32_t* kind,
                          uint32_t* bad, uint32_t* third) {
  *kind = 0u;
  *bad = 0u;
  *third = kInvalid;
  if (beyond == 0u) return true;
  if (beyond & (beyond - 1u)) return false;
  // 3-2 needs the edge to have degree 3 (see face_classify)
  const int b = (int)ctz32(beyond);
  const int pthird = face_vi(f, b == 0 ? 2 : b - 1);
  if (get4(tov, pthird) != get4(tov, f)) return false;
  *kind = 1u;
  *bad = (uint32_t)b;
  *third = opp_tet(*opp_word(M, t, (uint32_t)pthird));
  return true;
}

// ---------------------------------------------------------------------------
// execute a winning flip (src/shaders/flip.wgsl:531-845).  New tets reuse
// the old slots; a 2-3 flip takes one fresh slot, a 3-2 flip frees one.
// External faces keep the old neighbour pointer; flip_update_body fixes
// them once every flip of the iteration is written.
// s: the fresh slot of a 2-3 flip.  The caller queues the new tets (the
// reused slots were claimed by flip_decide_load).
// outk, the flip's record for the adjacency update (64 bytes: the update
// reads it in order instead of the new tets' own records): slots of the new
// tets (the third unused for 3-2) and the kind; the vertices o, a and (3-2)
// z; the six external neighbour pointers in flip_update_body's order
// ---------------------------------------------------------------------------
// The records a flip reads: vertices, neighbours and opposite vertices of
// its two (2-3) or three (3-2) tets.  Loading them is split from the flip so
// that a caller can issue the loads early and overlap them with other work.
struct FlipTets {
  uint4 tv, to, tov, nv, no, nov, mv, mo, mov;
};

template <class MS>
WT_HD void flip_load(const MS& M, const uint4& pr, FlipTets& F) {
  // a 2-3 flip has no third tet: its slot is replaced by t's, so every load
  // is of a valid slot and none depends on a branch
  uint32_t m = ((pr.y >> 2) & 1u) ? pr.w : pr.x;
  F.tv = TV(M, pr.x), F.to = TN(M, pr.x), F.tov = TOV(M, pr.x);
  F.nv = TV(M, pr.z), F.no = TN(M, pr.z), F.nov = TOV(M, pr.z);
  F.mv = TV(M, m), F.mo = TN(M, m), F.mov = TOV(M, m);
}

template <class MS>
WT_HD void flip_exec_loaded(const MS& M, const uint4 pr, const FlipTets& F, uint32_t it,
                            uint32_t s, uint4* outk) {
  uint32_t t = pr.x, f = pr.y & 3u, kind = (pr.y >> 2) & 1u, edge = (pr.y >> 3) & 3u;
  uint32_t n = pr.z;
  const uint4 tv = F.tv, to = F.to, tov = F.tov;
  const uint4 nv = F.nv, no = F.no, nov = F.nov;
  uint32_t nf = opp_face(get4(to, (int)f));
  uint32_t a = get4(tv, (int)f), o = get4(nv, (int)nf);
  int pos[3] = {face_vi((int)f, 0), face_vi((int)f, 1), face_vi((int)f, 2)};
  if (kind == 0) {
    uint32_t x = get4(tv, pos[0]), y = get4(tv, pos[1]), z = get4(tv, pos[2]);
    int qx = find4(nv, x), qy = find4(nv, y), qz = find4(nv, z);
    uint32_t Txy = t, Tyz = n, Tzx = s;
    TV(M, Txy) = make_uint4(x, y, o, a);
    TV(M, Tyz) = make_uint4(y, z, o, a);
    TV(M, Tzx) = make_uint4(z, x, o, a);
    // external faces keep the old tets' opposite vertices until
    // flip_update_body sees a neighbour that flipped too
    set_adj(M, Txy, make_uint4(enc_opp(Tyz, 1), enc_opp(Tzx, 0), get4(to, pos[2]), get4(no, qz)),
            make_uint4(z, z, get4(tov, pos[2]), get4(nov, qz)));
    set_adj(M, Tyz, make_uint4(enc_opp(Tzx, 1), enc_opp(Txy, 0), get4(to, pos[0]), get4(no, qx)),
            make_uint4(x, x, get4(tov, pos[0]), get4(nov, qx)));
    set_adj(M, Tzx, make_uint4(enc_opp(Txy, 1), enc_opp(Tyz, 0), get4(to, pos[1]), get4(no, qy)),
            make_uint4(y, y, get4(tov, pos[1]), get4(nov, qy)));
    uint4 mt = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
    set4(mt, pos[2], enc_opp(Txy, 2));
    set4(mt, pos[0], enc_opp(Tyz, 2));
    set4(mt, pos[1], enc_opp(Tzx, 2));
    uint4 mn = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
    set4(mn, qz, enc_opp(Txy, 3));
    set4(mn, qx, enc_opp(Tyz, 3));
    set4(mn, qy, enc_opp(Tzx, 3));
    set_msg(&TMSG(M, t), mt, o);
    set_msg(&TMSG(M, n), mn, a);
    FSTAMP(M, t) = it;
    FSTAMP(M, n) = it;
    TVOTE(M, s) = kVoteNone;
    FVOTE(M, s) = kVoteNone;
    TSPLIT(M, s) = make_uint2(0u, 0u);
    FSTAMP(M, s) = 0u;
    TQUEUE(M, s) = 0u;
    outk[0] = make_uint4(Txy, Tyz, Tzx, 0u);
    outk[1] = make_uint4(o, a, 0u, get4(to, pos[2]));
    outk[2] = make_uint4(get4(no, qz), get4(to, pos[0]), get4(no, qx), get4(to, pos[1]));
    outk[3].x = get4(no, qy);
  } else {
    // rotate the face triple so the offending edge is (x, y), third z
    uint32_t x = get4(tv, pos[edge]), y = get4(tv, pos[(edge + 1) % 3]),
             z = get4(tv, pos[(edge + 2) % 3]);
    int px = pos[edge], py = pos[(edge + 1) % 3];
    uint32_t m = pr.w;
    const uint4 mv = F.mv, mo = F.mo, mov = F.mov;
    int qx = find4(nv, x), qy = find4(nv, y);
    int mx = find4(mv, x), my = find4(mv, y);
    uint32_t A = t, B = n;
    TV(M, A) = make_uint4(a, z, o, x);
    TV(M, B) = make_uint4(z, a, o, y);
    set_adj(M, A, make_uint4(get4(no, qy), get4(mo, my), get4(to, py), enc_opp(B, 3)),
            make_uint4(get4(nov, qy), get4(mov, my), get4(tov, py), y));
    set_adj(M, B, make_uint4(get4(mo, mx), get4(no, qx), get4(to, px), enc_opp(A, 3)),
            make_uint4(get4(mov, mx), get4(nov, qx), get4(tov, px), x));
    uint4 mt = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
    set4(mt, py, enc_opp(A, 2));
    set4(mt, px, enc_opp(B, 2));
    uint4 mn = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
    set4(mn, qy, enc_opp(A, 0));
    set4(mn, qx, enc_opp(B, 1));
    uint4 mm = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid);
    set4(mm, my, enc_opp(A, 1));
    set4(mm, mx, enc_opp(B, 0));
    set_msg(&TMSG(M, t), mt, o);
    set_msg(&TMSG(M, n), mn, a);
    set_msg(&TMSG(M, m), mm, z);
    FSTAMP(M, t) = it;
    FSTAMP(M, n) = it;
    FSTAMP(M, m) = it;
    TQUEUE(M, m) = kFreed;
    TV(M, m).x = kInvalid;
    TFWD(M, m) = A;
    outk[0] = make_uint4(A, B, kInvalid, 1u);
    outk[1] = make_uint4(o, a, z, get4(no, qy));
    outk[2] = make_uint4(get4(mo, my), get4(to, py), get4(mo, mx), get4(no, qx));
    outk[3].x = get4(to, px);
  }
}

// A proposal wins when it holds the smallest vote of every tet it involves; the
// winner executes at once (its tets belong to no other winner), losers go
// back to the active list (src/shaders/mark_rejected_flips.wgsl:61-178 and
// src/shaders/flip.wgsl:531-845, one pass here).
// Decide proposal pr.  qid[0..*nq) are the tets to append to the next active
// list: the proposal's own, and for a winner its neighbour's slot unless that
// proposed too and so appends itself (it lost: its vote is the winner's).  For
// a 2-3 winner (*nslot = 1) the caller appends the fresh slot after qid.  A
// winner also loads its flip's tets (into F).
template <class MS>
WT_HD bool flip_decide_load(const MS& M, const uint4& pr, uint32_t it, uint32_t qid[2],
                            uint32_t* nq, uint32_t* nslot, FlipTets& F) {
  *nq = 0;
  *nslot = 0;
  qid[0] = qid[1] = kInvalid;
  if (pr.x == kInvalid) return false;
  uint64_t key = flip_key(it, pr.x);
  // a 2-3 flip reads its neighbour's words again for its third tet's: every
  // load is issued before the first is used
  const uint32_t m = ((pr.y >> 2) & 1u) ? pr.w : pr.z;
  const uint64_t vx = FVOTE(M, pr.x), vz = FVOTE(M, pr.z), vm = FVOTE(M, m);
  const uint32_t tag = TQUEUE(M, pr.z), tag_m = TQUEUE(M, m);
  // votes of older iterations are larger than every one of this
  const bool lost = (vx <= key) | (vz != key) | (vm != key) | ((tag == it) & (pr.z < pr.x)) |
                    ((tag_m == it) & (m < pr.x));
  const bool win = !lost;
  qid[0] = pr.x;
  qid[1] = pr.z;
  *nq = 1;
  if (win) {
    flip_load(M, pr, F);
    if ((tag & ~kWaits) != it) *nq = 2;
    if (((pr.y >> 2) & 1u) == 0u) *nslot = 1;
  }
  return win;
}

// The proposal of a tet that no kernel of this iteration decides: nobody
// votes for it, so it loses and stays in the active list.
template <class MS>
WT_HD uint4 requeue_proposal(const MS& M, uint32_t t, uint32_t it) {
  TQUEUE(M, t) = kWaits | it;
  return make_uint4(t, 0u, t, kInvalid);
}

// entry t of the list that iteration it begins with stays there over the
// round's splits
template <class MS>
WT_HD void mark_listed(const MS& M, uint32_t t, uint32_t it) {
  if (TQUEUE(M, t) != kFreed) TQUEUE(M, t) = kListed | it;
}

// src/shaders/update_opp.wgsl:73-220.  The flip's six external faces
// (tet T, face e, T's vertex vT opposite e): a face whose neighbour q
// flipped too takes the tet and vertex that q's flip left in its message;
// otherwise q's face points back at T.  Every load comes before the first
// store (the flip record, the stamps in the records that most faces then
// write, and the messages of the few neighbours that flipped): no
// thread of this kernel
// stores a word that one of these loads reads (stamps and messages are
// read-only here).
template <class MS>
WT_HD void flip_update_body(const MS& M, const uint4* out, uint32_t k, uint32_t it) {
  uint4 r = out[4 * (size_t)k];
  uint4 w = out[4 * (size_t)k + 1];  // o, a, z
  uint4 p = out[4 * (size_t)k + 2];
  // 2-3: new tets (x, y, o, a), external faces 2 (apex o) and 3 (apex a);
  // 3-2: A = (a, z, o, x), B = (z, a, o, y), external faces 0, 1, 2.
  // Selected without a branch, so the record is read in one round trip.
  bool k32 = r.w != 0u;
  uint32_t T[6] = {r.x, r.x, k32 ? r.x : r.y, r.y, k32 ? r.y : r.z, k32 ? r.y : r.z};
  uint32_t E[6] = {k32 ? 0u : 2u, k32 ? 1u : 3u, 2u, k32 ? 0u : 3u, k32 ? 1u : 2u, k32 ? 2u : 3u};
  uint32_t V[6] = {k32 ? w.y : w.x, k32 ? w.z : w.y, w.x, k32 ? w.z : w.y, k32 ? w.y : w.x,
                   k32 ? w.x : w.y};
  uint32_t ptr[6] = {w.w, p.x, p.y, p.z, p.w, out[4 * (size_t)k + 3].x}, fq[6];
  uint2 msg[6];
  for (int i = 0; i < 6; ++i) fq[i] = FSTAMP(M, opp_tet(ptr[i]));
  // Every lane loads, from one common line where its neighbour did not flip:
  // behind branches each of the six waited for itself.
  for (int i = 0; i < 6; ++i) {
    const uint32_t at = fq[i] == it ? ptr[i] : 0u;
    msg[i] = reinterpret_cast<const uint2*>(&TMSG(M, opp_tet(at)))[opp_face(at)];
  }
  // one 8-byte store per face, its slot and value chosen without a branch
  for (int i = 0; i < 6; ++i) {
    bool fl = fq[i] == it;
    uint32_t dt = fl ? T[i] : opp_tet(ptr[i]), df = fl ? E[i] : opp_face(ptr[i]);
    set_face(M, dt, df, fl ? msg[i].x : enc_opp(T[i], E[i]), fl ? msg[i].y : V[i]);
  }
}

// ---------------------------------------------------------------------------
// relocate points whose tet a flip replaced: a stochastic visibility walk
// (Devillers, Pion, Teillaud 2002) from the old slot.  Replaces the
// reference's flip-trace replay (src/shaders/relocate_points_fast.wgsl).
// ---------------------------------------------------------------------------
constexpr uint32_t kWalkLimit = 1u << 16;

// *state: 0 arrived, 1 step limit, 2 deferred (FAST filter undecided)
template <bool FAST, class MS>
WT_HD uint32_t walk_to_t(const MS& M, uint32_t t, uint32_t q, uint32_t seed, PredStats* st,
                         int* state) {
  float Q[3];
  uint32_t rq;
  load_pt(M, q, Q, &rq);
  for (uint32_t step = 0; step < kWalkLimit; ++step) {
    uint4 tv = TV(M, t);
    uint4 to = TN(M, t);
    uint32_t r0 = hash32(seed + step * 0x9E3779B9u) & 3u;
    // the tet's four points in one round trip, all four face tests, then
    // the step takes the first face in its random order (r0, r0 + 1, ...)
    // that q lies beyond, or defers if an undecided face comes first
    float P[4][3];
    uint32_t R[4];
    for (int k = 0; k < 4; ++k) load_pt(M, get4(tv, k), P[k], &R[k]);
    uint32_t beyond = 0u, undecided = 0u;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      int a = face_vi(f, 0), b = face_vi(f, 1), c = face_vi(f, 2);
      int o = o3s<FAST>(M, P[a], P[b], P[c], Q, R[a], R[b], R[c], rq, st);
      if (o == 2) undecided |= 1u << f;
      else if (o < 0) beyond |= 1u << f;
    }
    uint32_t m = beyond | undecided;
    if (!m) {
      *state = 0;
      return t;
    }
    uint32_t rot = ((m >> r0) | (m << (4u - r0))) & 0xFu;
    uint32_t f = ((uint32_t)ctz32(rot) + r0) & 3u;
    if (undecided & (1u << f)) {
      *state = 2;
      return t;
    }
    t = opp_tet(get4(to, (int)f));
  }
  *state = 1;
  return t;
}

// the live slot that a point of slot t walks from; false when no flip of
// this round replaced t.  it0: flip iterations before this round
template <class MS>
WT_HD bool walk_start(const MS& M, uint32_t it0, uint32_t* t) {
  if (FSTAMP(M, *t) <= it0) return false;
  for (int guard = 0; guard < 64 && TV(M, *t).x == kInvalid; ++guard) *t = TFWD(M, *t);
  return true;
}
WT_HD uint32_t walk_seed(uint32_t i) { return i * 0x85EBCA6Bu; }

template <bool FAST, class MS>
WT_HD bool relocate_body_t(const MS& M, const uint32_t* uvert, uint32_t* utet, uint32_t i,
                           uint32_t it0, PredStats* st) {
  uint32_t t = utet[i];
  if (!walk_start(M, it0, &t)) return false;
  int state = 0;
  t = walk_to_t<FAST>(M, t, uvert[i], walk_seed(i), st, &state);
  if (state == 2) {  // the full walk goes on from here
    utet[i] = t;
    return true;
  }
  if (state == 1) at_add_u32(&M.ctr[C_WALK_FAIL], 1u);
  utet[i] = t;
  return false;
}

// ---------------------------------------------------------------------------
// audit: every finite face, counted once from its lower slot
// (src/lib.rs:25-78 checks real-only pairs; this covers all finite faces)
// rec: (t << 2 | f) of violations, capacity cap.  FAST: FP32 filter only;
// returns true (nothing recorded) when a face is undecided, for the full
// pass to redo the tet.
// ---------------------------------------------------------------------------
template <bool FAST>
WT_HD bool audit_body_t(const Mesh& M, uint32_t t, uint32_t* rec, uint32_t cap, PredStats* st) {
  if (!slot_alive(M, t)) return false;
  uint4 tv = TV(M, t);
  if (tv.x == M.inf || tv.y == M.inf || tv.z == M.inf || tv.w == M.inf) return false;
  uint4 to = TN(M, t);
  uint4 tov = TOV(M, t);
  float P[4][3];
  uint32_t R[4];
  for (int k = 0; k < 4; ++k) load_pt(M, get4(tv, k), P[k], &R[k]);
  int bad[4] = {0, 0, 0, 0};
  for (int f = 0; f < 4; ++f) {
    uint32_t nt = opp_tet(get4(to, f));
    if (nt < t) continue;
    uint32_t o = get4(tov, f);
    if (o == M.inf) continue;
    float O[3];
    uint32_t ro;
    load_pt(M, o, O, &ro);
    int s = o4s<FAST>(M, P[0], P[1], P[2], P[3], O, R[0], R[1], R[2], R[3], ro, st);
    if (s == 2) return true;
    bad[f] = s < 0;
  }
  for (int f = 0; f < 4; ++f)
    if (bad[f]) {
      at_add_u32(&M.ctr[C_VIOL], 1u);
      uint32_t k = at_add_u32(&M.ctr[C_FAILREC], 1u);
      if (k < cap) rec[k] = (t << 2) | (uint32_t)f;
    }
  return false;
}

}  // namespace wtet
