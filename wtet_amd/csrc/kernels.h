// Launchers for the triangulation kernels (defined in kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "prep.h"

namespace wtet {

constexpr int kBlock = 256;  // 4 wavefronts of 64

inline uint32_t nblocks(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

// per-cloud bounding box only (the first kernels of launch_prepare): mm
// gets 6 order-preserving words per cloud (min xyz, max xyz)
void launch_minmax(const float* xyz, uint32_t n, const Clouds& K, uint32_t* mm, hipStream_t s);
// point preparation for one or many clouds (layout: prep.h):
// per-cloud normalization (src/lib.rs:313-337) and (cloud, Morton) keys
void launch_prepare(const float* xyz, uint32_t n, const Clouds& K, uint32_t* mm, float* xyzn,
                    uint64_t* keys, uint32_t* ids, hipStream_t s);
// sorted points -> vertices, plus every cloud's super vertices and infinity
void launch_gather_points(const float* xyzn, const uint32_t* ids, const uint64_t* keys,
                          uint32_t n, const Clouds& K, float4* pts, hipStream_t s);
// five start tets per cloud in slots 5c..5c+4
void launch_start_tets(const Mesh& M, const Clouds& K, hipStream_t s);
// stable radix sort of (key, id) pairs (sort.h): keys/ids in, keys_tmp/ids_tmp out
hipError_t sort_pairs(uint64_t* keys, uint32_t* ids, uint64_t* keys_tmp, uint32_t* ids_tmp,
                      uint32_t n, int end_bit, void* temp, size_t temp_bytes, hipStream_t s);
size_t sort_temp_bytes(uint32_t n, int end_bit);
size_t sort_temp_bytes_u32(uint32_t n, int end_bit);
// bits of an output sort key: clouds 0..C-1 and C for free slots
inline int cloud_key_bits(uint32_t C) {
  int bits = 1;
  while ((1ull << bits) <= C) ++bits;
  return bits;
}
// uninserted list = every point except redundant exact duplicates;
// ctr[C_NPTS] = its length
void launch_init_uninserted(const float4* pts, const uint64_t* keys, uint32_t n, const Clouds& K,
                            uint32_t* blk, uint32_t* uvert, uint32_t* utet, uint32_t* ctr,
                            hipStream_t s);

// Hilbert mode: reorder the uninserted list into the reference's
// stratified order, per cloud (scratch: key, key_tmp, val_tmp of U entries)
hipError_t launch_stratify(uint32_t* uvert, uint32_t* utet, uint32_t U, const Clouds& K,
                           uint64_t* key, uint64_t* key_tmp, uint32_t* val_tmp, void* temp,
                           size_t temp_bytes, hipStream_t s);

// rounds.  The round kernels read their counts and the round number from
// ctr (C_WIN, C_SURV, C_ROUND); the count arguments only bound the launch
// grids, a power of two of workgroups (round_grid), so a captured round
// replays for any count up to its bound.
uint32_t round_grid(uint64_t bound);
void launch_vote(const Mesh& M, const uint32_t* uvert, const uint32_t* utet, uint32_t U,
                 hipStream_t s);
// the two active lists, flip proposals and the executed flips of one
// iteration
struct FlipLists {
  uint32_t* act[2];
  uint4* prop;
  uint4* out;    // four uint4 per executed flip (flip_exec_loaded)
  uint32_t* slow;  // entries the lean check deferred
};
// begins the next round (C_ROUND) and counts its winners (C_WIN); they leave
// C_SURV, and take their slots from C_TETS, at the split.
// ring: insert only where no tet within `ring` face-steps has a smaller vote
// (blk: round_grid(U) entries)
void launch_pick(const Mesh& M, const uint32_t* uvert, const uint32_t* utet, uint32_t U,
                 uint2* wlist, uint32_t* uvert2, uint32_t* utet2, uint32_t* blk, int ring,
                 const FlipLists& L, hipStream_t s);
// appends the children to the active list after its ctr[C_LIST] entries
void launch_split(const Mesh& M, const uint2* wlist, uint32_t W, const FlipLists& L, hipStream_t s);
// filtered mode: an FP32-only kernel, then the full predicates on the points
// it deferred (slow, U entries of scratch); exact mode: one full kernel.
// begin > 0: also launch_batch_begin(begin)
void launch_split_points(const Mesh& M, const uint32_t* uvert, uint32_t* utet, uint32_t U,
                         uint64_t* st, uint32_t* slow, int begin, hipStream_t s);
// a batch of k <= kMaxBatch flip iterations = begin; check, (deferred check,)
// decide+execute, update for i = 0..k-1; end.  Counts, tags, round and
// parity are read from ctr (device-driven, graph-capturable); grid =
// persistent blocks of the list kernels
void launch_batch_begin(uint32_t* ctr, int k, hipStream_t s);
// filtered mode: the FP32-only check, deferring undecided tets to the full
// check that follows or, with requeue, to a later iteration (none follows);
// exact mode, or with full: the full check, nothing deferred
void launch_flip_check(const Mesh& M, const FlipLists& L, int i, bool requeue, bool full, uint32_t grid, uint64_t* st,
                       hipStream_t s);
void launch_flip_check_deferred(const Mesh& M, const FlipLists& L, int i, uint32_t grid, uint64_t* st,
                                hipStream_t s);
void launch_flip_decide_exec(const Mesh& M, const FlipLists& L, int i, uint32_t grid, hipStream_t s);
void launch_flip_update(const Mesh& M, const FlipLists& L, int i, uint32_t grid, hipStream_t s);
// sums (IterSum) += what the batch did; the list it left in C_LIST
void launch_batch_end(uint32_t* ctr, uint64_t* sums, int k, hipStream_t s);
// a batch of up to k iterations of a list of at most `limit` entries in one
// workgroup, begin and end included
void launch_flip_small(const Mesh& M, const FlipLists& L, uint64_t* st, uint64_t* sums, int k,
                       uint32_t limit, hipStream_t s);
// Insertion rounds of few points in one workgroup, from the vote (voted 0) or
// from the split of the winners a pick left (voted 1), until the rounds are
// over (ctr[C_RUN_DONE]) or, after a pick, the next one does not fit.
struct SmallRun {
  uint32_t* uvert[2];
  uint32_t* utet[2];
  uint2* wlist;
  uint32_t* slow;    // one entry per point
  uint32_t cur;      // the list that holds the points
  int voted;
  int k;             // flip iterations in a round
  int ring;          // insertion ring after the warmup rounds
  uint32_t warmup, max_round;
  uint32_t list;     // longest flip list a round may begin with
  uint32_t list_full;  // the same after a round that left more entries an
                       // iteration to the full predicates
  uint32_t limit;    // and an iteration of it
};
void launch_rounds_small(const Mesh& M, const FlipLists& L, const SmallRun& J, uint64_t* st, uint64_t* sums,
                         hipStream_t s);
// end > 0: also launch_batch_end(end).  ctr[C_SLOW_R] is 0 before (the split
// clears it)
void launch_relocate(const Mesh& M, const uint32_t* uvert, uint32_t* utet, uint32_t U,
                     uint64_t* st, uint32_t* slow, uint64_t* sums, int end, hipStream_t s);
// filtered mode: an FP32-only pass, then the full predicates on the tets it
// could not decide (slow: T entries of scratch); exact mode: one full pass
void launch_audit(const Mesh& M, uint32_t T, uint32_t* rec, uint32_t cap, uint64_t* st,
                  uint32_t* slow, hipStream_t s);

// output: live tets grouped by cloud (rows of cloud c from cstart[c],
// cstart[C] = ctr[C_ALIVE] = rows), cloud-local vertex ids and
// (row << 5) | face adjacency; slot2pos maps slots to rows
struct OutputBufs {
  uint32_t* blk;
  uint32_t* olist;     // T
  uint32_t* okey;      // T (many clouds)
  uint32_t* olist2;    // T (many clouds)
  uint32_t* okey2;     // T (many clouds)
  uint32_t* slot2pos;  // T
  uint32_t* cstart;    // C + 1
  void* temp;          // sort temporary (many clouds)
  size_t temp_bytes;
  uint32_t* out_tets;  // rows * 4 (null: only slot2pos / cstart)
  uint32_t* out_adj;
  uint32_t* vrank;     // scratch, one word per vertex (K.V + 1): each vertex's SoS rank
};
hipError_t launch_output(const Mesh& M, uint32_t T, const Clouds& K, const OutputBufs& B, hipStream_t s);

// violation records (slot << 2 | face) -> output indices
void launch_map_records(uint32_t* rec, uint32_t n, const uint32_t* slot2idx, hipStream_t s);
// rows within `rings` face-steps of the recorded faces' rows and of the last
// `tail` rows: list[0, *cnt) (mark: M words of scratch, bounds: rings + 2).
// more=true keeps the rows already listed and appends those around the new
// seeds that are not (list[old *cnt, new *cnt)).
void launch_neighbourhood(const uint32_t* rec, uint32_t nrec, uint32_t M, uint32_t tail, int rings,
                          const uint32_t* adj, uint32_t* mark, uint32_t* list, uint32_t* cnt,
                          uint32_t* bounds, bool more, hipStream_t s);
// packed (row, tet[4], adj[4]) records of the listed rows
void launch_nbr_gather(const uint32_t* list, uint32_t n, const uint32_t* tets, const uint32_t* adj,
                       uint32_t* out, hipStream_t s);
// write (slot, tet[4], adj[4]) records into the output arrays
void launch_apply_patch(const uint32_t* patch, uint32_t n, uint32_t* tets, uint32_t* adj,
                        hipStream_t s);

// counters
void launch_set_ctr(uint32_t* ctr, int idx, uint32_t v, int idx2, uint32_t v2, hipStream_t s);

// fills
void launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s);
void launch_fill_u64(uint64_t* p, uint64_t v, uint64_t n, hipStream_t s);
// plain streaming copy (16 B per lane), also the HBM-counter calibration kernel
void launch_copy16(uint4* dst, const uint4* src, uint64_t n, hipStream_t s);

// predicate batches (for checking the device predicates)
void launch_pred_batch(int kind, const float* pts, const uint32_t* idx, uint32_t n, int mode,
                       int32_t* out, uint64_t* st, hipStream_t s);

}  // namespace wtet
