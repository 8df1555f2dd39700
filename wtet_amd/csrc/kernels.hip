// HIP kernels of the triangulation loop (gfx950, wave64).
//
// Element-wise kernels wrap the bodies of ops.h.  List compaction uses
// wave ballots: each wavefront ranks its lanes with popcount(ballot & lt),
// wave totals are combined in LDS, block totals are scanned by one block,
// and a scatter pass writes every element once (stable order).
#include <algorithm>
#include <cstring>


#include "kernels.h"
#include "prep.h"
#include "sort.h"
#include "wave.h"

namespace wtet {

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n);

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------
// Thread of a grid of kBlock-thread blocks (blockDim.x is a load from the
// dispatch's arguments, a memory round trip before anything else).
__device__ __forceinline__ uint32_t gid() { return blockIdx.x * kBlock + threadIdx.x; }

// exclusive rank of `flag` within the block; *total = block count.
// Every thread of the block must call it.
__device__ __forceinline__ uint32_t block_rank(bool flag, uint32_t* total) {
  __shared__ uint32_t wsum[kBlock / 64];
  uint64_t m = __ballot(flag);
  int lane = __lane_id();
  int wave = threadIdx.x >> 6;
  uint32_t r = __popcll(m & ((1ull << lane) - 1ull));
  if (lane == 0) wsum[wave] = __popcll(m);
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    off += w < wave ? wsum[w] : 0u;
    tot += wsum[w];
  }
  *total = tot;
  return off + r;
}

// in-place exclusive scan of blk[0..nb) by one 1024-thread block
// mode 0: insertion round -> ctr[C_WIN] = total
// mode 1: output          -> ctr[C_ALIVE] = total
// mode 2: point list      -> ctr[C_NPTS] = total
// A thread takes 32 counts of each 32,768 in eight loads that wait for each other
// once.  A round of 2,048 clouds (up to 20,000 counts) 67 us, read and written
// one by one, now 12.
__global__ void __launch_bounds__(1024) k_scan_blocks(uint32_t* blk, uint32_t nb, uint32_t* ctr,
                                                     int mode) {
  constexpr uint32_t kQuads = 8, kStep = 1024u * 4u * kQuads;
  __shared__ uint32_t part[16];
  const uint32_t tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
  uint32_t total = 0;
  for (uint32_t b = 0; b < nb; b += kStep) {
    const uint32_t first = b + tid * 4u * kQuads;
    uint32_t v[4 * kQuads], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < kQuads; ++q) {
      const uint32_t i = first + 4u * q;
      uint4 x = make_uint4(0u, 0u, 0u, 0u);
      if (i + 4u <= nb) x = *reinterpret_cast<const uint4*>(blk + i);
      else if (i < nb) x = make_uint4(blk[i], i + 1u < nb ? blk[i + 1u] : 0u, i + 2u < nb ? blk[i + 2u] : 0u, 0u);
      v[4 * q] = x.x, v[4 * q + 1] = x.y, v[4 * q + 2] = x.z, v[4 * q + 3] = x.w;
    }
#pragma unroll
    for (uint32_t k = 0; k < 4u * kQuads; ++k) sum += v[k];
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off);
      if (lane >= (uint32_t)off) incl += y;
    }
    if (lane == 63u) part[wave] = incl;
    __syncthreads();
    uint32_t run = total + incl - sum;
#pragma unroll
    for (uint32_t w = 0; w < 16u; ++w) {
      run += w < wave ? part[w] : 0u;
      total += part[w];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kQuads; ++q) {
      const uint32_t i = first + 4u * q;
      uint4 x;
      x.x = run;
      x.y = x.x + v[4 * q];
      x.z = x.y + v[4 * q + 1];
      x.w = x.z + v[4 * q + 2];
      run = x.w + v[4 * q + 3];
      if (i + 4u <= nb) *reinterpret_cast<uint4*>(blk + i) = x;
      else {
        if (i < nb) blk[i] = x.x;
        if (i + 1u < nb) blk[i + 1u] = x.y;
        if (i + 2u < nb) blk[i + 2u] = x.z;
      }
    }
  }
  if (tid == 1023u) {
    if (mode == 0) {
      ctr[C_WIN] = total;
    } else if (mode == 1) {
      ctr[C_ALIVE] = total;
    } else {
      ctr[C_NPTS] = total;
    }
  }
}

// ---------------------------------------------------------------------------
// point preparation (layout of one or many clouds: prep.h)
// ---------------------------------------------------------------------------
__global__ void k_minmax_init(uint32_t* mm, uint32_t C) {
  uint32_t i = gid();
  if (i < 6u * C) mm[i] = (i % 6u) < 3u ? 0xFFFFFFFFu : 0u;
}

// Per-cloud min/max of each axis.  Lanes in the cloud of the wave's first
// lane combine with a wave reduction (one atomic per wave); lanes of other
// clouds (at most a few per cloud boundary) add their own atomics.
__global__ void k_minmax(const float* xyz, uint32_t n, Clouds K, uint32_t* mm) {
  uint32_t i = gid();
  uint32_t c = (i < n && K.C > 1) ? cloud_of_point(K.off, K.C, i) : 0u;
  uint32_t lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, hi[3] = {0u, 0u, 0u};
  if (i < n)
    for (int k = 0; k < 3; ++k) {
      float v = xyz[3 * (size_t)i + k];
      if (v == v) {
        uint32_t o = ord_f32(v);
        lo[k] = o;
        hi[k] = o;
      }
    }
  uint32_t c0 = __shfl(c, 0);
  bool same = c == c0;
  for (int k = 0; k < 3; ++k) {
    uint32_t l = same ? lo[k] : 0xFFFFFFFFu, h = same ? hi[k] : 0u;
    for (int off = 32; off > 0; off >>= 1) {
      l = min(l, (uint32_t)__shfl_xor(l, off));
      h = max(h, (uint32_t)__shfl_xor(h, off));
    }
    if (__lane_id() == 0) {
      atomicMin(&mm[6 * (size_t)c0 + k], l);
      atomicMax(&mm[6 * (size_t)c0 + 3 + k], h);
    }
    if (!same && i < n) {
      atomicMin(&mm[6 * (size_t)c + k], lo[k]);
      atomicMax(&mm[6 * (size_t)c + 3 + k], hi[k]);
    }
  }
}

__global__ void k_normalize(const float* xyz, uint32_t n, Clouds K, const uint32_t* mm,
                            float* xyzn, uint64_t* keys, uint32_t* ids) {
  uint32_t i = gid();
  if (i < n) normalize_body(xyz, i, K, mm, xyzn, keys, ids);
}

__global__ void k_gather_points(const float* xyzn, const uint32_t* ids, const uint64_t* keys,
                                uint32_t n, Clouds K, float4* pts) {
  uint32_t j = gid();
  if (j < n) gather_body(xyzn, ids, keys, j, K, pts);
}

__global__ void k_tail_points(Clouds K, float4* pts) {
  uint32_t g = gid();
  if (g <= 4u * K.C) tail_body(g, K, pts);
}

__global__ void k_start_tets(Mesh M, StartTets S, Clouds K) {
  uint32_t g = gid();
  if (g < 5u * K.C) start_tet_body(M, S, g, K);
}

// One cloud: every thread folds many points (grid-stride, coalesced), the
// block combines in LDS, and one lane per block issues the 6 atomics.
__global__ void __launch_bounds__(kBlock) k_minmax_single(const float* xyz, uint32_t n, uint32_t* mm) {
  __shared__ uint32_t red[6][kBlock / 64];
  uint32_t lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu}, hi[3] = {0u, 0u, 0u};
  uint32_t stride = gridDim.x * kBlock;
  for (uint32_t i = gid(); i < n; i += stride)
    for (int k = 0; k < 3; ++k) {
      float v = xyz[3 * (size_t)i + k];
      if (v == v) {
        uint32_t o = ord_f32(v);
        lo[k] = min(lo[k], o);
        hi[k] = max(hi[k], o);
      }
    }
  int wave = threadIdx.x >> 6;
  for (int k = 0; k < 3; ++k) {
    for (int off = 32; off > 0; off >>= 1) {
      lo[k] = min(lo[k], (uint32_t)__shfl_xor(lo[k], off));
      hi[k] = max(hi[k], (uint32_t)__shfl_xor(hi[k], off));
    }
    if (__lane_id() == 0) {
      red[k][wave] = lo[k];
      red[3 + k][wave] = hi[k];
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    int k = threadIdx.x;
    uint32_t v = k < 3 ? 0xFFFFFFFFu : 0u;
    for (int w = 0; w < kBlock / 64; ++w) v = k < 3 ? min(v, red[k][w]) : max(v, red[k][w]);
    if (k < 3) atomicMin(&mm[k], v);
    else atomicMax(&mm[k], v);
  }
}

void launch_minmax(const float* xyz, uint32_t n, const Clouds& K, uint32_t* mm, hipStream_t s) {
  k_minmax_init<<<nblocks(6u * K.C), kBlock, 0, s>>>(mm, K.C);
  if (K.C <= 1)
    k_minmax_single<<<std::max(1u, std::min(nblocks(n) / 16u, 1024u)), kBlock, 0, s>>>(xyz, n, mm);
  else
    k_minmax<<<nblocks(n), kBlock, 0, s>>>(xyz, n, K, mm);
}

void launch_prepare(const float* xyz, uint32_t n, const Clouds& K, uint32_t* mm, float* xyzn,
                    uint64_t* keys, uint32_t* ids, hipStream_t s) {
  launch_minmax(xyz, n, K, mm, s);
  k_normalize<<<nblocks(n), kBlock, 0, s>>>(xyz, n, K, mm, xyzn, keys, ids);
}

void launch_gather_points(const float* xyzn, const uint32_t* ids, const uint64_t* keys,
                          uint32_t n, const Clouds& K, float4* pts, hipStream_t s) {
  k_gather_points<<<nblocks(n), kBlock, 0, s>>>(xyzn, ids, keys, n, K, pts);
  k_tail_points<<<nblocks(4u * K.C + 1u), kBlock, 0, s>>>(K, pts);
}

void launch_start_tets(const Mesh& M, const Clouds& K, hipStream_t s) {
  static const StartTets S = make_start_tets();
  k_start_tets<<<nblocks(5u * K.C), kBlock, 0, s>>>(M, S, K);
}

size_t sort_temp_bytes(uint32_t n, int end_bit) { return radix_temp_bytes_u64(n, end_bit); }

hipError_t sort_pairs(uint64_t* keys, uint32_t* ids, uint64_t* keys_tmp, uint32_t* ids_tmp, uint32_t n,
                      int end_bit, void* temp, size_t temp_bytes, hipStream_t s) {
  return radix_sort_u64(keys, ids, keys_tmp, ids_tmp, n, end_bit, temp, temp_bytes, s);
}

size_t sort_temp_bytes_u32(uint32_t n, int end_bit) { return radix_temp_bytes_u32(n, end_bit); }

hipError_t sort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp,
                          uint32_t n, int end_bit, void* temp, size_t temp_bytes, hipStream_t s) {
  return radix_sort_u32(keys, vals, keys_tmp, vals_tmp, n, end_bit, temp, temp_bytes, s);
}

__global__ void k_uninit_count(const float4* pts, const uint64_t* keys, uint32_t n, Clouds K,
                               uint32_t* blk, uint32_t* ctr) {
  uint32_t j = gid();
  uint32_t capped = 0, c = 0;
  bool keep = keep_point(pts, keys, n, K, j, &c, &capped);
  if (capped) atomicAdd(&ctr[C_DUPSCAN], 1u);
  uint32_t tot;
  block_rank(keep, &tot);
  if (threadIdx.x == 0) blk[blockIdx.x] = tot;
}

__global__ void k_uninit_scatter(const float4* pts, const uint64_t* keys, uint32_t n, Clouds K,
                                 const uint32_t* blk, uint32_t* uvert, uint32_t* utet) {
  uint32_t j = gid();
  uint32_t capped = 0, c = 0;
  bool keep = keep_point(pts, keys, n, K, j, &c, &capped);
  uint32_t tot;
  uint32_t r = blk[blockIdx.x] + block_rank(keep, &tot);
  if (keep) {
    uvert[r] = j + 4u * c;
    utet[r] = 5u * c;  // every point starts in its cloud's super tet
  }
}

void launch_init_uninserted(const float4* pts, const uint64_t* keys, uint32_t n, const Clouds& K,
                            uint32_t* blk, uint32_t* uvert, uint32_t* utet, uint32_t* ctr,
                            hipStream_t s) {
  uint32_t nb = nblocks(n);
  k_uninit_count<<<nb, kBlock, 0, s>>>(pts, keys, n, K, blk, ctr);
  k_scan_blocks<<<1, 1024, 0, s>>>(blk, nb, ctr, 2);
  k_uninit_scatter<<<nb, kBlock, 0, s>>>(pts, keys, n, K, blk, uvert, utet);
}

// Reference insertion order of the Hilbert mode: within each cloud the
// uninserted list follows the stratified order of the sorted points
// (src/gpu/mod.rs:473-600).  key = (cloud, rank among all the cloud's points);
// after the sort each entry's start tet is its cloud's super tet again.
__global__ void k_stratify_keys(const uint32_t* uvert, uint32_t U, Clouds K, uint64_t* key) {
  uint32_t r = gid();
  if (r >= U) return;
  uint32_t v = uvert[r];
  uint32_t c = K.C > 1 ? cloud_of_vertex(K.off, K.C, v) : 0u;
  uint32_t nc = K.off[c + 1] - K.off[c];
  uint32_t jl = v - 4u * c - K.off[c];
  key[r] = ((uint64_t)c << 32) | stratified_rank(jl, nc, initial_stride(nc));
}

__global__ void k_list_from_sorted(const uint32_t* sv, uint32_t U, Clouds K, uint32_t* uvert,
                                   uint32_t* utet) {
  uint32_t r = gid();
  if (r >= U) return;
  uint32_t v = sv[r];
  uvert[r] = v;
  utet[r] = 5u * (K.C > 1 ? cloud_of_vertex(K.off, K.C, v) : 0u);
}

hipError_t launch_stratify(uint32_t* uvert, uint32_t* utet, uint32_t U, const Clouds& K, uint64_t* key,
                           uint64_t* key_tmp, uint32_t* val_tmp, void* temp, size_t temp_bytes,
                           hipStream_t s) {
  if (!U) return hipSuccess;
  k_stratify_keys<<<nblocks(U), kBlock, 0, s>>>(uvert, U, K, key);
  int bits = 32 + (K.C > 1 ? cloud_key_bits(K.C) : 0);
  hipError_t e = radix_sort_u64(key, uvert, key_tmp, val_tmp, U, bits, temp, temp_bytes, s);
  if (e != hipSuccess) return e;
  k_list_from_sorted<<<nblocks(U), kBlock, 0, s>>>(val_tmp, U, K, uvert, utet);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// insertion rounds
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kBlock) k_vote(Mesh M, const uint32_t* uvert, const uint32_t* utet) {
  vote_wave(M, uvert, utet, gid(), M.ctr[C_SURV]);
}

// Counts the winners of each block of points, and marks the tets left in the
// flip list.  Begins the round in the
// counters: no other thread of this kernel reads them.
__global__ void __launch_bounds__(kBlock) k_pick_count(Mesh M, const uint32_t* utet, uint32_t* blk, int ring,
                                                       FlipLists L) {
  const uint32_t U = M.ctr[C_SURV], A = M.ctr[C_LIST], it = M.ctr[C_IT] + 1u;
  const uint32_t* act = L.act[M.ctr[C_PAR] & 1u];
  for (uint32_t j = gid(); j < A; j += gridDim.x * kBlock) mark_listed(M, act[j], it);
  uint32_t i = gid();
  if (i == 0) {
    M.ctr[C_ROUND] += 1u;
    M.ctr[C_SLOW_P] = 0u;
  }
  bool w = i < U && is_winner(M, utet, i, ring);
  uint32_t tot;
  block_rank(w, &tot);
  if (threadIdx.x == 0) blk[blockIdx.x] = tot;
}

// SCANNED: blk holds each block's first winner; otherwise the blocks' counts,
// which every block adds up to its own (and the last one to C_WIN): a launch
// less, for grids whose counts are few enough to read in each block.
template <bool SCANNED>
__global__ void __launch_bounds__(kBlock) k_pick_scatter(Mesh M, const uint32_t* uvert, const uint32_t* utet,
                               uint2* wlist, uint32_t* uvert2, uint32_t* utet2, const uint32_t* blk,
                               int ring) {
  const uint32_t U = M.ctr[C_SURV], round = M.ctr[C_ROUND];
  uint32_t i = gid();
  uint32_t first = 0;
  if (SCANNED) {
    first = blk[blockIdx.x];
  } else {
    __shared__ uint32_t part[kBlock / 64];
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kBlock) first += blk[b];
    for (int off = 32; off > 0; off >>= 1) first += __shfl_xor(first, off);
    if (__lane_id() == 0) part[threadIdx.x >> 6] = first;
    __syncthreads();
    first = 0;
    for (int w = 0; w < kBlock / 64; ++w) first += part[w];
  }
  bool w = i < U && is_winner(M, utet, i, ring);
  uint32_t tot;
  uint32_t r = first + block_rank(w, &tot);
  if (!SCANNED && blockIdx.x == gridDim.x - 1u && threadIdx.x == 0) M.ctr[C_WIN] = first + tot;
  if (i >= U) return;
  uint32_t t = utet[i], v = uvert[i];
  if (w) {
    wlist[r] = make_uint2(t, v);
    TSPLIT(M, t) = make_uint2(round, M.ctr[C_TETS] + 3u * r);
    TPOINT(M, t) = v;
  } else {
    uvert2[i - r] = v;
    utet2[i - r] = t;
  }
}

// Launch grids of the round kernels: a power of two of workgroups covering
// the host's bound, so that a captured round can be replayed for any count
// up to that bound (the kernels read the counts from ctr).
uint32_t round_grid(uint64_t bound) {
  uint32_t want = std::max<uint32_t>(1u, nblocks(bound)), g = 1;
  while (g < want) g <<= 1;
  return g;
}

void launch_vote(const Mesh& M, const uint32_t* uvert, const uint32_t* utet, uint32_t U,
                 hipStream_t s) {
  k_vote<<<round_grid(U), kBlock, 0, s>>>(M, uvert, utet);
}

// Up to this many blocks every block of the scatter adds up the counts before
// its own (4,096 words from L2: 1M points); above, one block scans them.
constexpr uint32_t kScatterScan = 4096;

void launch_pick(const Mesh& M, const uint32_t* uvert, const uint32_t* utet, uint32_t U,
                 uint2* wlist, uint32_t* uvert2, uint32_t* utet2, uint32_t* blk, int ring,
                 const FlipLists& L, hipStream_t s) {
  // blocks past the count write zero block totals, so the scan may cover
  // the whole grid
  uint32_t nb = round_grid(U);
  k_pick_count<<<nb, kBlock, 0, s>>>(M, utet, blk, ring, L);
  if (nb <= kScatterScan) {
    k_pick_scatter<false><<<nb, kBlock, 0, s>>>(M, uvert, utet, wlist, uvert2, utet2, blk, ring);
  } else {
    k_scan_blocks<<<1, 1024, 0, s>>>(blk, nb, M.ctr, 0);
    k_pick_scatter<true><<<nb, kBlock, 0, s>>>(M, uvert, utet, wlist, uvert2, utet2, blk, ring);
  }
}

// The children join the active list with one counter atomic per wave, in
// child-major order within the wave (the wave's child-0 slots, then its
// child-1 slots, ...).  The order matters: the fresh slots of the flips
// that follow are numbered in list order, and lower slot ids win flip
// votes.  On co-spherical inputs a tet-major order left about four times
// as many faces stuck (1M points on a sphere: 3,150 against 866).
// Also takes the winners' slots and points off the counters, which no thread
// of this kernel reads.
__global__ void __launch_bounds__(kBlock) k_split(Mesh M, const uint2* wlist, FlipLists L) {
  const uint32_t W = M.ctr[C_WIN], round = M.ctr[C_ROUND], it = M.ctr[C_IT];
  uint32_t k = gid();
  if (k == 0) {
    M.ctr[C_IT0] = it;
    M.ctr[C_TETS] += 3u * W;
    M.ctr[C_SURV] -= W;
    M.ctr[C_SLOW_R] = 0u;
  }
  uint32_t c[4], m = 0u;
  if (k < W) m = split_body(M, wlist, k, round, it + 1u, c);
  uint64_t lt = (1ull << __lane_id()) - 1ull;
  uint64_t b0 = __ballot(m & 1u), bv = __ballot(m != 0u);
  uint32_t n0 = __popcll(b0), nv = __popcll(bv);
  uint32_t tot = n0 + 3u * nv;
  if (tot == 0u) return;
  uint32_t base = 0u;
  if (__lane_id() == 0) base = atomicAdd(&M.ctr[C_LIST], tot);
  base = __shfl(base, 0);
  uint32_t* act = L.act[M.ctr[C_PAR] & 1u];
  if (m & 1u) act[base + __popcll(b0 & lt)] = c[0];
  if (m) {
    uint32_t r = __popcll(bv & lt);
    for (uint32_t j = 1; j < 4; ++j) act[base + n0 + (j - 1u) * nv + r] = c[j];
  }
}

void launch_split(const Mesh& M, const uint2* wlist, uint32_t W, const FlipLists& L, hipStream_t s) {
  k_split<<<round_grid(W), kBlock, 0, s>>>(M, wlist, L);
}

// ---------------------------------------------------------------------------
// Batches of flip iterations, driven from the device: every count, the
// iteration tags, the round and the list parity are read from ctr, so a batch
// runs (and can be captured in a graph) without the host.  Iteration i of a
// batch has counters of its own (C_ITA + 32 i, ..): no kernel stands between
// two iterations to reset them, and one wave adds them up at the end.
// Measured with a one-thread kernel between iterations instead: 3 to 4 us
// each and the gap, 160 to 270 times a triangulation.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t* it_ctr(uint32_t* ctr, int which, int i) { return &ctr[which + 32 * i]; }

// the counters of a batch of k iterations; by one workgroup
__device__ __forceinline__ void batch_begin(uint32_t* ctr, int k) {
  for (int i = threadIdx.x; i < 4 * (k + 1); i += blockDim.x) {
    const int which = i / (k + 1), slot = i - which * (k + 1);
    *it_ctr(ctr, C_ITA + 65 * 32 * which, slot) = which == 0 && slot == 0 ? ctr[C_LIST] : 0u;
  }
  if (threadIdx.x == 0) ctr[C_TETS_IT] = ctr[C_TETS];
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// by one whole wave.  sums (IterSum): checked tets, flips, iterations, 2-3
// flips (a 2-3 flip takes one fresh slot, a 3-2 none)
__device__ __forceinline__ void batch_end(uint32_t* ctr, unsigned long long* sums, int k) {
  const int i = __lane_id();
  const bool run = i < k && *it_ctr(ctr, C_ITR, i) != 0u;
  const uint32_t a = run ? *it_ctr(ctr, C_ITA, i) : 0u, f = run ? *it_ctr(ctr, C_ITF, i) : 0u,
                 d = run ? *it_ctr(ctr, C_ITS, i) : 0u;
  const int n = __popcll(__ballot(run));  // iterations run: the first n
  uint64_t sa = a;
  uint32_t peak = a;
  for (int off = 32; off > 0; off >>= 1) {
    sa += (uint64_t)__shfl_xor((uint32_t)sa, off) | (uint64_t)__shfl_xor((uint32_t)(sa >> 32), off) << 32;
    peak = max(peak, (uint32_t)__shfl_xor(peak, off));
  }
  const uint32_t sf = wave_sum_u32(f), sd = wave_sum_u32(d), last = __shfl(d, n > 0 ? n - 1 : 0);
  if (i != 0) return;
  const uint32_t left = *it_ctr(ctr, C_ITA, n);
  sums[S_CHECKED] += sa;
  sums[S_FLIPS] += sf;
  sums[S_ITERS] += (unsigned long long)n;
  sums[S_FLIPS23] += ctr[C_TETS] - ctr[C_TETS_IT];
  ctr[C_SLOW_SUM] += sd;
  ctr[C_CHECK_SUM] += (uint32_t)sa;
  ctr[C_SLOW_LAST] = last;
  if (peak > ctr[C_PEAKA]) ctr[C_PEAKA] = peak;
  if (n < k && left > 0u) ctr[C_STOP] = 1u;  // the tet slots could not hold the next one
  ctr[C_LIST] = left;
  ctr[C_IT] += (uint32_t)n;  // the list left is that of the next iteration
  ctr[C_PAR] ^= (uint32_t)n & 1u;
}

__global__ void __launch_bounds__(kBlock) k_batch_begin(uint32_t* ctr, int k) { batch_begin(ctr, k); }
__global__ void k_batch_end(uint32_t* ctr, unsigned long long* sums, int k) { batch_end(ctr, sums, k); }

void launch_batch_begin(uint32_t* ctr, int k, hipStream_t s) { k_batch_begin<<<1, kBlock, 0, s>>>(ctr, k); }
void launch_batch_end(uint32_t* ctr, uint64_t* sums, int k, hipStream_t s) {
  k_batch_end<<<1, 64, 0, s>>>(ctr, reinterpret_cast<unsigned long long*>(sums), k);
}

// Point kernels in three forms: LEAN runs the FP32 filter alone and defers
// the points it cannot decide to `slow` (ctr[C_SLOW_P]); SLOW runs the full
// staged predicates on those; FULL runs them on every point (exact mode).
enum KForm : int { LEAN = 0, FULL = 1, SLOW = 2 };

// Grid of the point kernels' SLOW form, for the points the LEAN form
// deferred (their count is on the device): a quarter of the LEAN grid, at
// most 1,024 blocks.  Each deferred point keeps its thread in the full
// predicates for microseconds; degenerate input defers many (a 128^3
// lattice's relocation: 26.0 ms at a sixteenth and 256 blocks, 18.5 ms).
static uint32_t slow_grid(uint32_t g) { return std::min(g / 4u + 16u, 1024u); }

// The survivors of the round's pick (ctr[C_SURV]) in the round ctr[C_ROUND].
// Each clears the vote of its tet first: votes of tets whose winner was
// deferred must not survive into the next round (a split clears its own).
// begin > 0: the last form's first workgroup begins the batch of iterations.
template <int FORM>
__global__ void __launch_bounds__(kBlock) k_split_points(Mesh M, const uint32_t* uvert, uint32_t* utet,
                                                         uint64_t* st, uint32_t* slow, int begin) {
  const uint32_t U = M.ctr[C_SURV], round = M.ctr[C_ROUND];
  PredStats ls = {};
  if (FORM == SLOW) {
    uint32_t n = M.ctr[C_SLOW_P], stride = gridDim.x * kBlock;
    for (uint32_t k = gid(); k < n; k += stride)
      (void)split_points_body_t<false>(M, uvert, utet, slow[k], round, &ls);
  } else {
    uint32_t i = gid();
    bool defer = false;
    if (i < U) {
      TVOTE(M, utet[i]) = kVoteNone;
      defer = split_points_body_t<FORM == LEAN>(M, uvert, utet, i, round, &ls);
    }
    if (defer) slow[append_slot(&M.ctr[C_SLOW_P])] = i;
  }
  flush_stats(ls, st);
  if (FORM != LEAN && begin > 0 && blockIdx.x == 0) batch_begin(M.ctr, begin);
}

void launch_split_points(const Mesh& M, const uint32_t* uvert, uint32_t* utet, uint32_t U,
                         uint64_t* st, uint32_t* slow, int begin, hipStream_t s) {
  if (!U) return;
  uint32_t g = round_grid(U);
  if (M.mode == PRED_FILTERED) {
    k_split_points<LEAN><<<g, kBlock, 0, s>>>(M, uvert, utet, st, slow, 0);
    k_split_points<SLOW><<<slow_grid(g), kBlock, 0, s>>>(M, uvert, utet, st, slow, begin);
  } else {
    k_split_points<FULL><<<g, kBlock, 0, s>>>(M, uvert, utet, st, slow, begin);
  }
}

// ---------------------------------------------------------------------------
// flips: iteration i of a batch.  The kernels are persistent: a fixed grid
// strides over the current list.
// ---------------------------------------------------------------------------
// A kernel begins with its counters, and a load that only one side of a branch
// uses is moved there by the compiler, behind the loads of the branch's
// condition.  Here the values are complete: all of them come in one round trip.
__device__ __forceinline__ void loaded(uint32_t& a, uint32_t& b, uint32_t& c) {
  asm volatile("" : "+s"(a), "+s"(b), "+s"(c));
}

struct Iter {
  uint32_t n;    // entries (flips) of the list, 0 when the iteration does not run
  uint32_t it;   // tag
  uint32_t par;  // which active list is current
};
// The first kernel of an iteration decides whether it runs (C_TETS changes in
// decide_exec only) and says so to the others.
__device__ __forceinline__ Iter iter_first(uint32_t* ctr, int i) {
  uint32_t A = *it_ctr(ctr, C_ITA, i), tets = ctr[C_TETS], stop = ctr[C_STOP], cap = ctr[C_CAP], it = ctr[C_IT],
           par = ctr[C_PAR];
  loaded(A, tets, stop);
  loaded(cap, it, par);
  // worst case every proposal wins a 2-3 flip and takes a fresh slot
  const bool run = (A != 0u) & (stop == 0u) & ((uint64_t)tets + A + 64u <= (uint64_t)cap);
  if (run && gid() == 0) *it_ctr(ctr, C_ITR, i) = 1u;
  return Iter{run ? A : 0u, it + (uint32_t)i + 1u, (par + (uint32_t)i) & 1u};
}
// the others; which: the count (C_ITA, C_ITF, C_ITS) they run over
__device__ __forceinline__ Iter iter_next(uint32_t* ctr, int which, int i) {
  uint32_t run = *it_ctr(ctr, C_ITR, i), n = *it_ctr(ctr, which, i), it = ctr[C_IT], par = ctr[C_PAR];
  loaded(run, n, it);
  return Iter{run ? n : 0u, it + (uint32_t)i + 1u, (par + (uint32_t)i) & 1u};
}

// The filters of the flip check on every list entry, one thread per tet; the
// entries they leave go to L.slow.  100 VGPRs, 4 waves per SIMD (at 96 and 5
// waves, with two registers spilled, it took the same time).  1M uniform
// points: 6.68 ms of event time a triangulation with insphere_f32 and
// insphere_f64 per face and three orient3d after each (158 VGPRs), 5.60 ms
// with one set of cofactors per tet; 100k points 2.79 -> 2.05 ms.
// The neighbours stay in registers with the record they came in (read again for
// each proposal before): 1M points 21.1 -> 18.9 us a launch, on a sphere 8.7 -> 7.1.
// requeue: no kernel of this iteration runs the full predicates; an entry that
// needs them stays in the active list.
__global__ void __launch_bounds__(kBlock) k_flip_check(Mesh M, FlipLists L, int i, int requeue, uint64_t* st) {
  const Iter I = iter_first(M.ctr, i);
  const uint32_t* cur = I.par ? L.act[1] : L.act[0];
  const uint32_t stride = gridDim.x * kBlock;
  PredStats ls = {};
  for (uint32_t j = gid(); j < I.n; j += stride) {
    const uint32_t t = cur[j];
    if (flip_check_lean(M, t, L.prop, j, I.it, &ls)) {
      const uint32_t k = append_slot(it_ctr(M.ctr, C_ITS, i));
      if (requeue) L.prop[j] = requeue_proposal(M, t, I.it);
      else L.slow[k] = j;
    }
  }
  flush_stats(ls, st);
}

// The full predicates, four lanes per tet (flip_check_faces), on the entries
// the filters left or, with ALL, on every entry of the list (exact mode: one
// thread per tet and its faces in turn took 159 us a launch at 10,000 points,
// four lanes 41 us).  A wave's first k is a multiple of 64, so a tet's four
// lanes share a wave.  Where ALL runs beside filters (Run::full) it counts the
// tets that those would have left, one atomic a block.
template <bool ALL>
__global__ void __launch_bounds__(kBlock) k_flip_check_faces(Mesh M, FlipLists L, int i, uint64_t* st) {
  const Iter I = ALL ? iter_first(M.ctr, i) : iter_next(M.ctr, C_ITS, i);
  if (I.n == 0u) return;
  const uint32_t it = I.it;
  const uint32_t* cur = I.par ? L.act[1] : L.act[0];
  const uint32_t n4 = 4u * I.n, stride = gridDim.x * kBlock;
  PredStats ls = {};
  uint32_t left = 0u;
  for (uint32_t k = gid(); k < n4; k += stride) {
    const uint32_t before = ls.c[6] + ls.c[7];
    flip_check_faces(M, cur, L.prop, ALL ? k >> 2 : L.slow[k >> 2], (int)(k & 3u), it, &ls);
    uint64_t b = __ballot(ls.c[6] + ls.c[7] != before);  // lanes whose face took the exact insphere
    b |= b >> 1;
    b |= b >> 2;
    left += (uint32_t)__popcll(b & 0x1111111111111111ull);
  }
  flush_stats(ls, st);
  if (!ALL || M.mode != PRED_FILTERED) return;
  // a wave's active lanes are its first: lane 0 has counted them all
  __shared__ uint32_t part[kBlock / 64];
  if (__lane_id() == 0) part[threadIdx.x >> 6] = left;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < kBlock / 64; ++w) left += part[w];
  if (left) atomicAdd(it_ctr(M.ctr, C_ITS, i), left);
}

// Exclusive prefixes of three small counts in one pass (a, b in {0, 1},
// c in 0..3), packed 10, 10 and 12 bits (block totals of a and b stay
// below 1024, of c below 4096, for blocks of at most 512 threads).  Every
// thread of the block of BS threads must call it; w is LDS of BS/64.
template <int BS>
__device__ __forceinline__ uint32_t block_prefix3(uint32_t a, uint32_t b, uint32_t c, uint32_t* tot,
                                                  uint32_t* w) {
  uint64_t lt = (1ull << __lane_id()) - 1ull;
  uint64_t ba = __ballot(a), bb = __ballot(b), c0 = __ballot(c & 1u), c1 = __ballot(c & 2u);
  auto pack = [](uint32_t x, uint32_t y, uint32_t z) { return x | (y << 10) | (z << 20); };
  uint32_t r = pack(__popcll(ba & lt), __popcll(bb & lt), __popcll(c0 & lt) + 2u * __popcll(c1 & lt));
  int wave = threadIdx.x >> 6;
  if (__lane_id() == 0) w[wave] = pack(__popcll(ba), __popcll(bb), __popcll(c0) + 2u * __popcll(c1));
  __syncthreads();
  uint32_t off = 0, t = 0;
#pragma unroll
  for (int k = 0; k < BS / 64; ++k) {
    off += k < wave ? w[k] : 0u;
    t += w[k];
  }
  __syncthreads();
  *tot = t;
  return off + r;
}

// Decide every proposal; a winner loads its flip's tets at once, so those
// loads overlap the block's counter claims.  Then the
// block claims list space with one atomic per counter (flips, fresh slots,
// next active entries) -- the counters share a cache line, so per-wave
// atomics from every wave would serialize -- and every winner executes its
// own flip from registers.
// A tet's plain-stored fields are one 64-byte record (TetRec) and the update
// finds the external neighbours in the flip's own record.  Event time at 1M
// points against an array per field: flip_check 5.58 -> 4.28 ms (it reads one
// line of a tet instead of three, and no queued bit to clear), decide_exec 6.81
// -> 5.83 ms, flip_update 4.83 -> 4.39 ms.  With plain tags instead of an
// atomic maximum per queued tet and an atomic vote for the proposal's own:
// decide_exec 5.83 -> 5.20 ms, flip_check 4.28 -> 4.17 ms (1,024 clouds: 9.52 ->
// 8.69 and 11.6 -> 10.8).  Random lines bound both: this card serves 55 G/s
// of 64-byte reads, 27 G/s of atomics.
// Blocks of 512 threads: each tile of proposals claims its flips, fresh
// slots and queue entries with one atomic per counter, and those
// same-address atomics complete one at a time at the memory side; 512
// halves them against 256 (1M uniform device 26.0-26.1 -> 25.7-26.0 ms).
// Three lanes of one instruction make the three claims: from one lane the
// compiler waited for each, up to three of the launch's round trips
// (decide_exec at 100k points 10.7 -> 9.7 us, on a sphere 8.3 -> 7.7, at 1M 26.8
// -> 26.1).  Tried beside it: every proposal loading its tets beside the votes,
// instead of the winners after them (64 clouds 10.9 -> 11.2 us, 1M 26.9 -> 27.2).
constexpr uint32_t kDecBlock = 512;
static_assert(kDecBlock <= 512, "block_prefix3 packs totals of at most 512 threads");

__global__ void __launch_bounds__(kDecBlock) k_flip_decide_exec(Mesh M, FlipLists L, int i) {
  constexpr uint32_t kBS = kDecBlock;
  __shared__ uint32_t wsum[kBS / 64];
  __shared__ uint32_t base[3];
  const Iter I = iter_next(M.ctr, C_ITA, i);
  const uint32_t A = I.n, it = I.it;
  uint32_t* act_next = I.par ? L.act[0] : L.act[1];
  for (uint32_t b0 = blockIdx.x * kBS; b0 < A; b0 += gridDim.x * kBS) {
    uint32_t j = b0 + threadIdx.x;
    uint4 pr = make_uint4(kInvalid, 0u, 0u, 0u);
    if (j < A) pr = L.prop[j];
    uint32_t qid[2], nq, nslot;
    FlipTets F;
    bool win = flip_decide_load(M, pr, it, qid, &nq, &nslot, F);
    uint32_t nqa = nq + nslot;  // the fresh slot is queued too
    uint32_t tot;
    uint32_t r = block_prefix3<kBS>(win ? 1u : 0u, nslot, nqa, &tot, wsum);
    uint32_t rf = r & 1023u, rs = (r >> 10) & 1023u, rq = r >> 20;
    uint32_t tf = tot & 1023u, ts = (tot >> 10) & 1023u, tq = tot >> 20;
    if (threadIdx.x < 3u) {  // three lanes: one round trip, not one after another
      const uint32_t l = threadIdx.x, v = l == 0u ? tf : (l == 1u ? ts : tq);
      uint32_t* p = l == 0u ? it_ctr(M.ctr, C_ITF, i) : (l == 1u ? &M.ctr[C_TETS] : it_ctr(M.ctr, C_ITA, i + 1));
      base[l] = v ? atomicAdd(p, v) : 0u;
    }
    __syncthreads();
    uint32_t q = base[2] + rq;
    if (nq > 0u) act_next[q] = qid[0];
    if (nq > 1u) act_next[q + 1u] = qid[1];
    if (win) {
      uint32_t sl = nslot ? base[1] + rs : kInvalid;
      if (nslot) act_next[q + nq] = sl;
      flip_exec_loaded(M, pr, F, it, sl, &L.out[4 * (size_t)(base[0] + rf)]);
    }
    // the next tile's prefix sums synchronize before base is rewritten
  }
}

// Three round trips: records, stamps, messages.  With the messages behind a
// branch each (loaded only where the neighbour flipped) the compiler waited for
// each of the six; now a lane without one reads a line common to all: 1M points
// 22.0 -> 20.0 us a launch, 64 clouds 6.8 -> 6.1, 2,048 clouds 70.6 -> 67.2.
__global__ void __launch_bounds__(kBlock) k_flip_update(Mesh M, FlipLists L, int i) {
  const Iter I = iter_next(M.ctr, C_ITF, i);
  const uint32_t stride = gridDim.x * kBlock;
  for (uint32_t k = gid(); k < I.n; k += stride) flip_update_body(M, L.out, k, I.it);
}

// Up to k flip iterations of a short list in one workgroup
// (wg_flip_iteration), a whole batch.  Stops at the first iteration whose
// list is empty or longer than `limit`; a longer list stays for the next
// batch.  Event time at 100k points: 1.28 ms a triangulation with counters and
// atomics at the memory side (and the full predicates inline), 0.37 ms with
// LDS counters and atomics at workgroup scope.
constexpr int kFlipSmallBlock = 512;

__global__ void __launch_bounds__(kFlipSmallBlock) k_flip_small(WgMesh M, FlipLists L, uint64_t* st,
                                                                unsigned long long* sums, int k, uint32_t limit) {
  __shared__ WgCounters c;
  uint32_t* ctr = M.ctr;
  const uint32_t tets0 = ctr[C_TETS], cap = ctr[C_CAP], it0 = ctr[C_IT];
  uint32_t A = ctr[C_LIST], par = ctr[C_PAR] & 1u, tets = tets0, sa = 0, sf = 0, peak = 0, slow = 0, last = 0;
  bool stop = ctr[C_STOP] != 0u;
  int n = 0;
  if (threadIdx.x == 0) c.slots = tets0;
  for (; n < k && !stop && A > 0u && A <= limit; ++n) {
    if ((uint64_t)tets + A + 64u > (uint64_t)cap) {
      stop = true;
      break;
    }
    wg_flip_iteration<WgMesh, kFlipSmallBlock>(M, c, par ? L.act[1] : L.act[0], par ? L.act[0] : L.act[1], L.prop,
                                               L.slow, L.out, A, it0 + (uint32_t)n + 1u, st);
    sa += A;
    sf += c.flips;
    slow += c.slow;
    last = c.slow;
    peak = max(peak, A);
    A = c.act_next;
    tets = c.slots;
    par ^= 1u;
    __syncthreads();  // the counters are read before the next iteration resets them
  }
  if (threadIdx.x == 0) {
    sums[S_CHECKED] += sa;
    sums[S_FLIPS] += sf;
    sums[S_ITERS] += (unsigned long long)n;
    sums[S_FLIPS23] += tets - tets0;
    sums[S_SMALL_CHECKED] += sa;
    sums[S_SMALL_FLIPS] += sf;
    ctr[C_TETS] = tets;
    ctr[C_SLOW_SUM] += slow;
    ctr[C_CHECK_SUM] += sa;
    ctr[C_SLOW_LAST] = last;
    if (peak > ctr[C_PEAKA]) ctr[C_PEAKA] = peak;
    if (stop) ctr[C_STOP] = 1u;
    ctr[C_LIST] = A;
    ctr[C_IT] = it0 + (uint32_t)n;
    ctr[C_PAR] = par;
  }
}

void launch_flip_small(const Mesh& M, const FlipLists& L, uint64_t* st, uint64_t* sums, int k,
                       uint32_t limit, hipStream_t s) {
  k_flip_small<<<1, kFlipSmallBlock, 0, s>>>(WgMesh{M}, L, st, reinterpret_cast<unsigned long long*>(sums), k, limit);
}

// Rounds of few points: a round is nine launches and a read by the host, and
// its flips a batch, whatever it holds.  The phases are those of the list
// kernels in their order, with barriers in place of launches, counters in LDS
// and atomics at workgroup scope.  64 points: device 1.05 -> 0.74 ms, 1,000 points
// 2.47 -> 2.09 ms (10 and 20 rounds).
__global__ void __launch_bounds__(kFlipSmallBlock) k_rounds_small(WgMesh M, FlipLists L, SmallRun J, uint64_t* st,
                                                                  unsigned long long* sums) {
  constexpr int BS = kFlipSmallBlock;
  __shared__ WgCounters c;
  __shared__ uint32_t wsum[BS / 64];
  const uint32_t tid = threadIdx.x;
  const uint64_t lt = (1ull << __lane_id()) - 1ull;
  const bool filtered = M.mode == PRED_FILTERED;
  uint32_t* ctr = M.ctr;
  const uint32_t cap = ctr[C_CAP], tets0 = ctr[C_TETS];
  uint32_t U = ctr[C_SURV], W = ctr[C_WIN], A = ctr[C_LIST], par = ctr[C_PAR] & 1u, it = ctr[C_IT], it0 = ctr[C_IT0],
           round = ctr[C_ROUND], tets = tets0, cur = J.cur;
  bool crowded = false;
  uint32_t picks = 0, sumu = 0, sa = 0, sf = 0, peak = 0, slow = 0, last_slow = ctr[C_SLOW_LAST], done = 0, f23 = 0, iters = 0;
  bool stop = ctr[C_STOP] != 0u, voted = J.voted != 0;
  for (;;) {
    if (!voted) {
      // the vote and the pick: winners to wlist, the others to the second list,
      // both in list order
      const uint32_t* uv = cur ? J.uvert[1] : J.uvert[0];
      const uint32_t* ut = cur ? J.utet[1] : J.utet[0];
      uint32_t* uv2 = cur ? J.uvert[0] : J.uvert[1];
      uint32_t* ut2 = cur ? J.utet[0] : J.utet[1];
      for (uint32_t b = 0; b < U; b += BS) vote_wave(M, uv, ut, b + tid, U);
      for (uint32_t j = tid; j < A; j += BS) mark_listed(M, par ? L.act[1][j] : L.act[0][j], it + 1u);
      __syncthreads();
      ++round;
      const int ring = round <= J.warmup ? 0 : J.ring;
      W = 0;
      for (uint32_t b = 0; b < U; b += BS) {
        const uint32_t i = b + tid;
        const bool w = i < U && is_winner(M, ut, i, ring);
        uint32_t tot;
        const uint32_t r = W + wg_rank<BS>(w, &tot, wsum);
        if (i < U) {
          const uint32_t t = ut[i], v = uv[i];
          if (w) {
            J.wlist[r] = make_uint2(t, v);
            TSPLIT(M, t) = make_uint2(round, tets + 3u * r);
            TPOINT(M, t) = v;
          } else {
            uv2[i - r] = v;
            ut2[i - r] = t;
          }
        }
        W += tot;
      }
      ++picks;
      sumu += U;
      cur ^= 1u;
      __syncthreads();
      if (W == 0u) break;
    }
    voted = false;
    const uint32_t bound = crowded ? J.list_full : J.list;
    if (stop || (uint64_t)tets + 3u * W + 64u > (uint64_t)cap || A + 4u * W > bound) break;
    // the splits; the children join the active list as in k_split
    const uint32_t* uv = cur ? J.uvert[1] : J.uvert[0];
    uint32_t* ut = cur ? J.utet[1] : J.utet[0];
    uint32_t* act = par ? L.act[1] : L.act[0];
    if (tid == 0) {
      c.act_next = A;
      c.slow = 0u;
      c.slots = tets + 3u * W;
    }
    __syncthreads();
    it0 = it;
    for (uint32_t b = 0; b < W; b += BS) {
      const uint32_t k = b + tid;
      uint32_t ch[4], m = 0u;
      if (k < W) m = split_body(M, J.wlist, k, round, it + 1u, ch);
      const uint64_t b0 = __ballot(m & 1u), bv = __ballot(m != 0u);
      const uint32_t n0 = __popcll(b0), nv = __popcll(bv);
      uint32_t base = 0u;
      if (__lane_id() == 0 && nv) base = lds_add(&c.act_next, n0 + 3u * nv);
      base = __shfl(base, 0);
      if (m & 1u) act[base + __popcll(b0 & lt)] = ch[0];
      if (m) {
        const uint32_t r = __popcll(bv & lt);
        for (uint32_t j = 1; j < 4; ++j) act[base + n0 + (j - 1u) * nv + r] = ch[j];
      }
    }
    U -= W;
    tets += 3u * W;
    __syncthreads();
    A = c.act_next;
    uint32_t ns = U;
    if (filtered) {
      PredStats ls = {};
      for (uint32_t i = tid; i < U; i += BS) {
        TVOTE(M, ut[i]) = kVoteNone;
        if (split_points_body_t<true>(M, uv, ut, i, round, &ls)) J.slow[lds_slot(&c.slow)] = i;
      }
      flush_stats(ls, st);
      __syncthreads();
      ns = c.slow;
    } else {
      for (uint32_t i = tid; i < U; i += BS) TVOTE(M, ut[i]) = kVoteNone;
      __syncthreads();
    }
    if (ns) wg_slow_points<WgMesh, BS>(M, uv, ut, filtered ? J.slow : nullptr, ns, round, false, st);
    __syncthreads();
    // the flips of the round, the last round's to the end of the list
    done = U == 0u || round >= J.max_round ? 1u : 0u;
    const uint32_t n_it = done ? 4096u : (uint32_t)J.k;
    uint32_t round_slow = 0, round_it = 0;
    for (uint32_t n = 0; n < n_it && A > 0u && A <= J.limit; ++n) {
      if ((uint64_t)tets + A + 64u > (uint64_t)cap) {
        stop = true;
        break;
      }
      wg_flip_iteration<WgMesh, BS>(M, c, par ? L.act[1] : L.act[0], par ? L.act[0] : L.act[1], L.prop, L.slow, L.out, A,
                                    ++it, st);
      sa += A;
      sf += c.flips;
      slow += c.slow;
      last_slow = c.slow;
      peak = max(peak, A);
      ++iters;
      ++round_it;
      round_slow += c.slow;
      f23 += c.slots - tets;
      A = c.act_next;
      tets = c.slots;
      par ^= 1u;
      __syncthreads();  // the counters are read before the next iteration resets them
    }
    crowded = round_slow > J.list_full * round_it;
    if (U > 0u) {
      // points of flipped tets to the tets now holding them
      if (tid == 0) c.slow = 0u;
      __syncthreads();
      ns = U;
      if (filtered) {
        PredStats ls = {};
        for (uint32_t i = tid; i < U; i += BS)
          if (relocate_body_t<true>(M, uv, ut, i, it0, &ls)) J.slow[lds_slot(&c.slow)] = i;
        flush_stats(ls, st);
        __syncthreads();
        ns = c.slow;
      }
      if (ns) wg_slow_points<WgMesh, BS>(M, uv, ut, filtered ? J.slow : nullptr, ns, it0, true, st);
      __syncthreads();
    }
    W = 0u;
    if (done) break;
  }
  if (tid == 0) {
    sums[S_CHECKED] += sa;
    sums[S_FLIPS] += sf;
    sums[S_ITERS] += (unsigned long long)iters;
    sums[S_FLIPS23] += f23;
    sums[S_SMALL_CHECKED] += sa;
    sums[S_SMALL_FLIPS] += sf;
    ctr[C_TETS] = tets;
    ctr[C_SLOW_SUM] += slow;
    ctr[C_CHECK_SUM] += sa;
    ctr[C_SLOW_LAST] = last_slow;
    if (peak > ctr[C_PEAKA]) ctr[C_PEAKA] = peak;
    if (stop) ctr[C_STOP] = 1u;
    ctr[C_LIST] = A;
    ctr[C_IT] = it;
    ctr[C_IT0] = it0;
    ctr[C_PAR] = par;
    ctr[C_ROUND] = round;
    ctr[C_SURV] = U;
    ctr[C_WIN] = W;
    ctr[C_SLOW_P] = 0u;
    ctr[C_SLOW_R] = 0u;
    ctr[C_RUN_PICKS] = picks;
    ctr[C_RUN_SUMU] = sumu;
    ctr[C_RUN_DONE] = done;
    ctr[C_RUN_CROWDED] = crowded;
  }
}

void launch_rounds_small(const Mesh& M, const FlipLists& L, const SmallRun& J, uint64_t* st, uint64_t* sums,
                         hipStream_t s) {
  k_rounds_small<<<1, kFlipSmallBlock, 0, s>>>(WgMesh{M}, L, J, st, reinterpret_cast<unsigned long long*>(sums));
}

__global__ void k_set_ctr(uint32_t* ctr, int idx, uint32_t v, int idx2, uint32_t v2) {
  if (threadIdx.x == 0) {
    ctr[idx] = v;
    if (idx2 >= 0) ctr[idx2] = v2;
  }
}

void launch_set_ctr(uint32_t* ctr, int idx, uint32_t v, int idx2, uint32_t v2, hipStream_t s) {
  k_set_ctr<<<1, 64, 0, s>>>(ctr, idx, v, idx2, v2);
}

void launch_flip_check(const Mesh& M, const FlipLists& L, int i, bool requeue, bool full, uint32_t grid, uint64_t* st,
                       hipStream_t s) {
  if (M.mode == PRED_FILTERED && !full) k_flip_check<<<grid, kBlock, 0, s>>>(M, L, i, requeue ? 1 : 0, st);
  else k_flip_check_faces<true><<<std::min(4u * grid, 4096u), kBlock, 0, s>>>(M, L, i, st);
}
void launch_flip_check_deferred(const Mesh& M, const FlipLists& L, int i, uint32_t grid, uint64_t* st,
                                hipStream_t s) {
  if (M.mode == PRED_FILTERED) k_flip_check_faces<false><<<grid, kBlock, 0, s>>>(M, L, i, st);
}
// grid: blocks of kBlock threads, as the other list kernels; the same
// threads in blocks of kDecBlock
void launch_flip_decide_exec(const Mesh& M, const FlipLists& L, int i, uint32_t grid, hipStream_t s) {
  k_flip_decide_exec<<<std::max<uint32_t>(grid * kBlock / kDecBlock, 1u), kDecBlock, 0, s>>>(M, L, i);
}
void launch_flip_update(const Mesh& M, const FlipLists& L, int i, uint32_t grid, hipStream_t s) {
  k_flip_update<<<grid, kBlock, 0, s>>>(M, L, i);
}

// The uninserted points after the round's pick (ctr[C_SURV]) whose tet a flip
// since the split (ctr[C_IT0]) took apart.  end > 0: the last form's first workgroup ends the batch of
// `end` iterations, which none of these kernels reads the counters of.
template <int FORM>
__global__ void __launch_bounds__(kBlock) k_relocate(Mesh M, const uint32_t* uvert, uint32_t* utet,
                                                     uint64_t* st, uint32_t* slow, unsigned long long* sums, int end) {
  const uint32_t U = M.ctr[C_SURV], it0 = M.ctr[C_IT0];
  PredStats ls = {};
  if (FORM == SLOW) {
    uint32_t n = 4u * M.ctr[C_SLOW_R], stride = gridDim.x * kBlock;
    for (uint32_t k = gid(); k < n; k += stride) relocate_faces(M, uvert, utet, slow[k >> 2], (int)(k & 3u), it0, true, &ls);
  } else if (FORM == FULL) {
    uint32_t k = gid();
    if (k < 4u * U) relocate_faces(M, uvert, utet, k >> 2, (int)(k & 3u), it0, false, &ls);
  } else {
    uint32_t i = gid();
    bool defer = false;
    if (i < U) defer = relocate_body_t<true>(M, uvert, utet, i, it0, &ls);
    if (defer) slow[append_slot(&M.ctr[C_SLOW_R])] = i;
  }
  flush_stats(ls, st);
  if (FORM != LEAN && end > 0 && blockIdx.x == 0 && threadIdx.x < 64) batch_end(M.ctr, sums, end);
}

void launch_relocate(const Mesh& M, const uint32_t* uvert, uint32_t* utet, uint32_t U,
                     uint64_t* st, uint32_t* slow, uint64_t* sums, int end, hipStream_t s) {
  if (!U) return;
  uint32_t g = round_grid(U);
  unsigned long long* sm = reinterpret_cast<unsigned long long*>(sums);
  if (M.mode == PRED_FILTERED) {
    k_relocate<LEAN><<<g, kBlock, 0, s>>>(M, uvert, utet, st, slow, sm, 0);
    k_relocate<SLOW><<<slow_grid(g), kBlock, 0, s>>>(M, uvert, utet, st, slow, sm, end);
  } else {
    // four lanes per point; 4 g, as every grid, follows from the rounded bound
    // that a captured round is kept by (the rounded grid of 4 U does not: one
    // block for 64 points, four for 65)
    k_relocate<FULL><<<4u * g, kBlock, 0, s>>>(M, uvert, utet, st, slow, sm, end);
  }
}

// LEAN: every slot, FP32 filter, undecided tets to slow[ctr[C_SLOW_T]];
// SLOW: the full predicates on those; FULL: the full predicates on every slot
template <int FORM>
__global__ void __launch_bounds__(kBlock) k_audit(Mesh M, uint32_t T, uint32_t* rec, uint32_t cap,
                                                  uint64_t* st, uint32_t* slow) {
  PredStats ls = {};
  if (FORM == SLOW) {
    uint32_t n = M.ctr[C_SLOW_T], stride = gridDim.x * kBlock;
    for (uint32_t k = gid(); k < n; k += stride) (void)audit_body_t<false>(M, slow[k], rec, cap, &ls);
  } else {
    uint32_t t = gid();
    if (t < T && audit_body_t<FORM == LEAN>(M, t, rec, cap, &ls))
      slow[append_slot(&M.ctr[C_SLOW_T])] = t;
  }
  flush_stats(ls, st);
}

void launch_audit(const Mesh& M, uint32_t T, uint32_t* rec, uint32_t cap, uint64_t* st, uint32_t* slow,
                  hipStream_t s) {
  if (!T) return;
  if (M.mode == PRED_FILTERED) {
    k_set_ctr<<<1, 64, 0, s>>>(M.ctr, C_SLOW_T, 0u, -1, 0u);
    k_audit<LEAN><<<nblocks(T), kBlock, 0, s>>>(M, T, rec, cap, st, slow);
    k_audit<SLOW><<<std::min<uint32_t>(nblocks(T), 1024u), kBlock, 0, s>>>(M, T, rec, cap, st, slow);
  } else {
    k_audit<FULL><<<nblocks(T), kBlock, 0, s>>>(M, T, rec, cap, st, slow);
  }
}

// ---------------------------------------------------------------------------
// output
// ---------------------------------------------------------------------------
__global__ void k_alive_count(Mesh M, uint32_t T, uint32_t* blk) {
  uint32_t t = gid();
  bool a = t < T && slot_alive(M, t);
  uint32_t tot;
  block_rank(a, &tot);
  if (threadIdx.x == 0) blk[blockIdx.x] = tot;
}

// one cloud: live slots in slot order are the rows
__global__ void k_alive_scatter(Mesh M, uint32_t T, const uint32_t* blk, uint32_t* olist,
                                uint32_t* slot2pos) {
  uint32_t t = gid();
  bool a = t < T && slot_alive(M, t);
  uint32_t tot;
  uint32_t r = blk[blockIdx.x] + block_rank(a, &tot);
  if (t < T) {
    slot2pos[t] = a ? r : kInvalid;
    if (a) olist[r] = t;
  }
}

// many clouds: sort key per slot = cloud of a live tet, or C for a free slot
__global__ void k_slot_keys(Mesh M, uint32_t T, Clouds K, uint32_t* okey, uint32_t* oslot) {
  uint32_t t = gid();
  if (t >= T) return;
  okey[t] = slot_alive(M, t) ? cloud_of_tet(M, t, K) : K.C;
  oslot[t] = t;
}

// after the sort: row j holds slot olist[j]; cstart[c] = first row of
// cloud c (every cloud has live tets), cstart[C] = number of live tets
__global__ void k_row_positions(const uint32_t* okey, const uint32_t* olist, uint32_t T, uint32_t C,
                                uint32_t* slot2pos, uint32_t* cstart) {
  uint32_t j = gid();
  if (j >= T) return;
  uint32_t c = okey[j];
  slot2pos[olist[j]] = c < C ? j : kInvalid;
  if (c < C && (j == 0 || okey[j - 1] != c)) cstart[c] = j;
}

__global__ void k_cstart_tail(uint32_t* cstart, uint32_t C, const uint32_t* ctr) {
  if (threadIdx.x == 0) cstart[C] = ctr[C_ALIVE];
}

__global__ void k_output_rows(Mesh M, uint32_t T, const uint32_t* olist, const uint32_t* okey,
                              const uint32_t* cstart, const uint32_t* slot2pos, const uint32_t* vrank,
                              Clouds K, uint32_t* out_tets, uint32_t* out_adj) {
  uint32_t j = gid();
  if (j >= T || j >= M.ctr[C_ALIVE]) return;
  output_body(M, j, olist, okey, cstart, slot2pos, vrank, K, out_tets, out_adj);
}

__global__ void k_vertex_ranks(const float4* pts, uint32_t nv, uint32_t* vrank) {
  uint32_t v = gid();
  if (v < nv) vrank[v] = pt_rank(pts[v]);
}

hipError_t launch_output(const Mesh& M, uint32_t T, const Clouds& K, const OutputBufs& B, hipStream_t s) {
  uint32_t nb = nblocks(T);
  k_alive_count<<<nb, kBlock, 0, s>>>(M, T, B.blk);
  k_scan_blocks<<<1, 1024, 0, s>>>(B.blk, nb, M.ctr, 1);
  const uint32_t* olist;
  const uint32_t* okey = nullptr;
  if (K.C <= 1) {
    k_alive_scatter<<<nb, kBlock, 0, s>>>(M, T, B.blk, B.olist, B.slot2pos);
    k_fill_u32<<<1, kBlock, 0, s>>>(B.cstart, 0u, 1);
    k_cstart_tail<<<1, 64, 0, s>>>(B.cstart, 1u, M.ctr);
    olist = B.olist;
  } else {
    k_slot_keys<<<nb, kBlock, 0, s>>>(M, T, K, B.okey, B.olist);
    hipError_t e = sort_pairs_u32(B.okey, B.olist, B.okey2, B.olist2, T, cloud_key_bits(K.C), B.temp,
                                  B.temp_bytes, s);
    if (e != hipSuccess) return e;
    k_row_positions<<<nb, kBlock, 0, s>>>(B.okey2, B.olist2, T, K.C, B.slot2pos, B.cstart);
    k_cstart_tail<<<1, 64, 0, s>>>(B.cstart, K.C, M.ctr);
    olist = B.olist2;
    okey = B.okey2;
  }
  if (B.out_tets) {
    k_vertex_ranks<<<nblocks((uint64_t)K.V + 1u), kBlock, 0, s>>>(M.pts, K.V + 1u, B.vrank);
    k_output_rows<<<nb, kBlock, 0, s>>>(M, T, olist, okey, B.cstart, B.slot2pos, B.vrank, K, B.out_tets,
                                        B.out_adj);
  }
  return hipGetLastError();
}

__global__ void k_map_records(uint32_t* rec, uint32_t n, const uint32_t* slot2idx) {
  uint32_t i = gid();
  if (i < n) rec[i] = (slot2idx[rec[i] >> 2] << 2) | (rec[i] & 3u);
}

void launch_map_records(uint32_t* rec, uint32_t n, const uint32_t* slot2idx, hipStream_t s) {
  if (n) k_map_records<<<nblocks(n), kBlock, 0, s>>>(rec, n, slot2idx);
}

// ---------------------------------------------------------------------------
// neighbourhood of the rows the host repair will touch: the rows of the
// recorded faces and the last `tail` rows (moved into holes), grown ring by
// ring over the output adjacency.  list[0, cnt) holds each marked row once;
// ring k reads list[bounds[k], bounds[k+1]).
// ---------------------------------------------------------------------------
__global__ void k_nbr_seed(const uint32_t* rec, uint32_t nrec, uint32_t M, uint32_t tail,
                           uint32_t* mark, uint32_t* list, uint32_t* cnt) {
  uint32_t i = gid();
  uint32_t row = kInvalid;
  if (i < nrec) row = rec[i] >> 2;
  else if (i < nrec + tail) row = M - tail + (i - nrec);
  bool add = row < M && atomicOr(&mark[row], 1u) == 0u;
  if (add) list[append_slot(cnt)] = row;
}

__global__ void k_nbr_snap(const uint32_t* cnt, uint32_t* bounds, int k) {
  if (threadIdx.x == 0) bounds[k] = cnt[0];
}

__global__ void k_nbr_ring(const uint32_t* adj, uint32_t M, uint32_t* mark, uint32_t* list,
                           uint32_t* cnt, const uint32_t* bounds, int k) {
  uint32_t b = bounds[k], e = bounds[k + 1];
  uint32_t stride = gridDim.x * kBlock;
  for (uint32_t i = b + gid(); i < e; i += stride) {
    uint32_t r = list[i];
    for (int f = 0; f < 4; ++f) {
      uint32_t a = adj[4 * (size_t)r + f];
      if (a == kInvalid) continue;
      uint32_t nb = a >> 5;
      if (nb < M && atomicOr(&mark[nb], 1u) == 0u) list[append_slot(cnt)] = nb;
    }
  }
}

// rows list[0, n) of the output arrays -> packed (row, tet[4], adj[4])
__global__ void k_nbr_gather(const uint32_t* list, uint32_t n, const uint32_t* tets,
                             const uint32_t* adj, uint32_t* out) {
  uint32_t i = gid();
  if (i >= n) return;
  uint32_t r = list[i];
  uint32_t* q = out + 9 * (size_t)i;
  q[0] = r;
  uint4 t = reinterpret_cast<const uint4*>(tets)[r];
  uint4 a = reinterpret_cast<const uint4*>(adj)[r];
  q[1] = t.x; q[2] = t.y; q[3] = t.z; q[4] = t.w;
  q[5] = a.x; q[6] = a.y; q[7] = a.z; q[8] = a.w;
}

void launch_neighbourhood(const uint32_t* rec, uint32_t nrec, uint32_t M, uint32_t tail, int rings,
                          const uint32_t* adj, uint32_t* mark, uint32_t* list, uint32_t* cnt,
                          uint32_t* bounds, bool more, hipStream_t s) {
  if (!more) {
    k_fill_u32<<<nblocks(M), kBlock, 0, s>>>(mark, 0u, M);
    k_fill_u32<<<1, kBlock, 0, s>>>(cnt, 0u, 1);
  }
  k_nbr_snap<<<1, 64, 0, s>>>(cnt, bounds, 0);
  if (nrec + tail)
    k_nbr_seed<<<nblocks((uint64_t)nrec + tail), kBlock, 0, s>>>(rec, nrec, M, tail, mark, list, cnt);
  for (int k = 0; k < rings; ++k) {
    k_nbr_snap<<<1, 64, 0, s>>>(cnt, bounds, k + 1);
    k_nbr_ring<<<256, kBlock, 0, s>>>(adj, M, mark, list, cnt, bounds, k);
  }
}

void launch_nbr_gather(const uint32_t* list, uint32_t n, const uint32_t* tets, const uint32_t* adj,
                       uint32_t* out, hipStream_t s) {
  if (n) k_nbr_gather<<<nblocks(n), kBlock, 0, s>>>(list, n, tets, adj, out);
}

__global__ void k_apply_patch(const uint32_t* patch, uint32_t n, uint32_t* tets, uint32_t* adj) {
  uint32_t i = gid();
  if (i >= n) return;
  const uint32_t* q = patch + 9 * (size_t)i;
  uint32_t sl = q[0];
  reinterpret_cast<uint4*>(tets)[sl] = make_uint4(q[1], q[2], q[3], q[4]);
  reinterpret_cast<uint4*>(adj)[sl] = make_uint4(q[5], q[6], q[7], q[8]);
}

void launch_apply_patch(const uint32_t* patch, uint32_t n, uint32_t* tets, uint32_t* adj,
                        hipStream_t s) {
  if (n) k_apply_patch<<<nblocks(n), kBlock, 0, s>>>(patch, n, tets, adj);
}

// ---------------------------------------------------------------------------
// fills and predicate batches
// ---------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_fill_u64(uint64_t* p, uint64_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_copy16(uint4* dst, const uint4* src, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (; i < n; i += stride) dst[i] = src[i];
}
void launch_copy16(uint4* dst, const uint4* src, uint64_t n, hipStream_t s) {
  if (n) k_copy16<<<(uint32_t)std::min<uint64_t>(nblocks(n), 8192), kBlock, 0, s>>>(dst, src, n);
}

void launch_fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s) {
  if (n) k_fill_u32<<<nblocks(n), kBlock, 0, s>>>(p, v, n);
}
void launch_fill_u64(uint64_t* p, uint64_t v, uint64_t n, hipStream_t s) {
  if (n) k_fill_u64<<<nblocks(n), kBlock, 0, s>>>(p, v, n);
}

__global__ void k_pred_batch(int kind, const float* pts, const uint32_t* idx, uint32_t n, int mode,
                             int32_t* out, uint64_t* st) {
  uint32_t i = gid();
  PredStats ls = {};
  if (i < n) {
    if (kind == 0) {
      const float* q = pts + 12 * (size_t)i;
      const uint32_t* k = idx + 4 * (size_t)i;
      out[i] = orient3d_sos(q, q + 3, q + 6, q + 9, k[0], k[1], k[2], k[3], mode, &ls);
    } else if (kind == 1) {
      const float* q = pts + 15 * (size_t)i;
      const uint32_t* k = idx + 5 * (size_t)i;
      out[i] = orient4d(q, q + 3, q + 6, q + 9, q + 12, k[0], k[1], k[2], k[3], k[4], mode, &ls);
    } else if (kind == 2) {
      const float* q = pts + 12 * (size_t)i;
      out[i] = orient3d_raw(q, q + 3, q + 6, q + 9, mode, &ls);
    } else {
      const float* q = pts + 15 * (size_t)i;
      out[i] = insphere_raw(q, q + 3, q + 6, q + 9, q + 12, mode, &ls);
    }
  }
  flush_stats(ls, st);
}

void launch_pred_batch(int kind, const float* pts, const uint32_t* idx, uint32_t n, int mode,
                       int32_t* out, uint64_t* st, hipStream_t s) {
  if (n) k_pred_batch<<<nblocks(n), kBlock, 0, s>>>(kind, pts, idx, n, mode, out, st);
}

}  // namespace wtet
