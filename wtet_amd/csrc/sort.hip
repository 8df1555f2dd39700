// Stable LSD radix sort of (key, value) pairs, 8-bit digits (sort.h).
//
// Per pass, over tiles of pairs:
//  * k_radix_up: each tile's digit counts (LDS atomics), digit-major
//    (counts[d * tiles + tile]);
//  * k_radix_scan: one workgroup per digit turns its row into global
//    offsets: the pairs of smaller digits (from the all-pass histogram that
//    k_radix_hist builds once, before the first pass) plus the exclusive
//    prefix over earlier tiles;
//  * k_radix_down: each tile ranks its pairs stably, sorts them by digit in
//    LDS and writes each digit's run to its place.
// Ranks need no workgroup barrier: a wave owns a contiguous part of the tile
// and its own row of digit counters, and ranks 64 pairs at a time with wave
// ballots.  At most kSmallTile pairs are sorted by one workgroup in one
// launch (k_radix_small).  Equal digits keep their order in every pass, so
// the whole sort is stable.
//
// What bounds it: pass for pass 32 bytes a pair (key read twice, value read
// once, both written).  4M pairs of 63-bit keys: 720 us with per-slab
// barriers and a scatter straight from registers (8 passes of 56 + 15 us,
// histogram 86 us), 359 us now (27 + 8, 31).  4,000
// pairs: 26 launches of about 4 us each before, 51 us in one now.
#include "sort.h"

#include <algorithm>

namespace wtet {

namespace {

constexpr int kSortThreads = 256;  // histogram, upsweep and scan
constexpr int kDigitBits = 8;
constexpr int kRadix = 1 << kDigitBits;
constexpr int kMaxPasses = 8;
constexpr int kWaves = kSortThreads / 64;
static_assert(kSortThreads == kRadix, "one thread per digit in the per-digit steps");

// Tiles: 4,096 pairs (runs of 16 a digit on average, 128 bytes of 64-bit
// keys) where that gives most CUs one, 1,024 below.  63-bit keys, 1,024
// against 4,096 a tile: 300k pairs 142 and 156 us, 500k 154 and 163, 1M 202
// and 180.
constexpr uint32_t kBigTile = 4096, kLittleTile = 1024;
constexpr uint32_t kBigFrom = 192 * kBigTile;
constexpr uint32_t kSmallTile = 4096;

// Digits are counted by LDS atomics, which take the lanes of one address one
// after another: keys of equal digits (sorted clouds, heavy ties) made a wave's
// count 64 steps.  Lane l counts in copy l % kCopies of the counters, a digit's
// copies side by side.  20M equal 64-bit keys: histogram 524 us with one copy,
// 190 with four, 185 with eight, upsweep 78, 41 and 41; random keys 195 and 37
// with any.
constexpr int kCopies = 4;

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }
inline uint32_t tile_of(uint32_t n) { return n >= kBigFrom ? kBigTile : kLittleTile; }
inline uint32_t tiles_of(uint32_t n) { return (n + tile_of(n) - 1) / tile_of(n); }
__host__ __device__ inline int passes_of(int end_bit) { return (end_bit + kDigitBits - 1) / kDigitBits; }

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K key, int shift, uint32_t mask) {
  return (uint32_t)(key >> shift) & mask;
}

// lanes of this wave that hold a valid pair with digit d (this lane's own
// when it is valid); every lane of the wave must call it
__device__ __forceinline__ uint64_t peer_mask(uint32_t d, bool valid) {
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < kDigitBits; ++b) {
    bool bit = (d >> b) & 1u;
    uint64_t bm = __ballot(bit);
    m &= bit ? bm : ~bm;
  }
  return m;
}

// inclusive sum over the lanes of the wave up to this one
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  uint32_t lane = lane_id();
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(x, off);
    if (lane >= (uint32_t)off) x += y;
  }
  return x;
}

__global__ void k_radix_zero(uint32_t* p, uint32_t n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// digit histograms of every pass in one read of the keys
template <typename K>
__global__ void __launch_bounds__(kSortThreads) k_radix_hist(const K* keys, uint32_t n, int end_bit,
                                                             uint32_t* ghist) {
  __shared__ uint32_t lh[kMaxPasses * kRadix * kCopies];
  const int P = passes_of(end_bit);
  const uint32_t copy = lane_id() % kCopies;
  for (int i = threadIdx.x; i < P * kRadix * kCopies; i += kSortThreads) lh[i] = 0u;
  __syncthreads();
  for (uint32_t i = blockIdx.x * kSortThreads + threadIdx.x; i < n; i += gridDim.x * kSortThreads) {
    const K key = keys[i];
    for (int p = 0; p < P; ++p) {
      int shift = p * kDigitBits;
      int bits = min(kDigitBits, end_bit - shift);
      atomicAdd(&lh[(p * kRadix + digit_of(key, shift, (1u << bits) - 1u)) * kCopies + copy], 1u);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < P * kRadix; i += kSortThreads) {
    uint32_t v = 0u;
#pragma unroll
    for (int k = 0; k < kCopies; ++k) v += lh[i * kCopies + k];
    if (v) atomicAdd(&ghist[i], v);
  }
}

template <typename K, int ITEMS>
__global__ void __launch_bounds__(kSortThreads) k_radix_up(const K* keys, uint32_t n, int shift,
                                                           uint32_t mask, uint32_t tiles,
                                                           uint32_t* counts) {
  __shared__ uint32_t cnt[kRadix * kCopies];
  const uint32_t t = threadIdx.x, copy = lane_id() % kCopies;
  const uint32_t base = blockIdx.x * (kSortThreads * ITEMS);
#pragma unroll
  for (int k = 0; k < kCopies; ++k) cnt[k * kRadix + t] = 0u;
  K kk[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    uint32_t i = base + (uint32_t)k * kSortThreads + t;
    kk[k] = i < n ? keys[i] : (K)0;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ITEMS; ++k)
    if (base + (uint32_t)k * kSortThreads + t < n)
      atomicAdd(&cnt[digit_of(kk[k], shift, mask) * kCopies + copy], 1u);
  __syncthreads();
  uint32_t v = 0u;
#pragma unroll
  for (int k = 0; k < kCopies; ++k) v += cnt[t * kCopies + k];
  counts[(size_t)t * tiles + blockIdx.x] = v;
}

// block d: counts[d * tiles + b] -> pairs before tile b's first pair of digit d
__global__ void __launch_bounds__(kSortThreads) k_radix_scan(const uint32_t* hist, uint32_t tiles,
                                                             uint32_t* counts) {
  __shared__ uint32_t ws[kWaves];
  const uint32_t d = blockIdx.x, t = threadIdx.x, lane = lane_id(), wave = t >> 6;
  // pairs of smaller digits
  uint32_t x = wave_incl_scan(t < d ? hist[t] : 0u);
  if (lane == 63) ws[wave] = x;
  __syncthreads();
  uint32_t running = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) running += ws[w];
  __syncthreads();
  uint32_t* row = counts + (size_t)d * tiles;
  for (uint32_t c = 0; c < tiles; c += kSortThreads * 4) {
    uint32_t j = c + 4 * t;
    uint32_t a[4], sum = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[q] = j + q < tiles ? row[j + q] : 0u;
      sum += a[q];
    }
    uint32_t incl = wave_incl_scan(sum);
    if (lane == 63) ws[wave] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      before += (uint32_t)w < wave ? ws[w] : 0u;
      total += ws[w];
    }
    uint32_t e = running + before + incl - sum;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (j + q < tiles) row[j + q] = e;
      e += a[q];
    }
    running += total;
    __syncthreads();
  }
}

// A tile of T * I pairs in registers -- wave w holds pairs [64 I w, 64 I (w + 1)),
// 64 at a time -- sorted by one digit into LDS.
template <typename K, int T, int I>
struct TileSort {
  static constexpr int kW = T / 64;
  K key[T * I];
  uint32_t val[T * I];
  uint32_t wc[kW][kRadix];  // per wave: pairs of a digit so far, then its offset in the digit
  uint32_t dstart[kRadix];  // first pair of a digit in the tile
  uint32_t ws[4];

  __device__ void sort(const K* kk, const uint32_t* vv, uint32_t count, int shift, uint32_t mask) {
    const uint32_t t = threadIdx.x, lane = lane_id(), wave = t >> 6;
    const uint64_t lt = (1ull << lane) - 1ull;
    for (uint32_t i = t; i < (uint32_t)kW * kRadix; i += T) (&wc[0][0])[i] = 0u;
    __syncthreads();
    uint32_t rank[I];
#pragma unroll
    for (int k = 0; k < I; ++k) {
      const bool valid = wave * 64u * I + (uint32_t)k * 64u + lane < count;
      const uint32_t d = valid ? digit_of(kk[k], shift, mask) : 0u;
      const uint64_t peers = peer_mask(d, valid);
      // the wave's own counters: its LDS operations complete in order
      const uint32_t pre = __hip_atomic_load(&wc[wave][d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      rank[k] = pre + (uint32_t)__popcll(peers & lt);
      if (valid && (uint32_t)__builtin_ctzll(peers) == lane)
        __hip_atomic_store(&wc[wave][d], pre + (uint32_t)__popcll(peers), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // thread d: each wave's offset within digit d, and the digit's first place
    uint32_t total = 0, incl = 0;
    if (t < (uint32_t)kRadix) {
#pragma unroll
      for (int w = 0; w < kW; ++w) {
        const uint32_t y = wc[w][t];
        wc[w][t] = total;
        total += y;
      }
      incl = wave_incl_scan(total);
      if (lane == 63) ws[wave] = incl;
    }
    __syncthreads();
    if (t < (uint32_t)kRadix) {
      uint32_t before = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) before += (uint32_t)w < wave ? ws[w] : 0u;
      dstart[t] = before + incl - total;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < I; ++k) {
      if (wave * 64u * I + (uint32_t)k * 64u + lane >= count) continue;
      const uint32_t d = digit_of(kk[k], shift, mask);
      const uint32_t p = dstart[d] + wc[wave][d] + rank[k];
      key[p] = kk[k];
      val[p] = vv[k];
    }
    __syncthreads();
  }
};

template <typename K, int T, int I>
__global__ void __launch_bounds__(T) k_radix_down(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout,
                                                  uint32_t n, int shift, uint32_t mask, uint32_t tiles,
                                                  const uint32_t* offs) {
  __shared__ TileSort<K, T, I> sh;
  __shared__ uint32_t goff[kRadix];
  const uint32_t t = threadIdx.x, lane = lane_id(), wave = t >> 6;
  const uint32_t base = blockIdx.x * (uint32_t)(T * I), count = min(n - base, (uint32_t)(T * I));
  K kk[I];
  uint32_t vv[I];
#pragma unroll
  for (int k = 0; k < I; ++k) {
    const uint32_t i = wave * 64u * I + (uint32_t)k * 64u + lane;
    kk[k] = i < count ? kin[base + i] : (K)0;
    vv[k] = i < count ? vin[base + i] : 0u;
  }
  if (t < (uint32_t)kRadix) goff[t] = offs[(size_t)t * tiles + blockIdx.x];
  sh.sort(kk, vv, count, shift, mask);
#pragma unroll
  for (int k = 0; k < I; ++k) {
    const uint32_t p = (uint32_t)k * T + t;
    if (p >= count) continue;
    const K key = sh.key[p];
    const uint32_t d = digit_of(key, shift, mask);
    const uint32_t pos = goff[d] + (p - sh.dstart[d]);
    kout[pos] = key;
    vout[pos] = sh.val[p];
  }
}

// every pass of at most kSmallTile pairs in one workgroup
template <typename K>
__global__ void __launch_bounds__(512) k_radix_small(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout,
                                                     uint32_t n, int end_bit) {
  constexpr int T = 512, I = (int)kSmallTile / T;
  __shared__ TileSort<K, T, I> sh;
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
  K kk[I];
  uint32_t vv[I];
#pragma unroll
  for (int k = 0; k < I; ++k) {
    const uint32_t i = wave * 64u * I + (uint32_t)k * 64u + lane;
    kk[k] = i < n ? kin[i] : (K)0;
    vv[k] = i < n ? vin[i] : 0u;
  }
  for (int shift = 0; shift < end_bit; shift += kDigitBits) {
    sh.sort(kk, vv, n, shift, (1u << min(kDigitBits, end_bit - shift)) - 1u);
#pragma unroll
    for (int k = 0; k < I; ++k) {
      const uint32_t i = wave * 64u * I + (uint32_t)k * 64u + lane;
      if (i < n) {
        kk[k] = sh.key[i];
        vv[k] = sh.val[i];
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < I; ++k) {
    const uint32_t i = wave * 64u * I + (uint32_t)k * 64u + lane;
    if (i < n) {
      kout[i] = kk[k];
      vout[i] = vv[k];
    }
  }
}

// Enough for every smaller n too, since callers keep one workspace for lists
// that shrink (the points left after duplicates).  The tiles do not grow with
// n: 768 little ones just below kBigFrom, 192 big ones from there.
template <typename K>
size_t temp_bytes_t(uint32_t n, int end_bit) {
  (void)end_bit;
  uint32_t tiles = std::max(1u, std::max(tiles_of(n), tiles_of(std::min(n, kBigFrom - 1u))));
  return align256((size_t)kMaxPasses * kRadix * 4) + align256((size_t)kRadix * tiles * 4) +
         align256((size_t)n * sizeof(K)) + align256((size_t)n * 4);
}

template <typename K>
hipError_t sort_t(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout, uint32_t n, int end_bit,
                  void* temp, size_t temp_bytes, hipStream_t s) {
  if (n == 0) return hipSuccess;
  end_bit = std::max(0, std::min(end_bit, (int)(8 * sizeof(K))));
  if (temp_bytes < temp_bytes_t<K>(n, end_bit) || !temp) return hipErrorInvalidValue;
  const int P = passes_of(end_bit);
  if (P == 0) {
    hipError_t e = hipMemcpyAsync(kout, kin, (size_t)n * sizeof(K), hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
    return hipMemcpyAsync(vout, vin, (size_t)n * 4, hipMemcpyDeviceToDevice, s);
  }
  if (n <= kSmallTile) {
    k_radix_small<K><<<1, 512, 0, s>>>(kin, vin, kout, vout, n, end_bit);
    return hipGetLastError();
  }
  const uint32_t tiles = tiles_of(n);
  const bool big = tile_of(n) == kBigTile;
  char* tp = static_cast<char*>(temp);
  uint32_t* hist = reinterpret_cast<uint32_t*>(tp);
  tp += align256((size_t)kMaxPasses * kRadix * 4);
  uint32_t* counts = reinterpret_cast<uint32_t*>(tp);
  tp += align256((size_t)kRadix * tiles * 4);
  K* kalt = reinterpret_cast<K*>(tp);
  tp += align256((size_t)n * sizeof(K));
  uint32_t* valt = reinterpret_cast<uint32_t*>(tp);
  k_radix_zero<<<(P * kRadix + 255) / 256, 256, 0, s>>>(hist, (uint32_t)(P * kRadix));
  // a block for 8,192 keys, 256 to 1,024 of them: the counters each one adds at
  // its end take time, and so do long loops of loads that wait.  256, 512 and
  // 1,024 blocks: 1M 63-bit keys 14, 19, 30 us, 4M 31, 27, 34, 20M 200, 121, 85;
  // 20M 12-bit keys 153, 88, 63.
  uint32_t hgrid = std::min((n + kSortThreads - 1) / kSortThreads, std::min(std::max(n / 8192u, 256u), 1024u));
  k_radix_hist<K><<<hgrid, kSortThreads, 0, s>>>(kin, n, end_bit, hist);
  const K* ksrc = kin;
  const uint32_t* vsrc = vin;
  for (int p = 0; p < P; ++p) {
    // the last pass writes the caller's output; earlier ones alternate
    bool to_out = ((P - 1 - p) & 1) == 0;
    K* kd = to_out ? kout : kalt;
    uint32_t* vd = to_out ? vout : valt;
    int shift = p * kDigitBits;
    int bits = std::min(kDigitBits, end_bit - shift);
    uint32_t mask = (1u << bits) - 1u;
    if (big) k_radix_up<K, kBigTile / kSortThreads><<<tiles, kSortThreads, 0, s>>>(ksrc, n, shift, mask, tiles, counts);
    else k_radix_up<K, kLittleTile / kSortThreads><<<tiles, kSortThreads, 0, s>>>(ksrc, n, shift, mask, tiles, counts);
    k_radix_scan<<<kRadix, kSortThreads, 0, s>>>(hist + p * kRadix, tiles, counts);
    if (big) k_radix_down<K, 512, kBigTile / 512><<<tiles, 512, 0, s>>>(ksrc, vsrc, kd, vd, n, shift, mask, tiles, counts);
    else k_radix_down<K, 256, kLittleTile / 256><<<tiles, 256, 0, s>>>(ksrc, vsrc, kd, vd, n, shift, mask, tiles, counts);
    ksrc = kd;
    vsrc = vd;
  }
  return hipGetLastError();
}

}  // namespace

size_t radix_temp_bytes_u64(uint32_t n, int end_bit) { return temp_bytes_t<uint64_t>(n, end_bit); }
size_t radix_temp_bytes_u32(uint32_t n, int end_bit) { return temp_bytes_t<uint32_t>(n, end_bit); }

hipError_t radix_sort_u64(const uint64_t* keys_in, const uint32_t* vals_in, uint64_t* keys_out,
                          uint32_t* vals_out, uint32_t n, int end_bit, void* temp, size_t temp_bytes,
                          hipStream_t s) {
  return sort_t<uint64_t>(keys_in, vals_in, keys_out, vals_out, n, end_bit, temp, temp_bytes, s);
}

hipError_t radix_sort_u32(const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                          uint32_t* vals_out, uint32_t n, int end_bit, void* temp, size_t temp_bytes,
                          hipStream_t s) {
  return sort_t<uint32_t>(keys_in, vals_in, keys_out, vals_out, n, end_bit, temp, temp_bytes, s);
}

}  // namespace wtet
