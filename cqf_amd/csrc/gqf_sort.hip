// gqf_sort.hip -- hash + LSD radix sort + run-length reduce for the bulk path.
//
// Replaces hash_all + thrust::sort + thrust::fill/reduce_by_key of the
// reference bulk API (src/gqf.cu:2615-2637, 3206-3209, 3258-3284).
//
// Sort: least-significant-digit radix sort over only the bits a hash can
// have (q + 8 of them; all 64 for pre-hashed keys), always an even number of
// passes so the result lands back in the caller's buffer, as the reference
// leaves `keys` holding the ascending hashes (src/gqf.cu:3180-3181).
// Each pass is upsweep (per-tile digit histogram in LDS) -> scan of the
// [digit][tile] matrix -> downsweep (stable rank with wave ballots, staged in
// LDS so each digit's keys leave the tile as one contiguous run).
// The first pass hashes on the fly.
#include <type_traits>

#include "gqf_internal.h"
#include "gqf_launch.h"

namespace {
constexpr int kThreads = 256;
constexpr int kItems = 16;
constexpr int kTile = kThreads * kItems;  // 4096 keys
constexpr int kItemsSmall = 4;            // tiles of 1024 keys for inputs up to kSmallN
constexpr uint64_t kSmallN = 1ULL << 16;
constexpr uint32_t kScanSmallTiles = 64;  // one-workgroup scan up to this many tiles
constexpr int kWaves = kThreads / 64;
constexpr int kMaxRadix = 1024;           // digits of up to 10 bits

// hash_it: 0 keys as they are; 1 hash under `mask`, then shift left by
// `vshift` (the filter's value bits); 2 pre-hashed keys shifted by vshift,
// a key above `mask` becoming ~0 (past every region, flagged there).
__device__ inline uint64_t load_key(const uint64_t* in, uint64_t i, uint64_t n, int hash_it, uint64_t mask,
                                    int vshift) {
  if (i >= n) return ~0ULL;
  uint64_t k = in[i];
  if (hash_it == 1) return gqf_hash64(k, mask) << vshift;
  if (hash_it == 2) return (k & ~mask) ? ~0ULL : (k << vshift);
  return k;
}
}  // namespace

// Where tile `tile`'s count of digit d lives: [digit][tile] rows for the
// many-tile scan (gqf_sort_scan_rows, one workgroup per row), [tile][digit]
// up to kScanSmallTiles tiles, where ONE workgroup scans everything and
// strided rows made every wave access touch 64 lines (15 us per scan).
__device__ inline uint64_t hist_at(uint32_t d, uint32_t tile, uint32_t ntiles, int radix) {
  return ntiles <= kScanSmallTiles ? (uint64_t)tile * (uint32_t)radix + d : (uint64_t)d * ntiles + tile;
}

// per-tile digit histogram -> hist[hist_at(d, tile)]
template <int ITEMS>
__device__ __forceinline__ void upsweep_body(const uint64_t* __restrict__ in, uint64_t n, int shift, int bits,
                                             int hash_it, uint64_t mask, int vshift, uint32_t* __restrict__ hist,
                                             uint32_t ntiles) {
  __shared__ uint32_t h[kMaxRadix];
  const int radix = 1 << bits;
  for (int d = threadIdx.x; d < radix; d += kThreads) h[d] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * (kThreads * ITEMS);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll 4
  for (int k = 0; k < ITEMS; k++) {
    uint64_t i = base + (uint64_t)w * (64 * ITEMS) + (uint64_t)k * 64 + lane;
    if (i < n) {
      uint64_t key = load_key(in, i, n, hash_it, mask, vshift);
      atomicAdd(&h[(uint32_t)(key >> shift) & (radix - 1)], 1u);
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < radix; d += kThreads) hist[hist_at(d, blockIdx.x, ntiles, radix)] = h[d];
}

extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_upsweep(const uint64_t* __restrict__ in, uint64_t n, int shift, int bits, int hash_it,
                 uint64_t mask, int vshift, uint32_t* __restrict__ hist, uint32_t ntiles) {
  upsweep_body<kItems>(in, n, shift, bits, hash_it, mask, vshift, hist, ntiles);
}

extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_upsweep_small(const uint64_t* __restrict__ in, uint64_t n, int shift, int bits, int hash_it,
                       uint64_t mask, int vshift, uint32_t* __restrict__ hist, uint32_t ntiles) {
  upsweep_body<kItemsSmall>(in, n, shift, bits, hash_it, mask, vshift, hist, ntiles);
}

// Exclusive scan of each digit's row of tile counts; row totals -> totals[d].
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_scan_rows(uint32_t* __restrict__ hist, uint32_t ntiles, uint32_t* __restrict__ totals) {
  __shared__ uint32_t wsum[kWaves];
  uint32_t* row = hist + (uint64_t)blockIdx.x * ntiles;
  uint32_t carry = 0;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (uint32_t base = 0; base < ntiles; base += kThreads) {
    uint32_t i = base + threadIdx.x;
    uint32_t v = i < ntiles ? row[i] : 0;
    uint32_t incl = wave_scan_add(v);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (int k = 0; k < kWaves; k++) {
      if (k < w) before += wsum[k];
      total += wsum[k];
    }
    if (i < ntiles) row[i] = carry + before + incl - v;
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Exclusive scan in place of count (<= 4 * kThreads) values in LDS by one
// workgroup: each thread takes four consecutive entries, the threads' sums
// are scanned by wave shuffles and across the four waves.
__device__ __forceinline__ void block_exclusive_scan(uint32_t* s, int count) {
  __shared__ uint32_t wsum[kWaves];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint32_t v[4];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int d = 4 * t + k;
    v[k] = d < count ? s[d] : 0;
    sum += v[k];
  }
  uint32_t incl = wave_scan_add(sum);
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  uint32_t run = incl - sum;
  for (int k = 0; k < w; k++) run += wsum[k];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const int d = 4 * t + k;
    if (d < count) s[d] = run;
    run += v[k];
  }
  __syncthreads();
}

// Exclusive scan of the digit totals (one workgroup, radix <= 1024).
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_scan_totals(uint32_t* __restrict__ totals, int radix) {
  __shared__ uint32_t s[kMaxRadix];
  for (int d = threadIdx.x; d < radix; d += kThreads) s[d] = totals[d];
  __syncthreads();
  block_exclusive_scan(s, radix);
  for (int d = threadIdx.x; d < radix; d += kThreads) totals[d] = s[d];
}

// Both scans for up to kScanSmallTiles tiles in one workgroup, over the
// [tile][digit] histogram: each digit's column of tile counts becomes its
// exclusive prefix (loads and stores coalesced across the digits' threads),
// and the digit totals their exclusive scan (as gqf_sort_scan_totals).
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_scan_small(uint32_t* __restrict__ hist, uint32_t ntiles, int radix, uint32_t* __restrict__ totals) {
  __shared__ uint32_t s[kMaxRadix];
  for (int d = threadIdx.x; d < radix; d += kThreads) {
    uint32_t v[kScanSmallTiles];
#pragma unroll
    for (uint32_t i = 0; i < kScanSmallTiles; i++) v[i] = i < ntiles ? hist[(uint64_t)i * radix + d] : 0u;
    uint32_t run = 0;
#pragma unroll
    for (uint32_t i = 0; i < kScanSmallTiles; i++) {
      if (i < ntiles) hist[(uint64_t)i * radix + d] = run;
      run += v[i];
    }
    s[d] = run;
  }
  __syncthreads();
  block_exclusive_scan(s, radix);
  for (int d = threadIdx.x; d < radix; d += kThreads) totals[d] = s[d];
}

// Stable scatter of one tile.
template <int ITEMS>
__device__ __forceinline__ void downsweep_body(const uint64_t* __restrict__ in, uint64_t* __restrict__ out,
                                               uint64_t n, int shift, int bits, int hash_it, uint64_t mask,
                                               int vshift, const uint32_t* __restrict__ hist,
                                               const uint32_t* __restrict__ bin_base, uint32_t ntiles) {
  constexpr int TILE = kThreads * ITEMS;
  static_assert(TILE < 65536, "per-wave digit counts are 16-bit");
  // 16-bit per-wave counts keep the kernel at 48 KB of LDS: three
  // workgroups per CU instead of two
  __shared__ uint16_t wcnt[kWaves][kMaxRadix];
  __shared__ uint32_t tile_start[kMaxRadix];
  __shared__ uint32_t glob[kMaxRadix];
  __shared__ uint64_t stage[TILE];
  const int radix = 1 << bits;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int d = threadIdx.x; d < radix; d += kThreads) {
#pragma unroll
    for (int k = 0; k < kWaves; k++) wcnt[k][d] = 0;
    glob[d] = bin_base[d] + hist[hist_at(d, blockIdx.x, ntiles, radix)];
  }
  __syncthreads();

  const uint64_t base = (uint64_t)blockIdx.x * TILE;
  const uint64_t lt_mask = lane ? (~0ULL >> (64 - lane)) : 0ULL;
  uint64_t keys[ITEMS];
  uint32_t rank[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    uint64_t i = base + (uint64_t)w * (64 * ITEMS) + (uint64_t)k * 64 + lane;
    bool valid = i < n;
    uint64_t key = load_key(in, i, n, hash_it, mask, vshift);
    uint32_t d = (uint32_t)(key >> shift) & (radix - 1);
    // lanes holding the same digit (and a valid key)
    uint64_t peers = __ballot(valid);
    for (int b = 0; b < bits; b++) {
      uint64_t m = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? m : ~m;
    }
    uint32_t before = wcnt[w][d];
    rank[k] = before + (uint32_t)__popcll(peers & lt_mask);
    keys[k] = key;
    // lowest peer bumps the wave's digit counter
    if (valid && (peers & lt_mask) == 0) wcnt[w][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
  }
  __syncthreads();
  // prefix over waves per digit, tile totals -> tile_start (exclusive over digits)
  for (int d = threadIdx.x; d < radix; d += kThreads) {
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < kWaves; k++) {
      uint32_t t = wcnt[k][d];
      wcnt[k][d] = (uint16_t)run;
      run += t;
    }
    tile_start[d] = run;  // tile count, scanned below
  }
  __syncthreads();
  block_exclusive_scan(tile_start, radix);  // all waves, 4 digits per thread
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    uint64_t i = base + (uint64_t)w * (64 * ITEMS) + (uint64_t)k * 64 + lane;
    if (i < n) {
      uint32_t d = (uint32_t)(keys[k] >> shift) & (radix - 1);
      stage[tile_start[d] + wcnt[w][d] + rank[k]] = keys[k];
    }
  }
  __syncthreads();
  const uint32_t cnt = (uint32_t)min((uint64_t)TILE, n - base);
  for (uint32_t i = threadIdx.x; i < cnt; i += kThreads) {
    uint64_t key = stage[i];
    uint32_t d = (uint32_t)(key >> shift) & (radix - 1);
    out[(uint64_t)glob[d] + (i - tile_start[d])] = key;
  }
}

extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_downsweep(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, int shift,
                   int bits, int hash_it, uint64_t mask, int vshift, const uint32_t* __restrict__ hist,
                   const uint32_t* __restrict__ bin_base, uint32_t ntiles) {
  downsweep_body<kItems>(in, out, n, shift, bits, hash_it, mask, vshift, hist, bin_base, ntiles);
}

extern "C" __global__ void __launch_bounds__(kThreads)
gqf_sort_downsweep_small(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, int shift,
                         int bits, int hash_it, uint64_t mask, int vshift, const uint32_t* __restrict__ hist,
                         const uint32_t* __restrict__ bin_base, uint32_t ntiles) {
  downsweep_body<kItemsSmall>(in, out, n, shift, bits, hash_it, mask, vshift, hist, bin_base, ntiles);
}

// ---------------------------------------------------------------------------
// Top-digit split of hashed keys for the two-level sort.  Only the bucket
// of each key matters here: the bucket sort then orders every bucket in
// full, and keys with equal hashes are equal values, so the split need not
// be stable.  That lets it use big tiles (kMRound keys per round, up to 8
// rounds per workgroup: a 2 MB [digit][tile] histogram at 2^24 keys instead
// of 16.8 MB of scattered counts) and rank keys within a round by LDS
// atomics; each round's keys leave the workgroup grouped by digit, about
// 64 bytes per digit at 1024 digits.

namespace {
constexpr int kMThreads = 1024;
constexpr int kMWaves = kMThreads / 64;
constexpr int kMItems = 8;
constexpr uint32_t kMRound = kMThreads * kMItems;  // 8192 keys, 64 KB staged
constexpr int kMItemsSmall = 2;                    // rounds of 2048 keys below kMSmallN: more, shorter tiles
constexpr uint64_t kMSmallN = 1ULL << 18;
constexpr int kMRankShift = 48;                    // ranks < kMRound ride above the hash bits
static_assert(kMRound <= (1u << (64 - kMRankShift)), "rank fits above the hash");
static_assert(kMaxRadix <= kMThreads, "one digit per thread");
// Up to this many tiles, each scatter workgroup adds up its digits' counts
// over the tiles before its own by itself ([tile][digit] histogram, read from
// L2); more go through gqf_sort_scan_rows ([digit][tile])
constexpr uint32_t kMScanTiles = 128;

// The sorts below order by (hash bits, request tag) for sequenced keys (tag
// above bit GQF_SEQ_SHIFT: sequence number, delete bit), which is the stable
// order: a request's sequence number grows with its position, and equal
// (hash, tag) are equal keys.  order_bits turns such a key's tag into 16 low
// bits, sequence number first.
__device__ __forceinline__ uint64_t seq_order(uint64_t hash_bits, uint64_t key) {
  const uint32_t tag = (uint32_t)(key >> GQF_SEQ_SHIFT);
  return hash_bits << 16 | ((tag << 1 | tag >> 15) & 0xFFFFu);
}
__device__ __forceinline__ uint64_t seq_tag_of(uint64_t order) {  // the tag in its place
  const uint32_t r = (uint32_t)order & 0xFFFFu;
  return (uint64_t)((r >> 1 | r << 15) & 0xFFFFu) << GQF_SEQ_SHIFT;
}
}  // namespace

// per-tile digit histogram of the hashed (kTagged: tagged) keys; workgroup 0
// also clears the region list counts
template <int ITEMS, bool kTagged>
__device__ __forceinline__ void msd_count_body(const uint64_t* __restrict__ in, uint64_t n, uint64_t tile_keys,
                                               int shift, int bits, uint64_t mask, int vshift,
                                               uint32_t* __restrict__ hist, uint32_t ntiles,
                                               uint32_t* __restrict__ list_count) {
  constexpr uint32_t kRound = kMThreads * ITEMS;
  __shared__ uint32_t h[kMaxRadix];
  const int radix = 1 << bits;
  const int t = threadIdx.x;
  if (t < radix) h[t] = 0;
  if (list_count && blockIdx.x == 0 && t < 2) list_count[t] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * tile_keys;
  const uint64_t end = min(n, base + tile_keys);
  for (uint64_t r0 = base; r0 < end; r0 += kRound) {
    uint64_t key[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) key[k] = in[min(r0 + (uint64_t)(k * kMThreads + t), end - 1)];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const uint64_t i = r0 + (uint64_t)(k * kMThreads + t);
      const uint64_t v = kTagged ? key[k] : gqf_hash64(key[k], mask) << vshift;
      if (i < end) atomicAdd(&h[(uint32_t)(v >> shift) & (radix - 1)], 1u);
    }
  }
  __syncthreads();
  if (t < radix)
    hist[ntiles <= kMScanTiles ? (uint64_t)blockIdx.x * (uint32_t)radix + (uint32_t)t : (uint64_t)t * ntiles + blockIdx.x] = h[t];
}

extern "C" __global__ void __launch_bounds__(kMThreads)
gqf_msd_count(const uint64_t* __restrict__ in, uint64_t n, uint64_t tile_keys, int shift, int bits, uint64_t mask,
              int vshift, uint32_t* __restrict__ hist, uint32_t ntiles, uint32_t* __restrict__ list_count) {
  msd_count_body<kMItems, false>(in, n, tile_keys, shift, bits, mask, vshift, hist, ntiles, list_count);
}
extern "C" __global__ void __launch_bounds__(kMThreads)
gqf_msd_count_small(const uint64_t* __restrict__ in, uint64_t n, uint64_t tile_keys, int shift, int bits, uint64_t mask,
                    int vshift, uint32_t* __restrict__ hist, uint32_t ntiles, uint32_t* __restrict__ list_count) {
  msd_count_body<kMItemsSmall, false>(in, n, tile_keys, shift, bits, mask, vshift, hist, ntiles, list_count);
}
extern "C" __global__ void __launch_bounds__(kMThreads)
gqf_msd_count_tagged(const uint64_t* __restrict__ in, uint64_t n, uint64_t tile_keys, int shift, int bits, uint64_t mask,
                     int vshift, uint32_t* __restrict__ hist, uint32_t ntiles, uint32_t* __restrict__ list_count) {
  msd_count_body<kMItemsSmall, true>(in, n, tile_keys, shift, bits, mask, vshift, hist, ntiles, list_count);
}

// scatter of one tile into the digit buckets.  hist: the counts of
// gqf_msd_count, or, above kMScanTiles tiles, its rows scanned per digit, with
// the digit totals in `totals`.  starts[d] (written by workgroup 0) = first
// index of digit d's keys.
template <int ITEMS, bool kTagged>
__device__ __forceinline__ void msd_scatter_body(const uint64_t* __restrict__ in, uint64_t* __restrict__ out,
                                                 uint64_t n, uint64_t tile_keys, int shift, int bits, uint64_t mask,
                                                 int vshift, const uint32_t* __restrict__ hist,
                                                 const uint32_t* __restrict__ totals, uint32_t* __restrict__ starts,
                                                 uint32_t ntiles) {
  constexpr uint32_t kRound = kMThreads * ITEMS;
  __shared__ uint64_t stage[kRound];
  __shared__ uint32_t cnt[kMaxRadix];     // keys of the round per digit
  __shared__ uint32_t lstart[kMaxRadix];  // their first index in stage
  __shared__ uint32_t glob[kMaxRadix];    // next output index of each digit
  __shared__ uint32_t wsum[kMWaves];
  const int radix = 1 << bits;
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  // exclusive scan over the digits, one digit per thread (threads past the
  // radix bring 0)
  auto scan_digits = [&](uint32_t c) -> uint32_t {
    const uint32_t incl = wave_scan_add(c);
    __syncthreads();
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t before = incl - c;
    for (int k = 0; k < w; k++) before += wsum[k];
    return before;
  };
  {
    uint32_t mine = 0, total = 0;  // digit t: keys in earlier tiles, in all
    if (ntiles <= kMScanTiles) {
      // the threads split into kMThreads / radix groups, each adding up every
      // so-many-th tile
      if (t < radix) cnt[t] = lstart[t] = 0;
      __syncthreads();
      const int d = t & (radix - 1), groups = kMThreads >> bits;
      for (uint32_t i = (uint32_t)(t >> bits); i < ntiles; i += (uint32_t)groups) {
        const uint32_t c = hist[(uint64_t)i * (uint32_t)radix + (uint32_t)d];
        total += c;
        mine += i < blockIdx.x ? c : 0u;
      }
      if (groups > 1) {
        atomicAdd(&cnt[d], mine);
        atomicAdd(&lstart[d], total);
        __syncthreads();
        mine = t < radix ? cnt[t] : 0u;
        total = t < radix ? lstart[t] : 0u;
      }
    } else if (t < radix) {
      mine = hist[(uint64_t)t * ntiles + blockIdx.x];
      total = totals[t];
    }
    const uint32_t start = scan_digits(t < radix ? total : 0u);
    if (t < radix) {
      glob[t] = start + mine;
      if (blockIdx.x == 0) starts[t] = start;
    }
  }
  const uint64_t base = (uint64_t)blockIdx.x * tile_keys;
  const uint64_t end = min(n, base + tile_keys);
  for (uint64_t r0 = base; r0 < end; r0 += kRound) {
    // 32-bit offsets from the round's (uniform) base: one VGPR per address
    const uint64_t* __restrict__ src = in + r0;
    const uint32_t m = (uint32_t)min((uint64_t)kRound, end - r0);
    if (t < radix) cnt[t] = 0;
    __syncthreads();
    // each key's rank within its digit rides in bits 48.. of the key (the
    // hashes here are below 2^42), which keeps the kernel within 64 VGPRs;
    // tagged keys keep theirs beside them
    uint64_t key[ITEMS];
    uint32_t rank[kTagged ? ITEMS : 1];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) key[k] = src[min((uint32_t)(k * kMThreads + t), m - 1)];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const uint32_t i = (uint32_t)(k * kMThreads + t);
      const uint64_t h = kTagged ? key[k] : gqf_hash64(key[k], mask) << vshift;
      const uint32_t r = i < m ? atomicAdd(&cnt[(uint32_t)(h >> shift) & (radix - 1)], 1u) : 0u;
      if (kTagged) rank[k] = r;
      else key[k] = h | ((uint64_t)r << kMRankShift);
    }
    __syncthreads();
    const uint32_t c = t < radix ? cnt[t] : 0u;
    const uint32_t first = scan_digits(c);
    if (t < radix) lstart[t] = first;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const uint32_t i = (uint32_t)(k * kMThreads + t);
      const uint64_t h = kTagged ? key[k] : key[k] & ((1ULL << kMRankShift) - 1);
      const uint32_t r = kTagged ? rank[k] : (uint32_t)(key[k] >> kMRankShift);
      if (i < m) stage[lstart[(uint32_t)(h >> shift) & (radix - 1)] + r] = h;
    }
    __syncthreads();
    for (uint32_t i = t; i < m; i += kMThreads) {
      const uint64_t v = stage[i];
      const uint32_t d = (uint32_t)(v >> shift) & (radix - 1);
      out[(uint64_t)glob[d] + (i - lstart[d])] = v;
    }
    __syncthreads();
    if (t < radix) glob[t] += c;
  }
}

extern "C" __global__ void __launch_bounds__(kMThreads, 8)
gqf_msd_scatter(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, uint64_t tile_keys,
                int shift, int bits, uint64_t mask, int vshift, const uint32_t* __restrict__ hist,
                const uint32_t* __restrict__ totals, uint32_t* __restrict__ starts, uint32_t ntiles) {
  msd_scatter_body<kMItems, false>(in, out, n, tile_keys, shift, bits, mask, vshift, hist, totals, starts, ntiles);
}
extern "C" __global__ void __launch_bounds__(kMThreads, 8)
gqf_msd_scatter_small(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, uint64_t tile_keys,
                      int shift, int bits, uint64_t mask, int vshift, const uint32_t* __restrict__ hist,
                      const uint32_t* __restrict__ totals, uint32_t* __restrict__ starts, uint32_t ntiles) {
  msd_scatter_body<kMItemsSmall, false>(in, out, n, tile_keys, shift, bits, mask, vshift, hist, totals, starts, ntiles);
}
extern "C" __global__ void __launch_bounds__(kMThreads, 8)
gqf_msd_scatter_tagged(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, uint64_t tile_keys,
                       int shift, int bits, uint64_t mask, int vshift, const uint32_t* __restrict__ hist,
                       const uint32_t* __restrict__ totals, uint32_t* __restrict__ starts, uint32_t ntiles) {
  msd_scatter_body<kMItemsSmall, true>(in, out, n, tile_keys, shift, bits, mask, vshift, hist, totals, starts, ntiles);
}

// ---------------------------------------------------------------------------
// Two-level sort of hashed or tagged keys (batches of up to 2^24): the top-digit
// split above (gqf_msd_count / gqf_msd_scatter) puts the keys into 2^msd
// buckets by their top `msd` hash bits; then one workgroup per bucket sorts the bucket's remaining
// low bits (at most 32) in LDS -- up to kBucketCap keys as 32-bit values in
// two 68 KB buffers of gfx950's 160 KB -- with stable 8-bit LSD passes whose
// ranks come from wave ballots over peers of equal digit, as in the
// downsweep.  The bucket's top bits are its index, so the low bits order it.
// A bucket larger than kBucketCap (heavily repeated keys) runs the same
// passes over its 64-bit keys in global memory.

namespace {
constexpr int kBThreads = 1024;
constexpr int kBWaves = kBThreads / 64;
constexpr int kBItems = 8;                           // keys per lane per round
constexpr uint32_t kBRound = kBThreads * kBItems;    // 8192
constexpr uint32_t kBucketCap = 17408;               // 2^24 keys in 1024 buckets: mean 16384, sd 128
constexpr int kBMaxPasses = 7;

struct PassSmem {
  uint32_t wcnt[kBWaves][256];        // per wave digit counts, then positions
  uint32_t run[256];                  // next free position of each digit
};
struct BucketSmem {
  alignas(16) uint32_t buf[2][kBucketCap];
  uint32_t tot[kBMaxPasses][256];     // digit totals of every pass
  PassSmem pass;
};

// Stable scatter of src[0, m) into dst by digit (v >> sh) & 255, given the
// digit totals; every thread of the workgroup calls it.
template <typename V>
__device__ __forceinline__ void bucket_pass(const V* src, V* dst, uint32_t m, int sh, const uint32_t* tot,
                                            PassSmem& sm) {
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  if (w == 0) {  // exclusive scan of the totals, 4 digits per lane
    uint32_t v[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      v[k] = tot[4 * lane + k];
      sum += v[k];
    }
    uint32_t incl = wave_scan_add(sum);
    uint32_t r = incl - sum;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      sm.run[4 * lane + k] = r;
      r += v[k];
    }
  }
  __syncthreads();
  const uint64_t lt = lane ? (~0ULL >> (64 - lane)) : 0ULL;
  for (uint32_t base = 0; base < m; base += kBRound) {
    for (int d = lane; d < 256; d += 64) sm.wcnt[w][d] = 0;
    V keys[kBItems];
    uint32_t rank[kBItems];
#pragma unroll
    for (int k = 0; k < kBItems; k++) {
      const uint32_t i = base + (uint32_t)(w * 64 * kBItems + k * 64 + lane);
      const bool valid = i < m;
      const V key = valid ? src[i] : (V)0;
      const uint32_t d = (uint32_t)(key >> sh) & 255u;
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (int b = 0; b < 8; b++) {
        const uint64_t mb = __ballot((d >> b) & 1u);
        peers &= ((d >> b) & 1u) ? mb : ~mb;
      }
      const uint32_t before = sm.wcnt[w][d];
      rank[k] = before + (uint32_t)__popcll(peers & lt);
      keys[k] = key;
      if (valid && (peers & lt) == 0) sm.wcnt[w][d] = before + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    if (t < 256) {  // wave counts -> positions, in wave order
      uint32_t r = sm.run[t];
#pragma unroll
      for (int k = 0; k < kBWaves; k++) {
        const uint32_t x = sm.wcnt[k][t];
        sm.wcnt[k][t] = r;
        r += x;
      }
      sm.run[t] = r;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kBItems; k++) {
      const uint32_t i = base + (uint32_t)(w * 64 * kBItems + k * 64 + lane);
      if (i < m) dst[sm.wcnt[w][(uint32_t)(keys[k] >> sh) & 255u] + rank[k]] = keys[k];
    }
  }
}

// A bitonic network of `size` (a power of two) places: order(a, c, up) puts
// places a < c into ascending order if up, else descending.  Every thread of the
// workgroup calls it.
template <typename F>
__device__ __forceinline__ void lds_network(uint32_t size, F order) {
  for (uint32_t k = 2; k <= size; k *= 2) {
    for (uint32_t j = k / 2; j > 0; j /= 2) {
      for (uint32_t i = threadIdx.x; i < size / 2; i += kBThreads) {
        const uint32_t a = 2 * i - (i & (j - 1));  // the i-th pair at distance j
        order(a, a + j, (a & k) == 0);
      }
      __syncthreads();
    }
  }
}

// Sorts the m values of a by their low 8 * passes bits, between the LDS
// buffers a and b, and returns the one that holds the result; tot: `passes`
// rows of digit totals.  A digit that all values share takes no pass (few
// distinct keys, and of the request tags few bits, is what it is called for).
// Every thread of the workgroup calls it, with a complete (a barrier passed).
// Latency bound: buckets of 2,400 sequenced keys on 100 hashes 37 us, where a
// table of their distinct (hash, request) pairs took 285.
template <typename V>
__device__ __forceinline__ V* lds_sort(V* a, V* b, uint32_t m, int passes, uint32_t (*tot)[256], PassSmem& sm) {
  for (int k = threadIdx.x; k < passes * 256; k += kBThreads) (&tot[0][0])[k] = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63;
  for (uint32_t i0 = 0; i0 < m; i0 += kBThreads) {
    const uint32_t i = i0 + threadIdx.x;
    const V v = a[min(i, m - 1)];
    for (int p = 0; p < passes; p++) {
      // the wave's first digit once for all lanes that have it
      const uint32_t d = (uint32_t)(v >> (8 * p)) & 255u;
      const uint64_t same = __ballot(i < m && d == (uint32_t)__builtin_amdgcn_readfirstlane((int)d));
      if (i < m && (lane == 0 || !((same >> lane) & 1)))
        atomicAdd(&tot[p][d], lane == 0 ? (uint32_t)__popcll(same) : 1u);
    }
  }
  __syncthreads();
  const V any = a[0];
  for (int p = 0; p < passes; p++) {
    if (tot[p][(uint32_t)(any >> (8 * p)) & 255u] == m) continue;  // uniform
    bucket_pass<V>(a, b, m, 8 * p, tot[p], sm);
    __syncthreads();
    V* t = a;
    a = b;
    b = t;
  }
  return a;
}

}  // namespace

// start[r] of the regions whose bounds lie in bucket b's hash range
// [b << low_bits, (b + 1) << low_bits): the bucket's first index s plus
// below(bound - bucket base), the number of its keys whose low bits are
// below that; the last bucket's workgroup also writes n at the bounds at or
// past range and at r = nregions
template <typename F>
__device__ __forceinline__ void bucket_region_starts(const gqf_region_args& ra, uint32_t b, uint32_t nbuckets,
                                                     int low_bits, uint64_t s, uint64_t n, F below) {
  if (!ra.start) return;
  const uint64_t lo = (uint64_t)b << low_bits;
  const uint64_t hi = lo + (1ULL << low_bits);
  const uint64_t r0 = (lo + ra.step - 1) / ra.step;
  uint64_t r1 = (hi + ra.step - 1) / ra.step;
  if (r1 > ra.nregions) r1 = ra.nregions;
  for (uint64_t r = r0 + threadIdx.x; r < r1; r += blockDim.x) {
    const uint64_t bound = r * ra.step;
    if (bound < ra.range) ra.start[r] = (uint32_t)(s + below((uint32_t)(bound - lo)));
  }
  if (b + 1 == nbuckets)
    for (uint64_t r = (ra.range + ra.step - 1) / ra.step + threadIdx.x; r <= ra.nregions; r += blockDim.x)
      ra.start[r] = (uint32_t)n;
}

// Common case, two workgroups per CU: the bucket's keys stay in registers
// (17 per thread) while they are counted by sub-bucket -- the top (up to) 11
// of the low bits, ~8 keys each for uniform hashes -- then go to one LDS
// buffer in sub-bucket order (any order within), and each key's place in
// its sub-bucket is the number of keys there below it (ties by buffer
// index), so every key is written straight to its sorted position.  A
// bucket above kBucketCap keys, or with a sub-bucket above kSubCap
// (repeated keys), is flagged for gqf_sort_buckets_slow.
constexpr int kSubBitsMax = 11;
constexpr uint32_t kSubMax = 1u << kSubBitsMax;
constexpr uint32_t kSubCap = 64;
static_assert(kSubMax == 2 * kBThreads, "two sub-buckets per thread in the scan");

// A key as the bucket sort orders it: the bucket's low bits, for tagged keys
// with the 16 tag bits below them (8-byte values: kBucketCapTagged of them)
constexpr uint32_t kBucketCapTagged = 8192;

template <bool kTagged>
struct BucketKey {
  using V = std::conditional_t<kTagged, uint64_t, uint32_t>;
  static constexpr uint32_t kCap = kTagged ? kBucketCapTagged : kBucketCap;
  static constexpr int kLoad = (int)((kCap + kBThreads - 1) / kBThreads);
  static constexpr int kExtra = kTagged ? 16 : 0;  // bits below the hash's
  static __device__ __forceinline__ V of(uint64_t key, uint64_t hi) {
    if constexpr (kTagged) return seq_order((key & GQF_SEQ_HASH_MASK) - hi, key);
    else return (uint32_t)(key - hi);
  }
  static __device__ __forceinline__ uint64_t key(V v, uint64_t hi) {
    if constexpr (kTagged) return hi | v >> 16 | seq_tag_of(v);
    else return hi | v;
  }
  // `of` in two steps, the load by itself first (of an untagged key, its low
  // word: the bucket's low bits are its low bits)
  static __device__ __forceinline__ V load(const uint64_t* __restrict__ in, uint32_t i) {
    if constexpr (kTagged) return in[i];
    else return ((const uint32_t*)in)[2 * (size_t)i];
  }
  static __device__ __forceinline__ V loaded(V x, uint64_t hi, int low_bits) {
    if constexpr (kTagged) return of(x, hi);
    else return x & (0xFFFFFFFFu >> (32 - low_bits));
  }
  static __device__ __forceinline__ V bound(uint32_t x) { return (V)x << kExtra; }  // first value at low bits x
};

// Eight waves per SIMD (two workgroups a CU) need at most 80 SGPRs as well as
// 64 VGPRs: with 82 one workgroup was resident, and 2^24 keys took 104 us in
// place of 79 (hence the second launch bound).
template <bool kTagged>
__device__ __forceinline__ void sort_bucket(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n,
                                            int low_bits, const uint32_t* __restrict__ starts, uint32_t nbuckets,
                                            uint32_t* __restrict__ slow, const gqf_region_args& ra, uint64_t tag) {
  using K = BucketKey<kTagged>;
  using V = typename K::V;
  __shared__ V buf[K::kCap];
  __shared__ uint32_t sub_end[kSubMax];  // counts, then cursors: after the scatter, each sub-bucket's end
  __shared__ uint32_t wsum[kBWaves];
  __shared__ uint32_t oversize;
  const uint32_t b = blockIdx.x;
  const uint64_t s = starts[b];
  const uint64_t e = b + 1 < nbuckets ? (uint64_t)starts[b + 1] : n;
  if (e <= s) {
    bucket_region_starts(ra, b, nbuckets, low_bits, s, n, [](uint32_t) { return 0u; });
    return;
  }
  const uint32_t m = (uint32_t)(e - s);
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  if (m > K::kCap) {
    if (t == 0) slow[b] = 1;
    return;
  }
  const uint64_t hi = (uint64_t)b << low_bits;  // the bucket's top bits
  const int db = low_bits < kSubBitsMax ? low_bits : kSubBitsMax;
  const int sb = low_bits - db + K::kExtra;
  const uint32_t nsub = 1u << db;
  for (uint32_t d = t; d < nsub; d += kBThreads) sub_end[d] = 0;
  if (t == 0) oversize = 0;
  // clamped indexes: every load is in flight before the first is used
  V v[K::kLoad];
#pragma unroll
  for (int k = 0; k < K::kLoad; k++) v[k] = K::load(in + s, min((uint32_t)(k * kBThreads + t), m - 1));
#pragma unroll
  for (int k = 0; k < K::kLoad; k++) v[k] = K::loaded(v[k], hi, low_bits);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K::kLoad; k++)
    if ((uint32_t)(k * kBThreads + t) < m) atomicAdd(&sub_end[(uint32_t)(v[k] >> sb)], 1u);
  __syncthreads();
  {  // exclusive scan of the counts, two sub-buckets per thread
    const uint32_t d0 = 2 * (uint32_t)t;
    const uint32_t c0 = d0 < nsub ? sub_end[d0] : 0u;
    const uint32_t c1 = d0 + 1 < nsub ? sub_end[d0 + 1] : 0u;
    const uint32_t sum = c0 + c1;
    uint32_t incl = wave_scan_add(sum);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
    for (int k = 0; k < w; k++) run += wsum[k];
    if (d0 < nsub) sub_end[d0] = run;
    if (d0 + 1 < nsub) sub_end[d0 + 1] = run + c0;
    if (c0 > kSubCap || c1 > kSubCap) oversize = 1;
  }
  __syncthreads();
  if (oversize) {
    if (t == 0) slow[b] = 1;
    return;
  }
#pragma unroll
  for (int k = 0; k < K::kLoad; k++)
    if ((uint32_t)(k * kBThreads + t) < m) buf[atomicAdd(&sub_end[(uint32_t)(v[k] >> sb)], 1u)] = v[k];
  __syncthreads();
  for (uint32_t i = t; i < m; i += kBThreads) {
    const V x = buf[i];
    const uint32_t d = (uint32_t)(x >> sb);
    const uint32_t st = d ? sub_end[d - 1] : 0u;
    const uint32_t en = sub_end[d];
    uint32_t r = 0;
    for (uint32_t j = st; j < en; j++) {
      const V y = buf[j];
      r += (y < x || (y == x && j < i)) ? 1u : 0u;
    }
    out[s + st + r] = tag | K::key(x, hi);
  }
  bucket_region_starts(ra, b, nbuckets, low_bits, s, n, [&](uint32_t x) {
    const V v0 = K::bound(x);
    const uint32_t d = (uint32_t)(v0 >> sb);
    const uint32_t st = d ? sub_end[d - 1] : 0u, en = sub_end[d];
    uint32_t c = st;
    for (uint32_t j = st; j < en; j++) c += buf[j] < v0 ? 1u : 0u;
    return c;
  });
}

extern "C" __global__ void __launch_bounds__(kBThreads, 8)
gqf_sort_buckets(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, int low_bits,
                 const uint32_t* __restrict__ starts, uint32_t nbuckets, uint32_t* __restrict__ slow,
                 gqf_region_args ra, uint64_t tag) {
  sort_bucket<false>(in, out, n, low_bits, starts, nbuckets, slow, ra, tag);
}
extern "C" __global__ void __launch_bounds__(kBThreads, 8)
gqf_sort_buckets_tagged(const uint64_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n, int low_bits,
                        const uint32_t* __restrict__ starts, uint32_t nbuckets, uint32_t* __restrict__ slow,
                        gqf_region_args ra) {
  sort_bucket<true>(in, out, n, low_bits, starts, nbuckets, slow, ra, 0);
}

// A bucket that repeats few keys (at most kTableMax distinct ones, however
// many times each): its distinct values are counted in an LDS hash table, the
// table's entries are packed and sorted, and every value is written as often as
// it came.  Returns false, with nothing written, if there are more.
// Latency bound (a workgroup by itself): eight keys a thread are in flight, the
// network sorts no more than the distinct values need, and values with many
// copies are listed as they are met: buckets of 17,400 keys, 2,000 of them
// distinct, 114 us; with one key in flight, a network over the whole table and a
// second look at every value for the many copies 314 us, and the passes between
// global buffers 100 us at 17,400 keys but longer with every repeat.
constexpr uint32_t kTableCap = 8192;
constexpr uint32_t kTableMax = 6144;
constexpr uint32_t kTableMany = 4096;  // copies that the whole workgroup writes
constexpr uint32_t kManyList = 64;
struct BucketTable {
  uint64_t val[kTableCap];  // ~0: free
  uint32_t cnt[kTableCap];  // then the values' first output indexes
  uint32_t wsum[kBWaves];
  uint32_t many[kManyList];
  uint32_t used, n_many;
};
static_assert(sizeof(BucketTable) <= sizeof(BucketSmem), "shares the passes' LDS");

template <bool kTagged>
__device__ __forceinline__ bool sort_by_table(const uint64_t* in, uint64_t* out, uint64_t s, uint64_t n, uint32_t m,
                                              int low_bits, uint32_t b, uint32_t nbuckets, BucketTable& tb,
                                              const gqf_region_args& ra, uint64_t tag) {
  using K = BucketKey<kTagged>;
  const uint32_t t = threadIdx.x, w = t >> 6, lane = t & 63;
  const uint64_t hi = (uint64_t)b << low_bits;
  for (uint32_t i = t; i < kTableCap; i += kBThreads) {
    tb.val[i] = ~0ULL;
    tb.cnt[i] = 0;
  }
  if (t == 0) tb.used = tb.n_many = 0;
  __syncthreads();
  auto count = [&](uint64_t v, bool left) {
    // a wave's repeats of one value are added together (two values' worth,
    // the rest one by one)
    uint32_t add = left ? 1u : 0u;
    uint64_t open = __ballot(left);
#pragma unroll
    for (int k = 0; k < 2; k++) {
      if (!open) break;
      const int first = __builtin_ctzll(open);
      const uint64_t lead = __shfl(v, first, 64);
      const uint64_t same = __ballot(((open >> lane) & 1) && v == lead);
      if ((same >> lane) & 1) add = lane == (uint32_t)first ? (uint32_t)__popcll(same) : 0u;
      open &= ~same;
    }
    if (add) {
      uint32_t at = (uint32_t)((v * 0x9E3779B97F4A7C15ULL) >> 51);
      for (uint32_t k = 0; k < kTableCap; k++) {
        const uint64_t old = atomicCAS((unsigned long long*)&tb.val[at], ~0ULL, (unsigned long long)v);
        if (old == ~0ULL) atomicAdd(&tb.used, 1u);
        if (old == ~0ULL || old == v) {
          atomicAdd(&tb.cnt[at], add);
          break;
        }
        if (*(volatile uint32_t*)&tb.used > kTableMax) break;
        at = (at + 1) & (kTableCap - 1);
      }
    }
  };
  for (uint32_t i0 = 0; i0 < m; i0 += kBThreads * kBItems) {
    if (*(volatile uint32_t*)&tb.used > kTableMax) break;  // checked again below
    uint64_t v[kBItems];
#pragma unroll
    for (int k = 0; k < kBItems; k++) v[k] = in[s + min(i0 + (uint32_t)k * kBThreads + t, m - 1)];
#pragma unroll
    for (int k = 0; k < kBItems; k++)
      if (i0 + (uint32_t)k * kBThreads < m) count((uint64_t)K::of(v[k], hi), i0 + (uint32_t)k * kBThreads + t < m);
  }
  __syncthreads();
  if (tb.used > kTableMax) return false;
  // the entries to the front, then a bitonic network over them (~0 behind them)
  const uint32_t used = tb.used;
  constexpr int kE = kTableCap / kBThreads;  // entries of a thread
  {
    uint64_t val[kE];
    uint32_t cnt[kE], mine = 0;
#pragma unroll
    for (int k = 0; k < kE; k++) {
      val[k] = tb.val[k * kBThreads + t];
      cnt[k] = tb.cnt[k * kBThreads + t];
      mine += val[k] != ~0ULL ? 1u : 0u;
    }
    const uint32_t incl = wave_scan_add(mine);
    if (lane == 63) tb.wsum[w] = incl;
    __syncthreads();  // every entry is read
    uint32_t at = incl - mine;
    for (uint32_t k = 0; k < w; k++) at += tb.wsum[k];
#pragma unroll
    for (int k = 0; k < kE; k++) {
      if (val[k] == ~0ULL) continue;
      tb.val[at] = val[k];
      tb.cnt[at] = cnt[k];
      at++;
    }
  }
  uint32_t size = 2;
  while (size < used) size *= 2;
  for (uint32_t i = used + t; i < size; i += kBThreads) {
    tb.val[i] = ~0ULL;
    tb.cnt[i] = 0;
  }
  __syncthreads();
  lds_network(size, [&](uint32_t a, uint32_t c, bool up) {
    const uint64_t x = tb.val[a], y = tb.val[c];
    if ((x > y) == up) {
      tb.val[a] = y;
      tb.val[c] = x;
      const uint32_t z = tb.cnt[a];
      tb.cnt[a] = tb.cnt[c];
      tb.cnt[c] = z;
    }
  });
  // counts -> first indexes, eight entries a thread
  uint32_t c[kE], sum = 0;
#pragma unroll
  for (int k = 0; k < kE; k++) {
    const uint32_t e = kE * t + (uint32_t)k;
    c[k] = e < used ? tb.cnt[e] : 0u;
    sum += c[k];
  }
  const uint32_t incl = wave_scan_add(sum);
  if (lane == 63) tb.wsum[w] = incl;
  __syncthreads();
  uint32_t run = incl - sum;
  for (uint32_t k = 0; k < w; k++) run += tb.wsum[k];
#pragma unroll
  for (int k = 0; k < kE; k++) {
    if (kE * t + (uint32_t)k < used) tb.cnt[kE * t + (uint32_t)k] = run;
    run += c[k];
  }
  __syncthreads();
  auto begin = [&](uint32_t e) { return e < used ? tb.cnt[e] : m; };
  // a value's copies: a wave each, or, for many, the workgroup (a listed value;
  // more than the list holds stay with their waves)
  for (uint32_t e = w; e < used; e += kBWaves) {
    const uint32_t a = begin(e), z = begin(e + 1);
    if (z - a >= kTableMany) {
      uint32_t k = 0;
      if (lane == 0) k = atomicAdd(&tb.n_many, 1u);
      k = (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
      if (k < kManyList) {
        if (lane == 0) tb.many[k] = e;
        continue;
      }
    }
    const uint64_t key = tag | K::key((typename K::V)tb.val[e], hi);
    for (uint32_t i = a + lane; i < z; i += 64) out[s + i] = key;
  }
  __syncthreads();
  for (uint32_t k = 0; k < min(tb.n_many, kManyList); k++) {
    const uint32_t e = tb.many[k], a = begin(e), z = begin(e + 1);
    const uint64_t key = tag | K::key((typename K::V)tb.val[e], hi);
    for (uint32_t i = a + t; i < z; i += kBThreads) out[s + i] = key;
  }
  bucket_region_starts(ra, b, nbuckets, low_bits, s, n, [&](uint32_t x) {
    uint32_t lo = 0, up = used;  // first value at or above the bound
    while (lo < up) {
      const uint32_t mid = (lo + up) >> 1;
      if (tb.val[mid] < (uint64_t)K::bound(x)) lo = mid + 1; else up = mid;
    }
    return begin(lo);
  });
  return true;
}

template <bool kTagged>
__device__ __forceinline__ void sort_flagged_bucket(uint64_t* in, uint64_t* out, uint64_t n, int low_bits,
                                                 const uint32_t* __restrict__ starts, uint32_t nbuckets,
                                                 uint32_t* __restrict__ slow, uint32_t b, BucketSmem& sm,
                                                 const gqf_region_args& ra, uint64_t tag) {
  using K = BucketKey<kTagged>;
  const uint64_t s = starts[b];
  const uint64_t e = b + 1 < nbuckets ? (uint64_t)starts[b + 1] : n;
  const uint32_t m = (uint32_t)(e - s);
  const uint64_t hi = (uint64_t)b << low_bits;
  const int t = threadIdx.x;
  const int passes = (low_bits + K::kExtra + 7) / 8;
  __syncthreads();  // every thread has read the flag
  if (t == 0) slow[b] = 0;
  if (m <= K::kCap) {
    using V = typename K::V;
    V* const first = (V*)sm.buf[0];
    for (uint32_t i = t; i < m; i += kBThreads) first[i] = K::of(in[s + i], hi);
    __syncthreads();
    const V* sorted = lds_sort<V>(first, (V*)sm.buf[1], m, passes, sm.tot, sm.pass);
    for (uint32_t i = t; i < m; i += kBThreads) out[s + i] = tag | K::key(sorted[i], hi);
    bucket_region_starts(ra, b, nbuckets, low_bits, s, n, [&](uint32_t x) {
      uint32_t lo = 0, hi2 = m;
      while (lo < hi2) {
        const uint32_t mid = (lo + hi2) >> 1;
        if (sorted[mid] < K::bound(x)) lo = mid + 1; else hi2 = mid;
      }
      return lo;
    });
    return;
  }
  if (sort_by_table<kTagged>(in, out, s, n, m, low_bits, b, nbuckets, *(BucketTable*)&sm, ra, tag)) return;
  __syncthreads();
  for (int k = t; k < kBMaxPasses * 256; k += kBThreads) (&sm.tot[0][0])[k] = 0;
  __syncthreads();
  // too large for LDS: the same passes, over the keys as they are ordered,
  // between the bucket's ranges of in and out, plus a pass on a zero digit when
  // the count is even, so the result lands in out; other waves' stores are
  // published between passes with agent-scope fences around the barrier
  const int gpasses = passes | 1;
  uint64_t* a = in + s;
  uint64_t* o = out + s;
  for (uint32_t i = t; i < m; i += kBThreads) {
    const uint64_t v = K::of(a[i], hi);
    a[i] = v;
    for (int p = 0; p < gpasses; p++) atomicAdd(&sm.tot[p][(uint32_t)(v >> (8 * p)) & 255u], 1u);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  for (int p = 0; p < gpasses; p++) {
    bucket_pass<uint64_t>(p & 1 ? o : a, p & 1 ? a : o, m, 8 * p, sm.tot[p], sm.pass);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  bucket_region_starts(ra, b, nbuckets, low_bits, s, n, [&](uint32_t x) {
    uint32_t lo = 0, hi2 = m;
    while (lo < hi2) {
      const uint32_t mid = (lo + hi2) >> 1;
      if (o[mid] < (uint64_t)K::bound(x)) lo = mid + 1; else hi2 = mid;
    }
    return lo;
  });
  __syncthreads();  // the searches above read o as ordered
  for (uint32_t i = t; i < m; i += kBThreads) o[i] = tag | K::key((typename K::V)o[i], hi);
}

// The flagged buckets (skips the others, and clears the flags it takes):
// stable 8-bit passes over the bucket's low bits in two LDS buffers, or, for
// a bucket that they have no room for, its distinct keys by a table, or, for
// more of those, the passes over its 64-bit keys between its ranges of in and
// out in global memory.  A grid of at most one workgroup per CU strides over
// the buckets, so an all-clear call costs one short launch.
extern "C" __global__ void __launch_bounds__(kBThreads)
gqf_sort_buckets_slow(uint64_t* in, uint64_t* out, uint64_t n, int low_bits, const uint32_t* __restrict__ starts,
                      uint32_t nbuckets, uint32_t* __restrict__ slow, gqf_region_args ra, uint64_t tag) {
  __shared__ BucketSmem sm;
  for (uint32_t b = blockIdx.x; b < nbuckets; b += gridDim.x) {
    if (slow[b]) sort_flagged_bucket<false>(in, out, n, low_bits, starts, nbuckets, slow, b, sm, ra, tag);
    __syncthreads();
  }
}
extern "C" __global__ void __launch_bounds__(kBThreads)
gqf_sort_buckets_slow_tagged(uint64_t* in, uint64_t* out, uint64_t n, int low_bits, const uint32_t* __restrict__ starts,
                             uint32_t nbuckets, uint32_t* __restrict__ slow, gqf_region_args ra) {
  __shared__ BucketSmem sm;
  for (uint32_t b = blockIdx.x; b < nbuckets; b += gridDim.x) {
    if (slow[b]) sort_flagged_bucket<true>(in, out, n, low_bits, starts, nbuckets, slow, b, sm, ra, 0);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// One-workgroup sort of up to kTinyCap keys (hashed here, or tagged), which
// also lists their regions: a batch of a few thousand keys is then one launch
// instead of a dozen.  As the bucket sort: the keys are counted by their top
// (up to) 12 bits, put into sub-bucket order in LDS, and each one's place is
// its rank among the keys of its sub-bucket (two on average at 8192 uniform
// keys).  A sub-bucket above kSubCap keys (repeats) makes the workgroup sort all
// of them by digits instead (lds_sort), or, up to kTNetwork keys, by a bitonic
// network: a whole delete of 300 / 1,000 / 2,000 keys that repeat a few, 30 / 37 /
// 47 us by the network and 43 / 48 / 53 by digits; a reduce of 8,192 equal keys,
// 135 and 85.  Latency bound: 12 us for 5000 keys, against 63 us for the four
// passes (12 launches) of the LSD sort plus 9 for the region bounds.

namespace {
constexpr int kTThreads = 1024;
constexpr uint32_t kTinyCap = GQF_SORT_TINY;
constexpr int kTLoad = kTinyCap / kTThreads;
constexpr int kTSubBits = 12;
constexpr uint32_t kTSub = 1u << kTSubBits;
constexpr uint32_t kTNetwork = 2048;
constexpr int kTPasses = (42 + 16 + 7) / 8;  // of the widest tagged keys (gqf_sort_fast_fits)
static_assert(kTSub == 4 * kTThreads, "four sub-buckets per thread in the scan");
static_assert(kTThreads == kBThreads, "lds_sort's workgroup");
}  // namespace

template <bool kTagged>
__device__ __forceinline__ void sort_tiny(uint64_t* __restrict__ keys, uint32_t n, uint64_t mask, int vshift, int bits,
                                          const gqf_list_args& la) {
  __shared__ uint64_t buf[kTinyCap];
  __shared__ uint64_t sorted[kTinyCap];
  __shared__ union {
    uint32_t sub_end[kTSub];
    PassSmem pass;  // the digit passes come after the sub-buckets
  } u;
  __shared__ uint32_t tot[kTPasses][256];
  __shared__ uint32_t wsum[kTThreads / 64];
  uint32_t* const sub_end = u.sub_end;
  __shared__ uint32_t oversize, nlist[2];
  const uint32_t t = threadIdx.x, w = t >> 6, lane = t & 63;
  // tagged keys as seq_order has them: hash bits above 16 tag bits
  const int all = bits + (kTagged ? 16 : 0);
  const int sb = bits > kTSubBits ? all - kTSubBits : all - bits;
  uint64_t v[kTLoad];
#pragma unroll
  for (int k = 0; k < kTLoad; k++) v[k] = keys[min((uint32_t)k * kTThreads + t, n - 1)];
#pragma unroll
  for (int k = 0; k < 4; k++) sub_end[(uint32_t)k * kTThreads + t] = 0;
  if (t == 0) oversize = nlist[0] = nlist[1] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTLoad; k++) {
    const uint32_t i = (uint32_t)k * kTThreads + t;
    v[k] = kTagged ? seq_order(v[k] & GQF_SEQ_HASH_MASK, v[k]) : gqf_hash64(v[k], mask) << vshift;
    if (i < n) atomicAdd(&sub_end[(uint32_t)(v[k] >> sb)], 1u);
  }
  __syncthreads();
  {
    uint32_t c[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      c[k] = sub_end[4 * t + k];
      sum += c[k];
      if (c[k] > kSubCap) oversize = 1;
    }
    const uint32_t incl = wave_scan_add(sum);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
    for (uint32_t k = 0; k < w; k++) run += wsum[k];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      sub_end[4 * t + k] = run;
      run += c[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTLoad; k++)
    if ((uint32_t)k * kTThreads + t < n) buf[atomicAdd(&sub_end[(uint32_t)(v[k] >> sb)], 1u)] = v[k];
  const uint64_t* res = sorted;
  __syncthreads();
  if (oversize) {
    if (n <= kTNetwork) {
      uint32_t size = 2;
      while (size < n) size *= 2;
      for (uint32_t i = n + t; i < size; i += kTThreads) buf[i] = ~0ULL;
      __syncthreads();
      lds_network(size, [&](uint32_t a, uint32_t c, bool up) {
        const uint64_t x = buf[a], y = buf[c];
        if ((x > y) == up) {
          buf[a] = y;
          buf[c] = x;
        }
      });
      res = buf;
    } else {
      res = lds_sort<uint64_t>(buf, sorted, n, (all + 7) / 8, tot, u.pass);
    }
  } else {
    for (uint32_t i = t; i < n; i += kTThreads) {
      const uint64_t x = buf[i];
      const uint32_t d = (uint32_t)(x >> sb);
      const uint32_t st = d ? sub_end[d - 1] : 0u, en = sub_end[d];
      uint32_t r = st;
      for (uint32_t j = st; j < en; j++) {
        const uint64_t y = buf[j];
        r += (y < x || (y == x && j < i)) ? 1u : 0u;
      }
      sorted[r] = x;
    }
    __syncthreads();
  }
  constexpr int kExtra = kTagged ? 16 : 0;
  for (uint32_t i0 = 0; i0 < n; i0 += kTThreads) {
    const uint32_t i = i0 + t;
    const bool in = i < n;
    const uint64_t x = in ? res[i] : 0;
    if (in) keys[i] = kTagged ? (x >> 16 | seq_tag_of(x)) : x;
    if (!la.list) continue;
    // a key that opens its region lists it; it also ends the region of the
    // key before it
    const uint32_t r = (uint32_t)(x >> (kExtra + 14)) / la.region_blocks;
    const uint32_t before = in && i ? (uint32_t)(res[i - 1] >> (kExtra + 14)) / la.region_blocks : 0u;
    const bool head = in && (i == 0 || r != before);
#pragma unroll
    for (uint32_t par = 0; par < 2; par++) {
      const uint64_t hm = __ballot(head && (r & 1u) == par);
      if (!hm) continue;
      uint32_t at = 0;
      if (lane == 0) at = atomicAdd(&nlist[par], (uint32_t)__popcll(hm));
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
      if (head && (r & 1u) == par)
        la.list[par * la.stride + at + (uint32_t)__popcll(hm & ((1ULL << lane) - 1))] = r;
    }
    if (head) {
      la.start[r] = i;
      if (i) la.start[before + 1] = i;
    }
    if (in && i + 1 == n) la.start[r + 1] = n;
  }
  if (la.list) {
    __syncthreads();
    if (t < 2) la.count[t] = nlist[t];
  }
}

extern "C" __global__ void __launch_bounds__(kTThreads)
gqf_sort_tiny(uint64_t* __restrict__ keys, uint32_t n, uint64_t mask, int vshift, int bits, gqf_list_args la) {
  sort_tiny<false>(keys, n, mask, vshift, bits, la);
}
extern "C" __global__ void __launch_bounds__(kTThreads)
gqf_sort_tiny_tagged(uint64_t* __restrict__ keys, uint32_t n, int bits, gqf_list_args la) {
  sort_tiny<true>(keys, n, 0, 0, bits, la);
}

// The regions of n sorted keys, listed by the keys that open them (as
// gqf_sort_tiny lists them; counts cleared before): start[r] and start[r + 1]
// are written for the listed regions only.
extern "C" __global__ void __launch_bounds__(kTThreads)
gqf_region_heads(const uint64_t* __restrict__ keys, uint32_t n, uint64_t hmask, gqf_list_args la) {
  __shared__ uint32_t cnt[2], base[2];
  const uint32_t t = threadIdx.x, lane = t & 63;
  const uint32_t i = blockIdx.x * kTThreads + t;
  const bool in = i < n;
  const uint32_t r = in ? (uint32_t)((keys[i] & hmask) >> 14) / la.region_blocks : 0u;
  const uint32_t before = in && i ? (uint32_t)((keys[i - 1] & hmask) >> 14) / la.region_blocks : 0u;
  const bool head = in && (i == 0 || r != before);
  if (t < 2) cnt[t] = 0;
  __syncthreads();
  uint32_t at = 0;
#pragma unroll
  for (uint32_t par = 0; par < 2; par++) {
    const uint64_t hm = __ballot(head && (r & 1u) == par);
    uint32_t a = 0;
    if (lane == 0 && hm) a = atomicAdd(&cnt[par], (uint32_t)__popcll(hm));
    a = (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
    if (head && (r & 1u) == par) at = a + (uint32_t)__popcll(hm & ((1ULL << lane) - 1));
  }
  __syncthreads();
  if (t < 2) base[t] = cnt[t] ? atomicAdd(&la.count[t], cnt[t]) : 0u;
  __syncthreads();
  if (head) {
    la.list[(r & 1u) * la.stride + base[r & 1u] + at] = r;
    la.start[r] = i;
    if (i) la.start[before + 1] = i;
  }
  if (in && i + 1 == n) la.start[r + 1] = n;
}

// ---------------------------------------------------------------------------
// run-length reduce of sorted keys: unique keys + their multiplicities

extern "C" __global__ void __launch_bounds__(kThreads)
gqf_rle_count(const uint64_t* __restrict__ keys, uint64_t n, uint32_t* __restrict__ tile_heads) {
  __shared__ uint32_t c;
  if (threadIdx.x == 0) c = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * kTile;
  uint32_t mine = 0;
  for (int k = 0; k < kItems; k++) {
    uint64_t i = base + (uint64_t)k * kThreads + threadIdx.x;
    if (i < n && (i == 0 || keys[i] != keys[i - 1])) mine++;
  }
  atomicAdd(&c, mine);
  __syncthreads();
  if (threadIdx.x == 0) tile_heads[blockIdx.x] = c;
}

// exclusive scan of tile head counts (one workgroup); total -> *m
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_rle_scan(uint32_t* __restrict__ tile_heads, uint32_t ntiles, uint64_t* __restrict__ m) {
  __shared__ uint32_t wsum[kWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t carry = 0;
  for (uint32_t base = 0; base < ntiles; base += kThreads) {
    uint32_t i = base + threadIdx.x;
    uint32_t v = i < ntiles ? tile_heads[i] : 0;
    uint32_t incl = wave_scan_add(v);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (int k = 0; k < kWaves; k++) {
      if (k < w) before += wsum[k];
      total += wsum[k];
    }
    if (i < ntiles) tile_heads[i] = carry + before + incl - v;
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) *m = carry;
}

// write unique keys and the index where each run starts
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_rle_emit(const uint64_t* __restrict__ keys, uint64_t n, const uint32_t* __restrict__ tile_base,
             uint64_t* __restrict__ ukeys, uint64_t* __restrict__ upos) {
  __shared__ uint32_t wsum[kWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t base = (uint64_t)blockIdx.x * kTile;
  uint32_t carry = tile_base[blockIdx.x];
  const uint64_t lt_mask = lane ? (~0ULL >> (64 - lane)) : 0ULL;
  for (int k = 0; k < kItems; k++) {
    uint64_t i = base + (uint64_t)k * kThreads + threadIdx.x;
    bool head = i < n && (i == 0 || keys[i] != keys[i - 1]);
    uint64_t b = __ballot(head);
    if (lane == 0) wsum[w] = (uint32_t)__popcll(b);
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (int q = 0; q < kWaves; q++) {
      if (q < w) before += wsum[q];
      total += wsum[q];
    }
    if (head) {
      uint32_t u = carry + before + (uint32_t)__popcll(b & lt_mask);
      ukeys[u] = keys[i];
      upos[u] = i;
    }
    carry += total;
    __syncthreads();
  }
}

// counts[u] = next run start - this run start
extern "C" __global__ void gqf_rle_counts(const uint64_t* __restrict__ upos, const uint64_t* __restrict__ m,
                                          uint64_t n, uint64_t* __restrict__ counts) {
  uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint64_t mm = *m;
  if (u >= mm) return;
  uint64_t next = u + 1 < mm ? upos[u + 1] : n;
  counts[u] = next - upos[u];
}

// ---------------------------------------------------------------------------
// launchers

static inline uint32_t sort_ntiles(uint64_t n) { return (uint32_t)((n + kTile - 1) / kTile); }

// sized for the larger of the 4096-key tiling and the small-input tilings
uint64_t gqf_sort_hist_words(uint64_t n) {
  const uint64_t t = sort_ntiles(n);
  static_assert(kMScanTiles >= kScanSmallTiles, "the larger of the small tilings");
  return (uint64_t)kMaxRadix * (t > kMScanTiles ? t : kMScanTiles);
}

namespace {
// radix digit and number of passes for `bits` key bits; an even number of
// passes leaves the result in `keys`
void sort_shape(int bits, int digit_bits, int* passes, int* digit) {
  if (digit_bits >= 6 && digit_bits <= 10) {
    *digit = digit_bits;
    *passes = (bits + digit_bits - 1) / digit_bits;
    *passes += *passes & 1;
  } else if (bits <= 40) {
    *passes = 4;
    *digit = (bits + 3) / 4;
    if (*digit < 6) *digit = 6;
  } else {
    *passes = 8;
    *digit = 8;
  }
}
}  // namespace

void gqf_launch_sort(uint64_t* keys, uint64_t* tmp, uint64_t n, int hash_it, uint64_t mask, int vshift, int bits,
                     int digit_bits, uint32_t* hist, uint32_t* totals, hipStream_t s) {
  if (n == 0) return;
  int passes, digit;
  sort_shape(bits, digit_bits, &passes, &digit);
  // small inputs: 1024-key tiles (more workgroups, shorter tiles)
  const bool small = n <= kSmallN;
  const uint32_t tile = small ? kThreads * kItemsSmall : kTile;
  const uint32_t ntiles = (uint32_t)((n + tile - 1) / tile);
  const int radix = 1 << digit;
  uint64_t* in = keys;
  uint64_t* out = tmp;
  for (int p = 0; p < passes; p++) {
    const int shift = p * digit;
    const int h = p == 0 ? hash_it : 0;
    gqf_prof_begin("sort_pass", s);
    hipLaunchKernelGGL(small ? gqf_sort_upsweep_small : gqf_sort_upsweep, dim3(ntiles), dim3(kThreads), 0, s, in, n,
                       shift, digit, h, mask, vshift, hist, ntiles);
    if (ntiles <= kScanSmallTiles) {
      hipLaunchKernelGGL(gqf_sort_scan_small, dim3(1), dim3(kThreads), 0, s, hist, ntiles, radix, totals);
    } else {
      hipLaunchKernelGGL(gqf_sort_scan_rows, dim3(radix), dim3(kThreads), 0, s, hist, ntiles, totals);
      hipLaunchKernelGGL(gqf_sort_scan_totals, dim3(1), dim3(kThreads), 0, s, totals, radix);
    }
    hipLaunchKernelGGL(small ? gqf_sort_downsweep_small : gqf_sort_downsweep, dim3(ntiles), dim3(kThreads), 0, s,
                       (const uint64_t*)in, out, n, shift, digit, h, mask, vshift, (const uint32_t*)hist,
                       (const uint32_t*)totals, ntiles);
    gqf_prof_end("sort_pass", s);
    uint64_t* t = in;
    in = out;
    out = t;
  }
}

bool gqf_sort_fast_fits(uint64_t n, int bits, bool tagged) {
  if (n <= kTinyCap) return bits <= 42;
  return n <= (tagged ? 1ULL << 22 : 1ULL << 24) && bits >= 18 && bits <= 42;  // 1024 buckets of 4K / 16K keys
}

void gqf_launch_sort_fast(uint64_t* keys, uint64_t* tmp, uint64_t n, bool tagged, uint64_t mask, int vshift, int bits,
                          uint32_t* hist, uint32_t* totals, uint32_t* slow, hipStream_t s,
                          const gqf_region_args* regions, const gqf_list_args* lists, uint64_t tag) {
  if (n == 0) return;
  const gqf_list_args la = lists ? *lists : gqf_list_args{};
  const gqf_region_args ra = regions ? *regions : gqf_region_args{};
  if (n <= kTinyCap && !tag && !regions) {
    gqf_prof_begin("sort_pass", s);
    if (tagged)
      hipLaunchKernelGGL(gqf_sort_tiny_tagged, dim3(1), dim3(kTThreads), 0, s, keys, (uint32_t)n, bits, la);
    else
      hipLaunchKernelGGL(gqf_sort_tiny, dim3(1), dim3(kTThreads), 0, s, keys, (uint32_t)n, mask, vshift, bits, la);
    gqf_prof_end("sort_pass", s);
    return;
  }
  // 2^msd buckets (at most 1024), low bits <= 32: of about 12K keys, or 4K
  // below 2^20 keys (more workgroups) and for tagged ones (8 bytes in LDS)
  const uint64_t want = tagged || n < (1ULL << 20) ? 4096 : 12288;
  int msd = 2;
  while (msd < 10 && (n >> msd) > want) msd++;
  if (bits - msd > 32) msd = bits - 32;
  const int radix = 1 << msd;
  const uint32_t* starts = totals + kMaxRadix;
  // tiles of one short round below kMSmallN keys; above, about 512 tiles of
  // 1..8 rounds: 32K keys per tile at 2^24 keys.  The histogram (radix x
  // ntiles <= 1024 x n / 8192 words, or 128 x 128) fits the LSD sort's
  // (gqf_sort_hist_words)
  const bool small = tagged || n < kMSmallN;
  const uint64_t round = (uint64_t)kMThreads * (small ? kMItemsSmall : kMItems);
  uint64_t rounds = n / (round * 512);
  rounds = rounds < 1 ? 1 : (rounds > 8 ? 8 : rounds);
  if (small && n > round * kMScanTiles) rounds = (n + round * kMScanTiles - 1) / (round * kMScanTiles);
  const uint64_t tile_keys = rounds * round;
  const uint32_t ntiles = (uint32_t)((n + tile_keys - 1) / tile_keys);
  gqf_prof_begin("sort_pass", s);
  hipLaunchKernelGGL(tagged ? gqf_msd_count_tagged : (small ? gqf_msd_count_small : gqf_msd_count), dim3(ntiles),
                     dim3(kMThreads), 0, s, (const uint64_t*)keys, n, tile_keys, bits - msd, msd, mask, vshift, hist,
                     ntiles, la.count);
  if (ntiles > kMScanTiles)
    hipLaunchKernelGGL(gqf_sort_scan_rows, dim3(radix), dim3(kThreads), 0, s, hist, ntiles, totals);
  hipLaunchKernelGGL(tagged ? gqf_msd_scatter_tagged : (small ? gqf_msd_scatter_small : gqf_msd_scatter), dim3(ntiles),
                     dim3(kMThreads), 0, s, (const uint64_t*)keys, tmp, n, tile_keys, bits - msd, msd, mask, vshift,
                     (const uint32_t*)hist, (const uint32_t*)totals, totals + kMaxRadix, ntiles);
  gqf_prof_end("sort_pass", s);
  gqf_prof_begin("sort_buckets", s);
  const dim3 gslow(radix < 256 ? radix : 256);
  if (tagged) {
    hipLaunchKernelGGL(gqf_sort_buckets_tagged, dim3(radix), dim3(kBThreads), 0, s, (const uint64_t*)tmp, keys, n,
                       bits - msd, starts, (uint32_t)radix, slow, ra);
    hipLaunchKernelGGL(gqf_sort_buckets_slow_tagged, gslow, dim3(kBThreads), 0, s, tmp, keys, n, bits - msd, starts,
                       (uint32_t)radix, slow, ra);
  } else {
    hipLaunchKernelGGL(gqf_sort_buckets, dim3(radix), dim3(kBThreads), 0, s, (const uint64_t*)tmp, keys, n, bits - msd,
                       starts, (uint32_t)radix, slow, ra, tag);
    hipLaunchKernelGGL(gqf_sort_buckets_slow, gslow, dim3(kBThreads), 0, s, tmp, keys, n, bits - msd, starts,
                       (uint32_t)radix, slow, ra, tag);
  }
  gqf_prof_end("sort_buckets", s);
  if (la.list) {
    gqf_prof_begin("region_bounds", s);
    hipLaunchKernelGGL(gqf_region_heads, dim3((uint32_t)((n + kTThreads - 1) / kTThreads)), dim3(kTThreads), 0, s,
                       (const uint64_t*)keys, (uint32_t)n, tagged ? GQF_SEQ_HASH_MASK : ~0ULL, la);
    gqf_prof_end("region_bounds", s);
  }
}

void gqf_launch_rle(const uint64_t* keys, uint64_t n, uint32_t* tile_heads, uint64_t* ukeys, uint64_t* upos,
                    uint64_t* ucounts, uint64_t* m_dev, hipStream_t s) {
  if (n == 0) return;
  const uint32_t ntiles = sort_ntiles(n);
  hipLaunchKernelGGL(gqf_rle_count, dim3(ntiles), dim3(kThreads), 0, s, keys, n, tile_heads);
  hipLaunchKernelGGL(gqf_rle_scan, dim3(1), dim3(kThreads), 0, s, tile_heads, ntiles, m_dev);
  hipLaunchKernelGGL(gqf_rle_emit, dim3(ntiles), dim3(kThreads), 0, s, keys, n, (const uint32_t*)tile_heads, ukeys,
                     upos);
  const uint32_t g = (uint32_t)((n + 255) / 256);
  hipLaunchKernelGGL(gqf_rle_counts, dim3(g), dim3(256), 0, s, (const uint64_t*)upos, (const uint64_t*)m_dev, n,
                     ucounts);
}
