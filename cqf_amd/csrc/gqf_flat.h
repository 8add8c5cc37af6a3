// gqf_flat.h -- merge-rebuild of one region by a whole workgroup, a lane on a
// few slots, items or entries (internal; included by gqf_rebuild.hip).
//
// The single-wave rebuild (gqf_rebuild.hip) gives each block one lane, which
// walks the block's runs: right for a few items per block, but a batch that
// brings more items than the region cache holds makes every lane merge ~38
// runs one after another, twice, reading its items from global memory.
// Here the region is taken as a sorted sequence of entries (hash, count):
//
//   1. every counter of the old window becomes an entry: each thread holds
//      eight slots; a slot's quotient is the k-th occupied one of the window, k =
//      run ends before the slot (a popcount, and a table of the occupied
//      quotients by rank).  In a run whose bytes ascend, but for pairs of
//      equal ones, every byte is a counter of 1 and every pair one of 2; the
//      lane at the start of any other run marks its counter starts first;
//   2. every distinct item hash finds its place among the old entries of its
//      quotient's run; an entry that is there takes the new count, the others
//      get a place among them (a bit map of the merged sequence);
//   3. with L(e) slots per entry and S(e) the slots of the entries before it,
//      entry e starts at S(e) + max over e' <= e of (quotient(e') - S(e')):
//      each entry starts at its quotient or behind its predecessor, whichever
//      is later (the two agree inside a run), so a sum scan and a max scan
//      place every entry;
//   4. the counters are written to their slots in LDS, each run's first slot
//      marked, which gives run ends and used slots; occupied quotients and
//      block ends are collected on the way.
//
// The result is the same canonical image as the single-wave rebuild's.
//
// Bound by instruction issue, vector and LDS (9,900 VALU, 6,400 SALU and 950
// LDS instructions for a region of a served batch); 54 KB of LDS keep three
// workgroups, 24 waves, on a CU.  The serial walk it replaces in dense
// batches, per launch: 943,718 keys into an empty table of 2^20 slots 268 ->
// 20 us; 14.1 M items into a table of 2^25 slots in four chunks 214 -> 55 us a
// chunk on average; a served batch at 2^24 slots, 42 items a region, 114 ->
// 83 us.  On regions with few entries the other forms are ahead (counted items
// into a nearly empty table of 2^26 slots: 69 us by the walk, 184 here), hence
// dense_line.
// Decoding every counter of two slots, in code repeated for each of a
// thread's slots, took 94 us for the served batch and 62 us a chunk.
// One lane per slot with a scan per 64 slots took 294 us where the eight
// consecutive slots or entries a thread takes here, scanned once, take 213.
#pragma once

#include "gqf_internal.h"
#include "gqf_launch.h"

namespace gqf_flat {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kWin = 64;                 // window blocks: the region and its push blocks
constexpr int kSlots = kWin * 64;
constexpr int kPer = kSlots / kThreads;  // slots per thread
static_assert(kPer == 8, "a thread's slots are one 8-byte word of its block");
constexpr int kItems = 3968;             // items of a region held as entries (with more, three workgroups would not fit a CU)
constexpr int kBig = 64;                 // counts of kAuxBig or more in a window
constexpr uint32_t kAuxBig = 4095;       // a larger count is in the big table
constexpr int32_t kNone = INT32_MIN / 4;

enum Kind : int { kAdd = 0, kCounts = 1, kTagged = 2 };
enum Result : int { kOk = 0, kNeedWide = 1, kNoSpace = 2 };

struct Head {
  uint64_t occ[kWin];       // old header words
  uint64_t run[kWin];
  uint64_t used[kWin];
  uint64_t own[kWin];       // used slots of this window's quotients (the earlier regions' cleared)
  uint64_t cont[kWin];      // own slots that continue the run of the slot before
  uint64_t start[kWin + 1]; // own slots at which a counter starts (+ 1: none past the window)
  uint64_t multi[kWin];     // first slots of runs that hold counters of more than one slot
  uint64_t occ_new[kWin];
  uint64_t run_new[kWin];
  uint64_t used_new[kWin];
  uint32_t rbase[kWin];     // own run ends / occupied quotients / entries before block j
  uint32_t obase[kWin];
  uint32_t ebase[kWin];
  int32_t xold[kWin];       // end of the runs of quotients < 64 j, at least 64 j - 1
  int32_t xnew[kWin];
  int32_t xblk[kWin];       // last slot of the new runs of block j's quotients
  uint32_t wsum[2][kWaves];
  int32_t wmax[2][kWaves];
  uint32_t n_old, n_slots, any_multi, n_big, over;
  int32_t xend, bstar, bwrite, keep, result;
  uint32_t big_hash[kBig];
  uint64_t big_count[kBig];
};

constexpr int kSeqWords = (kSlots + kItems + 31) / 32;

struct Smem : Head {
  alignas(16) uint8_t sin[kSlots];  // old slots
  uint32_t old[kSlots];             // old entries, hash << 12 | min(count, kAuxBig)
  union {
    uint16_t rend[kSlots];          // old entries of the runs of rank <= k
    alignas(16) uint16_t out[kSlots + 8];  // the new slots, once the items have their places
  };
  union {
    uint16_t quot[kSlots];          // the occupied quotients by rank (until the entries are made)
    uint32_t item[kItems];          // the items' entries
  };
  uint32_t is_item[kSeqWords];      // places of the merged sequence that items take
  uint32_t items_before[kSeqWords]; // items in earlier words of it
};

__device__ __forceinline__ int32_t max_i(int32_t a, int32_t b) { return a > b ? a : b; }

// inclusive maximum over the lanes of a wave, on the DPP steps of wave_scan_add
__device__ __forceinline__ int32_t wave_scan_max(int32_t x) {
  x = max_i(x, __builtin_amdgcn_update_dpp(kNone, x, 0x111, 0xf, 0xf, false));
  x = max_i(x, __builtin_amdgcn_update_dpp(kNone, x, 0x112, 0xf, 0xf, false));
  x = max_i(x, __builtin_amdgcn_update_dpp(kNone, x, 0x114, 0xf, 0xf, false));
  x = max_i(x, __builtin_amdgcn_update_dpp(kNone, x, 0x118, 0xf, 0xf, false));
  x = max_i(x, __builtin_amdgcn_update_dpp(kNone, x, 0x142, 0xa, 0xf, false));
  x = max_i(x, __builtin_amdgcn_update_dpp(kNone, x, 0x143, 0xc, 0xf, false));
  return x;
}
__device__ __forceinline__ int32_t below_i(int32_t x, int32_t fill) {  // the value of the lane below
  return __builtin_amdgcn_update_dpp(fill, x, 0x138, 0xf, 0xf, false);
}
__device__ __forceinline__ uint64_t below_u64(uint64_t x) {  // the same, 0 into lane 0
  return (uint64_t)(uint32_t)below_i((int32_t)(uint32_t)x, 0) |
         (uint64_t)(uint32_t)below_i((int32_t)(uint32_t)(x >> 32), 0) << 32;
}

// slots of the counter (rem, count): gqf_counter_len in 32 bits, for the
// counts an entry holds itself
__device__ __forceinline__ uint32_t entry_len(uint32_t rem, uint32_t count) {
  if (count <= 3) return count;
  if (rem == 0) return count - 4 < 255u ? 4u : 5u;
  const uint32_t v = count - 3;
  uint32_t d = (v < 254u ? v : v / 254u) + 1;  // top digit; two digits reach kAuxBig
  if (d >= rem) d++;
  return (v < 254u ? 3u : 4u) + (d >= rem ? 1u : 0u);
}

// the last slot of the run that holds own slot p (the window's last slot if it ends past the window)
__device__ __forceinline__ int32_t run_end_of(const Head& sm, int32_t p, int nwin) {
  int b = p >> 6;
  uint64_t w = sm.run[b] & (~0ULL << (p & 63));
  while (!w) {
    if (++b >= nwin) return 64 * nwin - 1;
    w = sm.run[b];
  }
  return 64 * b + __builtin_ctzll(w);
}

__device__ __forceinline__ uint32_t push_count(Head& sm, uint32_t h, uint64_t c) {
  if (c < kAuxBig) return (uint32_t)c;
  const uint32_t k = atomicAdd(&sm.n_big, 1u);
  if (k < (uint32_t)kBig) {
    sm.big_hash[k] = h;
    sm.big_count[k] = c;
  } else {
    sm.over = 1;  // more of them than the table holds: the wide pass takes the region
  }
  return kAuxBig;
}
// the count of hash h (entry count `aux`) among the first n big ones
__device__ __forceinline__ uint64_t full_count(const Head& sm, uint32_t h, uint32_t aux, uint32_t n) {
  if (aux < kAuxBig) return aux;
  for (uint32_t k = 0; k < n && k < (uint32_t)kBig; k++)
    if (sm.big_hash[k] == h) return sm.big_count[k];
  return kAuxBig;
}

// What a thread keeps of its window: the eight slots 8 t .. 8 t + 7 (eight
// threads a block), and, in wave 0, block `lane`'s old offset; the end x0 of the
// earlier blocks' runs; the entries.
struct Window {
  uint2 slots;
  uint32_t off;
  int32_t x0;
  bool any;     // some run of the window's quotients
  uint32_t n;   // entries
  uint64_t sum; // !kStore: the counts of the entries in the thread's slots
};

// 1. Loads the window of nwin blocks from block B0 and makes the entries of
// its runs, in order, in sm.old; sm.rend[k] = entries of the runs of rank <= k.
// kRange: only the runs of quotients [q_lo, q_hi) of the window (which must
// end inside it).  All kThreads threads call it.  Returns false if the runs of
// earlier blocks, or those of the range, reach past the window.
// kStore: make the entries; else only count them, with the sum of this thread's
// counts in out.sum (no quotients needed: sm has no quot, old and rend then).
template <bool kRange, bool kStore, class S>
__device__ __forceinline__ bool window_entries(const QF& qf, uint64_t B0, int nwin, int32_t q_lo, int32_t q_hi, S& sm,
                                               Window& out) {
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nslots = 64 * nwin;
  const int j = tid >> 3, sh = (tid & 7) * 8;
  const GQF_GLOBAL uint4* g = gqf_block_ptr(qf, B0);
  uint2 x = make_uint2(0, 0);
  if (j < nwin) x = ((const GQF_GLOBAL uint2*)(g + (size_t)j * (GQF_BLOCK_BYTES / 16) + 4))[tid & 7];
  uint32_t off_j = 0;
  if (wave == 0) {
    uint4 h0 = make_uint4(0, 0, 0, 0), h1 = h0;
    if (lane < nwin) {
      h0 = g[(size_t)lane * (GQF_BLOCK_BYTES / 16)];
      h1 = g[(size_t)lane * (GQF_BLOCK_BYTES / 16) + 1];
    }
    const uint64_t occ = (uint64_t)h0.x | (uint64_t)h0.y << 32, run = (uint64_t)h0.z | (uint64_t)h0.w << 32;
    const uint64_t used = (uint64_t)h1.z | (uint64_t)h1.w << 32;
    off_j = h1.x;
    // slots [0, x0] of the window belong to earlier blocks' runs
    const int32_t first = (int32_t)__builtin_amdgcn_readfirstlane((int)off_j);
    auto from = [&](int32_t p) -> uint64_t {  // this block's slots at or after window slot p
      const int32_t d = p - 64 * lane;
      return d <= 0 ? ~0ULL : (d >= 64 ? 0ULL : ~0ULL << d);
    };
    const uint64_t own = used & from(first);
    const uint32_t nr = (uint32_t)__popcll(run & own), no = (uint32_t)__popcll(occ);
    const uint32_t rb = wave_scan_add(nr) - nr, ob = wave_scan_add(no) - no;
    uint64_t part = own;
    if (kRange) {
      // the runs of quotients < q end at the k-th own run end, k = occupied
      // quotients below q
      bool inside = true;
      auto end_before = [&](int32_t q) -> int32_t {  // first slot behind them
        uint32_t k = 0;
        if (q > 0) {
          const int l = q < 64 * kWin ? q >> 6 : kWin - 1;
          const uint64_t m = q < 64 * kWin ? (1ULL << (q & 63)) - 1 : ~0ULL;
          k = (uint32_t)__builtin_amdgcn_readlane((int)(ob + (uint32_t)__popcll(occ & m)), l);
        }
        if (k == 0) return first;
        const uint64_t has = __ballot(rb < k && k <= rb + nr);
        if (!has) {
          inside = false;
          return 64 * kWin;
        }
        const int l = __builtin_ctzll(has);
        const int32_t p = (rb < k && k <= rb + nr) ? 64 * lane + gqf_select64(run & own, (int)(k - rb) - 1) : 0;
        return __builtin_amdgcn_readlane(p, l) + 1;
      };
      const int32_t lo = end_before(q_lo), hi = end_before(q_hi);
      part = own & from(lo) & ~from(hi);
      if (lane == 0) sm.over = inside ? 0u : 1u;
    } else if (lane == 0) {
      sm.over = 0;
    }
    sm.occ[lane] = occ;
    sm.run[lane] = run;
    sm.used[lane] = used;
    sm.own[lane] = own;
    sm.cont[lane] = own & (own << 1 | below_u64(own) >> 63) & ~(run << 1 | below_u64(run) >> 63);
    sm.start[lane] = part;
    sm.multi[lane] = 0;
    sm.occ_new[lane] = 0;
    sm.xblk[lane] = kNone;
    sm.xold[lane] = 64 * lane - 1 + (int32_t)off_j;
    sm.rbase[lane] = rb;
    sm.obase[lane] = ob;
    const bool any = __ballot(part != 0) != 0;
    const uint32_t slots = (uint32_t)__popcll(part);
    const uint32_t all = wave_scan_add(slots);
    if (lane == 63) sm.n_slots = all;
    if (lane == 0) {
      sm.start[kWin] = 0;
      sm.n_old = any ? 1u : 0u;
      sm.any_multi = 0;
      sm.n_big = 0;
      sm.xend = (int32_t)off_j - 1;
    }
  }
  ((uint2*)sm.sin)[tid] = x;
  __syncthreads();
  out.slots = x;
  out.off = off_j;
  out.x0 = sm.xold[0];
  out.any = sm.n_old != 0;
  out.n = 0;
  out.sum = 0;
  if (out.x0 + 1 > nslots) return false;
  if (kRange && sm.over) return false;
  if (!out.any) return true;
  const uint64_t below = (1ULL << sh) - 1;
  // the occupied quotients by rank (the thread's eight quotients)
  if constexpr (kStore) {
    const uint64_t occ = sm.occ[j];
    uint32_t k = sm.obase[j] + (uint32_t)__popcll(occ & below);
    for (uint32_t b = (uint32_t)(occ >> sh) & 0xFFu; b; b &= b - 1)
      sm.quot[k++] = (uint16_t)(64 * j + sh + __builtin_ctz(b));
  }
  // A byte not above its predecessor in the run goes on with a counter: a
  // counter's first slot is above the remainder that ends the one before it.
  // Counters of three slots and more hold digits that may ascend as well: such
  // a counter drops right after its first slot (x > 0: to a lower digit or a
  // leading 0) or has two 0s in a row (x = 0), and its run is decoded below.
  {
    const uint32_t c = (uint32_t)((sm.cont[j] & sm.start[j]) >> sh) & 0xFFu;
    uint32_t prev = tid ? sm.sin[8 * tid - 1] : 0u;
    uint32_t same = 0, viol = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const uint32_t b = ((k < 4 ? x.x : x.y) >> (8 * (k & 3))) & 0xFFu;
      same |= b == prev ? 1u << k : 0u;
      viol |= b < max(prev, 1u) ? 1u << k : 0u;
      prev = b;
    }
    // (three equal bytes in a row are no counter's: decoded as well)
    viol |= same & (same << 1 | (tid && sm.sin[8 * tid - 1] == sm.sin[8 * tid - 2] ? 1u : 0u));
    if ((same | viol) & c) ((uint8_t*)sm.start)[tid] = (uint8_t)((uint32_t)(sm.start[j] >> sh) & ~((same | viol) & c));
    for (viol &= c; viol; viol &= viol - 1) {
      // the run starts behind the last run end or unused slot before the byte
      const int at = sh + __builtin_ctz(viol);
      int b = j;
      uint64_t w = (sm.run[j] | ~sm.used[j]) & ((1ULL << at) - 1);
      while (!w && b > 0) {
        b--;
        w = sm.run[b] | ~sm.used[b];
      }
      const int32_t rs = w ? 64 * b + 64 - __builtin_clzll(w) : 0;
      atomicOr((unsigned long long*)&sm.multi[rs >> 6], 1ULL << (rs & 63));
      sm.any_multi = 1;
    }
  }
  __syncthreads();
  if (sm.any_multi) {
    for (uint32_t mb = (uint32_t)(sm.multi[j] >> sh) & 0xFFu; mb; mb &= mb - 1) {
      const int32_t p = 8 * tid + __builtin_ctz(mb);
      const uint32_t len = (uint32_t)(run_end_of(sm, p, nwin) - p + 1);
      auto slot = [&](uint32_t k) -> uint64_t { return sm.sin[p + (int32_t)k]; };
      for (uint32_t k = 0; k < len;) {
        uint64_t rem, c;
        const uint32_t last = gqf_decode_counter(slot, len, k, &rem, &c);
        if (k) atomicOr((unsigned long long*)&sm.start[(p + (int32_t)k) >> 6], 1ULL << ((p + (int32_t)k) & 63));
        for (uint32_t y = k + 1; y <= last; y++) {
          const int32_t q = p + (int32_t)y;
          atomicAnd((unsigned long long*)&sm.start[q >> 6], ~(1ULL << (q & 63)));
        }
        k = last + 1;
      }
    }
    __syncthreads();
  }
  if (wave == 0) {
    const uint32_t n = (uint32_t)__popcll(sm.start[lane]);
    const uint32_t incl = wave_scan_add(n);
    sm.ebase[lane] = incl - n;
    if (lane == 63) sm.n_old = incl;
  }
  __syncthreads();
  out.n = sm.n_old;
  {
    const uint64_t st = sm.start[j], own = sm.own[j], run = sm.run[j] & own;
    const uint32_t e0 = sm.ebase[j] + (uint32_t)__popcll(st & below);
    const uint32_t k0 = sm.rbase[j] + (uint32_t)__popcll(run & below);
    const uint32_t stb = (uint32_t)(st >> sh) & 0xFFu, runb = (uint32_t)(run >> sh) & 0xFFu;
    // slots whose next slot continues their counter
    const uint64_t inner = own & ~st;
    const uint32_t nextb = (uint32_t)((inner >> sh) >> 1) & 0x7Fu;
    const uint32_t after = sh < 56 ? (uint32_t)(inner >> (sh + 8)) & 3u
                                   : (j + 1 < nwin ? (uint32_t)(sm.own[j + 1] & ~sm.start[j + 1]) & 3u : 0u);
    const uint32_t moreb = stb & ~runb & (nextb | (after & 1u) << 7);
    auto count_at = [&](int32_t p) -> uint64_t {  // of the counter of several slots at slot p
      const uint32_t len = (uint32_t)(run_end_of(sm, p, nwin) - p + 1);
      uint64_t rem, c;
      gqf_decode_counter([&](uint32_t k) -> uint64_t { return sm.sin[p + (int32_t)k]; }, len, 0, &rem, &c);
      return c;
    };
    // a counter of two slots is a count of 2
    const uint32_t longb = moreb & (nextb >> 1 | after << 6);
    if constexpr (!kStore) {
      out.sum = (uint64_t)__builtin_popcount(stb) + (uint64_t)__builtin_popcount(moreb & ~longb);
      for (uint32_t m = longb; m; m &= m - 1) out.sum += count_at(8 * tid + __builtin_ctz(m)) - 1;
      return true;
    } else {
      uint32_t q[8];
#pragma unroll
      for (int i = 0; i < 8; i++)
        if ((stb >> i) & 1u) q[i] = sm.quot[k0 + (uint32_t)__builtin_popcount(runb & ((1u << i) - 1))];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const uint32_t ei = e0 + (uint32_t)__builtin_popcount(stb & ((1u << i) - 1));
        if ((stb >> i) & 1u) {
          const uint32_t h = q[i] << 8 | (((i < 4 ? x.x : x.y) >> (8 * (i & 3))) & 0xFFu);
          sm.old[ei] = h << 12 | (1u + ((moreb >> i) & 1u));
        }
        if ((runb >> i) & 1u)
          sm.rend[k0 + (uint32_t)__builtin_popcount(runb & ((1u << i) - 1))] = (uint16_t)(ei + ((stb >> i) & 1u));
      }
      for (uint32_t m = longb; m; m &= m - 1) {
        const int i = __builtin_ctz(m);
        uint32_t& y = sm.old[e0 + (uint32_t)__builtin_popcount(stb & ((1u << i) - 1))];
        const uint32_t h = y >> 12;
        y = h << 12 | push_count(sm, h, count_at(8 * tid + i));
      }
    }
  }
  __syncthreads();
  return true;
}

// Rebuilds region r of `qf` with its items [s, e) of `items` (sorted hashes
// + tag; per-item counts for kCounts).  All kThreads threads call it; nothing
// is written unless it returns kOk.  Window and result as rebuild_region
// (gqf_rebuild.hip) with `concurrent` set.
__device__ __forceinline__ int rebuild(const QF& qf, uint64_t r, const uint64_t* __restrict__ items,
                                       const uint64_t* __restrict__ counts, uint64_t s, uint64_t e, int kind,
                                       uint64_t tag, Smem& sm) {
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int R = (int)qf.region_blocks;
  const uint64_t B0 = r * (uint64_t)R;
  const int nwin = (int)min((uint64_t)(2 * R < kWin ? 2 * R : kWin), qf.nblocks - B0);
  const int nslots = 64 * nwin;
  const bool table_end = B0 + (uint64_t)nwin >= qf.nblocks;
  const uint64_t hmask = kind == kTagged ? GQF_SEQ_HASH_MASK : ~0ULL;
  const uint64_t base = tag + (B0 << 14);

  for (int k = tid; k < kSeqWords; k += kThreads) sm.is_item[k] = 0;
  Window w;
  if (!window_entries<false, true>(qf, B0, nwin, 0, 0, sm, w)) return kNeedWide;  // spill-in longer than the window
  const int j = tid >> 3, sh = (tid & 7) * 8;
  const uint2 x = w.slots;
  const uint32_t off_j = w.off;
  const int32_t x0 = w.x0;
  const bool any_old = w.any;
  const uint32_t n_old = w.n;
  const uint32_t big_old = sm.n_big;
  __syncthreads();

  // ---- 2. the items, each wave a contiguous share, 64 at a time.  Item k
  // becomes entry k of sm.item and takes the place (k + the old entries before
  // it) in the merged sequence, marked in sm.is_item; a repeat, or an item
  // whose hash has an old entry, is an empty entry.  Where the entries would
  // not hold all items, the ordinals count distinct hashes only.
  const uint64_t n_items = e - s;
  const uint64_t share = ((n_items + kThreads - 1) / kThreads) * 64;
  const uint64_t i0 = s + min(n_items, share * (uint64_t)wave), i1 = s + min(n_items, share * (uint64_t)(wave + 1));
  auto head_at = [&](uint64_t i, uint64_t& v) -> bool {
    v = i < i1 ? items[i] & hmask : ~0ULL;
    uint64_t prev = below_u64(v);
    if (lane == 0 && i < i1 && i > s) prev = items[i - 1] & hmask;
    return i < i1 && (i == s || prev != v);
  };
  uint32_t ord = (uint32_t)(i0 - s), n_new = (uint32_t)n_items;  // ordinal of the wave's next item, all ordinals
  const bool sparse = n_items > (uint64_t)kItems;
  if (sparse) {
    uint32_t heads = 0;
    for (uint64_t i = i0; i < i1; i += 64) {
      uint64_t v;
      heads += (uint32_t)__popcll(__ballot(head_at(i + (uint64_t)lane, v)));
    }
    if (lane == 0) sm.wsum[0][wave] = heads;
    __syncthreads();
    ord = n_new = 0;
    for (int w = 0; w < kWaves; w++) {
      const uint32_t c = sm.wsum[0][w];
      ord += w < wave ? c : 0u;
      n_new += c;
    }
    if (n_new > (uint32_t)kItems) return kNeedWide;
  }
  for (uint64_t i = i0; i < i1; i += 64) {
    const uint64_t ii = i + (uint64_t)lane;
    uint64_t v;
    const bool head = head_at(ii, v);
    const uint64_t hm = __ballot(head);
    const bool active = sparse ? head : ii < i1;
    if (active) {
      const uint32_t h = (uint32_t)(v - base);
      // its place among the old entries: its quotient's run holds entries
      // [lo, hi)
      uint32_t lo = 0, hi = 0;
      if (any_old) {
        const uint32_t q = h >> 8;
        const uint64_t occ = sm.occ[q >> 6];
        const uint32_t rank = sm.obase[q >> 6] + (uint32_t)__popcll(occ & ((1ULL << (q & 63)) - 1));
        const bool has = (occ >> (q & 63)) & 1;
        // (a run that ends past the window has no entry: clamped, and the
        // region goes to the wide pass below)
        lo = rank ? min((uint32_t)sm.rend[rank - 1], n_old) : 0u;
        hi = has ? min((uint32_t)sm.rend[rank], n_old) : lo;
        while (lo < hi && (sm.old[lo] >> 12) < h) lo++;
      }
      const uint32_t oe = lo < hi ? sm.old[lo] : 0xFFFFFFFFu;
      const bool there = lo < hi && (oe >> 12) == h;
      uint32_t entry = 0;
      if (head) {
        // the items of this hash: up to the next head
        const uint64_t up = lane < 63 ? hm >> (lane + 1) : 0ULL;
        uint64_t next = ii + 1 + (up ? (uint64_t)__builtin_ctzll(up) : 0ULL);
        if (!up) {
          next = ii + 1 + min((uint64_t)(63 - lane), i1 - ii - 1);  // the rest of this step are repeats
          if (next < e && (items[next] & hmask) == v) {             // and more follow
            uint64_t a = next, b = e;  // first item past the hash
            while (a < b) {
              const uint64_t mid = (a + b) >> 1;
              if ((items[mid] & hmask) <= v) a = mid + 1; else b = mid;
            }
            next = a;
          }
        }
        const uint64_t c_old = there ? full_count(sm, h, oe & 0xFFFu, big_old) : 0ULL;
        uint64_t c_new = c_old;
        if (kind == kAdd) {
          c_new += next - ii;
        } else if (kind == kCounts) {
          for (uint64_t k = ii; k < next; k++) c_new += counts[k];
        } else {  // in order: +1, or -1 down to 0
          for (uint64_t k = ii; k < next; k++) {
            if (items[k] >> 63) c_new -= c_new ? 1 : 0;
            else c_new++;
          }
        }
        if (there) {
          uint32_t aux = (uint32_t)c_new;
          if (c_new >= kAuxBig) {
            uint32_t k = 0;
            while (k < big_old && k < (uint32_t)kBig && sm.big_hash[k] != h) k++;
            if ((oe & 0xFFFu) == kAuxBig && k < big_old && k < (uint32_t)kBig) {
              sm.big_count[k] = c_new;
              aux = kAuxBig;
            } else {
              aux = push_count(sm, h, c_new);
            }
          }
          sm.old[lo] = h << 12 | aux;
        } else {
          entry = h << 12 | push_count(sm, h, c_new);
        }
      }
      const uint32_t k = sparse ? ord + (uint32_t)__popcll(hm & ((1ULL << lane) - 1)) : ord + (uint32_t)lane;
      const uint32_t at = lo + (there ? 1u : 0u);
      sm.item[k] = entry;
      atomicOr(&sm.is_item[(k + at) >> 5], 1u << ((k + at) & 31));
    }
    ord += sparse ? (uint32_t)__popcll(hm) : 64u;
  }
  __syncthreads();
  if (sm.over) return kNeedWide;

  // ---- the merged sequence: place i holds item k, k = items marked before
  // it, or old entry i - k
  const uint32_t n_all = n_old + n_new;
  if (wave == 0) {
    constexpr int kW = (kSeqWords + 63) / 64;  // words a lane
    uint32_t c[kW], sum = 0;
#pragma unroll
    for (int k = 0; k < kW; k++) {
      c[k] = kW * lane + k < kSeqWords ? (uint32_t)__popc(sm.is_item[kW * lane + k]) : 0u;
      sum += c[k];
    }
    uint32_t before = wave_scan_add(sum) - sum;
#pragma unroll
    for (int k = 0; k < kW; k++) {
      if (kW * lane + k < kSeqWords) sm.items_before[kW * lane + k] = before;
      before += c[k];
    }
  }
  auto scan_add = [&](uint32_t v) -> uint32_t {  // exclusive, over the workgroup; one barrier
    const uint32_t incl = wave_scan_add(v);
    if (lane == 63) sm.wsum[1][wave] = incl;
    __syncthreads();
    uint32_t before = incl - v;
#pragma unroll
    for (int w = 0; w < kWaves; w++) before += w < wave ? sm.wsum[1][w] : 0u;
    return before;
  };
  uint16_t* out = sm.out;  // new slots: byte | 1 << 8 | (first of its run) << 9
  const uint32_t n_big = sm.n_big;
  ((uint4*)out)[tid] = make_uint4(0, 0, 0, 0);
  __syncthreads();

  // ---- 3. positions.  A thread takes an odd number of consecutive places (odd
  // strides spread the lanes over the LDS banks): it adds them up by itself,
  // and one scan over the threads places its share.
  {
    const uint32_t per = ((n_all + kThreads - 1) / kThreads) | 1u;
    const uint32_t a = min(n_all, per * (uint32_t)tid), b = min(n_all, a + per);
    const uint32_t ka = a < n_all ? sm.items_before[a >> 5] +
                                        (uint32_t)__popc(sm.is_item[a >> 5] & ((1u << (a & 31)) - 1))
                                  : 0u;
    // the entry at place i, k items before it
    auto entry_at = [&](uint32_t i, uint32_t& k) -> uint32_t {
      const bool item = (sm.is_item[i >> 5] >> (i & 31)) & 1u;
      const uint32_t y = item ? sm.item[k] : sm.old[i - k];
      k += item ? 1u : 0u;
      return y;
    };
    auto slots_of = [&](uint32_t y) -> uint32_t {
      const uint32_t rem = (y >> 12) & 0xFFu, aux = y & 0xFFFu;
      uint32_t len = aux;  // counts up to 3
      if (aux > 3) len = aux < kAuxBig ? entry_len(rem, aux) : gqf_counter_len(rem, full_count(sm, y >> 12, aux, n_big));
      return len;
    };
    uint32_t sum = 0;
    int32_t lead = kNone, lastq = -1;  // max of quotient - slots before it in the share; the last quotient
    uint32_t ki = ka;
    for (uint32_t i = a; i < b; i++) {
      const uint32_t y = entry_at(i, ki);
      const uint32_t len = slots_of(y);
      const int32_t q = (int32_t)(y >> 20);
      if (len) {
        lead = max_i(lead, q - (int32_t)sum);
        lastq = q;
      }
      sum += len;
    }
    uint32_t before = scan_add(sum);
    // the same over the threads before this one: largest quotient - slots
    // before it, and the last quotient (they ascend)
    const int32_t li = wave_scan_max(lead == kNone ? kNone : lead - (int32_t)before), qi = wave_scan_max(lastq);
    if (lane == 63) {
      sm.wmax[0][wave] = li;
      sm.wmax[1][wave] = qi;
    }
    __syncthreads();
    lead = max_i(below_i(li, kNone), x0 + 1);
    lastq = below_i(qi, -1);
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      lead = w < wave ? max_i(lead, sm.wmax[0][w]) : lead;
      lastq = w < wave ? max_i(lastq, sm.wmax[1][w]) : lastq;
    }
    int32_t last = kNone, blk = -1;  // last new slot, of quotients of block blk
    ki = ka;
    for (uint32_t i = a; i < b; i++) {
      const uint32_t y = entry_at(i, ki);
      const uint32_t len = slots_of(y);
      if (!len) continue;
      const int32_t q = (int32_t)(y >> 20);
      const uint32_t rem = (y >> 12) & 0xFFu;
      lead = max_i(lead, q - (int32_t)before);
      const int32_t p = (int32_t)before + lead;
      before += len;
      const bool first = q != lastq;
      lastq = q;
      if ((q >> 6) != blk) {
        if (blk >= 0) atomicMax(&sm.xblk[blk], last);
        blk = q >> 6;
      }
      last = p + (int32_t)len - 1;
      if (first) atomicOr(&((uint32_t*)sm.occ_new)[q >> 5], 1u << (q & 31));
      const uint32_t word = 0x100u | (first ? 0x200u : 0u);
      if (len <= 2) {  // r, or r r
        if (p < kSlots) out[p] = (uint16_t)(word | rem);
        if (len == 2 && p + 1 < kSlots) out[p + 1] = (uint16_t)(0x100u | rem);
      } else {
        gqf_emit_counter(rem, full_count(sm, y >> 12, y & 0xFFFu, n_big), [&](uint32_t i2, uint64_t v) {
          const int32_t at = p + (int32_t)i2;
          if (at < kSlots) out[at] = (uint16_t)((i2 ? 0x100u : word) | (uint32_t)(v & 0xFFu));
        });
      }
    }
    if (blk >= 0) {
      atomicMax(&sm.xblk[blk], last);
      atomicMax(&sm.xend, last);
    }
  }
  __syncthreads();

  // ---- 4. the new header words: a slot is a run's last where the next one
  // starts a run or is unused
  uint2 fresh_bytes;
  {
    const uint4 o = ((const uint4*)out)[tid];
    const uint32_t nx = tid + 1 < kThreads ? (uint32_t)out[8 * tid + 8] >> 8 : 0u;
    fresh_bytes.x = __builtin_amdgcn_perm(o.y, o.x, 0x06040200);
    fresh_bytes.y = __builtin_amdgcn_perm(o.w, o.z, 0x06040200);
    const uint32_t f0 = __builtin_amdgcn_perm(o.y, o.x, 0x07050301), f1 = __builtin_amdgcn_perm(o.w, o.z, 0x07050301);
    // bit 0 / bit 1 of four bytes -> four bits
    auto bits = [](uint32_t f) { return ((f & 0x01010101u) * 0x01020408u) >> 24; };
    const uint32_t used = bits(f0) | bits(f1) << 4;
    const uint32_t first = bits(f0 >> 1) | bits(f1 >> 1) << 4;
    const uint32_t used_next = used >> 1 | (nx & 1u) << 7, first_next = first >> 1 | (nx >> 1 & 1u) << 7;
    ((uint8_t*)sm.used_new)[tid] = (uint8_t)used;
    ((uint8_t*)sm.run_new)[tid] = (uint8_t)(used & (first_next | ~used_next));
  }
  if (wave == 0) {
    // end of the runs of quotients < 64 j
    const int32_t incl = wave_scan_max(sm.xblk[lane]);
    const int32_t xn = max_i(max_i(below_i(incl, kNone), x0), 64 * lane - 1);
    const int32_t xo = sm.xold[lane];
    sm.xnew[lane] = xn;
    // Where the new layout meets the old one: the first block past the region
    // whose earlier runs end where they did, inside the window; for batches
    // that the single-wave rebuild would walk, inside that block.  Which regions
    // need the wide pass has to be the same there and here: in a table too full
    // for a batch, what it keeps of the batch depends on the order.
    const bool walked = kind != kAdd || n_items > 256;
    const uint64_t meet = __ballot(lane >= R && lane < nwin && xn == xo && xo < nslots && (!walked || xo - 64 * lane < 63));
    if (lane == 0) {
      int res = kOk, bstar = nwin, bwrite = nwin;
      int32_t keep = INT32_MAX;
      if (meet) {
        bstar = __builtin_ctzll(meet);
        keep = sm.xold[bstar];
        bwrite = max_i(bstar, (keep >> 6) + 1);
      } else if (!table_end) {
        res = kNeedWide;
      } else if ((int64_t)(B0 * 64) + sm.xend >= (int64_t)qf.xnslots) {
        res = kNoSpace;
      }
      sm.bstar = bstar;
      sm.bwrite = bwrite;
      sm.keep = keep;
      sm.result = res;
    }
  }
  __syncthreads();
  const int res = sm.result;
  if (res != kOk) return res;

  // ---- store: the earlier regions' slots (up to x0) and those past the
  // meeting point stay as they are
  const int bstar = sm.bstar, bwrite = sm.bwrite;
  const int32_t keep = sm.keep;
  // new slots of block b: (x0, keep]
  auto fresh_of = [&](int b) -> uint64_t {
    const int32_t lo = x0 + 1 - 64 * b, hi = keep - 64 * b;
    const uint64_t from = lo <= 0 ? ~0ULL : (lo >= 64 ? 0ULL : ~0ULL << lo);
    return from & (hi < 0 ? 0ULL : (hi >= 63 ? ~0ULL : (2ULL << hi) - 1));
  };
  uint8_t* dst = qf.blocks + B0 * GQF_BLOCK_BYTES;
  if (j < bwrite) {
    const uint32_t fr = (uint32_t)(fresh_of(j) >> sh) & 0xFFu;
    uint2 v = fresh_bytes;
    if (fr != 0xFFu) {  // byte masks from bits
      auto mask = [](uint32_t b) { return ((b & 1u) | (b & 2u) << 7 | (b & 4u) << 14 | (b & 8u) << 21) * 0xFFu; };
      const uint32_t m0 = mask(fr), m1 = mask(fr >> 4);
      v.x = (v.x & m0) | (x.x & ~m0);
      v.y = (v.y & m1) | (x.y & ~m1);
    }
    ((GQF_GLOBAL uint2*)gqf_gptr_mut(dst + (size_t)j * GQF_BLOCK_BYTES + GQF_SLOT_BASE))[tid & 7] = v;
  }
  if (wave == 0 && lane < bwrite) {
    const uint64_t fresh = fresh_of(lane);
    const uint64_t occ = lane < bstar ? sm.occ_new[lane] : sm.occ[lane];
    const uint64_t run = (sm.run_new[lane] & fresh) | (sm.run[lane] & ~fresh);
    const uint64_t used = (sm.used_new[lane] & fresh) | (sm.used[lane] & ~fresh);
    const uint32_t off = lane < bstar ? (uint32_t)(sm.xnew[lane] - (64 * lane - 1)) : off_j;
    GQF_GLOBAL uint4* b = gqf_gptr_mut((uint4*)dst) + (size_t)lane * (GQF_BLOCK_BYTES / 16);
    b[0] = make_uint4((uint32_t)occ, (uint32_t)(occ >> 32), (uint32_t)run, (uint32_t)(run >> 32));
    b[1] = make_uint4(off, 0, (uint32_t)used, (uint32_t)(used >> 32));
  }
  return kOk;
}

}  // namespace gqf_flat
