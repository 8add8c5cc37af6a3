// gqf_enum.hip -- whole-table passes over a filter: enumeration of its items
// in ascending hash order, the item / count / used-slot statistics, and the
// cluster census.
//
// Enumeration replaces the reference's host iterator
// (qf_iterator_from_position src/gqf.cu:3655-3700, qfi_next :3814-3840,
// qfi_get_hash :3807, qfi_get_key :3791-3805).  Table order is hash order:
// runs sit in quotient order and a run's counters in remainder order, so
// the iterator's sequence is the table's counters read left to right.  A
// workgroup turns the runs of GQF_ENUM_BLOCKS blocks' quotients into entries
// in LDS, as the dense rebuild does (gqf_flat.h): one pass counts the groups'
// items, a scan gives each group's first rank, a second pass makes the entries
// again and writes them out in order.
//
// The census replaces src/cluster_length_test.cu:37-120, which walks the
// table with find_first_empty_slot (src/gqf.cu:728-771) from one thread:
// a cluster is a maximal stretch of used slots.  Here each block's used
// slots become a 64-bit mask; cluster starts are the mask's rising edges,
// and each start finds its cluster's end by scanning the masks forward.
#include "gqf_flat.h"
#include "gqf_internal.h"
#include "gqf_launch.h"

namespace {

constexpr int kThreads = 256;  // census: one thread per table block

// Visits the counters of the runs of block b's occupied quotients in
// [q_lo, q_hi), in table order: item(storage hash, count).  Returns the slots
// those runs use, or -1 if a run has no run end (a damaged table).  For the
// groups that do not fit a window (runs far longer than a table of random
// hashes has).
template <typename Item>
__device__ inline int64_t walk_items(const QF& f, uint64_t b, uint64_t q_lo, uint64_t q_hi, Item item) {
  uint64_t occ = gqf_point::occ_word(f, b);
  int64_t prev = gqf_point::end_before_block(f, b);
  int64_t used = 0;
  // run-end word of block cb, reloaded only when a run starts or ends in
  // another block (a load per run made a chain of ~38 dependent loads)
  uint64_t cb = ~0ULL, cw = 0;
  while (occ) {
    const uint64_t q = b * 64 + (uint64_t)__builtin_ctzll(occ);
    occ &= occ - 1;
    const uint64_t start = (int64_t)q > prev + 1 ? q : (uint64_t)(prev + 1);
    // the run ends at the first run end at or after start
    uint64_t bj = start >> 6;
    if (bj >= f.nblocks) return -1;
    if (bj != cb) {
      cb = bj;
      cw = gqf_point::run_word(f, bj);
    }
    uint64_t w = cw & (~0ULL << (start & 63));
    while (!w) {
      if (++bj >= f.nblocks) return -1;
      cb = bj;
      cw = gqf_point::run_word(f, bj);
      w = cw;
    }
    const int64_t e = (int64_t)(bj * 64) + __builtin_ctzll(w);
    prev = e;
    if (q < q_lo || q >= q_hi) continue;
    const uint32_t len = (uint32_t)(e - (int64_t)start + 1);
    used += len;
    auto at = [&](uint32_t k) -> uint64_t { return gqf_point::slot(f, start + k); };
    uint32_t idx = 0;
    while (idx < len) {
      uint64_t rem, cnt;
      const uint32_t last = gqf_decode_counter(at, len, idx, &rem, &cnt);
      item((q << 8) | rem, cnt);
      idx = last + 1;
    }
  }
  return used;
}

// workgroup exclusive scan of one u32 per thread; returns the prefix and
// writes the workgroup total to *total
__device__ inline uint32_t wg_exclusive_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t wsum[kThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t incl = wave_scan_add(v);
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  uint32_t before = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kThreads / 64; k++) {
    if (k < w) before += wsum[k];
    tot += wsum[k];
  }
  __syncthreads();
  *total = tot;
  return before + incl - v;
}

}  // namespace

// Output form of an item (storage hash S = (hash << value_bits) | value):
//   GQF_ENUM_OUT_HASH  S >> value_bits (qfi_get_hash's key), value to `values`
//   GQF_ENUM_OUT_KEY   hash_64i of that (qfi_get_key's key)
//   GQF_ENUM_OUT_MOVE  the storage hash of the same (hash, value) in a filter
//                      with `dst_vb` value bits (value truncated to them)
struct gqf_out_form {
  int mode;
  int vb;       // source value bits
  int dst_vb;   // MOVE: destination value bits
  uint64_t key_mask;
};

// gqf_hash64_inv for hashes of at most 42 bits: an xor-shift by s of a w-bit
// word is undone by ceil(w / s) - 1 steps
static __device__ __forceinline__ uint64_t hash64_inv42(uint64_t h, uint64_t mask) {
  constexpr uint64_t i31 = gqf_inv_odd((1ULL << 31) + 1);
  constexpr uint64_t i21 = gqf_inv_odd(21);
  constexpr uint64_t i265 = gqf_inv_odd(265);
  constexpr uint64_t ik = gqf_inv_odd((1ULL << 21) - 1);
  uint64_t k = (h * i31) & mask;
  k ^= k >> 28;
  k = (k * i21) & mask;
  k ^= (k ^ (k >> 14)) >> 14;
  k = (k * i265) & mask;
  k ^= k >> 24;
  return ((k + 1) * ik) & mask;
}

static __device__ inline uint64_t form_hash(const gqf_out_form& o, uint64_t s) {
  const uint64_t h = s >> o.vb;
  if (o.mode == GQF_ENUM_OUT_KEY)
    return o.key_mask >> 42 ? gqf_hash64_inv(h, o.key_mask) : hash64_inv42(h, o.key_mask);
  if (o.mode == GQF_ENUM_OUT_MOVE) return (h << o.dst_vb) | (s & gqf_mask((uint64_t)min(o.vb, o.dst_vb)));
  return h;
}

// Group u of an enumeration of quotients [q_lo, q_hi) over blocks [b_lo,
// b_hi): the quotients of blocks b_lo + u GQF_ENUM_BLOCKS .., in a window with
// the blocks behind them for runs that reach out.
constexpr int kGroupWaves = gqf_flat::kThreads / 64;
static_assert(GQF_ENUM_BLOCKS < gqf_flat::kWin, "blocks of the window past the group's");

struct CountSmem : gqf_flat::Head {
  alignas(16) uint8_t sin[gqf_flat::kSlots];
  uint64_t sums[kGroupWaves];
};
struct EnumSmem : gqf_flat::Head {
  alignas(16) uint8_t sin[gqf_flat::kSlots];
  uint16_t rend[gqf_flat::kSlots];
  uint16_t quot[gqf_flat::kSlots];
  uint32_t old[gqf_flat::kSlots];
};

struct EnumRange {
  uint64_t b_lo, b_hi, q_lo, q_hi;
};

// Makes group u's entries; false where they do not fit the window or its
// table of large counts.  b0: the group's first block.
template <bool kStore, class S>
static __device__ __forceinline__ bool group_entries(const QF& f, const EnumRange& r, uint64_t u, S& sm,
                                                     gqf_flat::Window& w, uint64_t& b0) {
  b0 = r.b_lo + u * GQF_ENUM_BLOCKS;
  const int nwin = (int)min((uint64_t)gqf_flat::kWin, f.nblocks - b0);
  const uint64_t q0 = b0 * 64;
  const int32_t lo = r.q_lo > q0 ? (int32_t)min(r.q_lo - q0, (uint64_t)(64 * GQF_ENUM_BLOCKS)) : 0;
  const uint64_t end = min(min((uint64_t)(64 * GQF_ENUM_BLOCKS), 64 * (r.b_hi - b0)), r.q_hi > q0 ? r.q_hi - q0 : 0ULL);
  return gqf_flat::window_entries<true, kStore>(f, b0, nwin, lo, (int32_t)min(end, (uint64_t)(64 * nwin)), sm, w) && !sm.over;
}

// The group's items block by block, from the table (wave 0, a block a lane):
// item(rank in the group, storage hash, count); returns the lane's items
template <typename Item>
static __device__ inline uint32_t walk_group(const QF& f, const EnumRange& r, uint64_t b0, uint32_t rank, Item item,
                                             uint64_t& used) {
  const uint64_t b = b0 + (threadIdx.x & 63);
  uint32_t n = 0;
  used = 0;
  if ((threadIdx.x & 63) < GQF_ENUM_BLOCKS && b < r.b_hi) {
    const int64_t u = walk_items(f, b, r.q_lo, r.q_hi, [&](uint64_t s, uint64_t c) {
      item(rank + n, s, c);
      n++;
    });
    if (u < 0) atomicOr(f.status, GQF_STATUS_CLUSTER_OVERFLOW);
    else used = (uint64_t)u;
  }
  return n;
}

// Items, sum of counts and used slots of every group
extern "C" __global__ void __launch_bounds__(gqf_flat::kThreads)
gqf_enum_count(const QF* __restrict__ qfp, EnumRange r, uint32_t* __restrict__ items, uint32_t* __restrict__ slots,
               uint64_t* __restrict__ sums) {
  __shared__ CountSmem sm;
  const QF& f = *qfp;
  const uint64_t u = blockIdx.x;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  gqf_flat::Window w;
  uint64_t b0;
  const bool fits = group_entries<false>(f, r, u, sm, w, b0);
  if (fits) {
    uint64_t sum = w.n;
    if (w.any && w.n != sm.n_slots) {  // else every entry counts one
      sum = w.sum;
      for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
      if (lane == 0) sm.sums[wave] = sum;
      __syncthreads();
      sum = 0;
      for (int k = 0; k < kGroupWaves; k++) sum += sm.sums[k];
    }
    if (tid == 0) {
      items[u] = w.n;
      slots[u] = w.any ? sm.n_slots : 0u;
      sums[u] = sum;
    }
  } else if (wave == 0) {
    uint64_t sum = 0, used;
    uint32_t n = walk_group(f, r, b0, 0, [&](uint32_t, uint64_t, uint64_t c) { sum += c; }, used);
    for (int d = 32; d >= 1; d >>= 1) {
      n += __shfl_xor(n, d, 64);
      sum += __shfl_xor(sum, d, 64);
      used += __shfl_xor(used, d, 64);
    }
    if (lane == 0) {
      items[u] = n;
      slots[u] = (uint32_t)used;
      sums[u] = sum;
    }
  }
}

// Exclusive scan of n u32 counts into u64 bases (one workgroup, eight counts a
// thread and step); the total goes to base[n], and, with `stats`, the totals
// of items, sums and slots to it.  A step's counts add up to less than 2^32:
// they are of some of the table's entries or clusters.
// Bound by one CU's loads: a thread's eight values in 16-byte loads and stores
// where the arrays are aligned (every caller's are); one by one, each fetched
// its lines eight times over (17,000 groups: 21 us, 11 us so).
extern "C" __global__ void __launch_bounds__(1024)
gqf_enum_scan(const uint32_t* __restrict__ cnt, const uint32_t* __restrict__ slots, const uint64_t* __restrict__ sums,
              uint32_t n, uint64_t* __restrict__ base, uint64_t* __restrict__ stats) {
  __shared__ uint32_t wsum[16];
  __shared__ uint64_t wstat[2][16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const bool aligned = (((uintptr_t)cnt | (uintptr_t)slots | (uintptr_t)sums | (uintptr_t)base) & 15) == 0;
  uint64_t carry = 0, tsum = 0, tslots = 0;
  for (uint32_t i0 = 0; i0 < n; i0 += 8192) {
    const uint32_t i = i0 + 8 * threadIdx.x;
    const bool whole = aligned && i + 8 <= n;
    uint32_t c[8];
    if (whole) {
      const uint4 a = ((const uint4*)(cnt + i))[0], b = ((const uint4*)(cnt + i))[1];
      c[0] = a.x; c[1] = a.y; c[2] = a.z; c[3] = a.w;
      c[4] = b.x; c[5] = b.y; c[6] = b.z; c[7] = b.w;
      if (stats) {
        const uint4 d = ((const uint4*)(slots + i))[0], e = ((const uint4*)(slots + i))[1];
        tslots += (uint64_t)d.x + d.y + d.z + d.w + e.x + e.y + e.z + e.w;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const ulonglong2 t = ((const ulonglong2*)(sums + i))[k];
          tsum += t.x + t.y;
        }
      }
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 8; k++) {
        const bool in = i + k < n;
        c[k] = in ? cnt[i + k] : 0u;
        if (stats && in) {
          tsum += sums[i + k];
          tslots += slots[i + k];
        }
      }
    }
    uint32_t v = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8; k++) v += c[k];
    const uint32_t incl = wave_scan_add(v);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t before = incl - v, tot = 0;
#pragma unroll
    for (int k = 0; k < 16; k++) {
      if (k < w) before += wsum[k];
      tot += wsum[k];
    }
    uint64_t run = carry + before;
    if (whole) {
#pragma unroll
      for (uint32_t k = 0; k < 8; k += 2) {
        ((ulonglong2*)(base + i))[k / 2] = make_ulonglong2(run, run + c[k]);
        run += (uint64_t)c[k] + c[k + 1];
      }
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 8; k++) {
        if (i + k < n) base[i + k] = run;
        run += c[k];
      }
    }
    carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) base[n] = carry;
  if (stats) {
    for (int d = 32; d >= 1; d >>= 1) {
      tsum += __shfl_xor(tsum, d, 64);
      tslots += __shfl_xor(tslots, d, 64);
    }
    if (lane == 0) {
      wstat[0][w] = tsum;
      wstat[1][w] = tslots;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      uint64_t a = 0, b = 0;
      for (int k = 0; k < 16; k++) {
        a += wstat[0][k];
        b += wstat[1][k];
      }
      stats[0] = carry;
      stats[1] = a;
      stats[2] = b;
    }
  }
}

// Writes the items of groups u0 .. u0 + gridDim.x - 1: item i of the
// enumeration to index i - skip of the output arrays, if that is below cap.
// Bound by HBM for the hashes (16 B an item written, 96 B a block read); the
// key form's inverse hash (four 64-bit products) costs about as much again.
// 2^26 slots at load 0.9, keys and counts: 711 us with a lane on a block and
// a walk over its runs, 276 us with the entries made by the group (the count
// of them before: 349 -> 114 us).
extern "C" __global__ void __launch_bounds__(gqf_flat::kThreads)
gqf_enum_emit(const QF* __restrict__ qfp, EnumRange r, uint64_t u0, const uint64_t* __restrict__ base, uint64_t skip,
              gqf_out_form o, uint64_t* __restrict__ hashes, uint64_t* __restrict__ counts,
              uint64_t* __restrict__ values, uint64_t cap) {
  __shared__ EnumSmem sm;
  const QF& f = *qfp;
  const uint64_t u = u0 + blockIdx.x;
  const uint64_t first = base[u] - skip;
  if (base[u + 1] == base[u] || first >= cap) return;
  gqf_flat::Window w;
  uint64_t b0;
  const bool fits = group_entries<true>(f, r, u, sm, w, b0);
  auto put = [&](uint64_t i, uint64_t s, uint64_t c) {
    if (i >= cap) return;
    if (hashes) hashes[i] = form_hash(o, s);
    if (counts) counts[i] = c;
    if (values) values[i] = s & gqf_mask((uint64_t)o.vb);
  };
  if (fits) {
    const uint32_t nbig = sm.n_big;
    for (uint32_t e = threadIdx.x; e < w.n; e += gqf_flat::kThreads) {
      const uint32_t y = sm.old[e];
      put(first + e, (b0 << 14) + (y >> 12), gqf_flat::full_count(sm, y >> 12, y & 0xFFFu, nbig));
    }
  } else if (threadIdx.x < 64) {
    uint64_t used;
    const uint32_t n = walk_group(f, r, b0, 0, [](uint32_t, uint64_t, uint64_t) {}, used);
    const uint32_t rank = wave_scan_add(n) - n;
    (void)walk_group(f, r, b0, rank, [&](uint32_t k, uint64_t s, uint64_t c) { put(first + k, s, c); }, used);
  }
}

// ---------------------------------------------------------------------------
// census

// used-slot mask of block b, slots >= xnslots excluded.  Slot 64 b + i is
// used iff the runs of earlier blocks reach it (i < offset) or some quotient
// of block b at or below it has not ended its run before it
// (offset_lower_bound != 0, src/gqf.cu:681-705).
static __device__ inline uint64_t used_mask(const QF& f, uint64_t b) {
  const gqf_header h = gqf_load_header(f, b);
  const uint64_t lim = f.xnslots - b * 64;
  return gqf_used_mask(h.occupieds, h.runends, h.offset, lim < 64 ? (uint32_t)lim : 64u);
}

// the mask every writer of the table keeps in the block's line
static __device__ inline uint64_t stored_used(const QF& f, uint64_t b) {
  return ((const GQF_GLOBAL uint64_t*)gqf_block_ptr(f, b))[3];
}

// Blocks whose stored used-slot mask (bytes 24..31) differs from the one
// their header implies: one thread per block, one atomic per mismatch.
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_check_used(const QF* __restrict__ qfp, unsigned long long* __restrict__ bad) {
  const QF& f = *qfp;
  const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= f.nblocks) return;
  if (stored_used(f, b) != used_mask(f, b)) atomicAdd(bad, 1ULL);
}

extern "C" __global__ void __launch_bounds__(kThreads)
gqf_census_mask(const QF* __restrict__ qfp, uint64_t* __restrict__ used, uint32_t* __restrict__ wg_starts) {
  const QF& f = *qfp;
  const uint64_t b = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  uint32_t starts = 0;
  if (b < f.nblocks) {
    const uint64_t u = stored_used(f, b);
    used[b] = u;
    const uint64_t prev = b ? stored_used(f, b - 1) >> 63 : 0;
    starts = (uint32_t)__builtin_popcountll(u & ~((u << 1) | prev));
  }
  uint32_t tot;
  (void)wg_exclusive_scan(starts, &tot);
  if (threadIdx.x == 0) wg_starts[blockIdx.x] = tot;
}

// Each workgroup takes runs of kThreads blocks, `step` workgroups apart, and
// adds its histogram and maximum to the result once: an atomic per thread on
// the one maximum took most of the pass (212 us at 2^26 slots,
// 49 us without).
extern "C" __global__ void __launch_bounds__(kThreads)
gqf_census_write(uint64_t nb, const uint64_t* __restrict__ used, const uint64_t* __restrict__ wg_base, uint32_t nwg,
                 uint64_t* __restrict__ lengths, uint64_t cap, unsigned long long* __restrict__ hist, uint32_t nbins,
                 unsigned long long* __restrict__ max_len) {
  extern __shared__ uint32_t lhist[];
  __shared__ unsigned long long wg_max;
  for (uint32_t i = threadIdx.x; i < nbins; i += kThreads) lhist[i] = 0;
  if (threadIdx.x == 0) wg_max = 0;
  __syncthreads();
  uint64_t my_max = 0;
  for (uint32_t g = blockIdx.x; g < nwg; g += gridDim.x) {
    const uint64_t b = (uint64_t)g * kThreads + threadIdx.x;
    uint64_t starts = 0, u = 0;
    if (b < nb) {
      u = used[b];
      starts = u & ~((u << 1) | (b ? used[b - 1] >> 63 : 0));
    }
    uint32_t tot;
    uint64_t r = wg_base[g] + wg_exclusive_scan((uint32_t)__builtin_popcountll(starts), &tot);
    while (starts) {
      const int i = __builtin_ctzll(starts);
      starts &= starts - 1;
      // first unused slot after 64 b + i
      uint64_t cb = b;
      uint64_t free_bits = ~u & (~0ULL << i);
      while (!free_bits && ++cb < nb) free_bits = ~used[cb];
      const uint64_t end = cb < nb ? cb * 64 + (uint64_t)__builtin_ctzll(free_bits) : nb * 64;
      const uint64_t len = end - (b * 64 + (uint64_t)i);
      if (lengths && r < cap) lengths[r] = len;
      r++;
      if (nbins) atomicAdd(&lhist[len < nbins ? len : nbins - 1], 1u);
      if (len > my_max) my_max = len;
    }
  }
  for (int d = 32; d >= 1; d >>= 1) {
    const uint64_t o = __shfl_xor(my_max, d, 64);
    my_max = o > my_max ? o : my_max;
  }
  if ((threadIdx.x & 63) == 0 && my_max) atomicMax(&wg_max, (unsigned long long)my_max);
  __syncthreads();
  if (hist)
    for (uint32_t i = threadIdx.x; i < nbins; i += kThreads)
      if (lhist[i]) atomicAdd(&hist[i], (unsigned long long)lhist[i]);
  if (threadIdx.x == 0 && wg_max) atomicMax(max_len, wg_max);
}

uint64_t gqf_enum_groups(uint64_t nblocks) { return (nblocks + GQF_ENUM_BLOCKS - 1) / GQF_ENUM_BLOCKS; }
uint64_t gqf_census_wgs(uint64_t nblocks) { return (nblocks + kThreads - 1) / kThreads; }

void gqf_launch_enum_count(const QF* qf_dev, uint64_t b_lo, uint64_t b_hi, uint64_t q_lo, uint64_t q_hi,
                           const gqf_enum_tables& t, hipStream_t s) {
  const uint64_t n = gqf_enum_groups(b_hi - b_lo);
  if (n == 0) return;
  gqf_prof_begin("enum_count", s);
  hipLaunchKernelGGL(gqf_enum_count, dim3((uint32_t)n), dim3(gqf_flat::kThreads), 0, s, qf_dev,
                     EnumRange{b_lo, b_hi, q_lo, q_hi}, t.items, t.slots, t.sums);
  gqf_prof_end("enum_count", s);
  hipLaunchKernelGGL(gqf_enum_scan, dim3(1), dim3(1024), 0, s, (const uint32_t*)t.items, (const uint32_t*)t.slots,
                     (const uint64_t*)t.sums, (uint32_t)n, t.base, t.stats);
}

void gqf_launch_enum_emit(const QF* qf_dev, uint64_t b_lo, uint64_t b_hi, uint64_t q_lo, uint64_t q_hi, uint64_t u0,
                          uint64_t u1, const uint64_t* base, uint64_t skip, int mode, int vb, int dst_vb,
                          uint64_t key_mask, uint64_t* hashes, uint64_t* counts, uint64_t* values, uint64_t cap,
                          hipStream_t s) {
  if (u1 <= u0) return;
  const gqf_out_form o{mode, vb, dst_vb, key_mask};
  gqf_prof_begin("enum_emit", s);
  hipLaunchKernelGGL(gqf_enum_emit, dim3((uint32_t)(u1 - u0)), dim3(gqf_flat::kThreads), 0, s, qf_dev,
                     EnumRange{b_lo, b_hi, q_lo, q_hi}, u0, base, skip, o, hashes, counts, values, cap);
  gqf_prof_end("enum_emit", s);
}

void gqf_launch_check_used(const QF* qf_dev, uint64_t nblocks, unsigned long long* bad, hipStream_t s) {
  if (nblocks == 0) return;
  hipLaunchKernelGGL(gqf_check_used, dim3((uint32_t)((nblocks + kThreads - 1) / kThreads)), dim3(kThreads), 0, s,
                     qf_dev, bad);
}

void gqf_launch_census(const QF* qf_dev, uint64_t nblocks, uint64_t* used, uint32_t* wg_starts, uint64_t* wg_base,
                       uint64_t* lengths, uint64_t cap, unsigned long long* hist, uint32_t nbins,
                       unsigned long long* max_len, hipStream_t s) {
  const uint64_t nwg = gqf_census_wgs(nblocks);
  if (nwg == 0) return;
  gqf_prof_begin("census_mask", s);
  hipLaunchKernelGGL(gqf_census_mask, dim3((uint32_t)nwg), dim3(kThreads), 0, s, qf_dev, used, wg_starts);
  gqf_prof_end("census_mask", s);
  hipLaunchKernelGGL(gqf_enum_scan, dim3(1), dim3(1024), 0, s, (const uint32_t*)wg_starts, (const uint32_t*)nullptr,
                     (const uint64_t*)nullptr, (uint32_t)nwg, wg_base, (uint64_t*)nullptr);
  gqf_prof_begin("census_write", s);
  hipLaunchKernelGGL(gqf_census_write, dim3((uint32_t)(nwg < 1024 ? nwg : 1024)), dim3(kThreads),
                     nbins * sizeof(uint32_t), s, nblocks, (const uint64_t*)used, (const uint64_t*)wg_base,
                     (uint32_t)nwg, lengths, cap, hist, nbins, max_len);
  gqf_prof_end("census_write", s);
}
