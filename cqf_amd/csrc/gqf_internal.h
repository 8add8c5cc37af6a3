// gqf_internal.h -- constants and helpers private to the libgqf kernels
// (counting quotient filter for gfx950).  The table layout, the filter
// descriptor and the shared device helpers live in the public device
// header gqf_device.h.
#pragma once

#define GQF_NO_POINT_BULK_KERNEL  // the library launches its own point kernels (gqf_point.hip)
#include "gqf_device.h"

#define GQF_REGION_BLOCKS 48      // default rebuild region; + 16 push blocks = one wave64
#define GQF_REGION_BLOCKS_MIN 16  // tunable range (the push window is min(64, 2 x region) - region blocks)
#define GQF_REGION_BLOCKS_MAX 56

// Largest batch one pass of the bulk pipeline takes (its region starts,
// sort histograms and reduce counts are 32-bit); longer batches are cut
// into pieces of this size.
#define GQF_MAX_PIECE (1ULL << 30)

// Cuts n keys into consecutive pieces of at most max_piece keys (max_piece
// >= 1): piece k is [starts[k], starts[k + 1]).  Returns the number of
// pieces p (0 for n = 0) and writes starts[0..p] when p + 1 <= cap; p is
// returned either way, so a caller can size the array.
static inline uint32_t gqf_batch_pieces(uint64_t n, uint64_t max_piece, uint64_t* starts, uint32_t cap) {
  if (max_piece == 0) return 0;
  const uint64_t p = n / max_piece + (n % max_piece ? 1 : 0);
  if (p + 1 <= cap && starts) {
    for (uint64_t k = 0; k < p; k++) starts[k] = k * max_piece;
    starts[p] = n;
  }
  return (uint32_t)p;
}

// status bits reported through qf_get_status()
#define GQF_STATUS_NO_SPACE QF_STATUS_NO_SPACE                  // a run would end past xnslots; region left unchanged
#define GQF_STATUS_CLUSTER_OVERFLOW QF_STATUS_CLUSTER_OVERFLOW  // push longer than the widest window
#define GQF_STATUS_BAD_HASH QF_STATUS_BAD_HASH                  // pre-hashed key >= range; key ignored
#define GQF_STATUS_POINT_FULL QF_STATUS_POINT_FULL              // a point insert found no empty slot

// The first of the n > 0 `items`, sorted by hash (their bits in hmask), whose
// hash is not below h, and `item`, that item (where it is not n).  Hashes are
// spread evenly, so it is looked for at h's share of the items' range (from
// h0 on, `per` items per hash value) and twice more at the distance that the
// item there shows (about sqrt(n) / 2 items off, then the square root of
// that, and its root), then between steps that widen from there, and by
// halves; items with few distinct hashes cost some steps more.
// Bound by its chain of loads, and in a sequenced batch's queries by the rate
// of loads that miss L1, as nearly all of these do (16 waves a CU pass through
// it): halving the whole batch takes 20 of them for 0.7 M items and took 127
// us for 1.65 M queries, this takes 8 and 77 us; the bounds of 11,000 regions
// among 4 M
// items 16 and 11 us.
__device__ __forceinline__ uint64_t gqf_first_item(const uint64_t* __restrict__ items, uint64_t n, uint64_t hmask,
                                                   uint64_t h, double h0, double per, uint64_t& item) {
  auto guess = [&](double x) -> uint64_t {
    return x > 0.0 ? (x < (double)n ? (uint64_t)x : n - 1) : 0ULL;
  };
  uint64_t g = guess(((double)h - h0) * per), v = items[g];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    g = guess((double)g + ((double)h - (double)(v & hmask)) * per);
    v = items[g];
  }
  const bool up = (v & hmask) < h;
  uint64_t lo = up ? g + 1 : 0, hi = up ? n : g;  // items before lo are below h, those from hi on are not
  item = v;                                       // item hi, where hi < n
  auto look = [&](uint64_t p) {
    const uint64_t t = items[p];
    const bool below = (t & hmask) < h;
    if (below) lo = p + 1; else hi = p, item = t;
    return below;
  };
  for (uint64_t step = 8; (up ? n - lo : hi) >= step; step *= 4)
    if (look(up ? lo + step - 1 : hi - step) != up) break;
  while (lo < hi) look((lo + hi) >> 1);
  return lo;
}

// Inclusive sum over the 64 lanes of a wave on DPP row shifts (1, 2, 4, 8
// within each row of 16 lanes) and row broadcasts (lane 15 into rows 1 and
// 3, then lane 31 into rows 2 and 3): six VALU steps that read the
// neighbouring lanes' registers, no LDS round trip.  All lanes must be
// active.
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return x;
}
