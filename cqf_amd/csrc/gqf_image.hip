// gqf_image.hip -- conversion from the device layout (128-byte blocks with an
// exact 32-bit offset) to the reference's packed 81-byte block image
// (include/gqf_int.cuh:38-57): offset u8 saturated at 255, occupieds u64,
// runends u64, 64 slot bytes.  This is the parity / serialisation format.
#include "gqf_internal.h"
#include "gqf_launch.h"

namespace {

// Each workgroup packs kExportBlocks blocks.  A thread loads one block's line
// (six 16-byte loads; the line's second half-header is not read) and writes
// its 81 bytes to an LDS row of 21 words: everything past the offset byte is
// the line's words moved up one byte, so a row is 20 funnel shifts, and an
// odd row length keeps the rows' columns on different banks.  The rows leave
// as 16-byte stores: a word of output is a funnel shift of two words of a
// row, or, at a row's end, of its tail and the next row's head.
// HBM bound (96 B read, 81 B written per block).  A gather of single bytes
// (one thread per 8 output bytes, eight dependent address computations) took
// 484 us at 2^28 slots and 29 us at 2^24; this takes 145 us (6.1 TB/s) and
// 14 us.
constexpr int kExportBlocks = 256;
constexpr int kExportRow = 21;

__global__ void __launch_bounds__(kExportBlocks) gqf_export_kernel(const QF* __restrict__ qfp, uint8_t* __restrict__ out) {
  __shared__ uint32_t rows[kExportBlocks * kExportRow + 1];  // + 1: the last row's look-ahead
  const QF& qf = *qfp;
  const uint64_t nblocks = qf.nblocks;
  const uint64_t b0 = (uint64_t)blockIdx.x * kExportBlocks;
  if (b0 >= nblocks) return;
  const uint32_t nb = (uint32_t)(nblocks - b0 < kExportBlocks ? nblocks - b0 : kExportBlocks);
  const uint32_t t = threadIdx.x;
  if (t < nb) {
    const GQF_GLOBAL uint4* p = gqf_block_ptr(qf, b0 + t);
    const uint4 h = p[0];
    const uint32_t off = ((const GQF_GLOBAL uint32_t*)p)[4];
    uint4 s[4];
#pragma unroll
    for (int k = 0; k < 4; k++) s[k] = p[4 + k];
    uint32_t w[21];
    w[0] = off < GQF_OFFSET_SAT ? off : GQF_OFFSET_SAT;
    w[0] <<= 24;  // the byte before the first word
    w[1] = h.x; w[2] = h.y; w[3] = h.z; w[4] = h.w;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      w[5 + 4 * k] = s[k].x; w[6 + 4 * k] = s[k].y; w[7 + 4 * k] = s[k].z; w[8 + 4 * k] = s[k].w;
    }
    uint32_t* row = rows + kExportRow * t;
#pragma unroll
    for (int k = 0; k < 20; k++) row[k] = __builtin_amdgcn_alignbit(w[k + 1], w[k], 24);
    row[20] = w[20] >> 24;
  }
  __syncthreads();
  const uint32_t bytes = nb * GQF_REF_BLOCK_BYTES;
  uint8_t* dst = out + b0 * GQF_REF_BLOCK_BYTES;
  // the output word at byte `at` of the workgroup's share (bytes past it are junk)
  auto word = [&](uint32_t at) {
    const uint32_t b = at / GQF_REF_BLOCK_BYTES, o = at - b * GQF_REF_BLOCK_BYTES;
    const uint32_t* r = rows + kExportRow * b + (o >> 2);
    // in a row's last word (o >= 80: one byte left) the next row's head follows
    const uint32_t sh = (o & 3u) * 8u;
    if (o < GQF_REF_BLOCK_BYTES - 3) return (uint32_t)__builtin_amdgcn_alignbit(r[1], r[0], sh);
    const uint32_t left = GQF_REF_BLOCK_BYTES - o;  // 1..3 bytes of this row
    const uint32_t* nx = rows + kExportRow * (b + 1 < nb ? b + 1 : b);
    const uint32_t mine = o == GQF_REF_BLOCK_BYTES - 1 ? r[0] : (uint32_t)__builtin_amdgcn_alignbit(r[1], r[0], sh);
    return (mine & (0xFFFFFFFFu >> (32 - 8 * left))) | (nx[0] << (8 * left));
  };
  if (((uintptr_t)dst & 15) == 0) {
    for (uint32_t at = 16 * t; at + 16 <= bytes; at += 16 * kExportBlocks)
      *(uint4*)(dst + at) = make_uint4(word(at), word(at + 4), word(at + 8), word(at + 12));
    for (uint32_t i = (bytes & ~15u) + t; i < bytes; i += kExportBlocks) dst[i] = (uint8_t)word(i);
  } else {
    for (uint32_t i = t; i < bytes; i += kExportBlocks) dst[i] = (uint8_t)word(i);
  }
}

}  // namespace

void gqf_launch_export(const QF* qf_dev, uint64_t nblocks, uint8_t* out, hipStream_t s) {
  const uint64_t grid = (nblocks + kExportBlocks - 1) / kExportBlocks;
  if (grid == 0) return;
  hipLaunchKernelGGL(gqf_export_kernel, dim3((uint32_t)grid), dim3(kExportBlocks), 0, s, qf_dev, out);
}
