// radix_tile.hpp — pieces that the workgroup-tile radix passes share: the
// transpose / COO -> CSR sorts (transpose.hip) and the scattered-product
// SpMV (spmv_scatter.hip).
#pragma once

#include "fs_common.hpp"

namespace fs {

__device__ inline int lane_id_t() {
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}
__device__ inline int count_below_t(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}
__device__ inline void wave_sync_t() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lanes among `active` whose digit equals this lane's, over the low bits
// set in `mask` (a uniform value, contiguous from bit 0, at most MAXBITS).
// Per bit: the bit spread over a word, its ballot m, and one three-input
// operation per half, peers & ~(m ^ spread) (truth table 0x90).  The kernels
// that rank entries are bound by VALU issue (4 cycles an instruction): 4
// instructions a bit instead of the 8 that selects and ands came to.
template <int MAXBITS>
__device__ inline uint64_t match_lanes(unsigned digit, uint64_t active, unsigned mask) {
  unsigned lo = (unsigned)active, hi = (unsigned)(active >> 32);
#pragma unroll
  for (int b = 0; b < MAXBITS; ++b) {
    if (!((mask >> b) & 1u)) break;
    const int spread = __builtin_amdgcn_sbfe((int)digit, b, 1);
    const uint64_t m = __ballot(spread != 0);
    lo = (unsigned)__builtin_amdgcn_bitop3_b32((int)lo, (int)(unsigned)m, spread, 0x90);
    hi = (unsigned)__builtin_amdgcn_bitop3_b32((int)hi, (int)(unsigned)(m >> 32), spread, 0x90);
  }
  return ((uint64_t)hi << 32) | lo;
}

// Tile of workgroup b out of n so that each of the 8 XCDs (to which
// workgroups are dealt in turn) walks one contiguous range of tiles: the
// runs that neighbouring tiles of a scatter write for one digit or panel
// are adjacent in the output, so they meet in the same L2 and leave it as
// whole lines.
__device__ inline int64_t xcd_tile(uint32_t b, uint32_t n) {
  constexpr uint32_t kXcds = 8;
  const uint32_t q = n / kXcds, r = n % kXcds, x = b % kXcds, i = b / kXcds;
  return x < r ? (int64_t)x * (q + 1) + i : (int64_t)r * (q + 1) + (int64_t)(x - r) * q + i;
}

__device__ inline int64_t block_exclusive_scan(int64_t v, int64_t* s_wave, int64_t& total) {
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  int64_t x = v;
  for (int off = 1; off < 64; off <<= 1) {
    int lo = __builtin_amdgcn_ds_bpermute((lane - off) << 2, (int)(x & 0xffffffff));
    int hi = __builtin_amdgcn_ds_bpermute((lane - off) << 2, (int)(x >> 32));
    int64_t y = ((int64_t)hi << 32) | (uint32_t)lo;
    if (lane >= off) x += y;
  }
  if (lane == 63) s_wave[w] = x;
  __syncthreads();
  int64_t wave_base = 0;
  total = 0;
  for (int k = 0; k < (int)(blockDim.x >> 6); ++k) {
    if (k < w) wave_base += s_wave[k];
    total += s_wave[k];
  }
  __syncthreads();
  return wave_base + x - v;
}

// Inclusive max-scan over the wave (DPP row shifts within 16-lane rows,
// then row broadcasts across them; lanes without a source read 0, the
// identity of an unsigned max).
template <int CTRL, int ROWMASK>
__device__ inline unsigned dpp_shift_u(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWMASK, 0xF, false);
}
__device__ inline unsigned umax_(unsigned a, unsigned b) { return a > b ? a : b; }
__device__ inline unsigned wave_max_scan(unsigned v) {
  v = umax_(v, dpp_shift_u<0x111, 0xF>(v));  // row_shr:1
  v = umax_(v, dpp_shift_u<0x112, 0xF>(v));  // row_shr:2
  v = umax_(v, dpp_shift_u<0x114, 0xF>(v));  // row_shr:4
  v = umax_(v, dpp_shift_u<0x118, 0xF>(v));  // row_shr:8
  v = umax_(v, dpp_shift_u<0x142, 0xA>(v));  // row_bcast:15 -> rows 1, 3
  v = umax_(v, dpp_shift_u<0x143, 0xC>(v));  // row_bcast:31 -> rows 2, 3
  return v;
}

// ---- workgroup-tile radix passes (the transpose of 4- and 8-byte values) ----
// A workgroup of kWgWaves waves sorts a tile of kWgTile entries per pass
// (wave w holds entries [w * kWgSub, (w + 1) * kWgSub) of the tile in
// registers, kWgChunks per lane, and ranks them as radix_scatter_kernel
// does, against its own LDS counters).  The larger tile allows more digits
// at the same run length per digit, up to 11 key bits per pass: the 20-bit
// columns of a 1M-column matrix take two passes instead of three.  The
// payload carries the entry's value and row (an 8-byte word for 4-byte
// values, 12 bytes for 8-byte values), built by the first pass from the
// CSR arrays and written out as the transposed values and rows by the last,
// and the last pass writes no keys: the column pointer comes from an atomic
// minimum of the first position of each column the tile holds, and a
// suffix minimum over the columns (empty columns take the next one's start).
#ifndef FS_WG_WAVES
#define FS_WG_WAVES 8
#endif
#ifndef FS_WG_CHUNKS
#define FS_WG_CHUNKS 12
#endif
#ifndef FS_WG_MIN_WAVES
#define FS_WG_MIN_WAVES 4
#endif
constexpr int kWgWaves = FS_WG_WAVES;
constexpr int kWgThreads = 64 * kWgWaves;
constexpr int kWgChunks = FS_WG_CHUNKS;
constexpr int64_t kWgSub = 64 * kWgChunks;
constexpr int64_t kWgTile = kWgWaves * kWgSub;
constexpr int kWgMaxBits = 11;
constexpr int kWgScanTiles = 16;  // tiles per block of the digit scan
constexpr int kWgMaxDigits = 1 << kWgMaxBits;
// staging buffer: row marks, wave counters, keys, then the payload in
// windows (a multiple of 8 and 12 bytes; half a tile of 12-byte payload, so
// the payload leaves in two windows)
constexpr int kWgBufHalf = (int)(kWgTile / 2) * 12;
constexpr int kWgBufMin = kWgWaves * kWgMaxDigits * 2 > kWgBufHalf ? kWgWaves * kWgMaxDigits * 2 : kWgBufHalf;
constexpr int kWgBufBytes = (kWgBufMin + 23) / 24 * 24;
// the wave counters hold two digits per word (16-bit counts: a wave ranks
// at most kWgSub entries, a tile at most kWgTile < 2^16)
static_assert(kWgTile < 65536, "16-bit digit counters");
static_assert(kWgWaves * kWgMaxDigits * 2 <= kWgBufBytes, "wave counters fit the staging buffer");
static_assert(kWgTile * 4 <= kWgBufBytes, "row marks and keys fit the staging buffer");

// Keys of a wave sub-tile: `cnt` entries from `base` (kind 1: 8-byte
// column indices below 2^32; otherwise 4-byte keys); one per-lane base
// pointer, the chunks at immediate offsets from it.
// (FULL: the sub-tile has all its entries, so no lane tests are made.)
template <bool FULL = false>
__device__ inline void wg_load_keys(const void* keys, int kind, int64_t base, int cnt, int lane,
                                    uint32_t (&key)[kWgChunks]) {
  if (kind == 5 || kind == 6) {  // one word of each 8- / 12-byte payload (`keys` points at it)
    const int W = kind == 5 ? 2 : 3;
    const uint32_t* p = static_cast<const uint32_t*>(keys) + (base + lane) * W;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) key[ch] = FULL || ch * 64 + lane < cnt ? p[ch * 64 * W] : 0u;
  } else if (kind == 1) {
    const int64_t* p = static_cast<const int64_t*>(keys) + base + lane;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) key[ch] = FULL || ch * 64 + lane < cnt ? (uint32_t)p[ch * 64] : 0u;
  } else {
    const uint32_t* p = static_cast<const uint32_t*>(keys) + base + lane;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) key[ch] = FULL || ch * 64 + lane < cnt ? p[ch * 64] : 0u;
  }
}

// Row of every entry of a wave sub-tile (rows r0..r1 touch it): each row
// starting inside marks its first entry with r - r0, and a wave max-scan
// carried across the chunks gives entry j the largest mark at or before j.
template <class P>
__device__ inline void wg_rows(const P* __restrict__ rowptr, int64_t r0, int64_t r1, int64_t base, int cnt,
                               unsigned* s_mark, int lane, uint32_t (&row)[kWgChunks]) {
  for (int j = lane; j < (int)kWgSub; j += 64) s_mark[j] = 0u;
  wave_sync_t();
  for (int64_t r = r0 + 1 + lane; r <= r1; r += 64) {
    const int64_t st = (int64_t)rowptr[r];
    // (st >= base on a valid row pointer; the test keeps a malformed one,
    // which the caller's structure check reports, inside the tile's marks)
    if (st >= base && st - base < cnt && (int64_t)rowptr[r + 1] > st) s_mark[st - base] = (unsigned)(r - r0);
  }
  wave_sync_t();
  unsigned carry = 0u;
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch) {
    const unsigned m = umax_(wave_max_scan(s_mark[ch * 64 + lane]), carry);
    carry = (unsigned)__builtin_amdgcn_readlane((int)m, 63);
    row[ch] = (uint32_t)(r0 + (int64_t)m);
  }
}

constexpr int kDigitScanBatch = 16;  // loads in flight per thread of the digit scan

// Exclusive scan of cnt[tile][d] in (digit, tile) order (nd digits, up to
// kWgMaxDigits): per-block digit sums over kWgScanTiles tiles, one
// workgroup per digit scanning its block sums, then the downsweep.
static __global__ __launch_bounds__(256) void wg_scan_reduce_kernel(const uint32_t* __restrict__ cnt, int64_t n_tiles,
                                                             int nd, uint32_t* __restrict__ partial) {
  const int64_t s0 = (int64_t)blockIdx.x * kWgScanTiles;
  const int64_t s1 = s0 + kWgScanTiles < n_tiles ? s0 + kWgScanTiles : n_tiles;
  for (int d = threadIdx.x; d < nd; d += 256) {
    uint32_t sum = 0;
    for (int64_t s = s0; s < s1; s += kDigitScanBatch) {
      uint32_t v[kDigitScanBatch];
#pragma unroll
      for (int k = 0; k < kDigitScanBatch; ++k) v[k] = s + k < s1 ? cnt[(s + k) * nd + d] : 0u;
#pragma unroll
      for (int k = 0; k < kDigitScanBatch; ++k) sum += v[k];
    }
    partial[(int64_t)blockIdx.x * nd + d] = sum;
  }
}

static __global__ __launch_bounds__(256) void wg_scan_column_kernel(uint32_t* __restrict__ partial, int64_t n_blocks, int nd,
                                                             uint32_t* __restrict__ totals) {
  __shared__ int64_t s_wave[4];
  const int d = blockIdx.x;
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < n_blocks; b0 += 256) {
    const int64_t b = b0 + threadIdx.x;
    const int64_t v = b < n_blocks ? (int64_t)partial[b * nd + d] : 0;
    int64_t sum;
    const int64_t ex = block_exclusive_scan(v, s_wave, sum);
    if (b < n_blocks) partial[b * nd + d] = (uint32_t)(carry + ex);
    carry += sum;
  }
  if (threadIdx.x == 0) totals[d] = (uint32_t)carry;
}

static __global__ __launch_bounds__(256) void wg_scan_down_kernel(uint32_t* __restrict__ cnt, int64_t n_tiles, int nd,
                                                           const uint32_t* __restrict__ partial,
                                                           const uint32_t* __restrict__ totals) {
  __shared__ int64_t s_wave[4];
  __shared__ uint32_t s_base[kWgMaxDigits];
  // digit starts: thread t scans digits [t q, t q + q)
  const int q = (nd + 255) / 256;
  const int d0 = threadIdx.x * q;
  int64_t mine = 0;
  for (int j = 0; j < q; ++j)
    if (d0 + j < nd) mine += totals[d0 + j];
  int64_t all;
  int64_t run = block_exclusive_scan(mine, s_wave, all);
  for (int j = 0; j < q; ++j)
    if (d0 + j < nd) {
      s_base[d0 + j] = (uint32_t)run;
      run += totals[d0 + j];
    }
  __syncthreads();
  const int64_t s0 = (int64_t)blockIdx.x * kWgScanTiles;
  const int64_t s1 = s0 + kWgScanTiles < n_tiles ? s0 + kWgScanTiles : n_tiles;
  for (int d = threadIdx.x; d < nd; d += 256) {
    uint32_t r = s_base[d] + partial[(int64_t)blockIdx.x * nd + d];
    for (int64_t s = s0; s < s1; s += kDigitScanBatch) {
      uint32_t v[kDigitScanBatch];
#pragma unroll
      for (int k = 0; k < kDigitScanBatch; ++k) v[k] = s + k < s1 ? cnt[(s + k) * nd + d] : 0u;
#pragma unroll
      for (int k = 0; k < kDigitScanBatch; ++k) {
        if (s + k < s1) cnt[(s + k) * nd + d] = r;
        r += v[k];
      }
    }
  }
}

}  // namespace fs
