// transpose.hip — CSR -> CSR of A^T (or A^H) on gfx950, bit-exact with a
// stable sort of the entries by column.
//
// Reference: _transpose_csr_for_spmv (spmv_csr.py:477-515) and
// _transpose_csr_for_spmm (spmm_csr.py:300-338) expand row ids
// (repeat_interleave), stable-argsort the column indices, gather data and
// row ids, and build the new indptr with bincount + cumsum; conj is applied
// to the data first (spmv_csr.py:615-618, spmm_csr.py:341-349).
//
// Here: an LSD radix sort over the column index.  Within a tile, lanes
// holding equal digits find each other with ballots ("peer masks") and take
// their ranks from one returning LDS atomic per group, in input order, so
// equal keys keep their input order: the result is the reference's stable
// argsort, bit for bit.  Per pass: per-tile digit counts -> exclusive scan
// over (digit, tile) -> a scatter that sorts the tile by digit in LDS first,
// so that every digit's entries leave as one contiguous run.
//  - 4- and 8-byte values (positions below 2^32): workgroup tiles of
//    kWgTile entries, up to 11 key bits per pass, the (value, row) payload
//    built by the first pass and written out by the last, the column pointer
//    from integer atomic minima and a suffix minimum (wg_* kernels);
//    COO -> CSR runs on the same passes (column, then row).
//  - otherwise: wave tiles of kSub entries, up to 8 bits per pass, positions
//    through the sort and a gather at the end, the column pointer read off
//    the sorted keys (radix_* kernels).
#include "fs_common.hpp"
#include "radix_tile.hpp"
#include "row_starts.hpp"

#include <algorithm>
#include <type_traits>
#include <cstring>

namespace fs {

constexpr int kRadixBits = 8;
constexpr int kDigits = 1 << kRadixBits;
#ifndef FS_RADIX_CHUNKS
#define FS_RADIX_CHUNKS 32
#endif
constexpr int kChunks = FS_RADIX_CHUNKS;    // 64-entry chunks per wave sub-tile
constexpr int64_t kSub = 64 * kChunks;      // entries per wave sub-tile
constexpr int kWavesPerBlock = 4;
constexpr int kScanItems = 16;              // per-thread items in the scan kernels
constexpr int64_t kScanTile = 256 * kScanItems;

// Key source: pass 0 reads the CSR column indices directly.
template <class K>
__device__ inline K load_key(const void* src, int kind, int64_t e) {
  if (kind == 0) return (K)(uint32_t) static_cast<const int32_t*>(src)[e];
  if (kind == 1) return (K)(uint64_t) static_cast<const int64_t*>(src)[e];
  return static_cast<const K*>(src)[e];
}

// A wave's sub-tile lives in registers: lane l holds entries l, l + 64, ...
// (chunk c = entries [64c, 64c + 64) of the sub-tile), loaded with all loads
// in flight before any is used.
template <class K>
__device__ inline void load_tile_keys(const void* keys, int kind, int64_t base, int64_t n, int lane,
                                      K (&key)[kChunks]) {
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const int64_t e = base + (int64_t)ch * 64 + lane;
    key[ch] = e < n ? load_key<K>(keys, kind, e) : (K)0;
  }
}

template <class K, class CT>
__global__ __launch_bounds__(256) void radix_count_kernel(const void* __restrict__ keys, int kind, int64_t n,
                                                          int shift, unsigned mask, int64_t n_sub,
                                                          CT* __restrict__ counts) {
  __shared__ unsigned s_hist[kWavesPerBlock][kDigits];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int64_t sub = (int64_t)blockIdx.x * kWavesPerBlock + w;
  if (sub >= n_sub) return;  // wave-local work only
  unsigned* hist = s_hist[w];
  for (int d = lane; d < kDigits; d += 64) hist[d] = 0;
  const int64_t base = sub * kSub;
  K key[kChunks];
  load_tile_keys<K>(keys, kind, base, n, lane, key);
  wave_sync_t();
  // Counts only (no ranks): one LDS integer atomic per entry.  Integer sums do
  // not depend on order, so the counts are deterministic; the stable ranks
  // come from the scatter pass.  (Ballot peer groups here measured 98 us per
  // pass on 33.5 M keys.)
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    if (base + (int64_t)ch * 64 + lane < n) atomicAdd(&hist[(unsigned)(key[ch] >> shift) & mask], 1u);
  }
  wave_sync_t();
  // sub-tile-major: the wave's 256 counts leave as one contiguous row (the
  // digit-major layout made them 256 scattered 8-byte stores per wave)
  for (int d = lane; d < kDigits; d += 64) counts[sub * kDigits + d] = (CT)hist[d];
}

// ---- exclusive scan of the counts in (digit, sub-tile) order ----
// The counts are stored sub-tile-major, cnt[sub][digit]; the scatter needs
// for every (sub, digit) the number of entries with a smaller digit, plus
// those with the same digit in earlier sub-tiles.  Thread t of a workgroup
// owns digit t, and a workgroup owns kDigitScanSubs consecutive sub-tiles,
// so every load and store is a coalesced row: per-block digit sums, one
// workgroup scanning those in (digit, block) order, then a downsweep.
constexpr int kDigitScanSubs = 64;

// (loads are issued kScanBatch at a time before they are summed: a plain
// loop over dependent sums left the one-workgroup top scan at 83 us on 256
// blocks)
constexpr int kScanBatch = 16;

template <class CT>
__global__ __launch_bounds__(256) void digit_scan_reduce_kernel(const CT* __restrict__ cnt, int64_t n_sub,
                                                                CT* __restrict__ partial) {
  const int t = threadIdx.x;
  const int64_t s0 = (int64_t)blockIdx.x * kDigitScanSubs;
  const int64_t s1 = s0 + kDigitScanSubs < n_sub ? s0 + kDigitScanSubs : n_sub;
  CT sum = 0;
  for (int64_t s = s0; s < s1; s += kScanBatch) {
    CT v[kScanBatch];
#pragma unroll
    for (int k = 0; k < kScanBatch; ++k) v[k] = s + k < s1 ? cnt[(s + k) * kDigits + t] : (CT)0;
#pragma unroll
    for (int k = 0; k < kScanBatch; ++k) sum += v[k];
  }
  partial[(int64_t)blockIdx.x * kDigits + t] = sum;
}

// One workgroup per digit: the exclusive prefix of that digit's block sums
// over the blocks (in place), and the digit's total into totals[digit].
// (A single workgroup walking every digit's column took 27 us per pass on
// C4: one CU's bandwidth.)
template <class CT>
__global__ __launch_bounds__(256) void digit_scan_column_kernel(CT* __restrict__ partial, int64_t n_blocks,
                                                                int64_t* __restrict__ totals) {
  __shared__ int64_t s_wave[4];
  const int d = blockIdx.x;
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < n_blocks; b0 += 256) {
    const int64_t b = b0 + threadIdx.x;
    const int64_t v = b < n_blocks ? (int64_t)partial[b * kDigits + d] : 0;
    int64_t sum;
    const int64_t ex = block_exclusive_scan(v, s_wave, sum);
    if (b < n_blocks) partial[b * kDigits + d] = (CT)(carry + ex);
    carry += sum;
  }
  if (threadIdx.x == 0) totals[d] = carry;
}

// Per block: every sub-tile's offset = the digit's base (the digits below it,
// from the 256 totals) + the block's prefix within the digit + the sub-tiles
// before it in the block.
template <class CT>
__global__ __launch_bounds__(256) void digit_scan_down_kernel(CT* __restrict__ cnt, int64_t n_sub,
                                                              const CT* __restrict__ partial,
                                                              const int64_t* __restrict__ totals) {
  __shared__ int64_t s_wave[4];
  const int t = threadIdx.x;
  int64_t all;
  const int64_t base = block_exclusive_scan(totals[t], s_wave, all);
  const int64_t s0 = (int64_t)blockIdx.x * kDigitScanSubs;
  const int64_t s1 = s0 + kDigitScanSubs < n_sub ? s0 + kDigitScanSubs : n_sub;
  CT run = (CT)(base + (int64_t)partial[(int64_t)blockIdx.x * kDigits + t]);
  for (int64_t s = s0; s < s1; s += kScanBatch) {
    CT v[kScanBatch];
#pragma unroll
    for (int k = 0; k < kScanBatch; ++k) v[k] = s + k < s1 ? cnt[(s + k) * kDigits + t] : (CT)0;
#pragma unroll
    for (int k = 0; k < kScanBatch; ++k) {
      if (s + k < s1) cnt[(s + k) * kDigits + t] = run;
      run += v[k];
    }
  }
}

// Exclusive scan of 256 per-digit counts held 4 per lane (digits 4l..4l+3);
// writes the starts to out[256].
__device__ inline void wave_digit_scan(const unsigned (&c)[4], int lane, unsigned* out) {
  const unsigned lane_sum = c[0] + c[1] + c[2] + c[3];
  unsigned incl = lane_sum;
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned y = (unsigned)__builtin_amdgcn_ds_bpermute((lane - off) << 2, (int)incl);
    if (lane >= off) incl += y;
  }
  unsigned run = incl - lane_sum;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    out[4 * lane + k] = run;
    run += c[k];
  }
}

// Extra inputs / outputs of the transpose's fused first and last passes
// (4-byte values with row ids below 2^32): the first pass builds each
// entry's (value, row) word from the CSR arrays itself, the last writes the
// transposed values and row indices straight from the words.
struct FusedIO {
  const uint32_t* vals;     // first pass: the CSR values (4-byte words)
  const void* rowptr;       // first pass: the CSR row pointer (type P)
  const int64_t* tile_row;  // first pass: row of each sub-tile's first entry
  int64_t n_rows;
  uint32_t* t_vals;         // last pass: transposed values
  void* t_cols;             // last pass: transposed column indices (type OI)
};

constexpr int kScatterPlain = 0;  // keys + payload in, keys + payload out
constexpr int kScatterFirst = 1;  // payload built from values and row ids
constexpr int kScatterLast = 2;   // payload out as transposed values / rows
constexpr int kScatterOnly = 3;   // first and last (a single pass)

// Row marks of a sub-tile (kSub entries from `base`, rows r0..r1 touching
// it): every row that starts inside the tile marks its first entry with
// r - r0 in s_mark (rows read with unit stride, empty rows mark nothing).
// The row of entry j is then r0 + the largest mark at or before j.
template <class P>
__device__ inline void tile_row_marks(const P* __restrict__ rowptr, int64_t r0, int64_t r1, int64_t base, int cnt,
                                      unsigned* s_mark, int lane) {
  for (int j = lane; j < (int)kSub; j += 64) s_mark[j] = 0u;
  wave_sync_t();
  for (int64_t r = r0 + 1 + lane; r <= r1; r += 64) {
    const int64_t st = (int64_t)rowptr[r];
    if (st - base < cnt && (int64_t)rowptr[r + 1] > st) s_mark[st - base] = (unsigned)(r - r0);
  }
  wave_sync_t();
}

// Stable scatter of one pass.  One wave per sub-tile (kSub entries):
//  1. keys / payload into registers (all loads in flight);
//  2. every entry's rank within its digit, chunk by chunk in input order:
//     the lanes of a chunk holding the same digit find each other with
//     ballots (peer masks); the lowest of them adds the group's size to the
//     digit's LDS counter with one returning atomic and hands the old value
//     to its peers.  A wave's LDS operations complete in issue order, so
//     chunk c sees every earlier chunk's additions and equal digits keep
//     their input order (the sort is stable) without a barrier per chunk;
//  3. the counters, now the tile's digit counts, scanned into digit starts;
//  4. the keys, then the payload, through one digit-sorted LDS copy of the
//     tile, written out in order: entry i of digit d goes to
//     offsets[sub][d] + (i - start[d]), so a digit's entries leave as one
//     contiguous run instead of single scattered stores.
// MODE kScatterFirst / kScatterLast / kScatterOnly fuse the transpose's
// (value, row) packing into the first pass and its unpacking into the last
// (FusedIO; Pos is then the 8-byte word, value in the low half).
template <class K, class Pos, class CT, int MODE = kScatterPlain, class P = int32_t, class OI = int32_t>
__global__ __launch_bounds__(64, 2) void radix_scatter_kernel(const void* __restrict__ keys_in, int kind,
                                                           const Pos* __restrict__ pos_in, int64_t n, int shift,
                                                           unsigned mask, int64_t n_sub, const CT* __restrict__ offsets,
                                                           K* __restrict__ keys_out, Pos* __restrict__ pos_out,
                                                           FusedIO io) {
  constexpr bool kFirst = MODE == kScatterFirst || MODE == kScatterOnly;
  constexpr bool kLast = MODE == kScatterLast || MODE == kScatterOnly;
  // One LDS buffer stages the keys, then the payload (the tile's footprint
  // is the larger of the two, not their sum); a byte per slot keeps its
  // digit, so the write-out loops need no registers per entry; the digit
  // starts overwrite the counters, and offsets are 32-bit while every one
  // fits.  20 KB per wave with an 8-byte payload: 8 waves per CU.  The fused
  // first pass computes the row ids in the buffer before all that.
  using Off = std::conditional_t<sizeof(CT) == 4, uint32_t, int64_t>;
  constexpr int kBufWords = (int)((kSub * (sizeof(Pos) > sizeof(K) ? sizeof(Pos) : sizeof(K))) / 8);
  static_assert(!kFirst || kSub * 4 <= kBufWords * 8, "row marks fit the staging buffer");
  __shared__ uint64_t s_buf[kBufWords];
  __shared__ unsigned s_cnt[kDigits];  // digit counts, then digit starts
  __shared__ Off s_off[kDigits];
  __shared__ uint8_t s_dig[kSub];
  K* s_key = reinterpret_cast<K*>(s_buf);
  Pos* s_pos = reinterpret_cast<Pos*>(s_buf);
  const int lane = threadIdx.x;
  const int64_t sub = xcd_tile(blockIdx.x, gridDim.x);
  if (sub >= n_sub) return;
  const int64_t base = sub * kSub;
  const int cnt = n - base < kSub ? (int)(n - base) : (int)kSub;
  K key[kChunks];
  Pos pos[kChunks];
  load_tile_keys<K>(keys_in, kind, base, n, lane, key);
  if constexpr (kFirst) {
    static_assert(sizeof(Pos) == 8, "the fused passes carry 8-byte (value, row) words");
#pragma unroll
    for (int ch = 0; ch < kChunks; ++ch) {
      const int64_t e = base + (int64_t)ch * 64 + lane;
      pos[ch] = (Pos)(e < n ? io.vals[e] : 0u);
    }
    const int64_t r0 = io.tile_row[sub];
    const int64_t r1 = sub + 1 < n_sub ? io.tile_row[sub + 1] : io.n_rows - 1;
    unsigned* s_mark = reinterpret_cast<unsigned*>(s_buf);
    tile_row_marks<P>(static_cast<const P*>(io.rowptr), r0, r1, base, cnt, s_mark, lane);
    // rows chunk by chunk: a wave max-scan of the marks, carried across chunks
    unsigned carry = 0u;
#pragma unroll
    for (int ch = 0; ch < kChunks; ++ch) {
      const unsigned m = umax_(wave_max_scan(s_mark[ch * 64 + lane]), carry);
      carry = (unsigned)__builtin_amdgcn_readlane((int)m, 63);
      pos[ch] |= (Pos)((uint64_t)(r0 + (int64_t)m) << 32);
    }
    wave_sync_t();
  } else {
#pragma unroll
    for (int ch = 0; ch < kChunks; ++ch) {
      const int64_t e = base + (int64_t)ch * 64 + lane;
      pos[ch] = e < n ? (pos_in ? pos_in[e] : (Pos)e) : (Pos)0;
    }
  }
  for (int d = lane; d < kDigits; d += 64) s_cnt[d] = 0;
  wave_sync_t();
  // 2. ranks within the digit, in input order
  unsigned local[kChunks];
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const bool valid = ch * 64 + lane < cnt;
    const uint64_t active = __ballot(valid);
    const unsigned digit = (unsigned)(key[ch] >> shift) & mask;
    const uint64_t peers = match_lanes<kRadixBits>(digit, active, mask);
    const int rank = count_below_t(peers);
    unsigned old = 0;
    if (valid && rank == 0) old = atomicAdd(&s_cnt[digit], (unsigned)__popcll(peers));
    const int leader = peers ? (int)__builtin_ctzll(peers) : lane;
    old = (unsigned)__builtin_amdgcn_ds_bpermute(leader << 2, (int)old);
    local[ch] = old + (unsigned)rank;
  }
  wave_sync_t();
  // 3. digit starts within the tile (over the counts: every lane holds its
  // four counts in registers before any start is stored), and each digit's
  // global base minus its start (never negative)
  unsigned c4[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) c4[k] = s_cnt[4 * lane + k];
  wave_digit_scan(c4, lane, s_cnt);
  wave_sync_t();
  for (int d = lane; d < kDigits; d += 64) s_off[d] = (Off)((int64_t)offsets[sub * kDigits + d] - (int64_t)s_cnt[d]);
  // 4. keys (and digits) to their slots of the digit-sorted LDS copy
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const unsigned digit = (unsigned)(key[ch] >> shift) & mask;
    local[ch] += s_cnt[digit];
    if (ch * 64 + lane < cnt) {
      s_key[local[ch]] = key[ch];
      s_dig[local[ch]] = (uint8_t)digit;
    }
  }
  wave_sync_t();
  // keys out as contiguous runs
  for (int i = lane; i < cnt; i += 64) keys_out[(int64_t)s_off[s_dig[i]] + i] = s_key[i];
  wave_sync_t();
  // the payload through the same buffer, out to the same slots
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch)
    if (ch * 64 + lane < cnt) s_pos[local[ch]] = pos[ch];
  wave_sync_t();
  for (int i = lane; i < cnt; i += 64) {
    const int64_t dst = (int64_t)s_off[s_dig[i]] + i;
    if constexpr (kLast) {
      const uint64_t w = (uint64_t)s_pos[i];
      io.t_vals[dst] = (uint32_t)w;
      static_cast<OI*>(io.t_cols)[dst] = (OI)(w >> 32);
    } else {
      pos_out[dst] = s_pos[i];
    }
  }
}

// ---- exclusive scan over int64 (reduce -> scan partials -> downsweep) ----
// Tile total: integer sums do not depend on order, so the loads are
// coalesced (item k * 256 + t of the tile to thread t).
__global__ __launch_bounds__(256) void scan_reduce_kernel(const int64_t* __restrict__ in, int64_t n,
                                                          int64_t* __restrict__ partial) {
  __shared__ int64_t s_wave[4];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x;
  int64_t v[kScanItems];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) v[k] = base + k * 256 < n ? in[base + k * 256] : 0;
  int64_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) s += v[k];
  int64_t total;
  block_exclusive_scan(s, s_wave, total);
  if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void scan_partials_kernel(int64_t* __restrict__ partial, int64_t n) {
  __shared__ int64_t s_wave[4];
  int64_t carry = 0;
  for (int64_t b = 0; b < n; b += 256) {
    const int64_t i = b + threadIdx.x;
    const int64_t v = i < n ? partial[i] : 0;
    int64_t total;
    const int64_t ex = block_exclusive_scan(v, s_wave, total);
    if (i < n) partial[i] = carry + ex;
    carry += total;
  }
}

// Tile scan: coalesced loads into LDS, each thread scans 16 consecutive
// items there (slot i + i / 16 keeps that stride-16 walk free of bank
// conflicts), then coalesced stores.
__device__ inline int scan_slot(int i) { return i + (i >> 4); }

__global__ __launch_bounds__(256) void scan_downsweep_kernel(int64_t* __restrict__ data, int64_t n,
                                                             const int64_t* __restrict__ partial) {
  __shared__ int64_t s_wave[4];
  __shared__ int64_t s_tile[kScanTile + kScanTile / 16];
  const int t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int i = k * 256 + t;
    s_tile[scan_slot(i)] = base + i < n ? data[base + i] : 0;
  }
  __syncthreads();
  int64_t v[kScanItems];
  int64_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = s_tile[scan_slot(t * kScanItems + k)];
    s += v[k];
  }
  int64_t total;
  int64_t run = partial[blockIdx.x] + block_exclusive_scan(s, s_wave, total);
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    s_tile[scan_slot(t * kScanItems + k)] = run;
    run += v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int i = k * 256 + t;
    if (base + i < n) data[base + i] = s_tile[scan_slot(i)];
  }
}

// ---- row ids, gather, column pointer ----
constexpr int kExpandItems = 16;

// Row id of every entry.  A workgroup covers kExpandTile entries; thread t
// walks entries [16t, 16t + 16) of the tile (one binary search for the first,
// then the row pointer), staging the ids in LDS (index padded by one per 16,
// so the stride-16 walk is free of bank conflicts); the tile then leaves with
// coalesced stores.
constexpr int kExpandTile = 256 * kExpandItems;
__device__ inline int expand_slot(int j) { return j + (j >> 4); }

// First row r in [lo, hi] whose end pointer exceeds e (rowptr[r + 1] > e).
template <class P>
__device__ inline int64_t row_of_entry(const P* __restrict__ rowptr, int64_t lo, int64_t hi, int64_t e) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)rowptr[mid + 1] <= e)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Row ids of the tile's entries into s_row (call with all 256 threads; it
// contains barriers).  The rows that start inside the tile are marked at
// their first entry (row + 1; the row pointer is read with unit stride, 256
// rows at a time, and empty rows start nowhere), then an inclusive max-scan
// over the tile fills every entry with the last row that started at or
// before it, seeded with the row of the tile's first entry.  No thread walks
// rows one dependent load at a time.
template <class P, class RT>
__device__ inline void expand_tile_rows(const P* __restrict__ rowptr, int64_t n_rows, int64_t nnz, int64_t base,
                                        RT* s_row) {
  __shared__ int64_t s_bounds[2];
  __shared__ RT s_wmax[4];
  const int tid = threadIdx.x;
  const int64_t end = base + kExpandTile < nnz ? base + kExpandTile : nnz;
  if (tid == 0) s_bounds[0] = row_of_entry<P>(rowptr, 0, n_rows - 1, base);
  if (tid == 64) s_bounds[1] = row_of_entry<P>(rowptr, 0, n_rows - 1, end - 1);
  for (int j = tid; j < kExpandTile; j += 256) s_row[expand_slot(j)] = 0;
  __syncthreads();
  const int64_t rlo = s_bounds[0], rhi = s_bounds[1];
  // rows rlo+1 .. rhi start inside the tile (after entry base) unless empty
  for (int64_t r = rlo + 1 + tid; r <= rhi; r += 256) {
    const int64_t st = (int64_t)rowptr[r];
    if ((int64_t)rowptr[r + 1] > st) s_row[expand_slot((int)(st - base))] = (RT)(r + 1);
  }
  __syncthreads();
  // inclusive max-scan: 16 consecutive entries per thread, then across
  // threads (wave shuffles, then the 4 wave totals)
  RT v[kExpandItems];
  RT run = 0;
#pragma unroll
  for (int k = 0; k < kExpandItems; ++k) {
    const RT m = s_row[expand_slot(tid * kExpandItems + k)];
    run = m > run ? m : run;
    v[k] = run;
  }
  RT incl = run;
  const int lane = tid & 63;
  for (int off = 1; off < 64; off <<= 1) {
    const RT y = __shfl_up(incl, off);
    if (lane >= off && y > incl) incl = y;
  }
  if (lane == 63) s_wmax[tid >> 6] = incl;
  __syncthreads();
  RT carry = (RT)(rlo + 1);
  for (int w = 0; w < (tid >> 6); ++w) carry = s_wmax[w] > carry ? s_wmax[w] : carry;
  const RT prev = __shfl_up(incl, 1);
  if (lane > 0 && prev > carry) carry = prev;
#pragma unroll
  for (int k = 0; k < kExpandItems; ++k)
    s_row[expand_slot(tid * kExpandItems + k)] = (v[k] > carry ? v[k] : carry) - (RT)1;
}

template <class P, class OI>
__global__ __launch_bounds__(256) void expand_rows_kernel(const P* __restrict__ rowptr, int64_t n_rows, int64_t nnz,
                                                          OI* __restrict__ rowid) {
  using RT = std::conditional_t<sizeof(OI) == 8, uint64_t, uint32_t>;  // LDS word as wide as the output index
  __shared__ RT s_row[kExpandTile + kExpandTile / 16];
  const int64_t base = (int64_t)blockIdx.x * kExpandTile;
  expand_tile_rows<P, RT>(rowptr, n_rows, nnz, base, s_row);
  __syncthreads();
  for (int j = threadIdx.x; j < kExpandTile; j += 256) {
    const int64_t e = base + j;
    if (e < nnz) rowid[e] = (OI)s_row[expand_slot(j)];
  }
}

template <class V, class OI, class Pos>
__global__ __launch_bounds__(256) void transpose_gather_kernel(const V* __restrict__ vals, const OI* __restrict__ rowid,
                                                               const Pos* __restrict__ perm, int64_t nnz, int conj,
                                                               V* __restrict__ t_vals, OI* __restrict__ t_cols) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const int64_t p = (int64_t)perm[k];
  V v = vals[p];
  if (conj) v = VT<V>::conj(v);
  t_vals[k] = v;
  t_cols[k] = rowid[p];
}

// 4-byte values with 4-byte output indices: each entry's (value, row) packed
// into one 8-byte word, so the permutation gather below is one random 8-byte
// read per entry instead of two random 4-byte reads.  Values are read and
// words written coalesced, through the same LDS tile as expand_rows_kernel.
template <class P, class V, class OI>
__global__ __launch_bounds__(256) void expand_pack_kernel(const P* __restrict__ rowptr, int64_t n_rows, int64_t nnz,
                                                          const V* __restrict__ vals, uint2* __restrict__ packed) {
  static_assert(sizeof(V) == 4, "packs a 4-byte value with a 4-byte row index (rows below 2^32)");
  __shared__ unsigned s_row[kExpandTile + kExpandTile / 16];
  __shared__ unsigned s_val[kExpandTile + kExpandTile / 16];
  const int64_t base = (int64_t)blockIdx.x * kExpandTile;
  for (int j = threadIdx.x; j < kExpandTile; j += 256) {
    const int64_t e = base + j;
    if (e < nnz) __builtin_memcpy(&s_val[expand_slot(j)], &vals[e], 4);
  }
  expand_tile_rows<P, unsigned>(rowptr, n_rows, nnz, base, s_row);
  __syncthreads();
  for (int j = threadIdx.x; j < kExpandTile; j += 256) {
    const int64_t e = base + j;
    if (e < nnz) packed[e] = make_uint2(s_val[expand_slot(j)], s_row[expand_slot(j)]);
  }
}

template <class V, class OI, class Pos>
__global__ __launch_bounds__(256) void transpose_gather_packed_kernel(const uint2* __restrict__ packed,
                                                                      const Pos* __restrict__ perm, int64_t nnz,
                                                                      V* __restrict__ t_vals, OI* __restrict__ t_cols) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const uint2 w = packed[(int64_t)perm[k]];
  V v;
  __builtin_memcpy(&v, &w.x, 4);
  t_vals[k] = v;  // real 4-byte values only: conj is the identity
  t_cols[k] = (OI)w.y;
}

// 8-byte values (f64, complex64) with row ids below 2^32: (value, row) in
// one 16-byte word, so the permutation gather is one random 16-byte read per
// entry instead of an 8-byte value read and an 8-byte row id read.
template <class P, class V>
__global__ __launch_bounds__(256) void expand_pack16_kernel(const P* __restrict__ rowptr, int64_t n_rows, int64_t nnz,
                                                            const V* __restrict__ vals, uint4* __restrict__ packed) {
  static_assert(sizeof(V) == 8, "packs an 8-byte value with a 4-byte row index");
  __shared__ unsigned s_row[kExpandTile + kExpandTile / 16];
  const int64_t base = (int64_t)blockIdx.x * kExpandTile;
  expand_tile_rows<P, unsigned>(rowptr, n_rows, nnz, base, s_row);
  __syncthreads();
  for (int j = threadIdx.x; j < kExpandTile; j += 256) {
    const int64_t e = base + j;
    if (e < nnz) {
      uint2 v;
      __builtin_memcpy(&v, &vals[e], 8);
      packed[e] = make_uint4(v.x, v.y, s_row[expand_slot(j)], 0u);
    }
  }
}

template <class V, class OI, class Pos>
__global__ __launch_bounds__(256) void transpose_gather_packed16_kernel(const uint4* __restrict__ packed,
                                                                        const Pos* __restrict__ perm, int64_t nnz,
                                                                        int conj, V* __restrict__ t_vals,
                                                                        OI* __restrict__ t_cols) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const uint4 w = packed[(int64_t)perm[k]];
  const uint2 vb = make_uint2(w.x, w.y);
  V v;
  __builtin_memcpy(&v, &vb, 8);
  if (conj) v = VT<V>::conj(v);
  t_vals[k] = v;
  t_cols[k] = (OI)w.z;
}

// Sorted packed (value, row) words out to the transposed arrays (coalesced).
template <class V, class OI>
__global__ __launch_bounds__(256) void unpack_kernel(const uint2* __restrict__ packed, int64_t nnz,
                                                     V* __restrict__ t_vals, OI* __restrict__ t_cols) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const uint2 w = packed[k];
  V v;
  __builtin_memcpy(&v, &w.x, 4);
  t_vals[k] = v;  // real 4-byte values only: conj is the identity
  t_cols[k] = (OI)w.y;
}

// colptr[c] = first position whose key is >= c.  Thread k owns positions
// [kW, kW + W) (one 16-byte load of its keys, plus the key before them) and
// writes the pointers of the columns that start there; the thread at nnz
// writes the trailing ones.
template <class K, class OP>
__global__ __launch_bounds__(256) void colptr_kernel(const K* __restrict__ keys, int64_t nnz, int64_t n_cols,
                                                     OP* __restrict__ colptr) {
  constexpr int W = 16 / (int)sizeof(K);
  const int64_t k0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * W;
  if (k0 > nnz) return;
  K kv[W];
  if (k0 + W <= nnz && ((uintptr_t)keys % 16) == 0) {
    typedef K vec_t __attribute__((ext_vector_type(W)));
    const vec_t v = *reinterpret_cast<const vec_t*>(keys + k0);
#pragma unroll
    for (int w = 0; w < W; ++w) kv[w] = v[w];
  } else {
#pragma unroll
    for (int w = 0; w < W; ++w) kv[w] = k0 + w < nnz ? keys[k0 + w] : (K)0;
  }
  int64_t prev = k0 > 0 ? (int64_t)keys[k0 - 1] : -1;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const int64_t k = k0 + w;
    if (k > nnz) break;
    const int64_t cur = k < nnz ? ((int64_t)kv[w] < n_cols ? (int64_t)kv[w] : n_cols) : n_cols;
    for (int64_t c = prev + 1; c <= cur; ++c) colptr[c] = (OP)k;
    prev = cur;
  }
}

template <class OP>
__global__ __launch_bounds__(256) void fill_kernel(OP* __restrict__ p, int64_t n, OP v) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = v;
}

template <class K>
__global__ __launch_bounds__(256) void identity_kernel(const void* __restrict__ cols, int kind, int64_t n,
                                                       K* __restrict__ keys) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) keys[k] = load_key<K>(cols, kind, k);
}

// The payload between passes: the entry's value word(s) and row.  (Records
// that also carried the key, so that a digit's run left as one block, measured
// slower: the next pass's count then reads the whole records.)
struct alignas(4) Pay12 {
  uint32_t v0, v1, r;
};
template <int VW>
struct WgPay;
template <>
struct WgPay<1> {
  using T = uint64_t;  // value | row << 32
};
template <>
struct WgPay<2> {
  using T = Pay12;
};

struct WgIO {
  const void* vals;         // first pass: CSR values (VW 4-byte words each)
  const void* rowptr;       // first pass: CSR row pointer
  int ptr64;
  const int64_t* tile_row;  // first pass: row of each wave sub-tile's first entry
  int64_t n_rows;
  int64_t n_sub;
  void* t_vals;             // last pass: transposed values
  void* t_cols;             // last pass: transposed column indices (the rows)
  int oi64;
  void* colptr;             // last pass: atomic minimum per column (null: the sorted keys go to keys_out)
  int op64;
  int64_t n_cols;
  uint32_t conj_mask;       // xor into the high word of 8-byte values (complex64 conj)
  const void* other;        // first pass: explicit second index per entry (COO), in place of rows from rowptr
  int other64;
  int swap;                 // this pass sorts by the payload's index: it and the key change places
};

// Row of the first entry of every wave sub-tile: thread r writes r for the
// sub-tiles whose first entry lies in row r (one coalesced pass over the row
// pointer instead of a binary search per sub-tile).  A malformed row pointer
// can leave slots unwritten; the scatter clamps what it reads.
// (The same launch fills the column pointer with nnz, its start value for
// the last pass's atomic minima: thread k < n_fill writes fill[k].)
// (With `check`, the fused structure check: each row whose pointer
// decreases adds one to check[2].)
template <class P, class OP>
__global__ __launch_bounds__(256) void wg_tile_rows_kernel(const P* __restrict__ rowptr, int64_t n_rows,
                                                           int64_t n_sub, int64_t* __restrict__ tile_row,
                                                           OP* __restrict__ fill, int64_t n_fill, OP fill_value,
                                                           unsigned long long* __restrict__ check) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n_fill) fill[r] = fill_value;
  if (r >= n_rows) return;
  const int64_t a = (int64_t)rowptr[r], b = (int64_t)rowptr[r + 1];
  if (check != nullptr && b < a) atomicAdd(&check[2], 1ull);  // malformed input only
  const int64_t end = row_sub_tile(b, kWgSub, n_sub);
  for (int64_t sub = row_sub_tile(a, kWgSub, n_sub); sub < end; ++sub) tile_row[sub] = r;
}

// The fused structure check's column test over one lane's column values
// (slots past a sub-tile hold 0): columns outside [0, n_cols) fold into the
// sign-flipped minimum / maximum in check[3] / check[4], one pair of atomics
// per wave that holds any, so a valid matrix issues none.  All lanes call it.
__device__ inline void check_columns(const int64_t (&col)[kWgChunks], uint64_t n_cols, int lane,
                                     unsigned long long* __restrict__ check) {
  unsigned long long lo = ~0ull, hi = 0ull;
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch) {
    if ((uint64_t)col[ch] >= n_cols) {
      const unsigned long long f = (unsigned long long)col[ch] ^ kSignFlip;
      lo = f < lo ? f : lo;
      hi = f > hi ? f : hi;
    }
  }
  if (__ballot(lo != ~0ull) != 0ull) {  // wave-uniform
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long olo = __shfl_xor(lo, off), ohi = __shfl_xor(hi, off);
      lo = olo < lo ? olo : lo;
      hi = ohi > hi ? ohi : hi;
    }
    if (lane == 0) {
      atomicMin(&check[3], lo);
      atomicMax(&check[4], hi);
    }
  }
}

// Fused structure check, first words: indptr[0], indptr[n_rows], no
// decreasing row yet, and a column range of [0, 0] that only an entry
// outside [0, n_cols) widens.
template <class P>
__global__ void fused_check_init_kernel(const P* __restrict__ rowptr, int64_t n_rows,
                                        unsigned long long* __restrict__ check) {
  const int k = threadIdx.x;
  if (k == 0) check[0] = (unsigned long long)(int64_t)rowptr[0];
  if (k == 1) check[1] = (unsigned long long)(int64_t)rowptr[n_rows];
  if (k == 2) check[2] = 0ull;
  if (k == 3 || k == 4) check[k] = kSignFlip;
}

// Per-tile digit counts, cnt[tile][nd] (nd = mask + 1 digits).  With
// `check` (the first pass over CSR columns), also the fused structure
// check's column test.  (16-byte key loads: C4's first count, the first read of
// the columns, 51 -> 30 us.)
__global__ __launch_bounds__(kWgThreads) void wg_count_kernel(const void* __restrict__ keys, int kind, int64_t n,
                                                              int shift, unsigned mask,
                                                              uint32_t* __restrict__ counts,
                                                              unsigned long long* __restrict__ check,
                                                              int64_t n_cols) {
  __shared__ unsigned s_hist[kWgMaxDigits];
  const int nd = (int)mask + 1;
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int64_t tile = blockIdx.x;
  for (int d = threadIdx.x; d < nd; d += kWgThreads) s_hist[d] = 0;
  __syncthreads();
  const int64_t base = tile * kWgTile + (int64_t)w * kWgSub;
  const int cnt = n - base >= kWgSub ? (int)kWgSub : (n - base > 0 ? (int)(n - base) : 0);
  // A full sub-tile of CSR columns (kinds 0 / 1) or keys (kind 2) is read
  // with 16-byte loads in any order (a count needs no order); otherwise as
  // the scatter reads it.
  uint32_t key[kWgChunks];
  int64_t col[kWgChunks];  // column values, for the fused check
  const bool checked = check != nullptr && kind <= 1;
  static_assert(kWgChunks % 4 == 0, "a sub-tile is whole 16-byte loads per lane");
  const bool full = cnt == (int)kWgSub && kind <= 2 && ((uintptr_t)keys % 16) == 0;
  if (full && kind == 1) {
    typedef int64_t L2 __attribute__((ext_vector_type(2)));
    const L2* p = reinterpret_cast<const L2*>(static_cast<const int64_t*>(keys) + base) + lane;
#pragma unroll
    for (int k = 0; k < kWgChunks / 2; ++k) {
      const L2 q = p[k * 64];
      col[2 * k] = q[0];
      col[2 * k + 1] = q[1];
    }
  } else if (full) {
    typedef uint32_t U4 __attribute__((ext_vector_type(4)));
    const U4* p = reinterpret_cast<const U4*>(static_cast<const uint32_t*>(keys) + base) + lane;
#pragma unroll
    for (int k = 0; k < kWgChunks / 4; ++k) {
      const U4 q = p[k * 64];
#pragma unroll
      for (int j = 0; j < 4; ++j) col[4 * k + j] = kind == 0 ? (int64_t)(int32_t)q[j] : (int64_t)q[j];
    }
  } else if (checked) {
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      const int64_t q = base + ch * 64 + lane;
      col[ch] = ch * 64 + lane >= cnt ? 0
                : kind == 1            ? static_cast<const int64_t*>(keys)[q]
                                       : (int64_t) static_cast<const int32_t*>(keys)[q];
    }
  }
  if (full || checked) {
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) key[ch] = (uint32_t)col[ch];
  } else {
    wg_load_keys(keys, kind, base, cnt, lane, key);
  }
  if (checked) check_columns(col, (uint64_t)n_cols, lane, check);
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch)
    if (full || ch * 64 + lane < cnt) atomicAdd(&s_hist[(key[ch] >> shift) & mask], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < nd; d += kWgThreads) counts[tile * nd + d] = s_hist[d];
}

// Stable scatter of one workgroup-tile pass (see above).  Steps: keys and
// payload into registers; per wave, ranks within the digit against the
// wave's LDS counters (16-bit, two digits per word); per digit, the waves'
// counts turned into wave bases plus the tile's digit start (one scan over
// the digits); the keys through a digit-sorted LDS copy, out as contiguous
// runs (or, in the last pass, the column starts to colptr); the payload
// through the same buffer in windows.
// FULL: a whole tile, without lane tests.  (The passes are bound by
// instruction issue and the barriers between their steps.)
constexpr int kScatterBufBytes = (int)kWgTile * 8;  // one window of 8-byte payload, two of 12-byte
static_assert(kScatterBufBytes >= kWgBufBytes, "marks, counters and keys fit");
template <int VW, int MODE, bool FULL>
__device__ inline void wg_scatter_tile(const void* __restrict__ keys_in, int kind,
                                       const typename WgPay<VW>::T* __restrict__ pay_in, int64_t tile, int tcnt,
                                       int shift, unsigned mask, const uint32_t* __restrict__ offsets,
                                       uint32_t* __restrict__ keys_out, typename WgPay<VW>::T* __restrict__ pay_out,
                                       const WgIO& io, uint8_t* s_buf, uint32_t* s_off, int64_t* s_wave) {
  using Pay = typename WgPay<VW>::T;
  constexpr bool kFirst = MODE == kScatterFirst || MODE == kScatterOnly;
  constexpr bool kLast = MODE == kScatterLast || MODE == kScatterOnly;
  constexpr int kWords = kWgMaxDigits / 2;  // counter words per wave
  const int nd = (int)mask + 1;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // scalar: so are the wave's base addresses
  const int64_t base = tile * kWgTile + (int64_t)w * kWgSub;
  const int left = tcnt - w * (int)kWgSub;
  const int cnt = FULL ? (int)kWgSub : (left < 0 ? 0 : (left < (int)kWgSub ? left : (int)kWgSub));
  // thread t owns digits [t q, t q + q), q even (both halves of a counter word)
  constexpr int kQMax = 2 * ((kWgMaxDigits + 2 * kWgThreads - 1) / (2 * kWgThreads));
  const int q = nd > 2 * kWgThreads ? kQMax : 2;
  const int d0 = t * q;
  uint32_t key[kWgChunks];
  Pay pay[kWgChunks];
  wg_load_keys<FULL>(keys_in, kind, base, cnt, lane, key);
  // digit offsets, loaded before they are needed (a first pass with 12-byte
  // payload has no registers left for them then)
  constexpr bool kEarly = !(kFirst && VW == 2);
  uint32_t off[kQMax];
  auto load_offsets = [&]() {
#pragma unroll
    for (int j = 0; j < kQMax; ++j) off[j] = j < q && d0 + j < nd ? offsets[tile * nd + d0 + j] : 0u;
  };
  if constexpr (kEarly) load_offsets();
  if constexpr (kFirst) {
    if constexpr (VW == 1) {
      const uint32_t* vp = static_cast<const uint32_t*>(io.vals) + base + lane;
#pragma unroll
      for (int ch = 0; ch < kWgChunks; ++ch) pay[ch] = (uint64_t)(FULL || ch * 64 + lane < cnt ? vp[ch * 64] : 0u);
    } else {
      const uint2* vp = static_cast<const uint2*>(io.vals) + base + lane;
#pragma unroll
      for (int ch = 0; ch < kWgChunks; ++ch) {
        const uint2 v = FULL || ch * 64 + lane < cnt ? vp[ch * 64] : make_uint2(0u, 0u);
        pay[ch].v0 = v.x;
        pay[ch].v1 = v.y;
      }
    }
    uint32_t row[kWgChunks];
    if (io.other) {
      wg_load_keys<FULL>(io.other, io.other64 ? 1 : 0, base, cnt, lane, row);
    } else if (cnt > 0) {
      const int64_t sub = tile * kWgWaves + w;
      auto clamp_row = [&](int64_t r) { return r < 0 ? (int64_t)0 : (r >= io.n_rows ? io.n_rows - 1 : r); };
      const int64_t r0 = clamp_row(io.tile_row[sub]);
      const int64_t r1 = sub + 1 < io.n_sub ? clamp_row(io.tile_row[sub + 1]) : io.n_rows - 1;
      unsigned* s_mark = reinterpret_cast<unsigned*>(s_buf) + w * kWgSub;
      if (io.ptr64)
        wg_rows<int64_t>(static_cast<const int64_t*>(io.rowptr), r0, r1, base, cnt, s_mark, lane, row);
      else
        wg_rows<int32_t>(static_cast<const int32_t*>(io.rowptr), r0, r1, base, cnt, s_mark, lane, row);
    } else {
#pragma unroll
      for (int ch = 0; ch < kWgChunks; ++ch) row[ch] = 0u;
    }
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      if constexpr (VW == 1) pay[ch] |= (uint64_t)row[ch] << 32;
      else pay[ch].r = row[ch];
    }
    // every wave is done with its row marks before any wave's counters
    // (which need not cover the same bytes) are written over them
    __syncthreads();
  } else {
    const Pay* pp = pay_in + base + lane;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) pay[ch] = FULL || ch * 64 + lane < cnt ? pp[ch * 64] : Pay{};
    if (io.swap) {
#pragma unroll
      for (int ch = 0; ch < kWgChunks; ++ch) {
        const uint32_t k = key[ch];
        if constexpr (VW == 1) {
          key[ch] = (uint32_t)(pay[ch] >> 32);
          pay[ch] = (pay[ch] & 0xffffffffull) | ((uint64_t)k << 32);
        } else {
          key[ch] = pay[ch].r;
          pay[ch].r = k;
        }
      }
    }
  }
  // ranks within the wave's digits, against wave w's own counters
  uint32_t* wc = reinterpret_cast<uint32_t*>(s_buf);
  uint32_t* my = wc + w * kWords;
  for (int j = lane; j < (nd + 1) / 2; j += 64) my[j] = 0u;
  wave_sync_t();
  unsigned local[kWgChunks];
  {
    // (the counter updates of all chunks are issued before the first is waited for)
    unsigned old[kWgChunks];
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      const bool valid = FULL || ch * 64 + lane < cnt;
      const unsigned digit = (key[ch] >> shift) & mask;
      const uint64_t peers = match_lanes<kWgMaxBits>(digit, FULL ? ~0ull : __ballot(valid), mask);
      const int rank = count_below_t(peers);
      const unsigned half = (digit & 1u) * 16u;
      old[ch] = 0u;
      if (valid && rank == 0) old[ch] = atomicAdd(&my[digit >> 1], (unsigned)__popcll(peers) << half) >> half;
      const int leader = FULL || peers ? (int)__builtin_ctzll(peers) : lane;
      local[ch] = (unsigned)rank | (unsigned)leader << 8;
    }
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      const unsigned o = (unsigned)__builtin_amdgcn_ds_bpermute((int)(local[ch] >> 8) << 2, (int)old[ch]);
      local[ch] = (o & 0xffffu) + (local[ch] & 0xffu);
    }
  }
  __syncthreads();
  // per digit pair: wave bases, then the tile's digit starts
  {
    uint32_t sums[kQMax];
    int64_t mine = 0;
#pragma unroll
    for (int j = 0; j < kQMax; j += 2) {
      sums[j] = sums[j + 1] = 0u;
      const int d = d0 + j;
      if (j < q && d < nd) {
        uint32_t pre = 0u;  // two 16-bit prefixes
        uint32_t c[kWgWaves];
#pragma unroll
        for (int v = 0; v < kWgWaves; ++v) c[v] = wc[v * kWords + (d >> 1)];
#pragma unroll
        for (int v = 0; v < kWgWaves; ++v) {
          wc[v * kWords + (d >> 1)] = pre;
          pre += c[v];
        }
        sums[j] = pre & 0xffffu;
        sums[j + 1] = pre >> 16;
        mine += sums[j] + sums[j + 1];
      }
    }
    if constexpr (!kEarly) load_offsets();
    int64_t all;
    uint32_t run = (uint32_t)block_exclusive_scan(mine, s_wave, all);
#pragma unroll
    for (int j = 0; j < kQMax; j += 2) {
      const int d = d0 + j;
      if (j < q && d < nd) {
        const uint32_t st0 = run, st1 = run + sums[j];
        const uint32_t add = st0 | (st1 << 16);  // starts < kWgTile < 2^16
#pragma unroll
        for (int v = 0; v < kWgWaves; ++v) wc[v * kWords + (d >> 1)] += add;
        s_off[d] = off[j] - st0;
        if (d + 1 < nd) s_off[d + 1] = off[j + 1] - st1;
        run += sums[j] + sums[j + 1];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch) {
    const unsigned digit = (key[ch] >> shift) & mask;
    local[ch] += (my[digit >> 1] >> ((digit & 1u) * 16u)) & 0xffffu;
  }
  __syncthreads();
  // keys into the digit-sorted copy; then thread t takes sorted positions
  // t, t + kWgThreads, ... and keeps their destinations in registers (the
  // payload windows below overwrite the keys)
  uint32_t* s_key = reinterpret_cast<uint32_t*>(s_buf);
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch)
    if (FULL || ch * 64 + lane < cnt) s_key[local[ch]] = key[ch];
  __syncthreads();
  static_assert(kWgTile == (int64_t)kWgChunks * kWgThreads, "one sorted position per thread and chunk");
  uint32_t dst[kWgChunks];
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch) {
    const int i = t + ch * kWgThreads;
    const uint32_t k = FULL || i < tcnt ? s_key[i] : 0u;
    dst[ch] = s_off[(k >> shift) & mask] + (uint32_t)i;
    if (FULL || i < tcnt) {
      if (!kLast || io.colptr == nullptr) {
        keys_out[dst[ch]] = k;
      } else if ((i == 0 || s_key[i - 1] != k) && (int64_t)k < io.n_cols) {
        // the first entry of each column in the tile: its position is a
        // candidate for the column's start (the smallest over tiles wins)
        if (io.op64)
          __hip_atomic_fetch_min(static_cast<uint64_t*>(io.colptr) + k, (uint64_t)dst[ch], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
        else
          __hip_atomic_fetch_min(static_cast<uint32_t*>(io.colptr) + k, dst[ch], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  __syncthreads();
  // the payload, in windows of the buffer (each window holds whole rounds
  // of sorted positions, so a thread's positions stay its own)
  constexpr int kRounds = kScatterBufBytes / (int)sizeof(Pay) / kWgThreads;  // rounds per window
  constexpr int kWin = kRounds * kWgThreads;
  Pay* s_pay = reinterpret_cast<Pay*>(s_buf);
#pragma unroll
  for (int r0 = 0; r0 < kWgChunks; r0 += kRounds) {
    const int w0 = r0 * kWgThreads;
    if (!FULL && w0 >= tcnt) break;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      const unsigned j = local[ch] - (unsigned)w0;
      if ((FULL || ch * 64 + lane < cnt) && (kRounds >= kWgChunks || j < (unsigned)kWin)) s_pay[j] = pay[ch];
    }
    __syncthreads();
#pragma unroll
    for (int ch = r0; ch < (r0 + kRounds < kWgChunks ? r0 + kRounds : kWgChunks); ++ch) {
      const int i = t + ch * kWgThreads;
      if (!FULL && i >= tcnt) continue;
      const Pay v = s_pay[i - w0];
      if constexpr (kLast) {
        uint32_t r;
        if constexpr (VW == 1) {
          static_cast<uint32_t*>(io.t_vals)[dst[ch]] = (uint32_t)v;
          r = (uint32_t)(v >> 32);
        } else {
          static_cast<uint2*>(io.t_vals)[dst[ch]] = make_uint2(v.v0, v.v1 ^ io.conj_mask);
          r = v.r;
        }
        if (io.oi64) static_cast<int64_t*>(io.t_cols)[dst[ch]] = (int64_t)r;
        else static_cast<int32_t*>(io.t_cols)[dst[ch]] = (int32_t)r;
      } else {
        pay_out[dst[ch]] = v;
      }
    }
    if (r0 + kRounds < kWgChunks) __syncthreads();
  }
}

template <int VW, int MODE>
__global__ __launch_bounds__(kWgThreads, FS_WG_MIN_WAVES) void wg_scatter_kernel(
    const void* __restrict__ keys_in, int kind, const typename WgPay<VW>::T* __restrict__ pay_in, int64_t n, int shift,
    unsigned mask, const uint32_t* __restrict__ offsets, uint32_t* __restrict__ keys_out,
    typename WgPay<VW>::T* __restrict__ pay_out, WgIO io) {
  __shared__ __attribute__((aligned(16))) uint8_t s_buf[kScatterBufBytes];
  __shared__ uint32_t s_off[kWgMaxDigits];
  __shared__ int64_t s_wave[kWgWaves];
  const int64_t tile = xcd_tile(blockIdx.x, gridDim.x);  // per-XCD tile ranges
  const int64_t left = n - tile * kWgTile;
  // us of the scatters, before (lane tests, digit offsets loaded late, counter
  // updates one at a time, two windows) and now: R-MAT 2^21 complex64 455 + 361
  // -> 456 + 273; COO, 16 M float64 entries, 342 -> 274 in the middle passes;
  // 33.5 M float32 entries 220 + 289 -> 213 + 286.  12-byte payloads are faster
  // with the lane tests (the last R-MAT pass 273 / 325 us: registers spill
  // without them).
  constexpr bool kWhole = VW == 1;
  if (kWhole && left >= kWgTile)
    wg_scatter_tile<VW, MODE, kWhole>(keys_in, kind, pay_in, tile, (int)kWgTile, shift, mask, offsets, keys_out,
                                      pay_out, io, s_buf, s_off, s_wave);
  else
    wg_scatter_tile<VW, MODE, false>(keys_in, kind, pay_in, tile, left < kWgTile ? (int)left : (int)kWgTile, shift,
                                     mask, offsets, keys_out, pay_out, io, s_buf, s_off, s_wave);
}

// colptr[c] = min(colptr[c], colptr[c + 1], ...): block minima, their
// suffix minima, then every block's suffix minimum with the minimum of the
// blocks after it.
constexpr int kMinItems = 4;
constexpr int64_t kMinTile = 256 * kMinItems;

template <class OP>
__global__ __launch_bounds__(256) void suffix_min_reduce_kernel(const OP* __restrict__ p, int64_t n,
                                                                OP* __restrict__ bmin) {
  __shared__ OP s[256];
  const int64_t b0 = (int64_t)blockIdx.x * kMinTile;
  OP m = p[b0 < n ? b0 : n - 1];
  for (int k = 0; k < kMinItems; ++k) {
    const int64_t i = b0 + (int64_t)k * 256 + threadIdx.x;
    if (i < n && p[i] < m) m = p[i];
  }
  s[threadIdx.x] = m;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off && s[threadIdx.x + off] < s[threadIdx.x]) s[threadIdx.x] = s[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) bmin[blockIdx.x] = s[0];
}

// Suffix minima of the block minima, in place (one workgroup, 256 blocks
// at a time from the end, with the running minimum carried).
template <class OP>
__global__ __launch_bounds__(256) void suffix_min_blocks_kernel(OP* __restrict__ bmin, int64_t n_blocks) {
  __shared__ OP s[256];
  const int t = threadIdx.x;
  OP carry = bmin[n_blocks - 1];
  for (int64_t hi = n_blocks; hi > 0; hi -= 256) {
    const int64_t b = hi - 256 + t;
    OP v = b >= 0 ? bmin[b] : carry;
    if (carry < v) v = carry;
    s[t] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      const OP o = t + off < 256 ? s[t + off] : carry;
      __syncthreads();
      if (o < s[t]) s[t] = o;
      __syncthreads();
    }
    if (b >= 0) bmin[b] = s[t];
    carry = s[0];
    __syncthreads();
  }
}

// scanned = 1: bsuf holds the suffix minima of the block minima; 0: the
// block minima themselves, and each block takes the minimum of those after
// it (a few thousand L2-resident reads per block, one launch less).
template <class OP>
__global__ __launch_bounds__(256) void suffix_min_down_kernel(OP* __restrict__ p, int64_t n,
                                                              const OP* __restrict__ bsuf, int64_t n_blocks,
                                                              int scanned) {
  __shared__ OP s[256];
  // the minimum over the blocks after this one (the last entry, nnz, bounds all)
  OP carry = (int64_t)blockIdx.x + 1 < n_blocks ? bsuf[blockIdx.x + 1] : p[n - 1];
  if (!scanned) {
    for (int64_t b = (int64_t)blockIdx.x + 2 + threadIdx.x; b < n_blocks; b += 256)
      if (bsuf[b] < carry) carry = bsuf[b];
    s[threadIdx.x] = carry;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
      if ((int)threadIdx.x < off && s[threadIdx.x + off] < s[threadIdx.x]) s[threadIdx.x] = s[threadIdx.x + off];
      __syncthreads();
    }
    carry = s[0];
    __syncthreads();
  }
  // thread t owns kMinItems consecutive entries: its own suffix minima, then
  // the minimum over the threads after it
  const int64_t i0 = (int64_t)blockIdx.x * kMinTile + (int64_t)threadIdx.x * kMinItems;
  OP v[kMinItems];
  OP m = carry;
  for (int k = kMinItems - 1; k >= 0; --k) {
    const int64_t i = i0 + k;
    v[k] = i < n ? p[i] : carry;
    if (v[k] < m) m = v[k];
  }
  s[threadIdx.x] = m;  // this thread's minimum (with the carry)
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const OP o = (int)threadIdx.x + off < 256 ? s[threadIdx.x + off] : carry;
    __syncthreads();
    if (o < s[threadIdx.x]) s[threadIdx.x] = o;
    __syncthreads();
  }
  OP after = (int)threadIdx.x + 1 < 256 ? s[threadIdx.x + 1] : carry;
  for (int k = kMinItems - 1; k >= 0; --k) {
    const int64_t i = i0 + k;
    if (v[k] < after) after = v[k];
    if (i < n) p[i] = after;
  }
}

// ---- host side ----
struct Layout {
  size_t key_bytes, pos_bytes, rowid_bytes;
  int64_t n_sub, n_counts, n_partials;
  size_t off_keys_a, off_keys_b, off_pos_a, off_pos_b, off_rowid, off_counts, off_partials, total;
  size_t off_prow = 0, off_tile_rows = 0;
  bool payload = false;
};

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// payload = true sizes the position slots for 8-byte words (the transpose
// carries packed (value, row) words through the sort instead of positions).
Layout make_layout(int64_t n_rows, int64_t n_cols, int64_t nnz, bool payload = false) {
  Layout L{};
  L.key_bytes = (n_cols > (int64_t)0xffffffffLL) ? 8 : 4;
  L.pos_bytes = (nnz > (int64_t)0xffffffffLL) ? 8 : 4;
  L.rowid_bytes = payload ? 16 : 8;  // the widest output index, or a packed 16-byte (value, row) word
  L.n_sub = ceil_div(nnz, kSub);
  L.n_counts = (int64_t)kDigits * L.n_sub;
  L.n_partials = ceil_div(L.n_counts, kScanTile);
  size_t o = 0;
  L.off_keys_a = o; o = align256(o + L.key_bytes * nnz);
  L.off_keys_b = o; o = align256(o + L.key_bytes * nnz);
  const size_t slot = payload ? 8 : L.pos_bytes;
  L.off_pos_a = o; o = align256(o + slot * nnz);
  L.off_pos_b = o; o = align256(o + slot * nnz);
  L.off_rowid = o; o = align256(o + L.rowid_bytes * nnz);
  L.off_counts = o; o = align256(o + sizeof(int64_t) * L.n_counts);
  // partials: the flat scan's tile totals, or the digit scan's per-block rows
  // (the digit scan's block rows, then its 256 digit totals)
  const int64_t n_part = std::max<int64_t>(L.n_partials + 1, ceil_div(L.n_sub, kDigitScanSubs) * kDigits + kDigits);
  L.off_partials = o; o = align256(o + sizeof(int64_t) * n_part);
  L.total = o;
  L.payload = payload;
  (void)n_rows;
  return L;
}

int device_exclusive_scan(int64_t* data, int64_t n, int64_t* partial, hipStream_t s) {
  if (n == 0) return FS_OK;
  const int64_t blocks = ceil_div(n, kScanTile);
  hipLaunchKernelGGL(scan_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, s, data, n, partial);
  FS_CHECK_LAUNCH("scan_reduce_kernel");
  hipLaunchKernelGGL(scan_partials_kernel, dim3(1), dim3(256), 0, s, partial, blocks);
  FS_CHECK_LAUNCH("scan_partials_kernel");
  hipLaunchKernelGGL(scan_downsweep_kernel, dim3((unsigned)blocks), dim3(256), 0, s, data, n, partial);
  FS_CHECK_LAUNCH("scan_downsweep_kernel");
  return FS_OK;
}

// Exclusive scan of cnt[sub][digit] in (digit, sub) order, in place.
template <class CT>
int digit_exclusive_scan(CT* cnt, int64_t n_sub, CT* partial, hipStream_t s) {
  if (n_sub == 0) return FS_OK;
  const int64_t blocks = ceil_div(n_sub, kDigitScanSubs);
  int64_t* totals = reinterpret_cast<int64_t*>(partial + blocks * kDigits);  // 256 more, 8-byte aligned
  hipLaunchKernelGGL((digit_scan_reduce_kernel<CT>), dim3((unsigned)blocks), dim3(256), 0, s, cnt, n_sub, partial);
  FS_CHECK_LAUNCH("digit_scan_reduce_kernel");
  hipLaunchKernelGGL((digit_scan_column_kernel<CT>), dim3(kDigits), dim3(256), 0, s, partial, blocks, totals);
  FS_CHECK_LAUNCH("digit_scan_column_kernel");
  hipLaunchKernelGGL((digit_scan_down_kernel<CT>), dim3((unsigned)blocks), dim3(256), 0, s, cnt, n_sub, partial,
                     totals);
  FS_CHECK_LAUNCH("digit_scan_down_kernel");
  return FS_OK;
}

int key_bits(int64_t n_cols) {
  int b = 0;
  while (b < 64 && ((n_cols - 1) >> b) > 0) ++b;  // bits needed for n_cols-1
  return b;
}

// The passes of the LSD sort.  With Fused (the transpose's 8-byte
// (value, row) payload, FusedIO io) the first pass builds the words from the
// CSR arrays and the last writes the transposed values and rows; *perm is
// then null.
template <class K, class Pos, class CT, bool Fused = false, class P = int32_t, class OI = int32_t>
int radix_passes(const Layout& L, char* ws, const void* cols, int col_kind, int64_t nnz, int total_bits, int passes,
                 const K** sorted_keys, const Pos** perm, hipStream_t s, const Pos* pos_init,
                 FusedIO io = FusedIO{}) {
  K* ka = reinterpret_cast<K*>(ws + L.off_keys_a);
  K* kb = reinterpret_cast<K*>(ws + L.off_keys_b);
  Pos* pa = reinterpret_cast<Pos*>(ws + L.off_pos_a);
  Pos* pb = reinterpret_cast<Pos*>(ws + L.off_pos_b);
  CT* counts = reinterpret_cast<CT*>(ws + L.off_counts);
  CT* partial = reinterpret_cast<CT*>(ws + L.off_partials);
  const unsigned blocks = (unsigned)ceil_div(L.n_sub, kWavesPerBlock);
  const void* kin = cols;
  int kind = col_kind;
  const Pos* pin = pos_init;  // null: positions 0, 1, ... on the first pass
  K* kout = ka;
  Pos* pout = pa;
  // The key bits split evenly over the passes (20 bits: 7 + 7 + 6, not
  // 8 + 8 + 4): fewer digits per pass make each digit's run in a sub-tile's
  // output longer, and the scattered runs write faster the longer they are.
  int shift = 0;
  for (int p = 0; p < passes; ++p) {
    const int bits = (total_bits - shift + (passes - p) - 1) / (passes - p);
    const unsigned mask = (1u << bits) - 1u;
    hipLaunchKernelGGL((radix_count_kernel<K, CT>), dim3(blocks), dim3(256), 0, s, kin, kind, nnz, shift, mask,
                       L.n_sub, counts);
    FS_CHECK_LAUNCH("radix_count_kernel");
    int rc = digit_exclusive_scan<CT>(counts, L.n_sub, partial, s);
    if (rc != FS_OK) return rc;
    const dim3 g((unsigned)L.n_sub);
    if constexpr (Fused) {
      if (passes == 1)
        hipLaunchKernelGGL((radix_scatter_kernel<K, Pos, CT, kScatterOnly, P, OI>), g, dim3(64), 0, s, kin, kind,
                           pin, nnz, shift, mask, L.n_sub, counts, kout, pout, io);
      else if (p == 0)
        hipLaunchKernelGGL((radix_scatter_kernel<K, Pos, CT, kScatterFirst, P, OI>), g, dim3(64), 0, s, kin, kind,
                           pin, nnz, shift, mask, L.n_sub, counts, kout, pout, io);
      else if (p == passes - 1)
        hipLaunchKernelGGL((radix_scatter_kernel<K, Pos, CT, kScatterLast, P, OI>), g, dim3(64), 0, s, kin, kind,
                           pin, nnz, shift, mask, L.n_sub, counts, kout, pout, io);
      else
        hipLaunchKernelGGL((radix_scatter_kernel<K, Pos, CT>), g, dim3(64), 0, s, kin, kind, pin, nnz, shift, mask,
                           L.n_sub, counts, kout, pout, io);
    } else {
      hipLaunchKernelGGL((radix_scatter_kernel<K, Pos, CT>), g, dim3(64), 0, s, kin, kind, pin, nnz, shift, mask,
                         L.n_sub, counts, kout, pout, io);
    }
    shift += bits;
    FS_CHECK_LAUNCH("radix_scatter_kernel");
    kin = kout;
    kind = 2;
    pin = pout;
    kout = (kout == ka) ? kb : ka;
    pout = (pout == pa) ? pb : pa;
  }
  *sorted_keys = static_cast<const K*>(kin);
  *perm = Fused ? nullptr : pin;
  return FS_OK;
}

template <class K, class Pos>
int radix_sort_cols(const Layout& L, char* ws, const void* cols, int col_kind, int64_t nnz, int64_t n_cols,
                    const K** sorted_keys, const Pos** perm, hipStream_t s, const Pos* pos_init = nullptr) {
  const int passes = (key_bits(n_cols) + kRadixBits - 1) / kRadixBits;
  if (passes == 0) {
    K* ka = reinterpret_cast<K*>(ws + L.off_keys_a);
    hipLaunchKernelGGL((identity_kernel<K>), dim3((unsigned)ceil_div(nnz, 256)), dim3(256), 0, s, cols, col_kind,
                       nnz, ka);
    FS_CHECK_LAUNCH("identity_kernel");
    *sorted_keys = ka;
    *perm = nullptr;
    return FS_OK;
  }
  // 32-bit counts and offsets while every offset fits
  if (nnz <= (int64_t)0xffffffffLL)
    return radix_passes<K, Pos, uint32_t>(L, ws, cols, col_kind, nnz, key_bits(n_cols), passes, sorted_keys, perm, s,
                                          pos_init);
  return radix_passes<K, Pos, uint64_t>(L, ws, cols, col_kind, nnz, key_bits(n_cols), passes, sorted_keys, perm, s,
                                        pos_init);
}

template <class Pos>
__global__ __launch_bounds__(256) void iota_kernel(Pos* __restrict__ p, int64_t n) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = (Pos)k;
}

// Packed payload through the sort (4-byte values, row ids below 2^32,
// widened on the way out for 8-byte output indices): the (value, row) words ride through every scatter pass in
// place of positions, so no random permutation gather follows the sort.
// FLAGSPARSE_TRANSPOSE_PAYLOAD=0 sorts positions and gathers instead (A/B).
// 16-byte (value, row) words for the gather of 8-byte values;
// FLAGSPARSE_TRANSPOSE_PACK16=0 gathers value and row id separately (A/B).
inline bool transpose_pack16_enabled() {
  const char* e = std::getenv("FLAGSPARSE_TRANSPOSE_PACK16");
  return !(e && std::atoi(e) == 0);
}

inline bool transpose_payload_enabled() {
  const char* e = std::getenv("FLAGSPARSE_TRANSPOSE_PAYLOAD");
  return !(e && std::atoi(e) == 0);
}

// ---- the workgroup-tile transpose (4- and 8-byte values) ----
struct WgLayout {
  int64_t n_tiles = 0, n_sub = 0, n_blocks = 0, n_min_blocks = 0;
  size_t off_keys_a = 0, off_keys_b = 0, off_pay_a = 0, off_pay_b = 0, off_counts = 0, off_partial = 0,
         off_totals = 0, off_tile_row = 0, off_bmin = 0, total = 0;
};

WgLayout make_wg_layout(int64_t n_cols, int64_t nnz) {
  WgLayout L;
  L.n_tiles = ceil_div(nnz, kWgTile);
  L.n_sub = ceil_div(nnz, kWgSub);
  L.n_blocks = ceil_div(L.n_tiles, kWgScanTiles);
  L.n_min_blocks = ceil_div(n_cols + 1, kMinTile);
  size_t o = 0;
  L.off_keys_a = o; o = align256(o + 4 * (size_t)nnz);
  L.off_keys_b = o; o = align256(o + 4 * (size_t)nnz);
  L.off_pay_a = o; o = align256(o + sizeof(Pay12) * (size_t)nnz);
  L.off_pay_b = o; o = align256(o + sizeof(Pay12) * (size_t)nnz);
  L.off_counts = o; o = align256(o + 4 * (size_t)L.n_tiles * kWgMaxDigits);
  L.off_partial = o; o = align256(o + 4 * (size_t)L.n_blocks * kWgMaxDigits);
  L.off_totals = o; o = align256(o + 4 * (size_t)kWgMaxDigits);
  L.off_tile_row = o; o = align256(o + 8 * (size_t)L.n_sub);
  L.off_bmin = o; o = align256(o + 8 * (size_t)L.n_min_blocks);
  L.total = o;
  return L;
}

// The workgroup-tile path takes 4- and 8-byte values with positions, rows
// and columns below 2^32; FLAGSPARSE_TRANSPOSE_WG=0 keeps the wave-tile
// passes (A/B).
inline bool transpose_wg_applies(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz) {
  if (const char* e = std::getenv("FLAGSPARSE_TRANSPOSE_WG"))
    if (std::atoi(e) == 0) return false;
  const int64_t lim = (int64_t)0xffffffffLL;
  return val_t != FS_C128 && nnz > 0 && nnz < lim && n_rows <= lim && n_cols <= lim + 1;
}

// FLAGSPARSE_TRANSPOSE_COLPTR=keys: the last pass writes the sorted keys and
// colptr_kernel reads the column pointer off them (A/B of the atomic minima).
inline bool colptr_from_keys() {
  const char* e = std::getenv("FLAGSPARSE_TRANSPOSE_COLPTR");
  return e && std::string(e) == "keys";
}

template <class OP>
int colptr_suffix_min(OP* colptr, int64_t n, OP* bmin, int64_t n_blocks, hipStream_t s) {
  hipLaunchKernelGGL((suffix_min_reduce_kernel<OP>), dim3((unsigned)n_blocks), dim3(256), 0, s, colptr, n, bmin);
  FS_CHECK_LAUNCH("suffix_min_reduce_kernel");
  const int scanned = n_blocks > 8192 ? 1 : 0;  // (few blocks: each reads the later minima itself)
  if (scanned) {
    hipLaunchKernelGGL((suffix_min_blocks_kernel<OP>), dim3(1), dim3(256), 0, s, bmin, n_blocks);
    FS_CHECK_LAUNCH("suffix_min_blocks_kernel");
  }
  hipLaunchKernelGGL((suffix_min_down_kernel<OP>), dim3((unsigned)n_blocks), dim3(256), 0, s, colptr, n, bmin,
                     n_blocks, scanned);
  FS_CHECK_LAUNCH("suffix_min_down_kernel");
  return FS_OK;
}

// Passes for `bits` key bits (at least one): two passes up to 2 x 11 - 1
// bits, beyond that at most 10 bits per pass.  Measured (ms): 22-bit C3
// columns 1.92 in two 11-bit passes against 1.44 in three (8 + 7 + 7: runs
// of 2048 digits are 3 entries long and the count table grows to 90 MB);
// 21-bit R-MAT / stencil columns 1.03 / 1.23 in two against 1.12 / 1.53 in
// three.  FLAGSPARSE_TRANSPOSE_PASS_BITS=8..11 caps the bits per pass (A/B).
inline int wg_passes(int bits) {
  int cap = bits <= 2 * kWgMaxBits - 1 ? kWgMaxBits : 10;
  if (const char* e = std::getenv("FLAGSPARSE_TRANSPOSE_PASS_BITS")) {
    const int v = std::atoi(e);
    if (v >= 8 && v <= kWgMaxBits) cap = v;
  }
  return bits == 0 ? 1 : (bits + cap - 1) / cap;
}

template <class T>
struct type_id {
  using type = T;
};

template <int VW>
int wg_launch_scatter(int mode, dim3 g, hipStream_t s, const void* kin, int kind, const void* pin, int64_t nnz,
                      int shift, unsigned mask, const uint32_t* counts, uint32_t* kout, void* pout,
                      const WgIO& io) {
  using Pay = typename WgPay<VW>::T;
  const Pay* pi = static_cast<const Pay*>(pin);
  Pay* po = static_cast<Pay*>(pout);
  switch (mode) {
    case kScatterFirst:
      hipLaunchKernelGGL((wg_scatter_kernel<VW, kScatterFirst>), g, dim3(kWgThreads), 0, s, kin, kind, pi, nnz, shift,
                         mask, counts, kout, po, io);
      break;
    case kScatterLast:
      hipLaunchKernelGGL((wg_scatter_kernel<VW, kScatterLast>), g, dim3(kWgThreads), 0, s, kin, kind, pi, nnz, shift,
                         mask, counts, kout, po, io);
      break;
    case kScatterOnly:
      hipLaunchKernelGGL((wg_scatter_kernel<VW, kScatterOnly>), g, dim3(kWgThreads), 0, s, kin, kind, pi, nnz, shift,
                         mask, counts, kout, po, io);
      break;
    default:
      hipLaunchKernelGGL((wg_scatter_kernel<VW, kScatterPlain>), g, dim3(kWgThreads), 0, s, kin, kind, pi, nnz, shift,
                         mask, counts, kout, po, io);
  }
  FS_CHECK_LAUNCH("wg_scatter_kernel");
  return FS_OK;
}

// check (may be null): the fused structure check's five words, written by
// the row-tile and first count kernels (bounded on any input, so the check
// need not run first).
int transpose_wg(char* ws, int val_t, int idx_t, int ptr_t, int oi_t, int op_t, int64_t n_rows, int64_t n_cols,
                 int64_t nnz, const void* vals, const void* cols, const void* indptr, int conj, void* t_vals,
                 void* t_cols, void* t_indptr, hipStream_t s, unsigned long long* check = nullptr) {
  const WgLayout L = make_wg_layout(n_cols, nnz);
  const int vw = val_t == FS_F32 ? 1 : 2;
  int64_t* tile_row = reinterpret_cast<int64_t*>(ws + L.off_tile_row);
  const int64_t n_ptr = n_cols + 1;
  const bool by_keys = colptr_from_keys();
  {
    // sub-tile rows, and (unless the keys give it) the column pointer filled with nnz
    const int64_t n_fill = by_keys ? 0 : n_ptr;
    const unsigned blocks = (unsigned)ceil_div(std::max(n_rows, n_fill), 256);
    auto go = [&](auto ptag, auto otag) {
      using P = typename decltype(ptag)::type;
      using OP = typename decltype(otag)::type;
      if (check != nullptr)
        hipLaunchKernelGGL((fused_check_init_kernel<P>), dim3(1), dim3(64), 0, s, static_cast<const P*>(indptr),
                           n_rows, check);
      hipLaunchKernelGGL((wg_tile_rows_kernel<P, OP>), dim3(blocks), dim3(256), 0, s, static_cast<const P*>(indptr),
                         n_rows, L.n_sub, tile_row, static_cast<OP*>(t_indptr), n_fill, (OP)nnz, check);
    };
    if (ptr_t == FS_I32 && op_t == FS_I32) go(type_id<int32_t>{}, type_id<int32_t>{});
    else if (ptr_t == FS_I32) go(type_id<int32_t>{}, type_id<int64_t>{});
    else if (op_t == FS_I32) go(type_id<int64_t>{}, type_id<int32_t>{});
    else go(type_id<int64_t>{}, type_id<int64_t>{});
    FS_CHECK_LAUNCH("wg_tile_rows_kernel");
  }
  WgIO io{vals,   indptr, ptr_t == FS_I64 ? 1 : 0, tile_row, n_rows, L.n_sub, t_vals, t_cols,
          oi_t == FS_I64 ? 1 : 0, by_keys ? nullptr : t_indptr, op_t == FS_I64 ? 1 : 0, n_cols,
          (conj && val_t == FS_C64) ? 0x80000000u : 0u, nullptr, 0, 0};
  uint32_t* counts = reinterpret_cast<uint32_t*>(ws + L.off_counts);
  uint32_t* partial = reinterpret_cast<uint32_t*>(ws + L.off_partial);
  uint32_t* totals = reinterpret_cast<uint32_t*>(ws + L.off_totals);
  uint32_t* ka = reinterpret_cast<uint32_t*>(ws + L.off_keys_a);
  uint32_t* kb = reinterpret_cast<uint32_t*>(ws + L.off_keys_b);
  void* pa = ws + L.off_pay_a;
  void* pb = ws + L.off_pay_b;
  const int bits = key_bits(n_cols);
  const int passes = wg_passes(bits);
  const void* kin = cols;  // the CSR columns, then the keys of the previous pass
  int kind = idx_t == FS_I32 ? 0 : 1;
  const void* pin = nullptr;
  uint32_t* kout = ka;
  void* pout = pa;
  const dim3 g((unsigned)L.n_tiles);
  int shift = 0;
  for (int p = 0; p < passes; ++p) {
    // the key bits split evenly over the passes (longer runs per digit)
    const int pbits = (bits - shift + (passes - p) - 1) / (passes - p);
    const unsigned mask = (1u << pbits) - 1u;
    const int nd = (int)mask + 1;
    hipLaunchKernelGGL(wg_count_kernel, g, dim3(kWgThreads), 0, s, kin, kind, nnz, shift, mask, counts,
                       p == 0 ? check : nullptr, n_cols);
    FS_CHECK_LAUNCH("wg_count_kernel");
    hipLaunchKernelGGL(wg_scan_reduce_kernel, dim3((unsigned)L.n_blocks), dim3(256), 0, s, counts, L.n_tiles, nd,
                       partial);
    FS_CHECK_LAUNCH("wg_scan_reduce_kernel");
    hipLaunchKernelGGL(wg_scan_column_kernel, dim3((unsigned)nd), dim3(256), 0, s, partial, L.n_blocks, nd, totals);
    FS_CHECK_LAUNCH("wg_scan_column_kernel");
    hipLaunchKernelGGL(wg_scan_down_kernel, dim3((unsigned)L.n_blocks), dim3(256), 0, s, counts, L.n_tiles, nd,
                       partial, totals);
    FS_CHECK_LAUNCH("wg_scan_down_kernel");
    const int mode = passes == 1 ? kScatterOnly : p == 0 ? kScatterFirst : p == passes - 1 ? kScatterLast
                                                                                            : kScatterPlain;
    const int rc = vw == 1 ? wg_launch_scatter<1>(mode, g, s, kin, kind, pin, nnz, shift, mask, counts, kout, pout, io)
                           : wg_launch_scatter<2>(mode, g, s, kin, kind, pin, nnz, shift, mask, counts, kout, pout, io);
    if (rc != FS_OK) return rc;
    shift += pbits;
    kin = kout;
    kind = 2;
    pin = pout;
    kout = kout == ka ? kb : ka;
    pout = pout == pa ? pb : pa;
  }
  if (by_keys) {
    const unsigned blocks = (unsigned)ceil_div(ceil_div(nnz + 1, 4), 256);
    if (op_t == FS_I32)
      hipLaunchKernelGGL((colptr_kernel<uint32_t, int32_t>), dim3(blocks), dim3(256), 0, s,
                         static_cast<const uint32_t*>(kin), nnz, n_cols, static_cast<int32_t*>(t_indptr));
    else
      hipLaunchKernelGGL((colptr_kernel<uint32_t, int64_t>), dim3(blocks), dim3(256), 0, s,
                         static_cast<const uint32_t*>(kin), nnz, n_cols, static_cast<int64_t*>(t_indptr));
    FS_CHECK_LAUNCH("colptr_kernel");
    return FS_OK;
  }
  if (op_t == FS_I32)
    return colptr_suffix_min<uint32_t>(static_cast<uint32_t*>(t_indptr), n_ptr,
                                       reinterpret_cast<uint32_t*>(ws + L.off_bmin), L.n_min_blocks, s);
  return colptr_suffix_min<uint64_t>(static_cast<uint64_t*>(t_indptr), n_ptr,
                                     reinterpret_cast<uint64_t*>(ws + L.off_bmin), L.n_min_blocks, s);
}

template <class P>
__global__ __launch_bounds__(256) void tile_rows_kernel(const P* __restrict__ rowptr, int64_t n_rows, int64_t n_sub,
                                                        int64_t* __restrict__ tile_row);

template <class V, class P, class OI, class OP, class K, class Pos>
int transpose_typed(const Layout& L, char* ws, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                    const void* vals, const void* cols, const void* indptr, int conj, void* t_vals, void* t_cols,
                    void* t_indptr, hipStream_t s) {
  const K* keys = nullptr;
  const unsigned expand_blocks = (unsigned)ceil_div(nnz, kExpandTile);
  if constexpr (sizeof(V) == 4) {
    if (L.payload && n_rows <= (int64_t)0xffffffffLL && key_bits(n_cols) > 0) {
      // The (value, row) words are built inside the first radix pass and
      // unpacked by the last: no packing or unpacking pass over the arrays.
      // The row of each sub-tile's first entry comes from one binary search
      // per sub-tile, in the slot the packed words used to take.
      int64_t* tile_row = reinterpret_cast<int64_t*>(ws + L.off_rowid);
      hipLaunchKernelGGL((tile_rows_kernel<P>), dim3((unsigned)ceil_div(L.n_sub, 256)), dim3(256), 0, s,
                         static_cast<const P*>(indptr), n_rows, L.n_sub, tile_row);
      FS_CHECK_LAUNCH("tile_rows_kernel");
      FusedIO io{static_cast<const uint32_t*>(vals), indptr, tile_row, n_rows, static_cast<uint32_t*>(t_vals), t_cols};
      const uint64_t* none = nullptr;
      const int bits = key_bits(n_cols);
      const int passes = (bits + kRadixBits - 1) / kRadixBits;
      const int kind = idx_t == FS_I32 ? 0 : 1;
      int rc = nnz <= (int64_t)0xffffffffLL
                   ? radix_passes<K, uint64_t, uint32_t, true, P, OI>(L, ws, cols, kind, nnz, bits, passes, &keys,
                                                                     &none, s, nullptr, io)
                   : radix_passes<K, uint64_t, uint64_t, true, P, OI>(L, ws, cols, kind, nnz, bits, passes, &keys,
                                                                     &none, s, nullptr, io);
      if (rc != FS_OK) return rc;
      hipLaunchKernelGGL((colptr_kernel<K, OP>), dim3((unsigned)ceil_div(ceil_div(nnz + 1, 16 / (int64_t)sizeof(K)), 256)), dim3(256), 0, s, keys, nnz,
                         n_cols, static_cast<OP*>(t_indptr));
      FS_CHECK_LAUNCH("colptr_kernel");
      (void)conj;  // real 4-byte values: conj is the identity
      return FS_OK;
    }
    if (L.payload && n_rows <= (int64_t)0xffffffffLL) {
      // one column: the order is unchanged
      uint2* packed = reinterpret_cast<uint2*>(ws + L.off_rowid);
      hipLaunchKernelGGL((expand_pack_kernel<P, V, OI>), dim3(expand_blocks), dim3(256), 0, s,
                         static_cast<const P*>(indptr), n_rows, nnz, static_cast<const V*>(vals), packed);
      FS_CHECK_LAUNCH("expand_pack_kernel");
      const uint64_t* sorted = nullptr;
      int rc = radix_sort_cols<K, uint64_t>(L, ws, cols, idx_t == FS_I32 ? 0 : 1, nnz, n_cols, &keys, &sorted, s,
                                            reinterpret_cast<const uint64_t*>(packed));
      if (rc != FS_OK) return rc;
      if (sorted == nullptr) sorted = reinterpret_cast<const uint64_t*>(packed);
      hipLaunchKernelGGL((unpack_kernel<V, OI>), dim3((unsigned)ceil_div(nnz, 256)), dim3(256), 0, s,
                         reinterpret_cast<const uint2*>(sorted), nnz, static_cast<V*>(t_vals),
                         static_cast<OI*>(t_cols));
      FS_CHECK_LAUNCH("unpack_kernel");
      hipLaunchKernelGGL((colptr_kernel<K, OP>), dim3((unsigned)ceil_div(ceil_div(nnz + 1, 16 / (int64_t)sizeof(K)), 256)), dim3(256), 0, s, keys, nnz,
                         n_cols, static_cast<OP*>(t_indptr));
      FS_CHECK_LAUNCH("colptr_kernel");
      (void)conj;
      return FS_OK;
    }
  }
  const Pos* perm = nullptr;
  int rc = radix_sort_cols<K, Pos>(L, ws, cols, idx_t == FS_I32 ? 0 : 1, nnz, n_cols, &keys, &perm, s);
  if (rc != FS_OK) return rc;
  if (perm == nullptr) {  // single column: order unchanged
    Pos* pa = reinterpret_cast<Pos*>(ws + L.off_pos_a);
    hipLaunchKernelGGL((iota_kernel<Pos>), dim3((unsigned)ceil_div(nnz, 256)), dim3(256), 0, s, pa, nnz);
    FS_CHECK_LAUNCH("iota_kernel");
    perm = pa;
  }
  if constexpr (sizeof(V) == 4 && sizeof(OI) == 4) {
    // the rowid slot holds 8 bytes per entry: room for the packed words
    uint2* packed = reinterpret_cast<uint2*>(ws + L.off_rowid);
    hipLaunchKernelGGL((expand_pack_kernel<P, V, OI>), dim3(expand_blocks), dim3(256), 0, s,
                       static_cast<const P*>(indptr), n_rows, nnz, static_cast<const V*>(vals), packed);
    FS_CHECK_LAUNCH("expand_pack_kernel");
    hipLaunchKernelGGL((transpose_gather_packed_kernel<V, OI, Pos>), dim3((unsigned)ceil_div(nnz, 256)), dim3(256), 0,
                       s, packed, perm, nnz, static_cast<V*>(t_vals), static_cast<OI*>(t_cols));
    FS_CHECK_LAUNCH("transpose_gather_packed_kernel");
    (void)conj;
  } else {
    if constexpr (sizeof(V) == 8) {
      if (n_rows <= (int64_t)0xffffffffLL && L.payload && transpose_pack16_enabled()) {
        // the payload layout's rowid slot holds 16 bytes per entry
        uint4* packed = reinterpret_cast<uint4*>(ws + L.off_rowid);
        hipLaunchKernelGGL((expand_pack16_kernel<P, V>), dim3(expand_blocks), dim3(256), 0, s,
                           static_cast<const P*>(indptr), n_rows, nnz, static_cast<const V*>(vals), packed);
        FS_CHECK_LAUNCH("expand_pack16_kernel");
        hipLaunchKernelGGL((transpose_gather_packed16_kernel<V, OI, Pos>), dim3((unsigned)ceil_div(nnz, 256)), dim3(256),
                           0, s, packed, perm, nnz, conj, static_cast<V*>(t_vals), static_cast<OI*>(t_cols));
        FS_CHECK_LAUNCH("transpose_gather_packed16_kernel");
        hipLaunchKernelGGL((colptr_kernel<K, OP>), dim3((unsigned)ceil_div(ceil_div(nnz + 1, 16 / (int64_t)sizeof(K)), 256)), dim3(256), 0, s, keys, nnz,
                           n_cols, static_cast<OP*>(t_indptr));
        FS_CHECK_LAUNCH("colptr_kernel");
        return FS_OK;
      }
    }
    OI* rowid = reinterpret_cast<OI*>(ws + L.off_rowid);
    hipLaunchKernelGGL((expand_rows_kernel<P, OI>), dim3(expand_blocks), dim3(256), 0, s,
                       static_cast<const P*>(indptr), n_rows, nnz, rowid);
    FS_CHECK_LAUNCH("expand_rows_kernel");
    hipLaunchKernelGGL((transpose_gather_kernel<V, OI, Pos>), dim3((unsigned)ceil_div(nnz, 256)), dim3(256), 0, s,
                       static_cast<const V*>(vals), rowid, perm, nnz, conj, static_cast<V*>(t_vals),
                       static_cast<OI*>(t_cols));
    FS_CHECK_LAUNCH("transpose_gather_kernel");
  }
  hipLaunchKernelGGL((colptr_kernel<K, OP>), dim3((unsigned)ceil_div(ceil_div(nnz + 1, 16 / (int64_t)sizeof(K)), 256)), dim3(256), 0, s, keys, nnz,
                     n_cols, static_cast<OP*>(t_indptr));
  FS_CHECK_LAUNCH("colptr_kernel");
  return FS_OK;
}

template <class V, class P, class OI, class OP>
int transpose_keys(const Layout& L, char* ws, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                   const void* vals, const void* cols, const void* indptr, int conj, void* tv, void* tc, void* tp,
                   hipStream_t s) {
  if (L.key_bytes == 4 && L.pos_bytes == 4)
    return transpose_typed<V, P, OI, OP, uint32_t, uint32_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr,
                                                             conj, tv, tc, tp, s);
  if (L.key_bytes == 4)
    return transpose_typed<V, P, OI, OP, uint32_t, uint64_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr,
                                                             conj, tv, tc, tp, s);
  if (L.pos_bytes == 4)
    return transpose_typed<V, P, OI, OP, uint64_t, uint32_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr,
                                                             conj, tv, tc, tp, s);
  return transpose_typed<V, P, OI, OP, uint64_t, uint64_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr,
                                                           conj, tv, tc, tp, s);
}

template <class V, class P>
int transpose_out(const Layout& L, char* ws, int idx_t, int oi, int op, int64_t n_rows, int64_t n_cols, int64_t nnz,
                  const void* vals, const void* cols, const void* indptr, int conj, void* tv, void* tc, void* tp,
                  hipStream_t s) {
  if (oi == FS_I32 && op == FS_I32)
    return transpose_keys<V, P, int32_t, int32_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, tv, tc, tp, s);
  if (oi == FS_I32)
    return transpose_keys<V, P, int32_t, int64_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, tv, tc, tp, s);
  if (op == FS_I32)
    return transpose_keys<V, P, int64_t, int32_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, tv, tc, tp, s);
  return transpose_keys<V, P, int64_t, int64_t>(L, ws, idx_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, tv, tc, tp, s);
}

template <class V>
int transpose_ptr(const Layout& L, char* ws, int idx_t, int ptr_t, int oi, int op, int64_t n_rows, int64_t n_cols,
                  int64_t nnz, const void* vals, const void* cols, const void* indptr, int conj, void* tv, void* tc,
                  void* tp, hipStream_t s) {
  if (ptr_t == FS_I32)
    return transpose_out<V, int32_t>(L, ws, idx_t, oi, op, n_rows, n_cols, nnz, vals, cols, indptr, conj, tv, tc, tp, s);
  return transpose_out<V, int64_t>(L, ws, idx_t, oi, op, n_rows, n_cols, nnz, vals, cols, indptr, conj, tv, tc, tp, s);
}


// ---- COO -> CSR (stable lexicographic sort by (row, col)) ----
template <class IR, class K>
__global__ __launch_bounds__(256) void coo_keys_kernel(const IR* __restrict__ rows, const IR* __restrict__ cols,
                                                       int64_t n, int64_t n_cols, K* __restrict__ keys) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) keys[k] = (K)((uint64_t)rows[k] * (uint64_t)n_cols + (uint64_t)cols[k]);
}

template <class V, class K, class Pos>
__global__ __launch_bounds__(256) void coo_gather_kernel(const V* __restrict__ vals, const K* __restrict__ keys,
                                                         const Pos* __restrict__ perm, int64_t n, int64_t n_cols,
                                                         V* __restrict__ out_vals, int32_t* __restrict__ out_cols) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int64_t p = perm ? (int64_t)perm[k] : k;
  out_vals[k] = vals[p];
  out_cols[k] = (int32_t)((uint64_t)keys[k] % (uint64_t)n_cols);
}

// indptr[r] = first position whose row >= r, read off the sorted keys.
template <class K>
__global__ __launch_bounds__(256) void coo_indptr_kernel(const K* __restrict__ keys, int64_t n, int64_t n_rows,
                                                         int64_t n_cols, int64_t* __restrict__ indptr) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k > n) return;
  const int64_t prev = k > 0 ? (int64_t)((uint64_t)keys[k - 1] / (uint64_t)n_cols) : -1;
  const int64_t cur = k < n ? (int64_t)((uint64_t)keys[k] / (uint64_t)n_cols) : n_rows;
  for (int64_t r = prev + 1; r <= cur; ++r) indptr[r] = k;
}

template <class V, class IR, class K, class Pos>
int coo_to_csr_typed(const Layout& L, char* ws, int64_t n, int64_t n_rows, int64_t n_cols, const void* vals,
                     const void* rows, const void* cols, int assume_sorted, void* out_vals, void* out_cols,
                     void* out_indptr, hipStream_t s) {
  K* keys0 = reinterpret_cast<K*>(ws + L.off_rowid);  // unsorted keys (rowid slot holds 8 B / entry)
  const unsigned blocks = (unsigned)ceil_div(n, 256);
  hipLaunchKernelGGL((coo_keys_kernel<IR, K>), dim3(blocks), dim3(256), 0, s, static_cast<const IR*>(rows),
                     static_cast<const IR*>(cols), n, n_cols, keys0);
  FS_CHECK_LAUNCH("coo_keys_kernel");
  const K* sorted = keys0;
  const Pos* perm = nullptr;
  if (!assume_sorted) {
    int rc = radix_sort_cols<K, Pos>(L, ws, keys0, 2, n, n_rows * n_cols, &sorted, &perm, s);
    if (rc != FS_OK) return rc;
  }
  hipLaunchKernelGGL((coo_gather_kernel<V, K, Pos>), dim3(blocks), dim3(256), 0, s, static_cast<const V*>(vals),
                     sorted, perm, n, n_cols, static_cast<V*>(out_vals), static_cast<int32_t*>(out_cols));
  FS_CHECK_LAUNCH("coo_gather_kernel");
  hipLaunchKernelGGL((coo_indptr_kernel<K>), dim3((unsigned)ceil_div(n + 1, 256)), dim3(256), 0, s, sorted, n, n_rows,
                     n_cols, static_cast<int64_t*>(out_indptr));
  FS_CHECK_LAUNCH("coo_indptr_kernel");
  return FS_OK;
}

template <class V, class IR>
int coo_to_csr_keys(const Layout& L, char* ws, int64_t n, int64_t n_rows, int64_t n_cols, const void* vals,
                    const void* rows, const void* cols, int assume_sorted, void* ov, void* oc, void* op,
                    hipStream_t s) {
  if (L.key_bytes == 4 && L.pos_bytes == 4)
    return coo_to_csr_typed<V, IR, uint32_t, uint32_t>(L, ws, n, n_rows, n_cols, vals, rows, cols, assume_sorted, ov, oc, op, s);
  if (L.key_bytes == 4)
    return coo_to_csr_typed<V, IR, uint32_t, uint64_t>(L, ws, n, n_rows, n_cols, vals, rows, cols, assume_sorted, ov, oc, op, s);
  if (L.pos_bytes == 4)
    return coo_to_csr_typed<V, IR, uint64_t, uint32_t>(L, ws, n, n_rows, n_cols, vals, rows, cols, assume_sorted, ov, oc, op, s);
  return coo_to_csr_typed<V, IR, uint64_t, uint64_t>(L, ws, n, n_rows, n_cols, vals, rows, cols, assume_sorted, ov, oc, op, s);
}

template <class V>
int coo_to_csr_idx(const Layout& L, char* ws, int idx_t, int64_t n, int64_t n_rows, int64_t n_cols, const void* vals,
                   const void* rows, const void* cols, int assume_sorted, void* ov, void* oc, void* op,
                   hipStream_t s) {
  if (idx_t == FS_I32)
    return coo_to_csr_keys<V, int32_t>(L, ws, n, n_rows, n_cols, vals, rows, cols, assume_sorted, ov, oc, op, s);
  return coo_to_csr_keys<V, int64_t>(L, ws, n, n_rows, n_cols, vals, rows, cols, assume_sorted, ov, oc, op, s);
}

// ---- column panels (stacked CSR: panel-major rows) ----
// Panel of an entry = col / panel_width.  A stable partition by panel keeps
// CSR order inside every panel, so the stacked matrix with rows
// (panel * n_rows + row) is again a CSR, read off the composite keys.  With
// at most 64 panels the partition is one counting pass: per wave sub-tile,
// count the entries of every panel, scan the [panel][sub-tile] counts, then
// scatter.  Within a 64-entry chunk, lanes of one panel write consecutive
// slots, so stores leave in at most one run per panel; the sources are read
// once, in order.
constexpr int kMaxPanels = 64;

// col / width for 0 <= col < 2^53: a double-precision estimate, corrected by
// one step either way (no 64-bit integer division).
__device__ inline int panel_of(int64_t c, int64_t width, double inv_width) {
  int64_t q = (int64_t)((double)c * inv_width);
  if (q * width > c) --q;
  else if ((q + 1) * width <= c) ++q;
  return (int)q;
}

template <class I>
__global__ __launch_bounds__(256) void panel_count_kernel(const I* __restrict__ cols, int64_t n, int64_t width,
                                                          double inv_width, int n_panels, int qbits, int64_t n_sub,
                                                          int64_t* __restrict__ counts) {
  __shared__ unsigned s_hist[kWavesPerBlock][kMaxPanels];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int64_t sub = (int64_t)blockIdx.x * kWavesPerBlock + w;
  if (sub >= n_sub) return;  // wave-local work only
  unsigned* hist = s_hist[w];
  hist[lane] = 0;
  const int64_t base = sub * kSub;
  I c[kChunks];
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const int64_t e = base + (int64_t)ch * 64 + lane;
    c[ch] = e < n ? __builtin_nontemporal_load(cols + e) : (I)0;
  }
  wave_sync_t();
  // Lanes of one panel find each other with qbits ballots; one LDS atomic per
  // panel present in the chunk (an atomic per entry on a handful of addresses
  // serialised: 137 us on C3).
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const bool valid = base + (int64_t)ch * 64 + lane < n;
    const uint64_t active = __ballot(valid);
    if (active == 0) break;
    const int q = valid ? panel_of((int64_t)c[ch], width, inv_width) : 0;
    uint64_t peers = active;
    for (int b = 0; b < qbits; ++b) {
      const bool bit = (q >> b) & 1;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    if (valid && count_below_t(peers) == 0) atomicAdd(&hist[q], (unsigned)__popcll(peers));
  }
  wave_sync_t();
  if (lane < n_panels) counts[(int64_t)lane * n_sub + sub] = hist[lane];
}

// Row of the first entry of every sub-tile (first r with rowptr[r + 1] > e),
// one independent binary search per thread, so that the scatter waves start
// from known bounds instead of each searching all rows.
template <class P>
__global__ __launch_bounds__(256) void tile_rows_kernel(const P* __restrict__ rowptr, int64_t n_rows, int64_t n_sub,
                                                        int64_t* __restrict__ tile_row) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_sub) return;
  const int64_t e = t * kSub;
  int64_t lo = 0, hi = n_rows - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)rowptr[mid + 1] <= e)
      lo = mid + 1;
    else
      hi = mid;
  }
  tile_row[t] = lo;
}

// One wave per sub-tile of kSub entries.
//  1. row id of every entry into LDS: lane l walks entries [32l, 32l + 32)
//     of the tile from one binary search between the first rows of this and
//     the next sub-tile (slot j + j/32 keeps that stride-32 walk free of bank
//     conflicts);
//  2. the global start of panel q's run in this sub-tile, offsets[q][sub]
//     (exclusive scan of panel_count_kernel's counts), into LDS;
//  3. chunk by chunk, rank = lanes of the same panel below this lane (peer
//     masks from ceil(log2 n_panels) ballots) plus the panel's cursor, which
//     keeps the partition stable; value, column and row id go to the
//     entry's slot of the stacked copy.
template <class V, class I, class P, class RT>
__global__ __launch_bounds__(64) void panel_scatter_kernel(const V* __restrict__ vals, const I* __restrict__ cols,
                                                           const P* __restrict__ rowptr, int64_t n_rows, int64_t n,
                                                           int64_t width, double inv_width, int n_panels,
                                                           int qbits, int64_t n_sub,
                                                           const int64_t* __restrict__ offsets,
                                                           const int64_t* __restrict__ tile_row,
                                                           V* __restrict__ p_vals, I* __restrict__ p_cols,
                                                           RT* __restrict__ prow) {
  constexpr int kItems = (int)(kSub / 64);
  __shared__ RT s_row[kSub + kSub / 32];
  __shared__ int64_t s_glob[kMaxPanels];
  __shared__ unsigned s_cur[kMaxPanels];
  __shared__ int64_t s_bounds[2];
  const int lane = threadIdx.x;
  const int64_t sub = xcd_tile(blockIdx.x, gridDim.x);
  if (sub >= n_sub) return;
  const int64_t base = sub * kSub;
  const int cnt = n - base < kSub ? (int)(n - base) : (int)kSub;
  I c[kChunks];
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const int e = ch * 64 + lane;
    c[ch] = e < cnt ? __builtin_nontemporal_load(cols + base + e) : (I)0;
  }
  s_glob[lane] = lane < n_panels ? offsets[(int64_t)lane * n_sub + sub] : 0;
  s_cur[lane] = 0;
  // rows of this and the next sub-tile's first entries bound every lane's search
  if (lane == 0) s_bounds[0] = tile_row[sub];
  if (lane == 1) s_bounds[1] = sub + 1 < n_sub ? tile_row[sub + 1] : n_rows - 1;
  wave_sync_t();
  {
    const int j0 = lane * kItems;
    if (j0 < cnt) {
      const int64_t e0 = base + j0;
      int64_t lo = s_bounds[0], hi = s_bounds[1];
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)rowptr[mid + 1] <= e0)
          lo = mid + 1;
        else
          hi = mid;
      }
      int64_t row = lo;
      int64_t rend = (int64_t)rowptr[row + 1];
      for (int k = 0; k < kItems && j0 + k < cnt; ++k) {
        const int64_t e = e0 + k;
        while (rend <= e) {
          ++row;
          rend = (int64_t)rowptr[row + 1];
        }
        const int j = j0 + k;
        s_row[j + (j >> 5)] = (RT)row;
      }
    }
  }
  wave_sync_t();
#pragma unroll
  for (int ch = 0; ch < kChunks; ++ch) {
    const int j = ch * 64 + lane;
    const bool valid = j < cnt;
    const uint64_t active = __ballot(valid);
    if (active == 0) break;
    const int q = valid ? panel_of((int64_t)c[ch], width, inv_width) : 0;
    uint64_t peers = active;
    for (int b = 0; b < qbits; ++b) {
      const bool bit = (q >> b) & 1;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const int rank = count_below_t(peers);
    if (valid) {
      const int64_t dst = s_glob[q] + (int64_t)s_cur[q] + rank;
      p_vals[dst] = vals[base + j];
      p_cols[dst] = c[ch];
      prow[dst] = s_row[j + (j >> 5)];
    }
    wave_sync_t();
    if (valid && rank == 0) s_cur[q] += (unsigned)__popcll(peers);
    wave_sync_t();
  }
}

// Stacked row pointer from the row id of every stacked entry.  The panel of
// position k is the last panel whose start (the scanned count of its first
// sub-tile) is <= k, so the entries carry only their row: 4 bytes per entry
// when row ids fit, instead of a composite (panel, row) key.
constexpr int kIndptrItems = 8;  // positions per thread (strided by 256 within the block's range)

template <class OP, class RT>
__global__ __launch_bounds__(256) void panel_indptr_kernel(const RT* __restrict__ prow, int64_t n, int64_t n_rows,
                                                           int n_panels, const int64_t* __restrict__ offsets,
                                                           int64_t n_sub, OP* __restrict__ indptr) {
  __shared__ int64_t s_start[kMaxPanels + 1];
  __shared__ int s_qrange[2];
  if (threadIdx.x < n_panels) s_start[threadIdx.x] = offsets[(int64_t)threadIdx.x * n_sub];
  __syncthreads();
  const int64_t block_first = (int64_t)blockIdx.x * (256 * kIndptrItems);
  auto panel_at = [&](int64_t e, int lo, int hi) -> int {  // last panel in [lo, hi] whose start is <= e
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_start[mid] <= e)
        lo = mid;
      else
        hi = mid - 1;
    }
    return lo;
  };
  // panels of the block's first (minus one) and last positions bound every
  // search; most blocks lie inside one panel and search nothing
  if (threadIdx.x == 0) s_qrange[0] = panel_at(block_first > 0 ? block_first - 1 : 0, 0, n_panels - 1);
  if (threadIdx.x == 64) s_qrange[1] = panel_at(block_first + 256 * kIndptrItems - 1, 0, n_panels - 1);
  __syncthreads();
  const int q_lo = s_qrange[0], q_hi = s_qrange[1];
  auto composite = [&](int64_t e) -> int64_t {
    if (e >= n) return (int64_t)n_panels * n_rows;
    return (int64_t)panel_at(e, q_lo, q_hi) * n_rows + (int64_t)prow[e];
  };
  const int64_t base = block_first + threadIdx.x;
#pragma unroll
  for (int i = 0; i < kIndptrItems; ++i) {
    // every lane computes its own key; the previous one comes from the lane
    // below (lane 0 computes it)
    const int64_t k = base + i * 256;
    const int64_t cur = composite(k);
    int64_t prev = __shfl_up(cur, 1);
    if ((threadIdx.x & 63) == 0) prev = k > 0 ? composite(k - 1) : -1;
    if (k <= n)
      for (int64_t r = prev + 1; r <= cur; ++r) indptr[r] = (OP)k;
  }
}

template <class OP>
__global__ void panel_starts_kernel(const OP* __restrict__ indptr, int64_t n_rows, int n_panels,
                                    int64_t* __restrict__ out) {
  const int q = threadIdx.x;
  if (q <= n_panels) out[q] = (int64_t)indptr[(int64_t)q * n_rows];
}

template <class V, class I, class P, class RT>
int panelize_typed(const Layout& L, char* ws, int64_t n_rows, int64_t n_cols, int64_t nnz, int n_panels,
                   const void* vals, const void* cols, const void* indptr, void* p_vals, void* p_cols,
                   void* p_indptr, hipStream_t s) {
  const int64_t width = ceil_div(n_cols, n_panels);
  const double inv_width = 1.0 / (double)width;
  int qbits = 0;
  while ((1 << qbits) < n_panels) ++qbits;
  int64_t* counts = reinterpret_cast<int64_t*>(ws + L.off_counts);
  int64_t* partial = reinterpret_cast<int64_t*>(ws + L.off_partials);
  RT* prow = reinterpret_cast<RT*>(ws + L.off_prow);
  hipLaunchKernelGGL((panel_count_kernel<I>), dim3((unsigned)ceil_div(L.n_sub, kWavesPerBlock)), dim3(256), 0, s,
                     static_cast<const I*>(cols), nnz, width, inv_width, n_panels, qbits, L.n_sub, counts);
  FS_CHECK_LAUNCH("panel_count_kernel");
  int rc = device_exclusive_scan(counts, L.n_counts, partial, s);
  if (rc != FS_OK) return rc;
  int64_t* tile_row = reinterpret_cast<int64_t*>(ws + L.off_tile_rows);
  hipLaunchKernelGGL((tile_rows_kernel<P>), dim3((unsigned)ceil_div(L.n_sub, 256)), dim3(256), 0, s,
                     static_cast<const P*>(indptr), n_rows, L.n_sub, tile_row);
  FS_CHECK_LAUNCH("tile_rows_kernel");
  hipLaunchKernelGGL((panel_scatter_kernel<V, I, P, RT>), dim3((unsigned)L.n_sub), dim3(64), 0, s,
                     static_cast<const V*>(vals), static_cast<const I*>(cols), static_cast<const P*>(indptr), n_rows,
                     nnz, width, inv_width, n_panels, qbits, L.n_sub, counts, tile_row, static_cast<V*>(p_vals),
                     static_cast<I*>(p_cols), prow);
  FS_CHECK_LAUNCH("panel_scatter_kernel");
  hipLaunchKernelGGL((panel_indptr_kernel<P, RT>), dim3((unsigned)ceil_div(nnz + 1, 256 * kIndptrItems)), dim3(256), 0,
                     s, prow, nnz,
                     n_rows, n_panels, counts, L.n_sub, static_cast<P*>(p_indptr));
  FS_CHECK_LAUNCH("panel_indptr_kernel");
  return FS_OK;
}

// Entry offsets of the panels in the stacked CSR, copied to the host.
template <class P>
int read_panel_starts(const void* p_indptr, int64_t n_rows, int n_panels, int64_t* dev_tmp, int64_t* host,
                      hipStream_t s) {
  hipLaunchKernelGGL((panel_starts_kernel<P>), dim3(1), dim3(128), 0, s, static_cast<const P*>(p_indptr), n_rows,
                     n_panels, dev_tmp);
  FS_CHECK_LAUNCH("panel_starts_kernel");
  FS_CHECK_HIP(hipMemcpyAsync(host, dev_tmp, sizeof(int64_t) * (n_panels + 1), hipMemcpyDeviceToHost, s));
  FS_CHECK_HIP(hipStreamSynchronize(s));
  return FS_OK;
}

template <class V, class I, class P>
int panelize_pos(const Layout& L, char* ws, int64_t n_rows, int64_t n_cols, int64_t nnz, int n_panels,
                 const void* vals, const void* cols, const void* indptr, void* pv, void* pc, void* pp, hipStream_t s) {
  if (n_rows <= (int64_t)0xffffffffLL)
    return panelize_typed<V, I, P, uint32_t>(L, ws, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, pv, pc, pp, s);
  return panelize_typed<V, I, P, uint64_t>(L, ws, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, pv, pc, pp, s);
}

template <class V>
int panelize_idx(const Layout& L, char* ws, int idx_t, int ptr_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                 int n_panels, const void* vals, const void* cols, const void* indptr, void* pv, void* pc, void* pp,
                 hipStream_t s) {
  if (idx_t == FS_I32 && ptr_t == FS_I32)
    return panelize_pos<V, int32_t, int32_t>(L, ws, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, pv, pc, pp, s);
  if (idx_t == FS_I32)
    return panelize_pos<V, int32_t, int64_t>(L, ws, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, pv, pc, pp, s);
  if (ptr_t == FS_I32)
    return panelize_pos<V, int64_t, int32_t>(L, ws, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, pv, pc, pp, s);
  return panelize_pos<V, int64_t, int64_t>(L, ws, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, pv, pc, pp, s);
}

}  // namespace fs

using namespace fs;

extern "C" size_t fs_csr_transpose_workspace_bytes(int64_t n_rows, int64_t n_cols, int64_t nnz) {
  if (nnz <= 0) return 0;
  return std::max(make_layout(n_rows, n_cols, nnz, true).total, make_wg_layout(n_cols, nnz).total);
}

extern "C" int fs_csr_transpose_bounded(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz) {
  // (the column pointer from atomic minima and a suffix minimum is monotone
  // and within [0, nnz] whatever the keys; read off sorted keys it is not)
  return transpose_wg_applies(val_t, n_rows, n_cols, nnz) && !colptr_from_keys() ? 1 : 0;
}

extern "C" int fs_csr_transpose(int val_t, int idx_t, int ptr_t, int out_idx_t, int out_ptr_t, int64_t n_rows,
                                int64_t n_cols, int64_t nnz, const void* vals, const void* cols, const void* indptr,
                                int conj, void* t_vals, void* t_cols, void* t_indptr, void* ws, size_t ws_bytes,
                                hipStream_t stream) {
  if (!valid_types(val_t, idx_t, ptr_t) || !(out_idx_t == FS_I32 || out_idx_t == FS_I64) ||
      !(out_ptr_t == FS_I32 || out_ptr_t == FS_I64))
    return fail(FS_E_INVALID, "fs_csr_transpose: bad type code");
  if (n_rows < 0 || n_cols < 0 || nnz < 0) return fail(FS_E_INVALID, "fs_csr_transpose: negative size");
  if (!t_indptr) return fail(FS_E_INVALID, "fs_csr_transpose: t_indptr is null");
  if (nnz == 0) {
    const int64_t n = n_cols + 1;
    if (out_ptr_t == FS_I32)
      hipLaunchKernelGGL((fill_kernel<int32_t>), dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream,
                         static_cast<int32_t*>(t_indptr), n, 0);
    else
      hipLaunchKernelGGL((fill_kernel<int64_t>), dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, stream,
                         static_cast<int64_t*>(t_indptr), n, (int64_t)0);
    FS_CHECK_LAUNCH("fill_kernel");
    return FS_OK;
  }
  if (!vals || !cols || !indptr || !t_vals || !t_cols) return fail(FS_E_INVALID, "fs_csr_transpose: null pointer");
  if (n_rows == 0 || n_cols == 0) return fail(FS_E_INVALID, "fs_csr_transpose: nnz > 0 with an empty dimension");
  if (transpose_wg_applies(val_t, n_rows, n_cols, nnz)) {
    if (!ws || ws_bytes < make_wg_layout(n_cols, nnz).total)
      return fail(FS_E_WORKSPACE, "fs_csr_transpose: workspace too small");
    return transpose_wg(static_cast<char*>(ws), val_t, idx_t, ptr_t, out_idx_t, out_ptr_t, n_rows, n_cols, nnz, vals,
                        cols, indptr, conj, t_vals, t_cols, t_indptr, stream);
  }
  const Layout L = make_layout(n_rows, n_cols, nnz, transpose_payload_enabled());
  if (!ws || ws_bytes < L.total) return fail(FS_E_WORKSPACE, "fs_csr_transpose: workspace too small");
  char* w = static_cast<char*>(ws);
  switch (val_t) {
    case FS_F32: return transpose_ptr<float>(L, w, idx_t, ptr_t, out_idx_t, out_ptr_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, t_vals, t_cols, t_indptr, stream);
    case FS_F64: return transpose_ptr<double>(L, w, idx_t, ptr_t, out_idx_t, out_ptr_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, t_vals, t_cols, t_indptr, stream);
    case FS_C64: return transpose_ptr<c32>(L, w, idx_t, ptr_t, out_idx_t, out_ptr_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, t_vals, t_cols, t_indptr, stream);
    default: return transpose_ptr<c64>(L, w, idx_t, ptr_t, out_idx_t, out_ptr_t, n_rows, n_cols, nnz, vals, cols, indptr, conj, t_vals, t_cols, t_indptr, stream);
  }
}

// fs_csr_transpose with the CSR structure check fused into its passes (the
// row-tile kernel tests the row pointers, the first count pass the
// columns): the five check words (fs_csr_check_bytes) are written to
// check_dev and copied to host_words, on the stream, for
// fs_csr_check_decode once it has drained.  For a valid matrix the decoded
// column range is [0, 0]; outside [0, n_cols) it holds the offending
// extremes.  Only where fs_csr_transpose_bounded holds (the transpose stays
// in bounds on any input, so the check need not run first), with nnz > 0.
extern "C" int fs_csr_transpose_checked(int val_t, int idx_t, int ptr_t, int out_idx_t, int out_ptr_t,
                                        int64_t n_rows, int64_t n_cols, int64_t nnz, const void* vals,
                                        const void* cols, const void* indptr, int conj, void* t_vals, void* t_cols,
                                        void* t_indptr, void* ws, size_t ws_bytes, void* check_dev,
                                        void* host_words, hipStream_t stream) {
  if (!valid_types(val_t, idx_t, ptr_t) || !(out_idx_t == FS_I32 || out_idx_t == FS_I64) ||
      !(out_ptr_t == FS_I32 || out_ptr_t == FS_I64))
    return fail(FS_E_INVALID, "fs_csr_transpose_checked: bad type code");
  if (n_rows <= 0 || n_cols <= 0 || nnz <= 0)
    return fail(FS_E_INVALID, "fs_csr_transpose_checked: needs rows, columns and entries");
  if (!fs_csr_transpose_bounded(val_t, n_rows, n_cols, nnz))
    return fail(FS_E_INVALID, "fs_csr_transpose_checked: not a bounded transpose (check with fs_csr_check_enqueue)");
  if (!vals || !cols || !indptr || !t_vals || !t_cols || !t_indptr || !check_dev || !host_words)
    return fail(FS_E_INVALID, "fs_csr_transpose_checked: null pointer");
  if (!ws || ws_bytes < make_wg_layout(n_cols, nnz).total)
    return fail(FS_E_WORKSPACE, "fs_csr_transpose_checked: workspace too small");
  unsigned long long* ck = static_cast<unsigned long long*>(check_dev);
  const int rc = transpose_wg(static_cast<char*>(ws), val_t, idx_t, ptr_t, out_idx_t, out_ptr_t, n_rows, n_cols, nnz,
                              vals, cols, indptr, conj, t_vals, t_cols, t_indptr, stream, ck);
  if (rc != FS_OK) return rc;
  FS_CHECK_HIP(hipMemcpyAsync(host_words, ck, 5 * sizeof(unsigned long long), hipMemcpyDeviceToHost, stream));
  return FS_OK;
}

// Key range of a COO matrix: n_rows * n_cols lexicographic keys.
static Layout coo_layout(int64_t n_rows, int64_t n_cols, int64_t nnz) {
  const int64_t range = (n_cols > 0 && n_rows > INT64_MAX / n_cols) ? INT64_MAX : n_rows * n_cols;
  return make_layout(n_rows, range, nnz);
}

// COO -> CSR on the workgroup-tile passes (4- and 8-byte values, sizes below
// 2^32): an LSD sort by column, then by row (stable both times, so the order
// is lexicographic by (row, col) and equal pairs keep their input order).
// The payload carries the value and the row; the first row pass swaps the
// row into the key and the column into the payload; the last pass writes
// values, columns and, through atomic minima and a suffix minimum, indptr.
inline bool coo_wg_applies(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz, int assume_sorted) {
  return !assume_sorted && transpose_wg_applies(val_t, n_rows, n_cols, nnz) && n_rows <= (int64_t)0xffffffffLL &&
         !colptr_from_keys();
}

// by_row: the row passes alone (entries of a row keep their input order).
int coo_to_csr_wg(char* ws, int val_t, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz, const void* vals,
                  const void* rows, const void* cols, void* out_vals, void* out_cols, void* out_indptr,
                  hipStream_t s, bool by_row = false) {
  const WgLayout L = make_wg_layout(std::max(n_rows, n_cols), nnz);
  const int vw = val_t == FS_F32 ? 1 : 2;
  const int64_t n_ptr = n_rows + 1;
  hipLaunchKernelGGL((fill_kernel<int64_t>), dim3((unsigned)ceil_div(n_ptr, 256)), dim3(256), 0, s,
                     static_cast<int64_t*>(out_indptr), n_ptr, (int64_t)nnz);
  FS_CHECK_LAUNCH("fill_kernel");
  const int idx_kind = idx_t == FS_I32 ? 0 : 1;
  const int col_bits = key_bits(n_cols), row_bits = key_bits(n_rows);
  const int col_passes = by_row || col_bits == 0 ? 0 : wg_passes(col_bits);
  const int row_passes = wg_passes(row_bits);
  const int passes = col_passes + row_passes;
  // the first pass reads its keys from the columns (or, without column
  // passes, from the rows) and its second index from the other array
  WgIO io{vals, nullptr, 0, nullptr, n_rows, 0, out_vals, out_cols, 0, out_indptr, 1, n_rows, 0u,
          col_passes > 0 ? rows : cols, idx_t == FS_I64 ? 1 : 0, 0};
  uint32_t* counts = reinterpret_cast<uint32_t*>(ws + L.off_counts);
  uint32_t* partial = reinterpret_cast<uint32_t*>(ws + L.off_partial);
  uint32_t* totals = reinterpret_cast<uint32_t*>(ws + L.off_totals);
  uint32_t* ka = reinterpret_cast<uint32_t*>(ws + L.off_keys_a);
  uint32_t* kb = reinterpret_cast<uint32_t*>(ws + L.off_keys_b);
  void* pa = ws + L.off_pay_a;
  void* pb = ws + L.off_pay_b;
  const void* kin = col_passes > 0 ? cols : rows;
  int kind = idx_kind;
  const void* pin = nullptr;
  uint32_t* kout = ka;
  void* pout = pa;
  const dim3 g((unsigned)L.n_tiles);
  for (int p = 0; p < passes; ++p) {
    const bool col_phase = p < col_passes;
    const int q = col_phase ? p : p - col_passes;              // pass within its phase
    const int nq = col_phase ? col_passes : row_passes;
    const int bits = col_phase ? col_bits : row_bits;
    // the phase's key bits split evenly over its passes
    int shift = 0;
    for (int j = 0; j < q; ++j) shift += (bits - shift + (nq - j) - 1) / (nq - j);
    const int pbits = (bits - shift + (nq - q) - 1) / (nq - q);
    const unsigned mask = pbits > 0 ? (1u << pbits) - 1u : 0u;
    const int nd = (int)mask + 1;
    io.swap = (!col_phase && q == 0 && col_passes > 0) ? 1 : 0;
    // a swapping pass counts the keys it will sort by: the rows, still in the payload
    const void* ckin = kin;
    int ckind = kind;
    if (io.swap) {
      ckin = static_cast<const char*>(pin) + 4 * (vw == 1 ? 1 : 2);
      ckind = vw == 1 ? 5 : 6;  // the row word of the 8- / 12-byte payload
    }
    hipLaunchKernelGGL(wg_count_kernel, g, dim3(kWgThreads), 0, s, ckin, ckind, nnz, shift, mask, counts,
                       (unsigned long long*)nullptr, (int64_t)0);
    FS_CHECK_LAUNCH("wg_count_kernel");
    hipLaunchKernelGGL(wg_scan_reduce_kernel, dim3((unsigned)L.n_blocks), dim3(256), 0, s, counts, L.n_tiles, nd,
                       partial);
    FS_CHECK_LAUNCH("wg_scan_reduce_kernel");
    hipLaunchKernelGGL(wg_scan_column_kernel, dim3((unsigned)nd), dim3(256), 0, s, partial, L.n_blocks, nd, totals);
    FS_CHECK_LAUNCH("wg_scan_column_kernel");
    hipLaunchKernelGGL(wg_scan_down_kernel, dim3((unsigned)L.n_blocks), dim3(256), 0, s, counts, L.n_tiles, nd,
                       partial, totals);
    FS_CHECK_LAUNCH("wg_scan_down_kernel");
    const int mode = passes == 1 ? kScatterOnly : p == 0 ? kScatterFirst : p == passes - 1 ? kScatterLast
                                                                                            : kScatterPlain;
    const int rc = vw == 1 ? wg_launch_scatter<1>(mode, g, s, kin, kind, pin, nnz, shift, mask, counts, kout, pout, io)
                           : wg_launch_scatter<2>(mode, g, s, kin, kind, pin, nnz, shift, mask, counts, kout, pout, io);
    if (rc != FS_OK) return rc;
    kin = kout;
    kind = 2;
    pin = pout;
    kout = kout == ka ? kb : ka;
    pout = pout == pa ? pb : pa;
  }
  return colptr_suffix_min<uint64_t>(static_cast<uint64_t*>(out_indptr), n_ptr,
                                     reinterpret_cast<uint64_t*>(ws + L.off_bmin), L.n_min_blocks, s);
}

extern "C" size_t fs_coo_to_csr_workspace_bytes(int64_t n_rows, int64_t n_cols, int64_t nnz) {
  if (nnz <= 0) return 0;
  return std::max(coo_layout(n_rows, n_cols, nnz).total, make_wg_layout(std::max(n_rows, n_cols), nnz).total);
}

extern "C" int fs_coo_to_csr(int val_t, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz, const void* vals,
                             const void* rows, const void* cols, int assume_sorted, void* out_vals, void* out_cols,
                             void* out_indptr, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!valid_types(val_t, idx_t, FS_I64)) return fail(FS_E_INVALID, "fs_coo_to_csr: bad type code");
  if (n_rows < 0 || n_cols < 0 || nnz < 0) return fail(FS_E_INVALID, "fs_coo_to_csr: negative size");
  if (n_cols > 0 && n_rows > INT64_MAX / n_cols) return fail(FS_E_INVALID, "fs_coo_to_csr: n_rows * n_cols overflows");
  if (!out_indptr) return fail(FS_E_INVALID, "fs_coo_to_csr: out_indptr is null");
  if (nnz == 0) {
    hipLaunchKernelGGL((fill_kernel<int64_t>), dim3((unsigned)ceil_div(n_rows + 1, 256)), dim3(256), 0, stream,
                       static_cast<int64_t*>(out_indptr), n_rows + 1, (int64_t)0);
    FS_CHECK_LAUNCH("fill_kernel");
    return FS_OK;
  }
  if (!vals || !rows || !cols || !out_vals || !out_cols) return fail(FS_E_INVALID, "fs_coo_to_csr: null pointer");
  if (coo_wg_applies(val_t, n_rows, n_cols, nnz, assume_sorted)) {
    if (!ws || ws_bytes < make_wg_layout(std::max(n_rows, n_cols), nnz).total)
      return fail(FS_E_WORKSPACE, "fs_coo_to_csr: workspace too small");
    return coo_to_csr_wg(static_cast<char*>(ws), val_t, idx_t, n_rows, n_cols, nnz, vals, rows, cols, out_vals,
                         out_cols, out_indptr, stream);
  }
  const Layout L = coo_layout(n_rows, n_cols, nnz);
  if (!ws || ws_bytes < L.total) return fail(FS_E_WORKSPACE, "fs_coo_to_csr: workspace too small");
  char* w = static_cast<char*>(ws);
  switch (val_t) {
    case FS_F32: return coo_to_csr_idx<float>(L, w, idx_t, nnz, n_rows, n_cols, vals, rows, cols, assume_sorted, out_vals, out_cols, out_indptr, stream);
    case FS_F64: return coo_to_csr_idx<double>(L, w, idx_t, nnz, n_rows, n_cols, vals, rows, cols, assume_sorted, out_vals, out_cols, out_indptr, stream);
    case FS_C64: return coo_to_csr_idx<c32>(L, w, idx_t, nnz, n_rows, n_cols, vals, rows, cols, assume_sorted, out_vals, out_cols, out_indptr, stream);
    default: return coo_to_csr_idx<c64>(L, w, idx_t, nnz, n_rows, n_cols, vals, rows, cols, assume_sorted, out_vals, out_cols, out_indptr, stream);
  }
}

extern "C" int fs_coo_to_csr_by_row(int val_t, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                                    const void* vals, const void* rows, const void* cols, void* out_vals,
                                    void* out_cols, void* out_indptr, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!valid_types(val_t, idx_t, FS_I64)) return fail(FS_E_INVALID, "fs_coo_to_csr_by_row: bad type code");
  if (n_rows <= 0 || n_cols <= 0 || !coo_wg_applies(val_t, n_rows, n_cols, nnz, 0))
    return fail(FS_E_INVALID, "fs_coo_to_csr_by_row: type or sizes not supported (use fs_coo_to_csr)");
  if (!vals || !rows || !cols || !out_vals || !out_cols || !out_indptr)
    return fail(FS_E_INVALID, "fs_coo_to_csr_by_row: null pointer");
  if (!ws || ws_bytes < make_wg_layout(std::max(n_rows, n_cols), nnz).total)
    return fail(FS_E_WORKSPACE, "fs_coo_to_csr_by_row: workspace too small");
  return coo_to_csr_wg(static_cast<char*>(ws), val_t, idx_t, n_rows, n_cols, nnz, vals, rows, cols, out_vals, out_cols,
                       out_indptr, stream, true);
}

// Range check of two index arrays: flag k is set when array k has an entry
// outside [0, n_k).  16-byte loads where an array is aligned.
template <class I>
__device__ inline bool any_outside(const I* __restrict__ p, int64_t n, uint64_t limit, int64_t t0, int64_t stride) {
  constexpr int kVec = (int)(16 / sizeof(I));
  using L = I __attribute__((ext_vector_type(kVec)));
  bool bad = false;
  int64_t done = 0;
  if (((uintptr_t)p % 16) == 0) {
    const L* v = reinterpret_cast<const L*>(p);
    const int64_t nv = n / kVec;
    constexpr int kAheadV = 4;
    for (int64_t i0 = t0; i0 < nv; i0 += kAheadV * stride) {
      L q[kAheadV];
#pragma unroll
      for (int u = 0; u < kAheadV; ++u) q[u] = v[i0 + u * stride < nv ? i0 + u * stride : i0];
#pragma unroll
      for (int u = 0; u < kAheadV; ++u)
#pragma unroll
        for (int j = 0; j < kVec; ++j) bad |= (uint64_t)(int64_t)q[u][j] >= limit;
    }
    done = nv * kVec;
  }
  for (int64_t i = done + t0; i < n; i += stride) bad |= (uint64_t)(int64_t)p[i] >= limit;
  return bad;
}

template <class I>
__global__ __launch_bounds__(256) void coo_range_kernel(const I* __restrict__ rows, const I* __restrict__ cols,
                                                        int64_t n, uint64_t n_rows, uint64_t n_cols,
                                                        int32_t* __restrict__ flags) {
  const int64_t t0 = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
  if (any_outside(rows, n, n_rows, t0, stride)) __hip_atomic_store(flags, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (any_outside(cols, n, n_cols, t0, stride))
    __hip_atomic_store(flags + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

extern "C" int fs_coo_check_ranges(int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz, const void* rows,
                                   const void* cols, int32_t* flags, hipStream_t stream) {
  if (!(idx_t == FS_I32 || idx_t == FS_I64)) return fail(FS_E_INVALID, "fs_coo_check_ranges: bad type code");
  if (n_rows < 0 || n_cols < 0 || nnz <= 0 || !rows || !cols || !flags)
    return fail(FS_E_INVALID, "fs_coo_check_ranges: negative size, no entries or null pointer");
  void* df = nullptr;
  FS_CHECK_HIP(hipHostGetDevicePointer(&df, flags, 0));
  flags[0] = flags[1] = 0;
  const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(nnz, 256 * 8), 2048);
  if (idx_t == FS_I64)
    hipLaunchKernelGGL((coo_range_kernel<int64_t>), dim3(blocks), dim3(256), 0, stream,
                       static_cast<const int64_t*>(rows), static_cast<const int64_t*>(cols), nnz, (uint64_t)n_rows,
                       (uint64_t)n_cols, static_cast<int32_t*>(df));
  else
    hipLaunchKernelGGL((coo_range_kernel<int32_t>), dim3(blocks), dim3(256), 0, stream,
                       static_cast<const int32_t*>(rows), static_cast<const int32_t*>(cols), nnz, (uint64_t)n_rows,
                       (uint64_t)n_cols, static_cast<int32_t*>(df));
  FS_CHECK_LAUNCH("coo_range_kernel");
  FS_CHECK_HIP(hipStreamSynchronize(stream));
  return FS_OK;
}

// Panel layout: the [panel][sub-tile] counts and their scan partials, the
// first row of every sub-tile, then the row id of every stacked entry (up to
// 8 bytes).
static Layout panel_layout(int64_t n_rows, int64_t n_panels, int64_t nnz) {
  (void)n_rows;
  Layout L{};
  L.n_sub = ceil_div(nnz, kSub);
  L.n_counts = n_panels * L.n_sub;
  L.n_partials = ceil_div(L.n_counts, kScanTile);
  size_t o = 0;
  L.off_counts = o;
  o = align256(o + sizeof(int64_t) * L.n_counts);
  L.off_partials = o;
  o = align256(o + sizeof(int64_t) * (L.n_partials + 1));
  L.off_tile_rows = o;
  o = align256(o + sizeof(int64_t) * L.n_sub);
  L.off_prow = o;  // also stages the n_panels + 1 panel starts afterwards
  o = align256(o + 8 * (size_t)std::max<int64_t>(nnz, n_panels + 1));
  L.total = o;
  return L;
}

extern "C" size_t fs_csr_panelize_workspace_bytes(int64_t n_rows, int64_t n_cols, int64_t nnz, int n_panels) {
  (void)n_cols;
  if (n_panels <= 0) return 0;
  if (nnz <= 0) return 256;  // the panel-start staging slot
  return panel_layout(n_rows, n_panels, nnz).total;
}

extern "C" int fs_csr_panelize(int val_t, int idx_t, int ptr_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                               int n_panels, const void* vals, const void* cols, const void* indptr, void* p_vals,
                               void* p_cols, void* p_indptr, int64_t* panel_nnz, void* ws, size_t ws_bytes,
                               hipStream_t stream) {
  if (!valid_types(val_t, idx_t, ptr_t)) return fail(FS_E_INVALID, "fs_csr_panelize: bad type code");
  if (n_rows < 0 || n_cols <= 0 || nnz < 0 || n_panels <= 0 || n_panels > 64)
    return fail(FS_E_INVALID, "fs_csr_panelize: bad size");
  if (!p_indptr || !panel_nnz) return fail(FS_E_INVALID, "fs_csr_panelize: p_indptr / panel_nnz is null");
  const int64_t n_out = (int64_t)n_panels * n_rows;
  if (!ws || ws_bytes < fs_csr_panelize_workspace_bytes(n_rows, n_cols, nnz, n_panels))
    return fail(FS_E_WORKSPACE, "fs_csr_panelize: workspace too small");
  if (nnz == 0) {
    if (ptr_t == FS_I32)
      hipLaunchKernelGGL((fill_kernel<int32_t>), dim3((unsigned)ceil_div(n_out + 1, 256)), dim3(256), 0, stream,
                         static_cast<int32_t*>(p_indptr), n_out + 1, 0);
    else
      hipLaunchKernelGGL((fill_kernel<int64_t>), dim3((unsigned)ceil_div(n_out + 1, 256)), dim3(256), 0, stream,
                         static_cast<int64_t*>(p_indptr), n_out + 1, (int64_t)0);
    FS_CHECK_LAUNCH("fill_kernel");
    for (int q = 0; q <= n_panels; ++q) panel_nnz[q] = 0;
    return FS_OK;
  }
  if (!vals || !cols || !indptr || !p_vals || !p_cols) return fail(FS_E_INVALID, "fs_csr_panelize: null pointer");
  const Layout L = panel_layout(n_rows, n_panels, nnz);
  char* w = static_cast<char*>(ws);
  int rc = FS_OK;
  switch (val_t) {
    case FS_F32: rc = panelize_idx<float>(L, w, idx_t, ptr_t, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, p_vals, p_cols, p_indptr, stream); break;
    case FS_F64: rc = panelize_idx<double>(L, w, idx_t, ptr_t, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, p_vals, p_cols, p_indptr, stream); break;
    case FS_C64: rc = panelize_idx<c32>(L, w, idx_t, ptr_t, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, p_vals, p_cols, p_indptr, stream); break;
    default: rc = panelize_idx<c64>(L, w, idx_t, ptr_t, n_rows, n_cols, nnz, n_panels, vals, cols, indptr, p_vals, p_cols, p_indptr, stream); break;
  }
  if (rc != FS_OK) return rc;
  // the composite-key slot is free once the indptr is built (stream order)
  int64_t* tmp = reinterpret_cast<int64_t*>(w + L.off_prow);
  if (ptr_t == FS_I32) return read_panel_starts<int32_t>(p_indptr, n_rows, n_panels, tmp, panel_nnz, stream);
  return read_panel_starts<int64_t>(p_indptr, n_rows, n_panels, tmp, panel_nnz, stream);
}
