// spmv_scatter.hip — SpMV by scattered products on gfx950: y[o(e)] += a(e) x[i(e)]
// over entries e in any order, without a sorted copy of the matrix.
//
// Serves the calls whose entries do not lie in output order: the unprepared
// y = A^T x / A^H x of a CSR matrix (reference: the argsort transpose of
// spmv_csr.py:477-515 followed by spmv_csr.py:679-723) and the unprepared COO
// SpMV (spmv_coo.py:425-474, 575-644, which sorts the entries first).
//
// Two passes over the entries:
//  1. scatter: a workgroup takes a tile of kWgTile entries in input order,
//     forms every product in the accumulator type and partitions them by
//     bucket, a bucket being 2^low_bits consecutive outputs (the tile is
//     sorted by bucket in LDS, as in the transpose's radix pass, so that a
//     bucket's products leave as one run); an entry leaves as its product and
//     a 16-bit output number within the bucket;
//  2. reduce: a workgroup takes a segment of one bucket's products, keeps the
//     bucket's sums in LDS (one copy per wave) and adds the products to them
//     in order; buckets cut into several segments are completed by a fix-up.
// Order of every addition is fixed (stable partition, lanes of equal output
// ranked by ballots, waves and segments in order): no atomics on values, and
// the result is the same bits on every run.
//
// Per entry the passes read A once (the output index twice) and write and read
// one (product, 16-bit number) pair; the transpose they replace moves (key,
// value, row) through two passes and ends in a random gather of x.  Both
// kernels are bound by instruction issue, not by HBM (a 1M x 1M matrix with 32
// uniform columns per row, float32: 209 + 108 us for 0.67 + 0.34 GB).
// Measured, us per call, before (transpose or sort, then SpMV) and now:
// A^T x of that matrix 875 -> 394; 500,000 rows of 32, complex64 904 -> 466,
// complex128 1438 -> 490; R-MAT 2^20 complex64 A^H x 1856 -> 690; the 27-point
// 100^3 stencil, float64, 674 -> 543; 3000 x 2000 ragged, float64, 93 -> 73;
// COO, 4 M float64 entries over 400,009 rows, 1180 -> 153; 5000 entries over
// 1000 rows 607 -> 66.
//
// Precision: float32 products are exact in float64 and are summed there, as
// everywhere else; float64 / complex128 products are rounded once and summed
// with a running compensation (hi + lo), which keeps the error below that of
// a plain chain of fused multiply-adds.
//
// Bounded on any input: buckets are masked digits, rows are clamped, stray
// x indices read x[0], outputs past the end are not written; what is wrong
// with the structure is reported through the flags and the caller discards y.
#include "fs_common.hpp"
#include "radix_tile.hpp"
#include "row_starts.hpp"
#include "scatter_segments.hpp"

#include <algorithm>
#include <type_traits>

namespace fs {

// ---- accumulators ---------------------------------------------------------
// Sum with compensation: hi is the plain running sum (so infinities and NaN
// behave as in a plain sum), lo the rounding errors of its additions.
struct alignas(16) Comp {
  double hi, lo;
};
struct alignas(16) Comp2 {
  Comp re, im;
};

__device__ inline void comp_add(Comp& a, double p) {
  const double s = a.hi + p;
  const double b = s - a.hi;
  a.lo += (a.hi - (s - b)) + (p - b);
  a.hi = s;
}
__device__ inline double comp_out(Comp a) {
  return __builtin_isfinite(a.hi) ? a.hi + a.lo : a.hi;  // lo is NaN once hi has overflowed
}

template <class V>
struct SA;  // P: the stored product, A: the accumulator
template <>
struct SA<float> {
  using P = double;
  using A = double;
  __device__ static void add(A& a, P p) { a += p; }
  __device__ static A join(A a, A b) { return a + b; }
  __device__ static float out(A a) { return (float)a; }
};
template <>
struct SA<c32> {
  using P = c64;
  using A = c64;
  __device__ static void add(A& a, P p) {
    a.re += p.re;
    a.im += p.im;
  }
  __device__ static A join(A a, A b) { return c64{a.re + b.re, a.im + b.im}; }
  __device__ static c32 out(A a) { return c32{(float)a.re, (float)a.im}; }
};
template <>
struct SA<double> {
  using P = double;
  using A = Comp;
  __device__ static void add(A& a, P p) { comp_add(a, p); }
  __device__ static A join(A a, A b) {
    comp_add(a, b.hi);
    a.lo += b.lo;
    return a;
  }
  __device__ static double out(A a) { return comp_out(a); }
};
template <>
struct SA<c64> {
  using P = c64;
  using A = Comp2;
  __device__ static void add(A& a, P p) {
    comp_add(a.re, p.re);
    comp_add(a.im, p.im);
  }
  __device__ static A join(A a, A b) {
    return Comp2{SA<double>::join(a.re, b.re), SA<double>::join(a.im, b.im)};
  }
  __device__ static c64 out(A a) { return c64{comp_out(a.re), comp_out(a.im)}; }
};

template <class T>
__device__ inline T shfl_words(const T& v, int src) {
  constexpr int W = (int)(sizeof(T) / 4);
  int w[W];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int k = 0; k < W; ++k) w[k] = __builtin_amdgcn_ds_bpermute(src << 2, w[k]);
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// Flags live in pinned host memory: system-scope stores reach it directly.
__device__ inline void raise_flag(int32_t* flags, int k) {
  __hip_atomic_store(flags + k, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Row of the first entry of every wave sub-tile, with the row pointer's part
// of the structure check: flag 0 a start other than 0, flag 1 an end other
// than nnz, flag 2 a decrease.  (A malformed pointer can leave slots
// unwritten; the scatter clamps what it reads.)
template <class P>
__global__ __launch_bounds__(256) void scatter_rows_kernel(const P* __restrict__ rowptr, int64_t n_rows, int64_t nnz,
                                                           int64_t n_sub, int64_t* __restrict__ tile_row,
                                                           int32_t* __restrict__ flags) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n_rows) return;
  const int64_t a = (int64_t)rowptr[r], b = (int64_t)rowptr[r + 1];
  if (r == 0 && a != 0) raise_flag(flags, 0);
  if (r == n_rows - 1 && b != nnz) raise_flag(flags, 1);
  if (b < a) raise_flag(flags, 2);
  const int64_t end = row_sub_tile(b, kWgSub, n_sub);
  for (int64_t sub = row_sub_tile(a, kWgSub, n_sub); sub < end; ++sub) tile_row[sub] = r;
}

// Bucket counts of every tile, cnt[tile][bucket], and the range check of the
// output indices (flag `flag`).
template <class I>
__global__ __launch_bounds__(kWgThreads) void scatter_count_kernel(const I* __restrict__ keys, int64_t n, int low_bits,
                                                                   unsigned mask, uint32_t* __restrict__ counts,
                                                                   uint64_t n_out, int32_t* __restrict__ flags,
                                                                   int flag) {
  __shared__ unsigned s_hist[kWgMaxDigits];
  const int nd = (int)mask + 1;
  const int t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * kWgTile;
  const int cnt = n - base < kWgTile ? (int)(n - base) : (int)kWgTile;
  for (int d = t; d < nd; d += kWgThreads) s_hist[d] = 0;
  __syncthreads();
  constexpr int kVec = (int)(16 / sizeof(I));  // a count needs no order: 16-byte loads of a full, aligned tile
  I key[kWgChunks];
  static_assert(kWgChunks % kVec == 0, "a tile is whole 16-byte loads per thread");
  if (cnt == (int)kWgTile && ((uintptr_t)keys % 16) == 0) {
    using L = I __attribute__((ext_vector_type(kVec)));
    const L* p = reinterpret_cast<const L*>(keys + base) + t;
#pragma unroll
    for (int k = 0; k < kWgChunks / kVec; ++k) {
      const L q = p[k * kWgThreads];
#pragma unroll
      for (int j = 0; j < kVec; ++j) key[k * kVec + j] = q[j];
    }
  } else {
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) key[ch] = ch * kWgThreads + t < cnt ? keys[base + ch * kWgThreads + t] : (I)-1;
  }
  bool bad = false;
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch) {
    const bool in = cnt == (int)kWgTile || ch * kWgThreads + t < cnt;
    if (in) {
      bad |= (uint64_t)(int64_t)key[ch] >= n_out;
      atomicAdd(&s_hist[((uint32_t)key[ch] >> low_bits) & mask], 1u);
    }
  }
  if (bad) raise_flag(flags, flag);
  __syncthreads();
  for (int d = t; d < nd; d += kWgThreads) counts[(int64_t)blockIdx.x * nd + d] = s_hist[d];
}

// Bucket starts, the segments of every bucket (scatter_bucket_segments) and the
// buckets of several (split[0 .. split[nd])).  One workgroup; n_seg =
// seg_first[nd] segments in all.
__global__ __launch_bounds__(256) void scatter_plan_kernel(const uint32_t* __restrict__ totals, int nd,
                                                           uint32_t seg_items, uint32_t* __restrict__ bucket_start,
                                                           uint32_t* __restrict__ seg_first,
                                                           uint32_t* __restrict__ seg_bucket,
                                                           uint32_t* __restrict__ split) {
  __shared__ int64_t s_wave[4];
  const int q = (nd + 255) / 256;
  const int d0 = threadIdx.x * q;
  int64_t items = 0, segs = 0;  // segs: segments << 12 | split buckets (at most kWgMaxDigits), one scan for both
  for (int j = 0; j < q; ++j)
    if (d0 + j < nd) {
      const uint32_t c = totals[d0 + j];
      const int64_t k = scatter_bucket_segments(c, seg_items);
      items += c;
      segs += k << 12 | (k > 1 ? 1 : 0);
    }
  int64_t all;
  int64_t run = block_exclusive_scan(items, s_wave, all);
  int64_t all_segs;
  const int64_t first = block_exclusive_scan(segs, s_wave, all_segs);
  int64_t seg = first >> 12, sp = first & 4095;
  for (int j = 0; j < q; ++j)
    if (d0 + j < nd) {
      const uint32_t c = totals[d0 + j];
      const int64_t k = scatter_bucket_segments(c, seg_items);
      bucket_start[d0 + j] = (uint32_t)run;
      seg_first[d0 + j] = (uint32_t)seg;
      for (int64_t u = 0; u < k; ++u) seg_bucket[seg + u] = (uint32_t)(d0 + j);
      if (k > 1) split[sp++] = (uint32_t)(d0 + j);
      run += c;
      seg += k;
    }
  if (threadIdx.x == 0) {
    bucket_start[nd] = (uint32_t)all;
    seg_first[nd] = (uint32_t)(all_segs >> 12);
    split[nd] = (uint32_t)(all_segs & 4095);
  }
}

struct ScatterIn {
  const void* vals;
  const void* keys;         // output index of every entry
  int key64;
  const void* other;        // x index of every entry (COO), or null: the rows of rowptr
  int other64;
  const void* rowptr;
  int ptr64;
  const int64_t* tile_row;
  int64_t n_sub;
  int64_t n_x;              // entries of x
  int conj;
};

// Pass 1 (see the top).  8 waves rank their 768 entries each against their own
// 16-bit LDS counters (in input order: the partition is stable), one scan
// over the buckets turns the counts into tile positions, and thread t owns
// sorted positions t, t + 512, ... whose destinations it keeps in registers
// while the products pass through the same LDS buffer.
// What bounds it is instruction issue (a SIMD is active 78% of the time; a
// VALU instruction of a wave takes 4 cycles) across phases that end in
// barriers, with two workgroups per CU at 128 VGPRs; hence the lane tests
// compiled out of full tiles, the bucket offsets loaded at the start, and the
// counter updates of all chunks issued before the first is waited for.
template <class V>
constexpr int scatter_buf_bytes() {  // all products of the tile at 8 bytes, half of them at 16
  return (int)kWgTile * 8;
}
static_assert(kWgWaves * kWgMaxDigits * 2 <= scatter_buf_bytes<float>(), "wave counters fit the buffer");

template <class V, bool FULL>
__device__ inline void scatter_tile(const ScatterIn& in, const V* __restrict__ x, int64_t tile, int tcnt, int low_bits,
                                    unsigned mask, const uint32_t* __restrict__ offsets,
                                    uint16_t* __restrict__ low_out, typename SA<V>::P* __restrict__ prod_out,
                                    int32_t* __restrict__ flags, int flag, uint8_t* s_buf, uint32_t* s_off,
                                    int64_t* s_wave) {
  using P = typename SA<V>::P;
  constexpr int kWords = kWgMaxDigits / 2;  // counter words per wave
  const int nd = (int)mask + 1;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // scalar: so are the wave's base addresses
  const int64_t base = tile * kWgTile + (int64_t)w * kWgSub;
  const int left = tcnt - w * (int)kWgSub;
  const int cnt = FULL ? (int)kWgSub : (left < 0 ? 0 : (left < (int)kWgSub ? left : (int)kWgSub));
  // thread t owns buckets [t q, t q + q), q even (both halves of a counter word)
  constexpr int kQMax = 2 * ((kWgMaxDigits + 2 * kWgThreads - 1) / (2 * kWgThreads));
  const int q = nd > 2 * kWgThreads ? kQMax : 2;
  const int d0 = t * q;
  uint32_t key[kWgChunks];
  wg_load_keys<FULL>(in.keys, in.key64 ? 1 : 0, base, cnt, lane, key);
  uint32_t off[kQMax];
#pragma unroll
  for (int j = 0; j < kQMax; ++j) off[j] = j < q && d0 + j < nd ? offsets[tile * nd + d0 + j] : 0u;
  P prod[kWgChunks];
  {
    V val[kWgChunks];
    const V* vp = static_cast<const V*>(in.vals) + base + lane;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) val[ch] = FULL || ch * 64 + lane < cnt ? vp[ch * 64] : V{};
    uint32_t src[kWgChunks];
    if (in.other) {
      bool bad = false;
      auto load = [&](auto tag) {
        using I = decltype(tag);
        const I* op = static_cast<const I*>(in.other) + base + lane;
        I raw[kWgChunks];
#pragma unroll
        for (int ch = 0; ch < kWgChunks; ++ch) raw[ch] = FULL || ch * 64 + lane < cnt ? op[ch * 64] : (I)0;
#pragma unroll
        for (int ch = 0; ch < kWgChunks; ++ch) {
          const bool out = (uint64_t)(int64_t)raw[ch] >= (uint64_t)in.n_x;
          bad |= out;
          src[ch] = out ? 0u : (uint32_t)raw[ch];
        }
      };
      if (in.other64) load(int64_t{});
      else load(int32_t{});
      if (bad) raise_flag(flags, flag);
    } else if (cnt > 0) {
      const int64_t sub = tile * kWgWaves + w;
      auto clamp_row = [&](int64_t r) { return r < 0 ? (int64_t)0 : (r >= in.n_x ? in.n_x - 1 : r); };
      const int64_t r0 = clamp_row(in.tile_row[sub]);
      const int64_t r1 = sub + 1 < in.n_sub ? clamp_row(in.tile_row[sub + 1]) : in.n_x - 1;
      unsigned* s_mark = reinterpret_cast<unsigned*>(s_buf) + w * kWgSub;
      // (a row is r0 plus a mark, and marks are at most r1 - r0: inside x)
      if (in.ptr64)
        wg_rows<int64_t>(static_cast<const int64_t*>(in.rowptr), r0, r1, base, cnt, s_mark, lane, src);
      else
        wg_rows<int32_t>(static_cast<const int32_t*>(in.rowptr), r0, r1, base, cnt, s_mark, lane, src);
    } else {
#pragma unroll
      for (int ch = 0; ch < kWgChunks; ++ch) src[ch] = 0u;
    }
    V xv[kWgChunks];
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) xv[ch] = x[src[ch]];
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) prod[ch] = VT<V>::mul(in.conj ? VT<V>::conj(val[ch]) : val[ch], xv[ch]);
    __syncthreads();  // every wave is done with its row marks
  }
  // ranks within the wave's buckets, against wave w's own counters
  uint32_t* wc = reinterpret_cast<uint32_t*>(s_buf);
  uint32_t* my = wc + w * kWords;
  for (int j = lane; j < (nd + 1) / 2; j += 64) my[j] = 0u;
  wave_sync_t();
  unsigned local[kWgChunks];
  {
    unsigned old[kWgChunks];
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      const bool valid = FULL || ch * 64 + lane < cnt;
      const unsigned digit = (key[ch] >> low_bits) & mask;
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
  // per bucket pair: wave bases, then the tile's bucket starts
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
    const unsigned digit = (key[ch] >> low_bits) & mask;
    local[ch] += (my[digit >> 1] >> ((digit & 1u) * 16u)) & 0xffffu;
  }
  __syncthreads();
  uint32_t* s_key = reinterpret_cast<uint32_t*>(s_buf);
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch)
    if (FULL || ch * 64 + lane < cnt) s_key[local[ch]] = key[ch];
  __syncthreads();
  const unsigned low_mask = (1u << low_bits) - 1u;
  uint32_t dst[kWgChunks];
#pragma unroll
  for (int ch = 0; ch < kWgChunks; ++ch) {
    const int i = t + ch * kWgThreads;
    const uint32_t k = FULL || i < tcnt ? s_key[i] : 0u;
    dst[ch] = s_off[(k >> low_bits) & mask] + (uint32_t)i;
    if (FULL || i < tcnt) low_out[dst[ch]] = (uint16_t)(k & low_mask);
  }
  __syncthreads();
  // the products, in windows of whole rounds of sorted positions
  constexpr int kRounds = scatter_buf_bytes<V>() / (int)sizeof(P) / kWgThreads;  // rounds per window
  constexpr int kWin = kRounds * kWgThreads;
  P* s_prod = reinterpret_cast<P*>(s_buf);
#pragma unroll
  for (int r0 = 0; r0 < kWgChunks; r0 += kRounds) {
    const int w0 = r0 * kWgThreads;
    if (!FULL && w0 >= tcnt) break;
#pragma unroll
    for (int ch = 0; ch < kWgChunks; ++ch) {
      const unsigned j = local[ch] - (unsigned)w0;
      if ((FULL || ch * 64 + lane < cnt) && (kRounds >= kWgChunks || j < (unsigned)kWin)) s_prod[j] = prod[ch];
    }
    __syncthreads();
#pragma unroll
    for (int ch = r0; ch < (r0 + kRounds < kWgChunks ? r0 + kRounds : kWgChunks); ++ch) {
      const int i = t + ch * kWgThreads;
      if (FULL || i < tcnt) prod_out[dst[ch]] = s_prod[i - w0];
    }
    if (r0 + kRounds < kWgChunks) __syncthreads();
  }
}

template <class V>
__global__ __launch_bounds__(kWgThreads, 4) void scatter_products_kernel(ScatterIn in, const V* __restrict__ x,
                                                                         int64_t n, int low_bits, unsigned mask,
                                                                         const uint32_t* __restrict__ offsets,
                                                                         uint16_t* __restrict__ low_out,
                                                                         typename SA<V>::P* __restrict__ prod_out,
                                                                         int32_t* __restrict__ flags, int flag) {
  __shared__ __attribute__((aligned(16))) uint8_t s_buf[scatter_buf_bytes<V>()];
  __shared__ uint32_t s_off[kWgMaxDigits];
  __shared__ int64_t s_wave[kWgWaves];
  const int64_t tile = xcd_tile(blockIdx.x, gridDim.x);  // per-XCD tile ranges
  const int64_t left = n - tile * kWgTile;
  if (left >= kWgTile)
    scatter_tile<V, true>(in, x, tile, (int)kWgTile, low_bits, mask, offsets, low_out, prod_out, flags, flag, s_buf,
                          s_off, s_wave);
  else
    scatter_tile<V, false>(in, x, tile, (int)left, low_bits, mask, offsets, low_out, prod_out, flags, flag, s_buf,
                           s_off, s_wave);
}

// Pass 2 (see the top): workgroup s sums segment s.  Each wave adds a
// contiguous part of the segment to its own LDS copy of the bucket's sums,
// 64 products at a time (kAhead such chunks loaded before any is added):
// lanes of the same output are ranked by ballots and add one after another.  A
// group of more than kCrowd lanes is first summed in registers: one such group
// over all lanes (6 exchanges), several of them together (as many exchanges as
// the largest group needs; one after another, 4.8 M entries in blocks of 8 rows
// of equal columns took, float32 / float64 / complex64 / complex128, 224 / 340
// / 371 / 611 us a call against 125 / 145 / 178 / 212; the joint exchanges alone,
// also for one group, cost blocks of 64 rows 141 us instead of 133).
constexpr int kAhead = 8;
constexpr int kCrowd = 6;
template <class V>
__global__ __launch_bounds__(256) void scatter_reduce_kernel(const uint16_t* __restrict__ low,
                                                             const typename SA<V>::P* __restrict__ prod,
                                                             const uint32_t* __restrict__ bucket_start,
                                                             const uint32_t* __restrict__ seg_first,
                                                             const uint32_t* __restrict__ seg_bucket, int nd,
                                                             uint32_t seg_items, int low_bits, int64_t n_out,
                                                             V* __restrict__ y,
                                                             typename SA<V>::A* __restrict__ partial) {
  using T = SA<V>;
  using A = typename T::A;
  using P = typename T::P;
  extern __shared__ __attribute__((aligned(16))) uint8_t r_lds[];
  A* sums = reinterpret_cast<A*>(r_lds);
  const uint32_t s = blockIdx.x;
  if (s >= seg_first[nd]) return;  // whole workgroup
  const int n_low = 1 << low_bits;
  const int t = threadIdx.x, lane = t & 63, waves = (int)(blockDim.x >> 6);
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // scalar: so are the wave's range and addresses
  const uint32_t b = seg_bucket[s];
  const uint32_t f0 = seg_first[b], f1 = seg_first[b + 1];
  const uint32_t start = bucket_start[b], end = bucket_start[b + 1];
  const uint32_t e0 = start + (s - f0) * seg_items;
  const uint32_t e1 = end - e0 < seg_items ? end : e0 + seg_items;
  const uint32_t part = (e1 - e0 + 64 * waves - 1) / (64 * waves) * 64;  // entries per wave, whole chunks
  const uint32_t w0 = e0 + w * part < e1 ? e0 + w * part : e1;
  const uint32_t w1 = e1 - w0 < part ? e1 : w0 + part;
  for (int k = t; k < n_low * waves; k += (int)blockDim.x) sums[k] = A{};
  __syncthreads();
  A* my = sums + (size_t)w * n_low;
  const unsigned low_mask = (unsigned)n_low - 1u;
  auto add_chunk = [&](unsigned o, P p, bool valid, uint64_t active) {
    const uint64_t peers = match_lanes<12>(o, active, low_mask);
    const int rank = count_below_t(peers);
    const uint64_t crowds = __ballot(valid && rank == kCrowd);  // one lane of every crowded group
    if (__builtin_expect(crowds != 0, 0)) {
      if ((crowds & (crowds - 1)) != 0) {
        // every group at once: a lane doubles the stretch of its group, itself
        // first, that it has summed, until the first lane's reaches the end
        const uint64_t above = peers & ~((2ull << lane) - 1ull);
        int next = valid && above != 0 ? (int)__builtin_ctzll(above) : 64;  // lane after the stretch, or 64
        A v{};
        T::add(v, p);
        for (int len = 1; __ballot(valid && rank >= len) != 0; len <<= 1) {  // len: lanes of a stretch
          const int src = next & 63;
          const A w = shfl_words(v, src);
          const int far = __builtin_amdgcn_ds_bpermute(src << 2, next);
          if (next < 64) {
            v = T::join(v, w);
            next = far;
          }
        }
        if (valid && rank == 0) my[o] = T::join(my[o], v);
        wave_sync_t();
        return;
      }
      const int l = (int)__builtin_ctzll(crowds);
      const uint64_t group = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(peers >> 32), l) << 32) |
                             (uint32_t)__builtin_amdgcn_readlane((int)peers, l);
      const bool in = (group >> lane) & 1u;
      A v{};
      if (in) T::add(v, p);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v = T::join(v, shfl_words(v, lane ^ off));
      if (lane == l) my[o] = T::join(my[o], v);
      if (in) valid = false;
      wave_sync_t();
    }
    for (int r = 0; __ballot(valid && rank >= r) != 0; ++r) {
      if (valid && rank == r) {
        A a = my[o];
        T::add(a, p);
        my[o] = a;
      }
      wave_sync_t();
    }
  };
  uint32_t c0 = w0;
  for (; w1 - c0 >= 64 * kAhead; c0 += 64 * kAhead) {  // whole groups of chunks: every lane holds an entry
    unsigned o[kAhead];
    P p[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      o[u] = (low + c0)[u * 64 + lane];
      p[u] = (prod + c0)[u * 64 + lane];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) add_chunk(o[u], p[u], true, ~0ull);
  }
  for (; c0 < w1; c0 += 64) {
    const bool valid = c0 + lane < w1;
    const unsigned o = valid ? (low + c0)[lane] : 0u;
    const P p = valid ? (prod + c0)[lane] : P{};
    add_chunk(o, p, valid, __ballot(valid));
  }
  __syncthreads();
  const bool whole = f1 - f0 == 1;
  for (int k = t; k < n_low; k += (int)blockDim.x) {
    A v = sums[k];
    for (int j = 1; j < waves; ++j) v = T::join(v, sums[(size_t)j * n_low + k]);
    const int64_t out = (int64_t)b * n_low + k;
    if (whole) {
      if (out < n_out) y[out] = T::out(v);
    } else {
      partial[(size_t)s * n_low + k] = v;
    }
  }
}

// Buckets of several segments: their partial sums.  A workgroup takes 64 outputs
// (or all of a smaller bucket) of one of them at a time; its threads take
// outputs x equal shares of the segments, joined in a fixed tree.  (One thread
// per output is a chain of up to 1,024 loads, a cache line each: A^T x with 4.8 M
// entries and 200 columns took 377 us a call in float32, 489 in complex128; 149
// and 235 shared.)
constexpr int kFixThreads = 1024;
template <class V>
__global__ __launch_bounds__(kFixThreads) void scatter_fixup_kernel(const uint32_t* __restrict__ seg_first,
                                                                    const uint32_t* __restrict__ split, int nd,
                                                                    int low_bits, int64_t n_out, V* __restrict__ y,
                                                                    const typename SA<V>::A* __restrict__ partial) {
  using T = SA<V>;
  using A = typename T::A;
  __shared__ __attribute__((aligned(16))) uint8_t s_raw[kFixThreads * sizeof(A)];
  A* s_sum = reinterpret_cast<A*>(s_raw);
  const int n_low = 1 << low_bits;
  const int width = n_low < 64 ? n_low : 64;
  const uint32_t groups = (uint32_t)(n_low / width), jobs = split[nd] * groups;
  const int tid = threadIdx.x, c = tid % width, shares = kFixThreads / width;
  const uint32_t share = (uint32_t)(tid / width);
  for (uint32_t job = blockIdx.x; job < jobs; job += gridDim.x) {
    const uint32_t b = split[job / groups];
    const int k = (int)(job % groups) * width + c;  // output within the bucket
    const uint32_t f0 = seg_first[b], f1 = seg_first[b + 1];
    const uint32_t len = (f1 - f0 + shares - 1) / shares;
    const uint32_t s0 = f0 + share * len < f1 ? f0 + share * len : f1;
    const uint32_t s1 = f1 - s0 < len ? f1 : s0 + len;
    A v{};
    for (uint32_t s = s0; s < s1; s += 4) {
      A w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = partial[(size_t)(s + u < s1 ? s + u : s1 - 1) * n_low + k];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s + u < s1) v = T::join(v, w[u]);
    }
    s_sum[tid] = v;
    for (int o = shares >> 1; o > 0; o >>= 1) {
      __syncthreads();
      if ((int)share < o) s_sum[tid] = T::join(s_sum[tid], s_sum[tid + o * width]);
    }
    const int64_t out = (int64_t)b * n_low + k;
    if (share == 0 && out < n_out) y[out] = T::out(s_sum[tid]);
    __syncthreads();
  }
}

// ---- host side ------------------------------------------------------------
struct ScatterLayout {
  int low_bits = 0, high_bits = 0, waves = 0;
  uint32_t seg_items = 0;
  int64_t n_tiles = 0, n_sub = 0, n_blocks = 0, max_segs = 0;
  size_t off_low = 0, off_prod = 0, off_counts = 0, off_partial = 0, off_totals = 0, off_tile_row = 0, off_start = 0,
         off_seg_first = 0, off_seg_bucket = 0, off_split = 0, off_sums = 0, total = 0;
};

inline size_t scatter_acc_bytes(int val_t) { return val_t == FS_F32 ? 8 : val_t == FS_C128 ? 32 : 16; }

// Outputs per bucket.  More buckets mean shorter runs to write, larger buckets
// fewer waves with a copy of the sums in LDS: scatter + reduce of 33.5 M
// float32 entries over 2^20 outputs take 297 + 107 us with 1024 buckets, 273 +
// 167 with 512, 263 + 450 with 256.  So 1024 buckets (fewer for few outputs: a
// bucket has at least 256), 2048 above 2^20 outputs.  The path ends where one
// wave's copy would pass 64 KB of LDS.
inline bool scatter_layout(int val_t, int64_t n_out, int64_t nnz, ScatterLayout& L) {
  if (n_out <= 0 || nnz <= 0 || nnz >= (int64_t)0xffffffffLL - kWgTile) return false;
  const size_t acc = scatter_acc_bytes(val_t);
  int bits = 0;
  while (bits < 62 && (int64_t(1) << bits) < n_out) ++bits;
  const int max_low = acc == 32 ? 11 : 12;
  if (bits > max_low + kWgMaxBits) return false;
  L.low_bits = std::min(bits, std::max(8, bits - 10));
  if (L.low_bits > 10) L.low_bits = std::max(10, bits - kWgMaxBits);
  L.high_bits = bits - L.low_bits;
  const int64_t nd = int64_t(1) << L.high_bits;
  L.waves = 4;
  while (L.waves > 1 && (acc << L.low_bits) * (size_t)L.waves > 65536) L.waves >>= 1;
  L.seg_items = scatter_segment_items(nnz, ceil_div(n_out, int64_t(1) << L.low_bits));
  L.max_segs = nd + ceil_div(nnz, (int64_t)L.seg_items);
  L.n_tiles = ceil_div(nnz, kWgTile);
  L.n_sub = ceil_div(nnz, kWgSub);
  L.n_blocks = ceil_div(L.n_tiles, (int64_t)kWgScanTiles);
  const size_t pbytes = (val_t == FS_F32 || val_t == FS_F64) ? 8 : 16;
  size_t o = 0;
  auto take = [&](size_t& off, size_t bytes) {
    off = o;
    o = (o + bytes + 255) & ~(size_t)255;
  };
  take(L.off_prod, pbytes * (size_t)nnz);
  take(L.off_low, 2 * (size_t)nnz);
  take(L.off_counts, 4 * (size_t)L.n_tiles * (size_t)nd);
  take(L.off_partial, 4 * (size_t)L.n_blocks * (size_t)nd);
  take(L.off_totals, 4 * (size_t)nd);
  take(L.off_tile_row, 8 * (size_t)L.n_sub);
  take(L.off_start, 4 * (size_t)(nd + 1));
  take(L.off_seg_first, 4 * (size_t)(nd + 1));
  take(L.off_seg_bucket, 4 * (size_t)L.max_segs);
  take(L.off_split, 4 * (size_t)(nd + 1));
  take(L.off_sums, (acc << L.low_bits) * (size_t)L.max_segs);
  L.total = o;
  return true;
}

template <class V>
int scatter_run(const ScatterLayout& L, char* ws, ScatterIn in, int val_t, int64_t n_out, int64_t nnz, const void* x,
                void* y, int32_t* flags, int key_flag, int other_flag, hipStream_t s) {
  using T = SA<V>;
  const unsigned mask = (1u << L.high_bits) - 1u;
  const int nd = (int)mask + 1;
  auto u32 = [&](size_t off) { return reinterpret_cast<uint32_t*>(ws + off); };
  uint32_t* counts = u32(L.off_counts);
  uint32_t* partial = u32(L.off_partial);
  uint32_t* totals = u32(L.off_totals);
  uint16_t* low = reinterpret_cast<uint16_t*>(ws + L.off_low);
  typename T::P* prod = reinterpret_cast<typename T::P*>(ws + L.off_prod);
  typename T::A* sums = reinterpret_cast<typename T::A*>(ws + L.off_sums);
  const dim3 tiles((unsigned)L.n_tiles);
  if (in.key64)
    hipLaunchKernelGGL((scatter_count_kernel<int64_t>), tiles, dim3(kWgThreads), 0, s,
                       static_cast<const int64_t*>(in.keys), nnz, L.low_bits, mask, counts, (uint64_t)n_out, flags,
                       key_flag);
  else
    hipLaunchKernelGGL((scatter_count_kernel<int32_t>), tiles, dim3(kWgThreads), 0, s,
                       static_cast<const int32_t*>(in.keys), nnz, L.low_bits, mask, counts, (uint64_t)n_out, flags,
                       key_flag);
  FS_CHECK_LAUNCH("scatter_count_kernel");
  hipLaunchKernelGGL(wg_scan_reduce_kernel, dim3((unsigned)L.n_blocks), dim3(256), 0, s, counts, L.n_tiles, nd, partial);
  FS_CHECK_LAUNCH("wg_scan_reduce_kernel");
  hipLaunchKernelGGL(wg_scan_column_kernel, dim3((unsigned)nd), dim3(256), 0, s, partial, L.n_blocks, nd, totals);
  FS_CHECK_LAUNCH("wg_scan_column_kernel");
  hipLaunchKernelGGL(wg_scan_down_kernel, dim3((unsigned)L.n_blocks), dim3(256), 0, s, counts, L.n_tiles, nd, partial,
                     totals);
  FS_CHECK_LAUNCH("wg_scan_down_kernel");
  hipLaunchKernelGGL(scatter_plan_kernel, dim3(1), dim3(256), 0, s, totals, nd, L.seg_items, u32(L.off_start),
                     u32(L.off_seg_first), u32(L.off_seg_bucket), u32(L.off_split));
  FS_CHECK_LAUNCH("scatter_plan_kernel");
  hipLaunchKernelGGL((scatter_products_kernel<V>), tiles, dim3(kWgThreads), 0, s, in, static_cast<const V*>(x), nnz,
                     L.low_bits, mask, counts, low, prod, flags, other_flag);
  FS_CHECK_LAUNCH("scatter_products_kernel");
  const size_t lds = (sizeof(typename T::A) << L.low_bits) * (size_t)L.waves;
  hipLaunchKernelGGL((scatter_reduce_kernel<V>), dim3((unsigned)L.max_segs), dim3(64 * L.waves), lds, s, low, prod,
                     u32(L.off_start), u32(L.off_seg_first), u32(L.off_seg_bucket), nd, L.seg_items, L.low_bits, n_out,
                     static_cast<V*>(y), sums);
  FS_CHECK_MAIN_LAUNCH("scatter_reduce_kernel");
  const int64_t fix_jobs = (int64_t)nd * std::max(1, (1 << L.low_bits) / 64);
  hipLaunchKernelGGL((scatter_fixup_kernel<V>), dim3((unsigned)std::min<int64_t>(fix_jobs, 512)), dim3(kFixThreads), 0,
                     s, u32(L.off_seg_first), u32(L.off_split), nd, L.low_bits, n_out, static_cast<V*>(y), sums);
  FS_CHECK_LAUNCH("scatter_fixup_kernel");
  return FS_OK;
}

// (the entry points hold the checks; `flags`: pinned host memory)
static int scatter_entry(const char* name, int val_t, ScatterIn in, int64_t n_src_rows, int64_t n_out, int64_t nnz,
                         const void* x, void* y, void* ws, size_t ws_bytes, int32_t* flags, int n_flags, int key_flag,
                         int other_flag, hipStream_t s) {
  ScatterLayout L;
  if (!scatter_layout(val_t, n_out, nnz, L)) return fail(FS_E_INVALID, std::string(name) + ": sizes not supported");
  if (!ws || ws_bytes < L.total) return fail(FS_E_WORKSPACE, std::string(name) + ": workspace too small");
  void* dflags = nullptr;
  FS_CHECK_HIP(hipHostGetDevicePointer(&dflags, flags, 0));
  for (int k = 0; k < n_flags; ++k) flags[k] = 0;
  int32_t* df = static_cast<int32_t*>(dflags);
  char* w = static_cast<char*>(ws);
  if (in.rowptr) {
    int64_t* tile_row = reinterpret_cast<int64_t*>(w + L.off_tile_row);
    in.tile_row = tile_row;
    in.n_sub = L.n_sub;
    const unsigned blocks = (unsigned)ceil_div(n_src_rows, 256);
    if (in.ptr64)
      hipLaunchKernelGGL((scatter_rows_kernel<int64_t>), dim3(blocks), dim3(256), 0, s,
                         static_cast<const int64_t*>(in.rowptr), n_src_rows, nnz, L.n_sub, tile_row, df);
    else
      hipLaunchKernelGGL((scatter_rows_kernel<int32_t>), dim3(blocks), dim3(256), 0, s,
                         static_cast<const int32_t*>(in.rowptr), n_src_rows, nnz, L.n_sub, tile_row, df);
    FS_CHECK_LAUNCH("scatter_rows_kernel");
  }
  int rc;
  switch (val_t) {
    case FS_F32: rc = scatter_run<float>(L, w, in, val_t, n_out, nnz, x, y, df, key_flag, other_flag, s); break;
    case FS_F64: rc = scatter_run<double>(L, w, in, val_t, n_out, nnz, x, y, df, key_flag, other_flag, s); break;
    case FS_C64: rc = scatter_run<c32>(L, w, in, val_t, n_out, nnz, x, y, df, key_flag, other_flag, s); break;
    default: rc = scatter_run<c64>(L, w, in, val_t, n_out, nnz, x, y, df, key_flag, other_flag, s); break;
  }
  if (rc != FS_OK) return rc;
  // the flags are in host memory once the stream has drained
  FS_CHECK_HIP(hipStreamSynchronize(s));
  return FS_OK;
}

}  // namespace fs

using namespace fs;

extern "C" size_t fs_spmv_scatter_workspace_bytes(int val_t, int64_t n_out, int64_t nnz) {
  if (val_t < FS_F32 || val_t > FS_C128) return 0;
  ScatterLayout L;
  return scatter_layout(val_t, n_out, nnz, L) ? L.total : 0;
}

extern "C" int fs_spmv_csr_scatter(int val_t, int idx_t, int ptr_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                                   const void* vals, const void* cols, const void* indptr, int conj, const void* x,
                                   void* y, void* ws, size_t ws_bytes, int32_t* flags, hipStream_t stream) {
  if (!valid_types(val_t, idx_t, ptr_t)) return fail(FS_E_INVALID, "fs_spmv_csr_scatter: bad type code");
  if (n_rows <= 0 || n_cols <= 0 || nnz <= 0 || n_rows > (int64_t)0xffffffffLL)
    return fail(FS_E_INVALID, "fs_spmv_csr_scatter: sizes not supported");
  if (!vals || !cols || !indptr || !x || !y || !flags) return fail(FS_E_INVALID, "fs_spmv_csr_scatter: null pointer");
  ScatterIn in{};
  in.vals = vals;
  in.keys = cols;
  in.key64 = idx_t == FS_I64;
  in.rowptr = indptr;
  in.ptr64 = ptr_t == FS_I64;
  in.n_x = n_rows;
  in.conj = conj;
  return scatter_entry("fs_spmv_csr_scatter", val_t, in, n_rows, n_cols, nnz, x, y, ws, ws_bytes, flags, 4, 3, 3,
                       stream);
}

extern "C" int fs_spmv_coo_scatter(int val_t, int out_idx_t, int x_idx_t, int64_t n_out, int64_t n_x, int64_t nnz,
                                   const void* vals, const void* out_idx, const void* x_idx, int conj, const void* x,
                                   void* y, void* ws, size_t ws_bytes, int32_t* flags, hipStream_t stream) {
  if (!valid_types(val_t, out_idx_t, x_idx_t)) return fail(FS_E_INVALID, "fs_spmv_coo_scatter: bad type code");
  if (n_out <= 0 || n_x <= 0 || nnz <= 0 || n_x > (int64_t)0xffffffffLL)
    return fail(FS_E_INVALID, "fs_spmv_coo_scatter: sizes not supported");
  if (!vals || !out_idx || !x_idx || !x || !y || !flags)
    return fail(FS_E_INVALID, "fs_spmv_coo_scatter: null pointer");
  ScatterIn in{};
  in.vals = vals;
  in.keys = out_idx;
  in.key64 = out_idx_t == FS_I64;
  in.other = x_idx;
  in.other64 = x_idx_t == FS_I64;
  in.n_x = n_x;
  in.conj = conj;
  return scatter_entry("fs_spmv_coo_scatter", val_t, in, 0, n_out, nnz, x, y, ws, ws_bytes, flags, 4, 0, 1, stream);
}
