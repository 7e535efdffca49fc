// spmm_group.hpp — the lane-group SpMM kernel, its fix-up and its launch, for
// every value type (spmm_group.hip: float32, float64, complex64, complex128;
// spmm_half.hip: float16, bfloat16).
#pragma once

#include "fs_common.hpp"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace fs {

template <class T>
__device__ inline T readlane_any(const T& v, int lane) {
  constexpr int W = (int)(sizeof(T) / 4);
  int w[W];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int k = 0; k < W; ++k) w[k] = __builtin_amdgcn_readlane(w[k], lane);
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// ---------------------------------------------------------------------------
// Lane-group SpMM (the default kernel).
//
// A wave is split into G = 64 / LPR groups of LPR lanes.  Each lane owns EPL
// consecutive columns of B / C (EPL * sizeof(V) = 16 bytes, so a B-row slice
// is one 16-byte load per lane: 64 lanes gather G rows per instruction).
// Every group walks its own merge-path sub-tile of S items (rows + nnz), so
// one load instruction gathers G different B rows and no FMA is predicated
// per group.  The sub-tile's row ends are staged in LDS (2-byte offsets from
// the sub-tile's first nnz); column / value chunks of LPR entries sit one per
// lane and reach the group's lanes by ds_bpermute (readlane when G == 1).
// Gathers are double buffered (U steps per batch).  Rows that cross
// sub-tiles leave head / tail fragments, summed in sub-tile order by
// spmm_group_fixup_kernel: deterministic, no floating-point atomics.
//
// B(k, n) is B[k * sbk + n * sbn] and C(m, n) is C[m * scm + n * scn]: the
// row-major fast path (sbn == scn == 1, 16-byte aligned) uses vector loads
// and stores, any other layout (column-major B / C) element accesses.
// ---------------------------------------------------------------------------
// The type a lane holds A's values in (cross-lane moves take whole words).
template <class V>
using held_t = std::conditional_t<sizeof(V) == 2, float, V>;

// Bytes of a B / C row slice per lane, and its elements.
template <class V>
struct group_slice {
  static constexpr int bytes = 16;
};
template <class V>
constexpr int group_epl() {
  return (int)(group_slice<V>::bytes / sizeof(V));
}

template <class T>
__device__ inline T bcast_lane(const T& v, int src_lane) {
  constexpr int W = (int)(sizeof(T) / 4);
  int w[W];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int k = 0; k < W; ++k) w[k] = __builtin_amdgcn_ds_bpermute(src_lane << 2, w[k]);
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// VEC: 16-byte vector loads / stores of row-major slices; otherwise element
// accesses at any strides.  Measured alternatives, not kept: 16-byte buffer
// loads with 32-bit offsets (C4 1.264 / 1.275 ms, R-MAT complex64 N = 32
// 1.447 / 1.400 ms), two gathers per batch instead of four (more waves per
// SIMD; C4 1.33 ms against 1.26), a residency bound through
// amdgpu_waves_per_eu (spills registers).
template <class V, int LPR, int U, bool VEC, class I, class T = VT<V>>
__global__ __launch_bounds__(256) void spmm_group_kernel(
    const V* __restrict__ vals, const I* __restrict__ cols, const void* __restrict__ rowptr_raw, int ptr64,
    const V* __restrict__ B, int64_t sbk, int64_t sbn, V* __restrict__ C, int64_t scm, int64_t scn,
    int64_t n_dense, const int64_t* __restrict__ part, int sub_items,
    typename T::acc* __restrict__ head, typename T::acc* __restrict__ tail, int64_t n_rows,
    int64_t nnz, int64_t n_sub, int xcd_cols, int row_ranges) {
  using A = typename T::acc;
  using H = held_t<V>;
  constexpr int G = 64 / LPR;
  constexpr int EPL = group_epl<V>();
  // one load or store of a whole slice
  using L4 = __attribute__((ext_vector_type(group_slice<V>::bytes / 4))) unsigned int;
  extern __shared__ uint16_t lds_re[];
  const int lane = threadIdx.x & 63;
  const int g = lane / LPR;
  const int gl = lane % LPR;
  const int64_t ctile = xcd_cols > 0 ? (int64_t)(blockIdx.x % (unsigned)xcd_cols) : (int64_t)blockIdx.y;
  // row_ranges (2-D grid only): each XCD walks one contiguous range of tile
  // blocks, so the rows in flight on an XCD at any moment are adjacent
  const int64_t tblk = xcd_cols > 0 ? (int64_t)(blockIdx.x / (unsigned)xcd_cols)
                                    : (row_ranges ? xcd_range_block(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x);
  const int64_t wid = tblk * 4 + (threadIdx.x >> 6);
  if (wid * G >= n_sub) return;  // wave-uniform; no barriers below
  const int64_t st = wid * G + g;
  const bool live = st < n_sub;
  const int64_t col0 = ctile * (int64_t)(LPR * EPL) + (int64_t)gl * EPL;
  const int64_t vrem = n_dense - col0;
  const int valid = vrem <= 0 ? 0 : (vrem >= EPL ? EPL : (int)vrem);
  // Loads are unconditional (so the compiler can count the ones in flight):
  // lanes past the last column read column 0's slice and discard it, steps
  // past a group's last nnz read B row 0.
  const int64_t col0_ld = valid > 0 ? col0 : 0;

  // sub-tile coordinates (merge path).  The prologue's loads are
  // unconditional, and each waits only on what its address needs: the
  // partition entries, then at once the row pointers and the first entry
  // chunks (a load in a branch is waited for at the branch's end).
  const int64_t st_ld = live ? st : n_sub - 1;
  const int64_t p0 = part[st_ld], p1 = part[st_ld + 1];
  int64_t r0 = 0, r1 = 0, n0 = 0;
  int nz = 0, R = 0;
  if (live) {
    r0 = p0;
    r1 = p1;
    const int64_t d0 = st * (int64_t)sub_items;
    const int64_t total = n_rows + nnz;
    const int64_t dend = d0 + sub_items < total ? d0 + sub_items : total;
    n0 = d0 - r0;
    nz = (int)(dend - r1 - n0);
    R = (int)(r1 - r0);
  }
  // Row pointer entries, int32 or int64, by one 8-byte load either way: an
  // int32 entry is read from the aligned 8-byte word that holds it (which
  // never crosses a page).
  auto rp = [&](int64_t i) -> int64_t {
    const unsigned char* a = static_cast<const unsigned char*>(rowptr_raw) + (i << (ptr64 ? 3 : 2));
    const uintptr_t mis = (uintptr_t)a & 7;
    const uint64_t w = *reinterpret_cast<const uint64_t*>(a - mis);
    return ptr64 ? (int64_t)w : (int64_t)(int32_t)(uint32_t)(mis ? w >> 32 : w);
  };

  const I* colp = cols + n0;
  const V* valp = vals + n0;
  // Entry chunks: LPR entries per group, one per lane; chunk c + 1 is loaded
  // while chunk c is walked.  Every global load below is unconditional, so
  // the compiler counts the ones in flight exactly and waits for a gather
  // only when its row is consumed: past a group's nnz, chunk entries re-read
  // entry 0 of the matrix (it exists whenever the kernel runs) and the steps
  // that use them are skipped.
  auto load_chunk = [&](int ch, I& cc, H& vv) {
    const int q = ch * LPR + gl;
    const bool in = q < nz;
    cc = *(in ? colp + q : cols);
    if constexpr (sizeof(V) == 2) vv = T::widen(*(in ? valp + q : vals));
    else vv = *(in ? valp + q : vals);
  };
  I colC, colN;
  H valC, valN;
  load_chunk(0, colC, valC);
  load_chunk(1, colN, valN);

  const int64_t row_start = rp(r0);
  // row ends of the sub-tile -> LDS, as offsets from n0 (<= nz <= sub_items),
  // four loads in flight per lane; the first four go out with the loads
  // above (an index clamped to R - 1 reads a real entry, r0 itself when R
  // is 0)
  uint16_t* re_tab = lds_re + (size_t)((threadIdx.x >> 6) * G + g) * (size_t)sub_items;
  auto row_ends = [&](int k0) {
    int64_t e[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + u * LPR + gl;
      e[u] = rp(r0 + 1 + (k < R ? k : R - 1));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + u * LPR + gl;
      if (k < R) re_tab[k] = (uint16_t)(e[u] - n0);
    }
  };
  row_ends(0);
  for (int k0 = 4 * LPR; k0 < R; k0 += 4 * LPR) row_ends(k0);
  const bool head_partial = R > 0 && row_start < n0;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  int maxnz = nz;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) maxnz = max(maxnz, __shfl_xor(maxnz, off));
  maxnz = __builtin_amdgcn_readfirstlane(maxnz);

  const V* Bl = B + col0_ld * sbn;
  const uint32_t row_bytes = (uint32_t)(sbk * (int64_t)sizeof(V));
  int row = 0;
  int re = R > 0 ? (int)re_tab[0] : 0x7fffffff;

  A acc[EPL];
#pragma unroll
  for (int k = 0; k < EPL; ++k) acc[k] = T::zero();
  auto emit = [&]() {
    if (valid > 0) {
      if (row == 0 && head_partial) {
        A* h = head + st * n_dense + col0;
#pragma unroll
        for (int k = 0; k < EPL; ++k)
          if (k < valid) h[k] = acc[k];
      } else {
        V* c = C + (r0 + row) * scm + col0 * scn;
        if constexpr (VEC) {
          V o[EPL];
#pragma unroll
          for (int k = 0; k < EPL; ++k) o[k] = T::out(acc[k]);
          L4 q;
          __builtin_memcpy(&q, o, sizeof(q));
          *reinterpret_cast<L4*>(c) = q;
        } else {
#pragma unroll
          for (int k = 0; k < EPL; ++k)
            if (k < valid) c[k * scn] = T::out(acc[k]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < EPL; ++k) acc[k] = T::zero();
  };
  auto next_row = [&]() {
    ++row;
    re = row < R ? (int)re_tab[row] : 0x7fffffff;
  };

  // Gathers of batch b (U steps) of a chunk held in (cc, vv).
  auto issue = [&](int b, const I& cch, const H& vch, V (&bb)[U][EPL], H (&aa)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int li = b * U + u;
      I cc;
      if constexpr (G == 1) {
        cc = readlane_any(cch, li);
        aa[u] = readlane_any(vch, li);
      } else {
        cc = bcast_lane(cch, g * LPR + li);
        aa[u] = bcast_lane(vch, g * LPR + li);
      }
      if constexpr (VEC) {
        // one 32 x 32 + 64-bit multiply-add per gather (the host takes this
        // path only when columns and the row stride in bytes fit 32 bits)
        const char* pb = reinterpret_cast<const char*>(Bl) + (uint64_t)(uint32_t)cc * (uint64_t)row_bytes;
        L4 q = *reinterpret_cast<const L4*>(pb);
        __builtin_memcpy(bb[u], &q, sizeof(q));
      } else {
        const V* p = Bl + (int64_t)cc * sbk;
#pragma unroll
        for (int k = 0; k < EPL; ++k) bb[u][k] = p[(k < valid ? k : 0) * sbn];
      }
    }
  };
  auto consume = [&](int s0, V (&bb)[U][EPL], H (&aa)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      if (s < nz) {
        while (re <= s) {  // rows that end before nnz s (empty rows included)
          emit();
          next_row();
        }
#pragma unroll
        for (int k = 0; k < EPL; ++k) acc[k] = T::fma(aa[u], bb[u][k], acc[k]);
      }
    }
  };

  constexpr int NB = LPR / U;  // batches per chunk (even)
  static_assert(NB % 2 == 0, "an even number of batches per chunk");
  const int n_chunks = (maxnz + LPR - 1) / LPR;
  V bA[U][EPL], bB[U][EPL];
  H aA[U], aB[U];
  issue(0, colC, valC, bA, aA);
  for (int c = 0; c < n_chunks; ++c) {
#pragma unroll
    for (int b = 0; b < NB; b += 2) {
      issue(b + 1, colC, valC, bB, aB);
      consume(c * LPR + b * U, bA, aA);
      if (b + 2 < NB) issue(b + 2, colC, valC, bA, aA);
      else issue(0, colN, valN, bA, aA);  // first batch of the next chunk (unused after the last)
      consume(c * LPR + (b + 1) * U, bB, aB);
    }
    colC = colN;
    valC = valN;
    load_chunk(c + 2, colN, valN);
  }
  while (row < R) {  // rows ending at the sub-tile's last nnz, and trailing empty rows
    emit();
    next_row();
  }
  if (live && r1 < n_rows && valid > 0) {
    A* tl = tail + st * n_dense + col0;
#pragma unroll
    for (int k = 0; k < EPL; ++k)
      if (k < valid) tl[k] = acc[k];
  }
}

// Rows that cross sub-tiles: C[row] = tail[f] + ... + tail[t-1] + head[t], one
// wave per sub-tile t, lanes over columns.  A row of more than kFixShort
// fragments is the workgroup's: its threads take columns x equal shares of the
// fragments, joined in a fixed tree (of kFixWaves sub-tiles in a row at most one
// ends such a row: the next one to end started after it).  One wave adding them
// all is a chain of loads that outlasts what small sub-tiles win.  us per
// prepared float32 call on an arrow matrix of 100,000 rows (its dense row up to
// 3,125 fragments), 2048-item waves / sized sub-tiles, one wave / 4 waves / 16
// waves: N = 1 121 / 103 / 24 / 24, N = 17 145 / 142 / 51 / 46, N = 64 178 / 94 /
// 50 / 43, N = 256 75 / 94 / 71 / 68.  4 waves, as graphs with hubs and the many
// ordinary rows count for more: the fix-up of R-MAT 2^19, N = 3, one wave / 4 / 16
// takes 12.4 / 12.3 / 17.6 us, of 2^21 complex64, N = 32 23.0 / 20.4 / 27.9.
constexpr int kFixWaves = 4;
constexpr int kFixThreads = 64 * kFixWaves;
constexpr int64_t kFixShort = 128;
static_assert((kFixWaves & (kFixWaves - 1)) == 0 && kFixWaves <= kFixShort, "lanes over sub-tiles, one long row");
__device__ inline int64_t lane_i64(int64_t v, int lane) {
  return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32 |
                   (uint32_t)__builtin_amdgcn_readlane((int)v, lane));
}
template <class V, class T = VT<V>>
__global__ __launch_bounds__(kFixThreads) void spmm_group_fixup_kernel(
    const void* __restrict__ rowptr_raw, int ptr64, const int64_t* __restrict__ part, int sub_items,
    const typename T::acc* __restrict__ head, const typename T::acc* __restrict__ tail,
    V* __restrict__ C, int64_t scm, int64_t scn, int64_t n_dense, int64_t n_sub) {
  using A = typename T::acc;
  __shared__ A s_sum[kFixThreads];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t0 = (int64_t)blockIdx.x * kFixWaves, t = t0 + w;
  // Every wave finds the workgroup's long row by itself, from loads that go out
  // with its own: the row that ends in sub-tile k has more than kFixShort
  // fragments if sub-tile k - kFixShort starts in it.  (A barrier here held every
  // workgroup for its slowest wave: R-MAT 2^21 bfloat16, N = 3 39 us instead of 30.)
  const int64_t j = t0 + (lane & (kFixWaves - 1)), k = j < n_sub ? j : n_sub - 1;
  const int64_t rk = part[k], rk_end = part[k + 1], rk_before = part[k > kFixShort ? k - kFixShort : 0];
  const uint64_t found =
      __ballot(lane < kFixWaves && j < n_sub && k > kFixShort && rk_end != rk && rk_before == rk);
  if (t < n_sub && !((found >> w) & 1)) {
    const int64_t r0 = lane_i64(rk, w);
    const bool ends = lane_i64(rk_end, w) != r0;
    const int64_t n0 = t * (int64_t)sub_items - r0;
    const int64_t start = !ends ? n0
                          : ptr64 ? static_cast<const int64_t*>(rowptr_raw)[r0]
                                  : (int64_t) static_cast<const int32_t*>(rowptr_raw)[r0];
    if (start < n0) {
      const int64_t f = fixup_start_tile(part, t, r0);
      for (int64_t col = (int64_t)blockIdx.y * 64 + lane; col < n_dense; col += (int64_t)gridDim.y * 64) {
        A sum = tail[f * n_dense + col];
        sum = sum_fragments(tail + col, n_dense, f + 1, t, sum);  // in sub-tile order
        sum = add(sum, head[t * n_dense + col]);
        C[r0 * scm + col * scn] = T::out(sum);
      }
    }
  }
  if (found == 0) return;  // whole workgroup
  const int64_t lt = t0 + (int)__builtin_ctzll(found), row = part[lt], lf = fixup_start_tile(part, lt, row);
  for (int64_t c0 = (int64_t)blockIdx.y * 64; c0 < n_dense; c0 += (int64_t)gridDim.y * 64) {
    const int nc = n_dense - c0 < 64 ? (int)(n_dense - c0) : 64;
    int width = 1;  // threads per share: the columns, rounded up to a power of two
    while (width < nc) width <<= 1;
    const int shares = kFixThreads / width, share = tid / width, c = tid % width;
    const int64_t len = (lt - lf + shares - 1) / shares;
    const int64_t k0 = lf + share * len < lt ? lf + share * len : lt;
    const int64_t k1 = lt - k0 < len ? lt : k0 + len;
    A sum = T::zero();
    if (c < nc) sum = sum_fragments(tail + c0 + c, n_dense, k0, k1, sum);
    s_sum[tid] = sum;
    for (int o = shares >> 1; o > 0; o >>= 1) {
      __syncthreads();
      if (share < o) s_sum[tid] = add(s_sum[tid], s_sum[tid + o * width]);
    }
    if (share == 0 && c < nc) {
      sum = add(s_sum[tid], head[lt * n_dense + c0 + c]);
      C[row * scm + (c0 + c) * scn] = T::out(sum);
    }
    __syncthreads();
  }
}

template <class V, int LPR, class T>
int launch_spmm_group(const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                      const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm, int64_t scn,
                      int64_t n_dense, const int64_t* part, int sub_items, int64_t n_sub, void* ws,
                      hipStream_t stream) {
  using A = typename T::acc;
  constexpr int G = 64 / LPR;
  constexpr int EPL = group_epl<V>();
  A* head = static_cast<A*>(ws);
  A* tail = head + n_sub * n_dense;
  const int64_t col_tiles = ceil_div(n_dense, (int64_t)LPR * EPL);
  const int64_t waves = ceil_div(n_sub, G);
  const int64_t blocks = ceil_div(waves, 4);
  if (blocks > 0x7fffffffLL || col_tiles > 65535) return fail(FS_E_INVALID, "fs_spmm_csr: grid too large");
  int xcd_cols = (col_tiles == 2 || col_tiles == 4 || col_tiles == 8) ? (int)col_tiles : 0;
  if (const char* e = std::getenv("FLAGSPARSE_SPMM_XCD")) xcd_cols = std::atoi(e) != 0 ? (int)col_tiles : 0;
  if (xcd_cols > 0 && blocks * col_tiles > 0x7fffffffLL) xcd_cols = 0;
  int row_ranges = 0;
  if (const char* e = std::getenv("FLAGSPARSE_SPMM_ROW_RANGES")) row_ranges = std::atoi(e) != 0;
  dim3 grid = xcd_cols > 0 ? dim3((unsigned)(blocks * col_tiles)) : dim3((unsigned)blocks, (unsigned)col_tiles);
  size_t lds = (size_t)4 * G * (size_t)sub_items * sizeof(uint16_t);
  if (const char* e = std::getenv("FLAGSPARSE_SPMM_WG_CAP")) lds = std::max(lds, lds_pad_for_cap(std::atoi(e), 0));
  // vector path: every lane's B / C slice is EPL unit-stride elements, 16-byte aligned
  // (and 32-bit gather offsets: column indices and B's row stride in bytes fit 32 bits)
  const bool vec = sbn == 1 && scn == 1 && (n_dense % EPL) == 0 && (sbk % EPL) == 0 && (scm % EPL) == 0 &&
                   ((uintptr_t)B % group_slice<V>::bytes) == 0 &&
                   ((uintptr_t)C % group_slice<V>::bytes) == 0 && plan->n_cols <= (int64_t(1) << 32) &&
                   sbk * (int64_t)sizeof(V) < (int64_t(1) << 32);
  const int ptr64 = plan->ptr_t == FS_I64 ? 1 : 0;
  auto go = [&](auto icode) {
    using I = std::conditional_t<decltype(icode)::value, int64_t, int32_t>;
    auto launch = [&](auto vcode) {
      hipLaunchKernelGGL((spmm_group_kernel<V, LPR, 4, decltype(vcode)::value, I, T>), grid, dim3(256), lds, stream,
                         static_cast<const V*>(vals), static_cast<const I*>(cols), indptr, ptr64,
                         static_cast<const V*>(B), sbk, sbn, static_cast<V*>(C), scm, scn, n_dense, part, sub_items,
                         head, tail, plan->n_rows, plan->nnz, n_sub, xcd_cols, row_ranges);
    };
    if (vec) launch(std::true_type{});
    else launch(std::false_type{});
  };
  if (plan->idx_t == FS_I64) go(std::true_type{});
  else go(std::false_type{});
  FS_CHECK_MAIN_LAUNCH("spmm_group_kernel");
  const int64_t fix_blocks = ceil_div(n_sub, (int64_t)kFixWaves);
  const int64_t fix_cols = ceil_div(n_dense, 64) < 64 ? ceil_div(n_dense, 64) : 64;
  hipLaunchKernelGGL((spmm_group_fixup_kernel<V, T>), dim3((unsigned)fix_blocks, (unsigned)fix_cols),
                     dim3(kFixThreads), 0, stream, indptr, plan->ptr_t == FS_I64 ? 1 : 0, part, sub_items, head, tail,
                     static_cast<V*>(C), scm, scn, n_dense, n_sub);
  FS_CHECK_LAUNCH("spmm_group_fixup_kernel");
  return FS_OK;
}

// 16-bit B rows of up to 64 columns, or not of whole 16-byte slices: 8-byte
// slices (spmm_half.hip).
inline bool half_narrow(int64_t n_dense) { return n_dense <= 64 || n_dense % 8 != 0; }

}  // namespace fs
