// merge_tile.hpp — one wave's merge-path tile of the SpMV: its loads, its walk
// over 512 items (row ends + nnz) and the fix-up of rows that span tiles.
// Shared by the merge-path kernels (spmv.hip) and the two-phase gather SpMV
// (spmv_gather.hip).
#pragma once

#include "fs_common.hpp"

#include <type_traits>

namespace fs {

constexpr int kSlabs = 8;
constexpr int kMergeTile = kSlabs * 64;
constexpr int kMergeWaves = 4;

__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ inline int count_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// DPP-shifted copy of a 32-bit value; lanes whose source is outside the
// enabled rows / row bounds receive 0.
template <int CTRL, int ROWMASK>
__device__ inline int dpp_shift(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWMASK, 0xF, false);
}

template <int CTRL, int ROWMASK>
__device__ inline double dpp_shift(double v) {
  int lo = dpp_shift<CTRL, ROWMASK>(__double2loint(v));
  int hi = dpp_shift<CTRL, ROWMASK>(__double2hiint(v));
  return __hiloint2double(hi, lo);
}

template <int CTRL, int ROWMASK>
__device__ inline c64 dpp_shift(c64 v) {
  return c64{dpp_shift<CTRL, ROWMASK>(v.re), dpp_shift<CTRL, ROWMASK>(v.im)};
}

// One step of the segmented scan: lanes that have not yet reached their
// segment head absorb the shifted partial and its head flag.
template <int CTRL, int ROWMASK, class A>
__device__ inline void seg_step(A& v, int& f) {
  A pv = dpp_shift<CTRL, ROWMASK>(v);
  int pf = dpp_shift<CTRL, ROWMASK>(f);
  if (!f) {
    v = add(v, pv);
    f = pf;
  }
}

// Segmented inclusive scan over the wave; f = 1 marks a segment head.
// row_shr 1,2,4,8 scan each 16-lane row; row_bcast15 / row_bcast31 carry
// across rows (the standard CDNA wave-scan sequence).
template <class A>
__device__ inline A seg_scan(A v, int f) {
  seg_step<0x111, 0xF>(v, f);  // row_shr:1
  seg_step<0x112, 0xF>(v, f);  // row_shr:2
  seg_step<0x114, 0xF>(v, f);  // row_shr:4
  seg_step<0x118, 0xF>(v, f);  // row_shr:8
  seg_step<0x142, 0xA>(v, f);  // row_bcast:15 -> rows 1,3
  seg_step<0x143, 0xC>(v, f);  // row_bcast:31 -> rows 2,3
  return v;
}

template <class A>
__device__ inline A readlane_acc(A v, int lane);
template <>
__device__ inline double readlane_acc<double>(double v, int lane) { return readlane_f64(v, lane); }
template <>
__device__ inline c64 readlane_acc<c64>(c64 v, int lane) {
  return c64{readlane_f64(v.re, lane), readlane_f64(v.im, lane)};
}

// Item layout of a tile: item d (0..511) is a row end if bit d of the
// tile mask is set, otherwise the next nnz.  Lane l walks items
// [8l, 8l+8) sequentially; the products it needs were staged in LDS by
// coalesced loads (index padded by j/8 so that lanes starting 8 products
// apart hit different banks).
__device__ inline int prod_slot(int j) { return j + (j >> 3); }

// Row results go to y as the value type, or (for column-panel partials)
// as the accumulator type, so that a later reduction rounds only once.
template <class V, class Y>
__device__ inline void store_row(Y* y, int64_t row, typename VT<V>::acc v) {
  if constexpr (std::is_same<Y, typename VT<V>::acc>::value)
    y[row] = v;
  else
    y[row] = VT<V>::out(v);
}

// Geometry of merge tile t: its first row r0 = part[t], its row ends
// r0 .. r1-1, its first nnz n0, R row ends and Nz nnz.
struct TileGeom {
  int64_t r0, r1, n0;
  int R, Nz;
};
__device__ inline TileGeom tile_geom(int64_t t, int64_t r0, int64_t r1, int64_t total) {
  const int64_t d0 = t * kMergeTile;
  const int64_t dend = d0 + kMergeTile < total ? d0 + kMergeTile : total;
  TileGeom g;
  g.r0 = r0;
  g.r1 = r1;
  g.n0 = d0 - r0;
  g.R = (int)(r1 - r0);
  g.Nz = (int)(dend - r1 - g.n0);
  return g;
}

// The tile's own loads: values and columns of its nnz (coalesced, read
// once: non-temporal, which keeps x in L2, power-law 0.608 -> 0.591 ms),
// and the row pointers of its row ends (lane-striped), plus rowptr[r0].
template <class V, class I, class P>
__device__ inline void tile_loads(const V* __restrict__ vals, const I* __restrict__ cols,
                                  const P* __restrict__ rowptr, const TileGeom& g, V (&av)[kMergeTile / 64],
                                  I (&cv)[kMergeTile / 64], P (&rp)[kMergeTile / 64], P& rp0) {
  constexpr int kIpt = kMergeTile / 64;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < kIpt; ++k) {
    const int j = k * 64 + lane;
    if (j < g.Nz) {  // lanes past the tile keep stale registers, never read
      av[k] = load_stream(vals + g.n0 + j);
      cv[k] = __builtin_nontemporal_load(cols + g.n0 + j);
    }
  }
#pragma unroll
  for (int i = 0; i < kIpt; ++i) {
    const int k = lane + 64 * i;
    if (k < g.R) rp[i] = rowptr[g.r0 + 1 + k];
  }
  rp0 = g.R > 0 ? rowptr[g.r0] : P(0);
}

// tile_loads without branches, for the pipelined loop: lanes past the
// tile's nnz re-read the matrix's last entry and lanes past its row ends the
// last row pointer (n_rows_total = rows of the CSR), so every load is issued
// and the compiler can count loads in flight exactly (a load skipped on
// some path makes it wait for all of them).  Needs nnz >= 1.
template <class V, class I, class P>
__device__ inline void tile_loads_all(const V* __restrict__ vals, const I* __restrict__ cols,
                                      const P* __restrict__ rowptr, const TileGeom& g, int64_t nnz,
                                      int64_t n_rows_total, V (&av)[kMergeTile / 64], I (&cv)[kMergeTile / 64],
                                      P (&rp)[kMergeTile / 64], P& rp0) {
  constexpr int kIpt = kMergeTile / 64;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < kIpt; ++k) {
    const int j = k * 64 + lane;
    const int64_t e = j < g.Nz ? g.n0 + j : nnz - 1;
    av[k] = load_stream(vals + e);
    cv[k] = __builtin_nontemporal_load(cols + e);
  }
#pragma unroll
  for (int i = 0; i < kIpt; ++i) {
    const int k = lane + 64 * i;
    rp[i] = rowptr[k < g.R ? g.r0 + 1 + k : n_rows_total];
  }
  rp0 = rowptr[g.r0];
}

// Everything after the x gathers of one tile: row-end mask, products in
// LDS, per-lane walk, carry scan, row stores and head / tail fragments.
// FULL: the tile has all its 512 items: no lane tests on items, the products
// past Nz are written and never read, and row ends beyond the first 64 are
// handled only where there are any.
template <class V, class P, class Y, bool FULL = false>
__device__ inline void tile_finish(Y* __restrict__ y, typename VT<V>::acc* __restrict__ head,
                                   typename VT<V>::acc* __restrict__ tail, int64_t n_rows, int64_t t,
                                   const TileGeom& g, const V (&av)[kMergeTile / 64], const V (&xv)[kMergeTile / 64],
                                   const P (&rp)[kMergeTile / 64], P rp0, unsigned* msk,
                                   typename VT<V>::acc* prod) {
  using T = VT<V>;
  using A = typename T::acc;
  constexpr int kIpt = kMergeTile / 64;  // items per lane
  const int lane = threadIdx.x & 63;
  const int64_t r0 = g.r0;
  const int R = g.R;
  const int Nz = g.Nz;
  const int items = R + Nz;
  // row-end mask (one ds_or per row end).
  if (lane < kMergeTile / 32) msk[lane] = 0u;
  wave_sync();
#pragma unroll
  for (int i = 0; i < kIpt; ++i) {
    if (FULL && i > 0 && R <= 64 * i) break;
    const int k = lane + 64 * i;
    if (k < R) {
      const int q = (int)(k + (int64_t)rp[i] - g.n0);
      atomicOr(&msk[q >> 5], 1u << (q & 31));
    }
  }
  const bool head_partial = R > 0 && (int64_t)rp0 < g.n0;
#pragma unroll
  for (int k = 0; k < kIpt; ++k) {
    const int j = k * 64 + lane;
    if (FULL || j < Nz) prod[prod_slot(j)] = T::mul(av[k], xv[k]);
  }
  wave_sync();
  // sequential walk of this lane's 8 items.  Row ends before the lane:
  // popcounts of the 16 mask words, scanned over lanes 0..15 with DPP row
  // shifts (one 16-lane row), read back from lane d/32 by a permute.
  static_assert(kMergeTile / 32 == 16, "word scan covers one DPP row");
  const int d = kIpt * lane;                          // first item of the lane
  const unsigned word = msk[d >> 5];
  const int cnt = lane < 16 ? __popc(msk[lane]) : 0;
  int inc = cnt;
  inc += dpp_shift<0x111, 0xF>(inc);  // row_shr:1
  inc += dpp_shift<0x112, 0xF>(inc);  // row_shr:2
  inc += dpp_shift<0x114, 0xF>(inc);  // row_shr:4
  inc += dpp_shift<0x118, 0xF>(inc);  // row_shr:8
  const int word_pre = __shfl(inc - cnt, d >> 5);
  const unsigned pattern = (word >> (d & 31)) & 0xFFu;  // 8 items never straddle a word
  const int i_l = word_pre + __popc(word & ((1u << (d & 31)) - 1u));
  int j = d - i_l;                                     // tile-local nnz index
  int ends = 0;
  A acc = T::zero(), first = T::zero();
#pragma unroll
  for (int u = 0; u < kIpt; ++u) {
    if (FULL || d + u < items) {
      if ((pattern >> u) & 1u) {
        if (ends == 0) {
          first = acc;
        } else {
          store_row<V>(y, r0 + i_l + ends, acc);
        }
        ++ends;
        acc = T::zero();
      } else {
        acc = add(acc, prod[prod_slot(j)]);
        ++j;
      }
    }
  }

  // carry across lanes: inclusive segmented scan of lane tails (a lane
  // with a row end starts a new segment), shifted to exclusive.
  const A incl = seg_scan(acc, ends > 0 ? 1 : 0);
  A carry_in = shfl(incl, lane > 0 ? lane - 1 : 0);
  if (lane == 0) carry_in = T::zero();
  if (ends > 0) {
    const A v = add(carry_in, first);
    const int64_t row = r0 + i_l;
    if (row == r0 && head_partial)
      head[t] = v;
    else
      store_row<V>(y, row, v);
  }
  if (lane == 63 && g.r1 < n_rows) tail[t] = incl;
}

// Rows that span tiles: y[row] = tail[f] + ... + tail[t-1] + head[t], where
// tiles f..t-1 all end inside `row` and tile t holds its row end.
template <class V, class P, class Y = V>
__global__ __launch_bounds__(256) void merge_fixup_kernel(
    const P* __restrict__ rowptr, const int64_t* __restrict__ part,
    const typename VT<V>::acc* __restrict__ head, const typename VT<V>::acc* __restrict__ tail,
    Y* __restrict__ y, int64_t n_tiles, int64_t tile_items) {
  using T = VT<V>;
  using A = typename T::acc;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_tiles) return;
  const int64_t r0 = part[t];
  if (part[t + 1] == r0) return;  // tile holds no row end
  const int64_t n0 = t * tile_items - r0;
  if ((int64_t)rowptr[r0] >= n0) return;  // row r0 starts inside tile t
  const int64_t f = fixup_start_tile(part, t, r0);
  A sum = sum_fragments(tail, 1, f + 1, t, tail[f]);
  sum = add(sum, head[t]);
  store_row<V>(y, r0, sum);
}

}  // namespace fs
