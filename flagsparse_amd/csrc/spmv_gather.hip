// spmv_gather.hip — two-phase SpMV on gfx950 for a prepared matrix whose
// columns spread over an x larger than L2 serves well.
//
// A gather of x from L2 costs one L1 miss per entry: the vector L1s stall on
// outstanding misses long before HBM is busy (a power-law matrix with 70 M
// float32 entries and a 16.8 MB x spent 0.45 of its 0.57 ms there).  Here x is
// gathered from LDS instead, in two streaming passes over a plan built once:
//
//  1. gather: the columns are cut into slices of x that fit LDS.  A workgroup
//     loads a slice and walks the entries of that slice, reading only a 16-bit
//     column number per entry and writing x[col] to the entry's place in its
//     region.  Entries move in quads (four of one slice and one region; a
//     quad's place in the regions is one 32-bit number), so every access is a
//     contiguous 8-, 4- or 16-byte one.
//  2. reduce: a region holds the gathered values of kTiles consecutive
//     merge-path tiles (the caller's rows and entries, in CSR order), sorted by
//     slice.  A workgroup copies its region into LDS and walks its tiles as the
//     merge-path kernel does, taking an entry's x from the region at the
//     entry's 16-bit position.  Products, sums, their order and the fix-up of
//     rows that span tiles are the merge-path kernel's: the same bits.
//
// us per call, one-pass kernels -> two-phase: power-law 4 M float32 563 -> 331;
// R-MAT 2^21 float32 290 -> 178, float64 513 -> 330, complex64 603 -> 374; 16
// uniform columns in each of 4,000,000 rows float32 870 -> 315, float64 1057 ->
// 594; 1 M rows float32 95 -> 82, float64 188 -> 116.  complex128 gained on none but
// R-MAT 2^21 (283 -> 368 on 1 M uniform rows) and does not take this path.
//
// Values are read from the caller's array; the plan holds 5 bytes per entry
// (position, column number, quarter of a quad's place).  HBM traffic per
// entry: 3 + s_v (gather) + 2 + 2 s_v (reduce).
#include "fs_common.hpp"
#include "merge_tile.hpp"
#include "radix_tile.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>

namespace fs {

constexpr int kGatherMaxSlices = 256;
constexpr int kGatherThreads = 1024;
constexpr int kSliceBytesLog2 = 17;  // 128 KB of x per slice

// Tiles per region: up to 32 KB of gathered values, so that two to three
// reduce workgroups fit a CU's LDS.  Power-law 4 M float32 (70 M entries), us
// gather + reduce: 122 + 201; 16 KB regions (shorter runs to write) 145 + 202,
// 64 KB 110 + 386; slices of 64 KB 152 + 200.
template <class V>
constexpr int region_tiles() {
  return (int)(64 / sizeof(V));
}
inline int region_tiles_of(int val_t) { return val_t == FS_F32 ? region_tiles<float>() : region_tiles<double>(); }
inline int slice_log2(int val_t) { return kSliceBytesLog2 - (val_t == FS_F32 ? 2 : 3); }

// Entries [n0, n1) of region g (tiles [g T, g T + T)).
__device__ inline void region_entries(const int64_t* __restrict__ part, int64_t g, int T, int64_t n_tiles,
                                      int64_t total, int64_t& n0, int64_t& n1) {
  const int64_t t0 = g * T, t1 = t0 + T < n_tiles ? t0 + T : n_tiles;
  const int64_t d1 = t1 * kMergeTile < total ? t1 * kMergeTile : total;
  n0 = t0 * kMergeTile - part[t0];
  n1 = d1 - part[t1];
}

// Plan, pass 1: quads of every (region, slice), cnt[region][slice]; per region
// the quads in all and the slices it touches (what the caller's choice of this
// path is judged on).
template <class I>
__global__ __launch_bounds__(256) void gather_count_kernel(const I* __restrict__ cols,
                                                           const int64_t* __restrict__ part, int T, int64_t n_tiles,
                                                           int64_t total, int log2w, int ns,
                                                           uint32_t* __restrict__ cnt, int32_t* __restrict__ quads,
                                                           int32_t* __restrict__ touched) {
  __shared__ unsigned s_hist[kGatherMaxSlices];
  __shared__ int s_sum[2];
  const int t = threadIdx.x;
  const int64_t g = blockIdx.x;
  if (t < ns) s_hist[t] = 0u;
  if (t < 2) s_sum[t] = 0;
  __syncthreads();
  int64_t n0, n1;
  region_entries(part, g, T, n_tiles, total, n0, n1);
  for (int64_t e = n0 + t; e < n1; e += 256) atomicAdd(&s_hist[(unsigned)((int64_t)cols[e] >> log2w)], 1u);
  __syncthreads();
  if (t < ns) {
    const unsigned q = (s_hist[t] + 3) / 4;
    cnt[g * ns + t] = q;
    if (q) {
      atomicAdd(&s_sum[0], (int)q);
      atomicAdd(&s_sum[1], 1);
    }
  }
  __syncthreads();
  if (t == 0) {
    quads[g] = s_sum[0];
    touched[g] = s_sum[1];
  }
}

// Plan, pass 2: the positions, column numbers and quad places.  `start` is
// cnt after its (slice, region) scan: the first quad of every run in the
// slice-major stream; region_q[g] is the first quad of region g.  Ranks within
// a run come from LDS counters in any order: where an entry's x lies does not
// change the sum.  The column numbers are put together in LDS in region order
// and leave as whole quads (stored one by one, each store was a request of its
// own: 842 us for 64 M entries).
constexpr int kRegionMaxEntries = 16 * kMergeTile;  // float32's region; the others' are smaller
constexpr int kRegionMaxQuads = kRegionMaxEntries / 4 + kGatherMaxSlices;
template <class I>
__global__ __launch_bounds__(256) void gather_fill_kernel(const I* __restrict__ cols,
                                                          const int64_t* __restrict__ part, int T, int64_t n_tiles,
                                                          int64_t total, int log2w, int ns,
                                                          const uint32_t* __restrict__ start,
                                                          const int32_t* __restrict__ region_q,
                                                          uint16_t* __restrict__ pos, uint2* __restrict__ idx,
                                                          uint32_t* __restrict__ place) {
  __shared__ unsigned s_next[kGatherMaxSlices];   // entries so far, per slice
  __shared__ unsigned s_first[kGatherMaxSlices];  // first quad within the region
  __shared__ unsigned s_shift[kGatherMaxSlices];  // stream quad - region quad, per slice
  __shared__ uint2 s_idx[kRegionMaxQuads];
  __shared__ uint8_t s_slice[kRegionMaxQuads];
  __shared__ int64_t s_wave[4];
  const int t = threadIdx.x;
  const int64_t g = blockIdx.x;
  if (t < ns) s_next[t] = 0u;
  __syncthreads();
  int64_t n0, n1;
  region_entries(part, g, T, n_tiles, total, n0, n1);
  for (int64_t e = n0 + t; e < n1; e += 256) atomicAdd(&s_next[(unsigned)((int64_t)cols[e] >> log2w)], 1u);
  __syncthreads();
  const unsigned n = t < ns ? s_next[t] : 0u;
  const unsigned q = (n + 3) / 4;
  int64_t all;
  const unsigned first = (unsigned)block_exclusive_scan((int64_t)q, s_wave, all);
  const unsigned quads = (unsigned)all;
  if (t < ns) {
    s_first[t] = first;
    s_next[t] = 0u;
    s_shift[t] = start[g * ns + t] - first;
    for (unsigned k = 0; k < q; ++k) s_slice[first + k] = (uint8_t)t;
  }
  for (unsigned k = t; k < quads; k += 256) s_idx[k] = make_uint2(0u, 0u);  // padding gathers the slice's first entry
  __syncthreads();
  uint16_t* s_one = reinterpret_cast<uint16_t*>(s_idx);
  for (int64_t e = n0 + t; e < n1; e += 256) {
    const int64_t c = (int64_t)cols[e];
    const unsigned p = (unsigned)(c >> log2w);
    const unsigned at = s_first[p] * 4 + atomicAdd(&s_next[p], 1u);
    pos[e] = (uint16_t)at;
    s_one[at] = (uint16_t)(c & (((int64_t)1 << log2w) - 1));
  }
  __syncthreads();
  for (unsigned k = t; k < quads; k += 256) {
    const unsigned at = k + s_shift[s_slice[k]];
    idx[at] = s_idx[k];
    place[at] = (uint32_t)region_q[g] + k;
  }
}

// Phase 1.  Workgroup b takes quads [b q_wg, (b + 1) q_wg) of the stream and
// loads each slice they belong to (one or two for evenly spread columns).
template <class V>
struct alignas(16) Quad {
  V v[4];
};
template <class V>
__global__ __launch_bounds__(kGatherThreads) void spmv_gather_kernel(const V* __restrict__ x, int64_t n_x,
                                                                     const uint2* __restrict__ idx,
                                                                     const uint32_t* __restrict__ place,
                                                                     const uint32_t* __restrict__ slice_q, int ns,
                                                                     uint32_t n_quads, uint32_t q_wg, int log2w,
                                                                     Quad<V>* __restrict__ xg) {
  extern __shared__ __attribute__((aligned(16))) uint8_t g_lds[];
  V* s_x = reinterpret_cast<V*>(g_lds);
  const int t = threadIdx.x;
  uint32_t q = blockIdx.x * q_wg;
  const uint32_t q_end = n_quads - q < q_wg ? n_quads : q + q_wg;  // (the grid has no empty workgroup)
  int p = 0;
  while (p + 1 < ns && slice_q[p + 1] <= q) ++p;  // the last slice starting at or before q
  while (q < q_end) {
    while (slice_q[p + 1] <= q) ++p;  // (slice_q[ns] = n_quads > q)
    const int64_t x0 = (int64_t)p << log2w;
    const int len = n_x - x0 < ((int64_t)1 << log2w) ? (int)(n_x - x0) : 1 << log2w;
    constexpr int kPer = 8;
    for (int k0 = t; k0 < len; k0 += kPer * kGatherThreads) {
      V r[kPer];
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int k = k0 + u * kGatherThreads;
        r[u] = x[x0 + (k < len ? k : len - 1)];
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int k = k0 + u * kGatherThreads;
        if (k < len) s_x[k] = r[u];
      }
    }
    __syncthreads();
    const uint32_t stop = slice_q[p + 1] < q_end ? slice_q[p + 1] : q_end;
    constexpr int kAheadQ = 4;
    for (uint32_t k0 = q + t; k0 < stop; k0 += kAheadQ * kGatherThreads) {
      uint2 i[kAheadQ];
      uint32_t d[kAheadQ];
#pragma unroll
      for (int u = 0; u < kAheadQ; ++u) {
        const uint32_t k = k0 + u * kGatherThreads < stop ? k0 + u * kGatherThreads : stop - 1;
        i[u] = idx[k];
        d[u] = place[k];
      }
#pragma unroll
      for (int u = 0; u < kAheadQ; ++u) {
        Quad<V> o;
        o.v[0] = s_x[i[u].x & 0xffffu];
        o.v[1] = s_x[i[u].x >> 16];
        o.v[2] = s_x[i[u].y & 0xffffu];
        o.v[3] = s_x[i[u].y >> 16];
        if (k0 + u * kGatherThreads < stop) xg[d[u]] = o;
      }
    }
    __syncthreads();  // before the next slice overwrites this one
    q = stop;
  }
}

// A tile's loads for the region walk.  A whole tile away from the end of the
// matrix reads 512 entries from its first (scalar base, no lane tests; those
// past its own are not used) and the row ends it has; any other tile reads as
// the pipelined merge-path walk does.
template <class V, class P>
__device__ inline bool region_tile_loads(const V* __restrict__ vals, const uint16_t* __restrict__ pos,
                                         const P* __restrict__ rowptr, const TileGeom& g, int64_t nnz, int64_t n_rows,
                                         V (&av)[kMergeTile / 64], uint16_t (&cv)[kMergeTile / 64],
                                         P (&rp)[kMergeTile / 64], P& rp0) {
  constexpr int kIpt = kMergeTile / 64;
  const int lane = threadIdx.x & 63;
  const bool full = g.R + g.Nz == kMergeTile && g.n0 + kMergeTile <= nnz;
  if (!full) {
    tile_loads_all<V, uint16_t, P>(vals, pos, rowptr, g, nnz, n_rows, av, cv, rp, rp0);
    return false;
  }
  const V* v = vals + g.n0;
  const uint16_t* c = pos + g.n0;
#pragma unroll
  for (int k = 0; k < kIpt; ++k) {
    av[k] = load_stream(v + k * 64 + lane);
    cv[k] = __builtin_nontemporal_load(c + k * 64 + lane);
  }
  const P* r = rowptr + g.r0;
  rp0 = r[0];
  const int last = n_rows - g.r0 < kMergeTile ? (int)(n_rows - g.r0) : kMergeTile;
  rp[0] = r[lane + 1 < last ? lane + 1 : last];
#pragma unroll
  for (int i = 1; i < kIpt; ++i) {
    if (g.R <= 64 * i) break;
    const int k = 64 * i + lane + 1;
    rp[i] = r[k < last ? k : last];
  }
  return true;
}

// Phase 2: one region per workgroup.  A wave's first tile is loaded before the
// region is waited for, and tile i + 1 before tile i is walked.  It moves
// 4.3 TB/s (power-law 4 M float32: 862 MB in 200 us); with lane tests in whole
// tiles it was bound by instruction issue (212 us, SIMDs active 88%).
template <class V, class P>
__global__ __launch_bounds__(256) void spmv_region_kernel(const V* __restrict__ vals, const uint16_t* __restrict__ pos,
                                                          const P* __restrict__ rowptr,
                                                          const uint8_t* __restrict__ xg,
                                                          const int32_t* __restrict__ region_q, V* __restrict__ y,
                                                          const int64_t* __restrict__ part,
                                                          typename VT<V>::acc* __restrict__ head,
                                                          typename VT<V>::acc* __restrict__ tail, int64_t n_rows,
                                                          int64_t nnz, int64_t n_tiles) {
  using A = typename VT<V>::acc;
  using L4 = __attribute__((ext_vector_type(4))) unsigned int;
  constexpr int T = region_tiles<V>();
  constexpr int kIpt = kMergeTile / 64;
  __shared__ unsigned s_mask[kMergeWaves][kMergeTile / 32];
  __shared__ A s_prod[kMergeWaves][kMergeTile + kMergeTile / 8];
  extern __shared__ __attribute__((aligned(16))) uint8_t r_lds[];
  const V* s_x = reinterpret_cast<const V*>(r_lds);
  const int t = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int64_t g = blockIdx.x;
  const int64_t total = n_rows + nnz;
  const int64_t t_end = (g + 1) * T < n_tiles ? (g + 1) * T : n_tiles;
  int64_t tile = g * T + w;
  const int64_t tile0 = tile < t_end ? tile : t_end - 1;  // a wave without a tile loads (and drops) the last one
  TileGeom gm = tile_geom(tile0, part[tile0], part[tile0 + 1], total);
  V av[kIpt];
  uint16_t cv[kIpt];
  P rp[kIpt];
  P rp0;
  bool full = region_tile_loads<V, P>(vals, pos, rowptr, gm, nnz, n_rows, av, cv, rp, rp0);
  {
    const int32_t q0 = region_q[g];
    const int n16 = (region_q[g + 1] - q0) * (int)(sizeof(Quad<V>) / 16);
    const L4* src = reinterpret_cast<const L4*>(xg) + (int64_t)q0 * (int)(sizeof(Quad<V>) / 16);
    L4* dst = reinterpret_cast<L4*>(r_lds);
    constexpr int kPer = 8;
    for (int k0 = t; k0 < n16; k0 += kPer * 256) {
      L4 r[kPer];
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int k = k0 + u * 256;
        r[u] = __builtin_nontemporal_load(src + (k < n16 ? k : n16 - 1));
      }
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int k = k0 + u * 256;
        if (k < n16) dst[k] = r[u];
      }
    }
  }
  __syncthreads();
  while (tile < t_end) {
    // (positions of lanes past the tile's entries may belong to another
    // region but stay inside the LDS allocation, which holds the largest)
    V xv[kIpt];
#pragma unroll
    for (int k = 0; k < kIpt; ++k) xv[k] = s_x[cv[k]];
    const int64_t tn = tile + kMergeWaves < t_end ? tile + kMergeWaves : tile;
    const TileGeom gn = tile_geom(tn, part[tn], part[tn + 1], total);
    V avn[kIpt];
    uint16_t cvn[kIpt];
    P rpn[kIpt];
    P rp0n;
    const bool fulln = region_tile_loads<V, P>(vals, pos, rowptr, gn, nnz, n_rows, avn, cvn, rpn, rp0n);
    if (full)
      tile_finish<V, P, V, true>(y, head, tail, n_rows, tile, gm, av, xv, rp, rp0, s_mask[w], s_prod[w]);
    else
      tile_finish<V, P, V, false>(y, head, tail, n_rows, tile, gm, av, xv, rp, rp0, s_mask[w], s_prod[w]);
    wave_sync();  // this tile's LDS reads are done before the next tile's writes
    gm = gn;
    full = fulln;
#pragma unroll
    for (int k = 0; k < kIpt; ++k) {
      av[k] = avn[k];
      cv[k] = cvn[k];
      rp[k] = rpn[k];
    }
    rp0 = rp0n;
    tile += kMergeWaves;
  }
}

inline size_t gather_acc_bytes(int val_t) { return val_t == FS_C64 ? sizeof(c64) : sizeof(double); }
inline size_t gather_val_bytes(int val_t) { return val_t == FS_F32 ? 4 : 8; }

template <class V, class P>
int launch_gather_spmv(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz, const void* vals, const void* indptr,
                       const void* x, void* y, const int64_t* part, const uint16_t* pos, const uint2* idx,
                       const uint32_t* place, const uint32_t* slice_q, const int32_t* region_q, int64_t n_quads,
                       int64_t max_region_quads, char* ws, hipStream_t s) {
  using A = typename VT<V>::acc;
  const int64_t n_tiles = ceil_div(n_rows + nnz, (int64_t)kMergeTile);
  const int64_t regions = ceil_div(n_tiles, (int64_t)region_tiles<V>());
  const int log2w = slice_log2(val_t);
  const int ns = (int)ceil_div(n_cols, int64_t(1) << log2w);
  uint8_t* xg = reinterpret_cast<uint8_t*>(ws);
  A* head = reinterpret_cast<A*>(ws + (size_t)n_quads * sizeof(Quad<V>));
  A* tail = head + n_tiles;
  // one workgroup per CU (its slice takes most of the LDS), even shares
  const int64_t wgs = std::min<int64_t>(ceil_div(n_quads, (int64_t)kGatherThreads), 256);
  const uint32_t q_wg = (uint32_t)ceil_div(n_quads, wgs);
  const size_t slice_lds = (size_t)std::min<int64_t>(n_cols, int64_t(1) << log2w) * sizeof(V);
  FS_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&spmv_gather_kernel<V>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 1 << kSliceBytesLog2));
  hipLaunchKernelGGL((spmv_gather_kernel<V>), dim3((unsigned)ceil_div(n_quads, (int64_t)q_wg)), dim3(kGatherThreads),
                     slice_lds, s, static_cast<const V*>(x), n_cols, idx, place, slice_q, ns, (uint32_t)n_quads, q_wg,
                     log2w, reinterpret_cast<Quad<V>*>(xg));
  FS_CHECK_LAUNCH("spmv_gather_kernel");
  const size_t region_lds = (size_t)max_region_quads * sizeof(Quad<V>);
  FS_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&spmv_region_kernel<V, P>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 96 << 10));
  hipLaunchKernelGGL((spmv_region_kernel<V, P>), dim3((unsigned)regions), dim3(256), region_lds, s,
                     static_cast<const V*>(vals), pos, static_cast<const P*>(indptr), xg, region_q,
                     static_cast<V*>(y), part, head, tail, n_rows, nnz, n_tiles);
  FS_CHECK_MAIN_LAUNCH("spmv_region_kernel");
  hipLaunchKernelGGL((merge_fixup_kernel<V, P, V>), dim3((unsigned)ceil_div(n_tiles, 256)), dim3(256), 0, s,
                     static_cast<const P*>(indptr), part, head, tail, static_cast<V*>(y), n_tiles,
                     (int64_t)kMergeTile);
  FS_CHECK_LAUNCH("merge_fixup_kernel");
  return FS_OK;
}

inline bool gather_sizes_ok(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz) {
  return val_t >= FS_F32 && val_t < FS_C128 && n_rows > 0 && n_cols > 0 && nnz > 0 && nnz < (int64_t(1) << 31) &&
         n_rows < (int64_t(1) << 31) && ceil_div(n_cols, int64_t(1) << slice_log2(val_t)) <= kGatherMaxSlices;
}

}  // namespace fs

using namespace fs;

extern "C" int fs_spmv_gather_slices(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz, int64_t* n_regions) {
  if (!n_regions || !gather_sizes_ok(val_t, n_rows, n_cols, nnz)) return 0;
  *n_regions = ceil_div(ceil_div(n_rows + nnz, (int64_t)kMergeTile), (int64_t)region_tiles_of(val_t));
  return (int)ceil_div(n_cols, int64_t(1) << slice_log2(val_t));
}

extern "C" size_t fs_spmv_gather_plan_bytes(int val_t, int64_t n_rows, int64_t n_cols, int64_t nnz) {
  int64_t regions = 0;
  const int ns = fs_spmv_gather_slices(val_t, n_rows, n_cols, nnz, &regions);
  return ns == 0 ? 0 : 4 * (size_t)ns * (size_t)(regions + ceil_div(regions, (int64_t)kWgScanTiles));
}

extern "C" int fs_spmv_gather_count(int val_t, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                                    const void* cols, const void* part_dev, int32_t* quads, int32_t* touched,
                                    uint32_t* totals, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!valid_types(val_t, idx_t, FS_I32)) return fail(FS_E_INVALID, "fs_spmv_gather_count: bad type code");
  int64_t regions = 0;
  const int ns = fs_spmv_gather_slices(val_t, n_rows, n_cols, nnz, &regions);
  if (ns == 0) return fail(FS_E_INVALID, "fs_spmv_gather_count: sizes not supported");
  if (!cols || !part_dev || !quads || !touched || !totals) return fail(FS_E_INVALID, "fs_spmv_gather_count: null pointer");
  if (!ws || ws_bytes < fs_spmv_gather_plan_bytes(val_t, n_rows, n_cols, nnz))
    return fail(FS_E_WORKSPACE, "fs_spmv_gather_count: workspace too small");
  uint32_t* cnt = static_cast<uint32_t*>(ws);
  uint32_t* partial = cnt + (size_t)ns * regions;
  const int64_t* part = static_cast<const int64_t*>(part_dev);
  const int64_t total = n_rows + nnz, n_tiles = ceil_div(total, (int64_t)kMergeTile);
  const int T = region_tiles_of(val_t), log2w = slice_log2(val_t);
  if (idx_t == FS_I64)
    hipLaunchKernelGGL((gather_count_kernel<int64_t>), dim3((unsigned)regions), dim3(256), 0, stream,
                       static_cast<const int64_t*>(cols), part, T, n_tiles, total, log2w, ns, cnt, quads, touched);
  else
    hipLaunchKernelGGL((gather_count_kernel<int32_t>), dim3((unsigned)regions), dim3(256), 0, stream,
                       static_cast<const int32_t*>(cols), part, T, n_tiles, total, log2w, ns, cnt, quads, touched);
  FS_CHECK_LAUNCH("gather_count_kernel");
  const int64_t blocks = ceil_div(regions, (int64_t)kWgScanTiles);
  hipLaunchKernelGGL(wg_scan_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, cnt, regions, ns, partial);
  FS_CHECK_LAUNCH("wg_scan_reduce_kernel");
  hipLaunchKernelGGL(wg_scan_column_kernel, dim3((unsigned)ns), dim3(256), 0, stream, partial, blocks, ns, totals);
  FS_CHECK_LAUNCH("wg_scan_column_kernel");
  hipLaunchKernelGGL(wg_scan_down_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, cnt, regions, ns, partial,
                     totals);
  FS_CHECK_LAUNCH("wg_scan_down_kernel");
  return FS_OK;
}

extern "C" int fs_spmv_gather_fill(int val_t, int idx_t, int64_t n_rows, int64_t n_cols, int64_t nnz,
                                   const void* cols, const void* part_dev, const void* ws, const int32_t* region_q,
                                   void* pos, void* idx, void* place, hipStream_t stream) {
  if (!valid_types(val_t, idx_t, FS_I32)) return fail(FS_E_INVALID, "fs_spmv_gather_fill: bad type code");
  int64_t regions = 0;
  const int ns = fs_spmv_gather_slices(val_t, n_rows, n_cols, nnz, &regions);
  if (ns == 0) return fail(FS_E_INVALID, "fs_spmv_gather_fill: sizes not supported");
  if (!cols || !part_dev || !ws || !region_q || !pos || !idx || !place)
    return fail(FS_E_INVALID, "fs_spmv_gather_fill: null pointer");
  const int64_t* part = static_cast<const int64_t*>(part_dev);
  const int64_t total = n_rows + nnz, n_tiles = ceil_div(total, (int64_t)kMergeTile);
  const int T = region_tiles_of(val_t), log2w = slice_log2(val_t);
  const uint32_t* start = static_cast<const uint32_t*>(ws);
  if (idx_t == FS_I64)
    hipLaunchKernelGGL((gather_fill_kernel<int64_t>), dim3((unsigned)regions), dim3(256), 0, stream,
                       static_cast<const int64_t*>(cols), part, T, n_tiles, total, log2w, ns, start, region_q,
                       static_cast<uint16_t*>(pos), static_cast<uint2*>(idx), static_cast<uint32_t*>(place));
  else
    hipLaunchKernelGGL((gather_fill_kernel<int32_t>), dim3((unsigned)regions), dim3(256), 0, stream,
                       static_cast<const int32_t*>(cols), part, T, n_tiles, total, log2w, ns, start, region_q,
                       static_cast<uint16_t*>(pos), static_cast<uint2*>(idx), static_cast<uint32_t*>(place));
  FS_CHECK_LAUNCH("gather_fill_kernel");
  return FS_OK;
}

extern "C" size_t fs_spmv_gather_workspace_bytes(int val_t, int64_t n_rows, int64_t nnz, int64_t n_quads) {
  if (val_t < FS_F32 || val_t >= FS_C128) return 0;
  const int64_t n_tiles = ceil_div(n_rows + nnz, (int64_t)kMergeTile);
  return (size_t)n_quads * 4 * gather_val_bytes(val_t) + 2 * (size_t)n_tiles * gather_acc_bytes(val_t);
}

extern "C" int fs_spmv_csr_gather(int val_t, int ptr_t, int64_t n_rows, int64_t n_cols, int64_t nnz, const void* vals,
                                  const void* indptr, const void* x, void* y, const void* part_dev, const void* pos,
                                  const void* idx, const void* place, const void* slice_q, const void* region_q,
                                  int64_t n_quads, int64_t max_region_quads, void* ws, size_t ws_bytes,
                                  hipStream_t stream) {
  if (!valid_types(val_t, FS_I32, ptr_t)) return fail(FS_E_INVALID, "fs_spmv_csr_gather: bad type code");
  if (!gather_sizes_ok(val_t, n_rows, n_cols, nnz) || n_quads <= 0 || n_quads >= (int64_t(1) << 31) ||
      max_region_quads <= 0 || (size_t)max_region_quads * 4 * gather_val_bytes(val_t) > (96u << 10))
    return fail(FS_E_INVALID, "fs_spmv_csr_gather: sizes not supported");
  if (!vals || !indptr || !x || !y || !part_dev || !pos || !idx || !place || !slice_q || !region_q)
    return fail(FS_E_INVALID, "fs_spmv_csr_gather: null pointer");
  if (!ws || ws_bytes < fs_spmv_gather_workspace_bytes(val_t, n_rows, nnz, n_quads))
    return fail(FS_E_WORKSPACE, "fs_spmv_csr_gather: workspace too small");
  auto go = [&](auto vtag, auto ptag) {
    using V = decltype(vtag);
    using P = decltype(ptag);
    return launch_gather_spmv<V, P>(val_t, n_rows, n_cols, nnz, vals, indptr, x, y,
                                    static_cast<const int64_t*>(part_dev), static_cast<const uint16_t*>(pos),
                                    static_cast<const uint2*>(idx), static_cast<const uint32_t*>(place),
                                    static_cast<const uint32_t*>(slice_q), static_cast<const int32_t*>(region_q),
                                    n_quads, max_region_quads, static_cast<char*>(ws), stream);
  };
  auto by_ptr = [&](auto vtag) { return ptr_t == FS_I64 ? go(vtag, int64_t{}) : go(vtag, int32_t{}); };
  switch (val_t) {
    case FS_F32: return by_ptr(float{});
    case FS_F64: return by_ptr(double{});
    default: return by_ptr(c32{});
  }
}
