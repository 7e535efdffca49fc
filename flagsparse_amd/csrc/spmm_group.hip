// spmm_group.hip — CSR SpMM (C = A B) for gfx950: the lane-group kernel
// and the C-ABI entry points.
//
// Replaces the reference's base SpMM (spmm_csr.py:2684-2789 with
// _spmm_csr_real_kernel / _spmm_csr_complex_kernel, spmm_csr.py:134-237,
// whose B / C strides, spmm_csr.py:134-176, this kernel takes too) and the
// bucketed opt kernels (spmm_csr.py:2792-3109, spmm_csr_opt_alg2.py:438-729).
#include "fs_common.hpp"
#include "spmm_group.hpp"

#include <algorithm>
#include <cstdlib>
#include <string>
#include <type_traits>

namespace fs {

constexpr int kMergeTileItems = 512;  // tile of the merge-path kernel in spmm.hip

int spmm_half_dispatch(int lpr, const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                       const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm, int64_t scn, int64_t n_dense,
                       const int64_t* part, int sub_items, int64_t n_sub, void* ws, hipStream_t stream);

int spmm_merge_dispatch(const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                        const void* B, int64_t ldb, void* C, int64_t ldc, int64_t n_dense, const int64_t* part,
                        int64_t n_tiles, void* ws, hipStream_t stream);

// C = 0 for a matrix without entries (any strides).
template <class V>
__global__ __launch_bounds__(256) void spmm_zero_kernel(V* __restrict__ C, int64_t scm, int64_t scn, int64_t n_rows,
                                                        int64_t n_dense) {
  const int64_t total = n_rows * n_dense;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / n_dense, c = i - r * n_dense;
    C[r * scm + c * scn] = V{};
  }
}

// Lanes per group for a dense width: twice the lanes whose 16-byte slices
// cover n_dense, at least 16 and at most 64 (wider B runs several column
// tiles of 64 lanes).  The idle upper half of a group re-reads its first
// slice, which shares the row's cache lines; fewer groups per wave walk
// fewer sub-tiles side by side.  Measured on MI355X (kernel ms, lanes per
// group 16 / 32): 1M x 1M with 32 uniform columns per row, f32, N = 64:
// 1.32 / 1.26; R-MAT 2^21 complex64 N = 32: 1.55 / 1.39.
// FLAGSPARSE_SPMM_LPR forces a width (8, 16, 32 or 64).
inline int spmm_value_bytes(int val_t) {
  const int esz[] = {4, 8, 8, 16, 2, 2};
  return esz[val_t];
}
inline bool spmm_half(int val_t) { return val_t == FS_F16 || val_t == FS_BF16; }
inline int group_lpr(int val_t, int64_t n_dense) {
  const int epl = spmm_half(val_t) && half_narrow(n_dense) ? 4 : 16 / spmm_value_bytes(val_t);
  int need = 1;
  while (need < 64 && (int64_t)need * epl < n_dense) need <<= 1;
  // (16-bit values: no idle half, it would double the VALU work that bounds
  // them; bfloat16 N = 128, 16 / 32 lanes: 250,007 rows of 24 245 / 267 us,
  // R-MAT 2^19 429 / 485, 1 M uniform rows of 32 1305 / 1258)
  int lpr = std::min(64, std::max(16, spmm_half(val_t) ? need : 2 * need));
  if (const char* e = std::getenv("FLAGSPARSE_SPMM_LPR")) {
    const int v = std::atoi(e);
    if ((v == 8 && !spmm_half(val_t)) || v == 16 || v == 32 || v == 64) lpr = v;
  }
  return lpr;
}

// Items per sub-tile: a wave covers kGroupWaveItems items whatever its
// group count (FLAGSPARSE_SPMM_WAVE_ITEMS overrides, 256..16384).
constexpr int kGroupWaveItems = 2048;
constexpr int64_t kGroupSkewNnz = 1 << 20;  // from here on a caller may find skewed columns (merge kernel, 512 items)
inline int group_sub_items(int val_t, int64_t n_dense) {
  int wave_items = kGroupWaveItems;
  if (const char* e = std::getenv("FLAGSPARSE_SPMM_WAVE_ITEMS")) {
    const int v = std::atoi(e);
    if (v >= 256 && v <= 16384) wave_items = v;
  }
  return wave_items * group_lpr(val_t, n_dense) / 64;
}

// Kernel choice.  The lane-group kernel is the default.  For B rows of at
// least 512 bytes on matrices with skewed columns (the caller sets
// plan->spmm_wg_cap when a few columns hold much of the matrix) the
// merge-path kernel wins: two columns per lane in XCD-affine column tiles
// under a residency cap keep more hot B rows in L2.  Kernel ms, merge /
// lane-group, R-MAT 2^20: f32 N = 128 1.27 / 1.37, N = 256 2.50 / 3.14;
// complex64 N = 64 1.26 / 1.38, N = 128 2.66 / 3.15; on uniform columns
// the lane-group kernel ties or wins (complex64 N = 128: 6.63 / 5.85).
// Both kernels use 512-item tiles for such rows, so the partition does not
// depend on the choice; the merge kernel reads row-major B / C only.
// FLAGSPARSE_SPMM_KERNEL=merge|group forces one.
inline int forced_kernel() {  // 0 none, 1 merge, 2 group
  const char* e = std::getenv("FLAGSPARSE_SPMM_KERNEL");
  if (!e) return 0;
  if (std::string(e) == "merge") return 1;
  if (std::string(e) == "group") return 2;
  return 0;
}
inline bool wide_rows(int val_t, int64_t n_dense) {
  return n_dense * spmm_value_bytes(val_t) >= 512 && !spmm_half(val_t);
}
inline int spmm_tile_items_for(int val_t, int64_t n_dense) {
  const int f = spmm_half(val_t) ? 2 : forced_kernel();  // 16-bit values: the lane-group kernel always
  if (f == 1 || (f == 0 && wide_rows(val_t, n_dense))) return kMergeTileItems;
  return group_sub_items(val_t, n_dense);
}

// Items per sub-tile for a matrix of this size: the size above, halved while
// the matrix gives fewer waves than fill the chip (a group walks its sub-tile
// one entry after another, so a small matrix in 2048-item waves is a serial
// chain on a few CUs), down to 128 items per wave.  Measured (us per prepared
// call, 2048 items always / at least 1024 / 2048 / 4096 / 8192 waves): 2000
// rows of 9, f32, N = 17: 106 / 24 / 20 / 21 / 21; 100,000 of 16, f32, N = 8:
// 75 / 45 / 37 / 39 / 50, N = 64 118 / 69 / 85 / 75 / 75; 300,000 of 20, f32,
// N = 32: 128 / 128 / 128 / 137 / 149, f64, N = 32: 295 / 295 / 295 / 280 /
// 253.  Smaller sub-tiles cost row fragments, more for narrow B rows: at least
// 2048 waves there, 4096 with 32 lanes or more per row.  With 32 lanes, whole
// slices and short rows, 2048 to 3072 waves stay as they are: they run at once
// (3 a SIMD), and half the size would be a round and a third of them.  us, as
// they are / halved: 600,000 rows of 6, 2049 waves, f32 N = 64 166 / 191, f64 N =
// 32 160 / 188; 400,009 of 10 174 / 186, 175 / 183; 100,000 of 10 (512 items)
// 49 / 53, 48 / 52; but 600,000 of 10 (3221 waves) 350 / 293, 44,000 of 50 c128
// N = 16 99 / 86, and at N = 33 (element loads) 400,009 of 10 289 / 242.
// With fewer lanes and longer rows 1792 waves are enough: they are nearly two on
// every SIMD, and halved a round and a half.  us, 2048 waves at least / 1792: rows
// of 100, 4 M entries f64 N = 16 73 / 67, N = 3 80 / 78, 2 M 42 / 39, 1 M 35 / 24;
// rows of 1000, 4 M f64 N = 16 80 / 71, f32 N = 32 78 / 72; banded rows of 125, 4 M
// 87 / 78, 89 / 77.  Not with short rows (500,000 of 6, 1709 waves, f64 N = 16 77
// halved, 94 not; banded rows of 9 60 / 83) nor on 16-bit values (rows of 30, N =
// 16 62 / 78), and not with 32 lanes, where halving costs 5% on random columns
// (rows of 100, 4 M, f32 N = 64 138 / 134) but gains 20% on banded ones (127 / 152).
constexpr int kGroupMinWaveItems = 128;
constexpr int64_t kGroupSlots = 3072;
inline int spmm_tile_items_sized(int val_t, int64_t n_dense, int64_t n_rows, int64_t nnz) {
  const int base = spmm_tile_items_for(val_t, n_dense);
  if (forced_kernel() != 0 || std::getenv("FLAGSPARSE_SPMM_WAVE_ITEMS")) return base;
  if (wide_rows(val_t, n_dense) && nnz >= kGroupSkewNnz) return base;
  const int lpr = group_lpr(val_t, n_dense);
  const int bytes = spmm_value_bytes(val_t);
  const bool half = spmm_half(val_t), short_rows = nnz / (bytes == 16 ? 12 : 24) <= n_rows;
  const int64_t fill = lpr >= 32 ? 4096 : half || short_rows ? 2048 : 1792;
  const bool one_round = lpr == 32 && !half && short_rows && n_dense % (16 / bytes) == 0;
  int wave_items = base * 64 / lpr;
  for (; wave_items > kGroupMinWaveItems; wave_items >>= 1) {
    const int64_t waves = ceil_div(n_rows + nnz, (int64_t)wave_items);
    if (waves >= fill || (one_round && waves >= 2048 && waves <= kGroupSlots)) break;
  }
  return wave_items * lpr / 64;
}

template <class V, class T>
int launch_spmm_group_lpr_t(int lpr, const fs_csr_plan* plan, const void* vals, const void* cols,
                            const void* indptr, const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm,
                            int64_t scn, int64_t n_dense, const int64_t* part, int sub_items, int64_t n_sub,
                            void* ws, hipStream_t s) {
  switch (lpr) {
    case 8: return launch_spmm_group<V, 8, T>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
    case 16: return launch_spmm_group<V, 16, T>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
    case 32: return launch_spmm_group<V, 32, T>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
    case 64: return launch_spmm_group<V, 64, T>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
  }
  return fail(FS_E_INVALID, "fs_spmm_csr: unsupported lane-group width");
}

// native = 1: float32 / complex64 accumulate in their own precision (VN);
// otherwise, and always for float64 / complex128, in VT's.
template <class V>
int launch_spmm_group_lpr(int lpr, int native, const fs_csr_plan* plan, const void* vals, const void* cols,
                          const void* indptr, const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm,
                          int64_t scn, int64_t n_dense, const int64_t* part, int sub_items, int64_t n_sub,
                          void* ws, hipStream_t s) {
  if constexpr (std::is_same_v<V, float> || std::is_same_v<V, c32>) {
    if (native)
      return launch_spmm_group_lpr_t<V, VN<V>>(lpr, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense,
                                               part, sub_items, n_sub, ws, s);
  }
  return launch_spmm_group_lpr_t<V, VT<V>>(lpr, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part,
                                           sub_items, n_sub, ws, s);
}

}  // namespace fs

using namespace fs;

extern "C" int fs_spmm_tile_items(int val_t, int64_t n_dense) {
  if (val_t < FS_F32 || val_t > FS_BF16) return kMergeTileItems;
  return spmm_tile_items_for(val_t, n_dense);
}

extern "C" int fs_spmm_tile_items_sized(int val_t, int64_t n_dense, int64_t n_rows, int64_t nnz) {
  if (val_t < FS_F32 || val_t > FS_BF16) return kMergeTileItems;
  return spmm_tile_items_sized(val_t, n_dense, n_rows, nnz);
}

extern "C" size_t fs_spmm_workspace_bytes(int val_t, int64_t n_tiles, int64_t n_dense) {
  const size_t acc = (val_t == FS_C64 || val_t == FS_C128) ? sizeof(c64) : sizeof(double);
  return (size_t)n_tiles * (size_t)n_dense * 2 * acc;
}

extern "C" int fs_spmm_csr_strided(const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                                   const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm, int64_t scn,
                                   int64_t n_dense, const void* part_dev, int tile_items, int64_t n_tiles, void* ws,
                                   size_t ws_bytes, hipStream_t stream) {
  if (!plan) return fail(FS_E_INVALID, "fs_spmm_csr: plan is null");
  const bool half = spmm_half(plan->val_t);
  if (!valid_types(half ? FS_F32 : plan->val_t, plan->idx_t, plan->ptr_t))
    return fail(FS_E_INVALID, "fs_spmm_csr: bad type code");
  if (n_dense < 0 || sbk < 0 || sbn < 0 || scm < 0 || scn < 0) return fail(FS_E_INVALID, "fs_spmm_csr: negative size");
  if (plan->n_rows == 0 || n_dense == 0) return FS_OK;
  const int forced = half ? 2 : forced_kernel();
  const bool merge = forced == 1 || (forced == 0 && wide_rows(plan->val_t, n_dense) && plan->spmm_wg_cap > 0);
  const bool group = !merge || sbn != 1 || scn != 1;
  if (tile_items != fs_spmm_tile_items(plan->val_t, n_dense) &&
      (!group || tile_items != spmm_tile_items_sized(plan->val_t, n_dense, plan->n_rows, plan->nnz)))
    return fail(FS_E_INVALID, "fs_spmm_csr: tile_items must come from fs_spmm_tile_items");
  if (n_tiles != ceil_div(plan->n_rows + plan->nnz, tile_items))
    return fail(FS_E_INVALID, "fs_spmm_csr: n_tiles does not match the matrix");
  // C must not overlap itself: distinct (row, column) pairs map to distinct elements.
  const bool c_rowmajor = scn == 1 && scm >= n_dense;
  const bool c_colmajor = scm == 1 && scn >= plan->n_rows;
  if (!(c_rowmajor || c_colmajor) && !(n_dense == 1 && scm >= 1) && !(plan->n_rows == 1 && scn >= 1))
    return fail(FS_E_INVALID, "fs_spmm_csr: C strides overlap (leading dimension smaller than the other extent)");
  if (!indptr || !C || !part_dev || (plan->nnz > 0 && (!vals || !cols || !B)))
    return fail(FS_E_INVALID, "fs_spmm_csr: null pointer");
  if (ws_bytes < fs_spmm_workspace_bytes(plan->val_t, n_tiles, n_dense) || (!ws && n_tiles > 0))
    return fail(FS_E_WORKSPACE, "fs_spmm_csr: workspace too small");
  const int64_t* part = static_cast<const int64_t*>(part_dev);
  if (half)
    return spmm_half_dispatch(group_lpr(plan->val_t, n_dense), plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn,
                              n_dense, part, tile_items, n_tiles, ws, stream);
  if (plan->nnz == 0) {
    const int64_t blocks = std::min<int64_t>(ceil_div(plan->n_rows * n_dense, 256), 65536);
    switch (plan->val_t) {
      case FS_F32: hipLaunchKernelGGL(spmm_zero_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, stream, static_cast<float*>(C), scm, scn, plan->n_rows, n_dense); break;
      case FS_F64: hipLaunchKernelGGL(spmm_zero_kernel<double>, dim3((unsigned)blocks), dim3(256), 0, stream, static_cast<double*>(C), scm, scn, plan->n_rows, n_dense); break;
      case FS_C64: hipLaunchKernelGGL(spmm_zero_kernel<c32>, dim3((unsigned)blocks), dim3(256), 0, stream, static_cast<c32*>(C), scm, scn, plan->n_rows, n_dense); break;
      default: hipLaunchKernelGGL(spmm_zero_kernel<c64>, dim3((unsigned)blocks), dim3(256), 0, stream, static_cast<c64*>(C), scm, scn, plan->n_rows, n_dense); break;
    }
    FS_CHECK_LAUNCH("spmm_zero_kernel");
    return FS_OK;
  }
  if (group) {
    const int lpr = group_lpr(plan->val_t, n_dense);
    int native = 0;
    if (const char* e = std::getenv("FLAGSPARSE_SPMM_ACC")) native = std::string(e) == "native";
    switch (plan->val_t) {
      case FS_F32: return launch_spmm_group_lpr<float>(lpr, native, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, tile_items, n_tiles, ws, stream);
      case FS_F64: return launch_spmm_group_lpr<double>(lpr, native, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, tile_items, n_tiles, ws, stream);
      case FS_C64: return launch_spmm_group_lpr<c32>(lpr, native, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, tile_items, n_tiles, ws, stream);
      default: return launch_spmm_group_lpr<c64>(lpr, native, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, tile_items, n_tiles, ws, stream);
    }
  }
  // Merge-path kernel (FLAGSPARSE_SPMM_KERNEL=merge): row-major B / C only.
  if (sbn != 1 || scn != 1) return fail(FS_E_INVALID, "fs_spmm_csr: the merge kernel takes row-major B and C only");
  if (scm < n_dense || (plan->n_cols > 0 && sbk < n_dense))
    return fail(FS_E_INVALID, "fs_spmm_csr: leading dimension smaller than n_dense");
  return spmm_merge_dispatch(plan, vals, cols, indptr, B, sbk, C, scm, n_dense, part, n_tiles, ws, stream);
}

extern "C" int fs_spmm_csr(const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                           const void* B, int64_t ldb, void* C, int64_t ldc, int64_t n_dense,
                           const void* part_dev, int tile_items, int64_t n_tiles, void* ws, size_t ws_bytes,
                           hipStream_t stream) {
  if (plan && plan->n_rows > 0 && n_dense > 0 && (ldc < n_dense || (plan->n_cols > 0 && ldb < n_dense)))
    return fail(FS_E_INVALID, "fs_spmm_csr: leading dimension smaller than n_dense");
  return fs_spmm_csr_strided(plan, vals, cols, indptr, B, ldb, 1, C, ldc, 1, n_dense, part_dev, tile_items, n_tiles,
                             ws, ws_bytes, stream);
}
