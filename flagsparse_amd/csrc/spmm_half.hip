// spmm_half.hip — the lane-group SpMM on float16 / bfloat16 as they are.
//
// The reference computes 16-bit products in wider precision and rounds once
// (spmm_csr.py:2716-2719); so does this: values and B rows are read in 16
// bits, widened in registers, accumulated in float64, and a result is rounded
// to float32 and then to 16 bits, the same bits as converting A and B to
// float32, multiplying and converting back, which cost three passes over
// memory and gathered B rows twice as wide.  us per prepared call, converted and
// now, bfloat16: 250,007 rows of 24, N = 16 / 64 / 128 / 256: 125 / 274 / 526 /
// 1053 and 102 / 122 / 244 / 472; R-MAT 2^19, N = 64 456 and 255; 1 M uniform
// rows of 32, N = 128 2618 and 1297 (bound by the gathers of 256-byte rows, as
// float32 at N = 64).
#include "spmm_group.hpp"

namespace fs {

struct h16 {
  _Float16 v;
};
struct b16 {
  uint16_t bits;
};
static_assert(sizeof(h16) == 2 && sizeof(b16) == 2, "16-bit values");

template <>
struct VT<h16> {
  using acc = double;
  static constexpr bool complex = false;
  __device__ static acc zero() { return 0.0; }
  __device__ static float widen(h16 a) { return (float)a.v; }
  __device__ static acc fma(float a, h16 x, acc s) { return __builtin_fma((double)a, (double)(float)x.v, s); }
  __device__ static h16 out(acc s) {
    float f = (float)s;
    asm("" : "+v"(f));  // two roundings, two instructions: folded, float64 -> float16 is a long sequence
    return h16{(_Float16)f};
  }
};
template <>
struct VT<b16> {
  using acc = double;
  static constexpr bool complex = false;
  __device__ static acc zero() { return 0.0; }
  __device__ static float widen(b16 a) { return __uint_as_float((uint32_t)a.bits << 16); }
  __device__ static acc fma(float a, b16 x, acc s) { return __builtin_fma((double)a, (double)widen(x), s); }
  __device__ static b16 out(acc s) {
    float f = (float)s;
    asm("" : "+v"(f));
    const __bf16 h = (__bf16)f;  // to nearest even, one instruction
    b16 r;
    __builtin_memcpy(&r, &h, 2);
    return r;
  }
};

// The same types with 8-byte slices, for narrow B and for widths that are not
// multiples of 8: a lane's work is its slice's elements whatever N is, and
// 16-byte slices are eight of them, widened and multiplied in float64 (VALU
// bound: N = 16 took 163 us on the matrix above where float32 takes 107).
struct h16n : h16 {};
struct b16n : b16 {};
template <>
struct group_slice<h16n> {
  static constexpr int bytes = 8;
};
template <>
struct group_slice<b16n> {
  static constexpr int bytes = 8;
};
template <>
struct VT<h16n> : VT<h16> {
  __device__ static h16n out(acc s) { return h16n{VT<h16>::out(s)}; }
};
template <>
struct VT<b16n> : VT<b16> {
  __device__ static b16n out(acc s) { return b16n{VT<b16>::out(s)}; }
};

template <class V>
int launch_half(int lpr, const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm, int64_t scn, int64_t n_dense,
                const int64_t* part, int sub_items, int64_t n_sub, void* ws, hipStream_t s) {
  switch (lpr) {
    case 16: return launch_spmm_group<V, 16, VT<V>>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
    case 32: return launch_spmm_group<V, 32, VT<V>>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
    case 64: return launch_spmm_group<V, 64, VT<V>>(plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws, s);
  }
  return fail(FS_E_INVALID, "fs_spmm_csr: unsupported lane-group width");
}

// (the entry point has checked sizes, strides and workspace; without entries
// the caller clears C)
int spmm_half_dispatch(int lpr, const fs_csr_plan* plan, const void* vals, const void* cols, const void* indptr,
                       const void* B, int64_t sbk, int64_t sbn, void* C, int64_t scm, int64_t scn, int64_t n_dense,
                       const int64_t* part, int sub_items, int64_t n_sub, void* ws, hipStream_t stream) {
  if (plan->nnz == 0) return fail(FS_E_INVALID, "fs_spmm_csr: 16-bit values need entries");
  const bool narrow = half_narrow(n_dense);
  if (plan->val_t == FS_F16 && narrow)
    return launch_half<h16n>(lpr, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub,
                             ws, stream);
  if (narrow)
    return launch_half<b16n>(lpr, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub,
                             ws, stream);
  if (plan->val_t == FS_F16)
    return launch_half<h16>(lpr, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub,
                            ws, stream);
  return launch_half<b16>(lpr, plan, vals, cols, indptr, B, sbk, sbn, C, scm, scn, n_dense, part, sub_items, n_sub, ws,
                          stream);
}

}  // namespace fs
