"""COO SpMM C = A @ B on the HIP kernels (reference: sparse_operations/spmm_coo.py).

The reference coalesces duplicate (row, col) entries, lex-sorts them and
runs a row-run Triton kernel (complex dtypes through an atomic kernel),
spmm_coo.py:101-142, 417-595.  Here one device radix sort by row
(``fs_coo_to_csr_by_row``, stable) turns the COO into the
CSR the SpMM kernels walk; duplicates stay separate entries of the same
row, which is the same product up to rounding (the sum distributes), and
the merge-path SpMM kernel accumulates them in a fixed order (no atomics,
bit-reproducible).

Signature, argument checks and messages follow
``flagsparse_spmm_coo`` / ``_prepare_spmm_coo_inputs`` / ``_run_spmm_coo_route``
(spmm_coo.py:335-395, 597-724).  Compute precision: float16 / bfloat16 in
float32, float32 in float64, complex64 in complex128 components, as the
reference's compute-dtype rule (spmm_coo.py:11-18).
"""

import time

import torch

from . import _lib
from ._common import _INDEX_LIMIT_INT32, SUPPORTED_INDEX_DTYPES
from ._csr import CsrPlan
from .coo import coo_to_csr_for_spmv
from .spmm_csr import SUPPORTED_SPMM_VALUE_DTYPES, _hip_spmm, _SpmmPlan
from .spmv_csr import _oneshot_flags


def _prepare_spmm_coo_inputs(data, row, col, B, shape):
    """spmm_coo.py:335-394 (checks in the same order, same messages)."""
    if len(shape) != 2:
        raise ValueError("shape must be a 2-tuple: (n_rows, n_cols)")
    if data.ndim != 1 or row.ndim != 1 or col.ndim != 1:
        raise ValueError("data, row, and col must be 1D tensors")
    if B.ndim != 2:
        raise ValueError("B must be a 2D dense tensor")
    n_rows, n_cols = int(shape[0]), int(shape[1])
    if n_rows < 0 or n_cols < 0:
        raise ValueError("shape dimensions must be non-negative")
    if data.numel() != row.numel() or data.numel() != col.numel():
        raise ValueError("data, row, and col must have the same length (nnz)")
    if B.shape[0] != n_cols:
        raise ValueError(f"B.shape[0] must be n_cols={n_cols}, got {B.shape[0]}")
    if not all(t.is_cuda for t in (data, row, col, B)):
        raise ValueError("data, row, col, and B must be CUDA tensors")
    if not all(t.device == data.device for t in (row, col, B)):
        raise ValueError("data, row, col, and B must be on the same CUDA device")
    if data.dtype not in SUPPORTED_SPMM_VALUE_DTYPES:
        raise TypeError("data dtype must be one of: float16, bfloat16, float32, float64, complex64, complex128")
    if B.dtype != data.dtype:
        raise TypeError("B dtype must match data dtype")
    if row.dtype not in SUPPORTED_INDEX_DTYPES:
        raise TypeError("row dtype must be torch.int32 or torch.int64")
    if col.dtype not in SUPPORTED_INDEX_DTYPES:
        raise TypeError("col dtype must be torch.int32 or torch.int64")
    nnz = data.numel()
    if nnz > _INDEX_LIMIT_INT32:
        # same limit and message as the reference's COO kernel contract
        raise ValueError("nnz exceeds the int32 range supported by the Triton COO kernel")
    if nnz > 0 and max(n_rows, n_cols) <= _INDEX_LIMIT_INT32:
        idx_dtype = torch.promote_types(row.dtype, col.dtype)
        row, col = row.to(idx_dtype).contiguous(), col.to(idx_dtype).contiguous()
        flags = _oneshot_flags()
        _lib.check(
            _lib.lib().fs_coo_check_ranges(_lib.index_code(idx_dtype), n_rows, n_cols, nnz, _lib.ptr(row), _lib.ptr(col),
                                           flags.data_ptr(), _lib.stream_handle(data.device)),
            "fs_coo_check_ranges",
        )
        bad_row, bad_col = flags.tolist()[:2]
        if bad_row:
            raise IndexError("row indices out of range for n_rows")
        if bad_col:
            raise IndexError("col indices out of range for n_cols")
    elif nnz > 0:
        lo_hi = torch.stack(
            [row.min().to(torch.int64), row.max().to(torch.int64), col.min().to(torch.int64), col.max().to(torch.int64)]
        ).cpu().tolist()
        min_row, max_row, min_col, max_col = (int(v) for v in lo_hi)
        if min_row < 0 or max_row >= n_rows:
            raise IndexError("row indices out of range for n_rows")
        if min_col < 0 or max_col >= n_cols:
            raise IndexError("col indices out of range for n_cols")
        if max_row > _INDEX_LIMIT_INT32:
            raise ValueError("row indices exceed the int32 range supported by the Triton kernel")
        if max_col > _INDEX_LIMIT_INT32:
            raise ValueError("column indices exceed the int32 range supported by the Triton kernel")
    return data.contiguous(), row.contiguous(), col.contiguous(), B.contiguous(), n_rows, n_cols, int(B.shape[1])


def _check_out(out, device, n_rows, n_dense, dtype):
    """spmm_coo.py:619-625."""
    if not out.is_cuda:
        raise ValueError("out must be a CUDA tensor")
    if out.device != device:
        raise ValueError("out must be on the same CUDA device as the inputs")
    if out.shape != (n_rows, n_dense) or out.dtype != dtype:
        raise ValueError("out shape/dtype must match result")


def _rows_together(data, row, col, shape):
    """CSR of valid COO entries, each row's in their input order: the product
    needs rows, not sorted columns, so the sort's column passes are left out
    (two passes instead of four for 2^19 rows and columns) where the type and
    sizes allow."""
    n_rows, n_cols = shape
    nnz = data.numel()
    if nnz == 0 or data.dtype == torch.complex128 or max(shape) > _INDEX_LIMIT_INT32:
        return coo_to_csr_for_spmv(data, row, col, shape)
    lib = _lib.lib()
    out_data, out_cols = torch.empty_like(data), torch.empty(nnz, dtype=torch.int32, device=data.device)
    indptr = torch.empty(n_rows + 1, dtype=torch.int64, device=data.device)
    idx_dtype = torch.promote_types(row.dtype, col.dtype)
    row, col = row.to(idx_dtype), col.to(idx_dtype)
    ws = _lib.workspace(lib.fs_coo_to_csr_workspace_bytes(n_rows, n_cols, nnz), data.device)
    rc = lib.fs_coo_to_csr_by_row(
        _lib.value_code(data.dtype), _lib.index_code(idx_dtype), n_rows, n_cols, nnz, _lib.ptr(data), _lib.ptr(row),
        _lib.ptr(col), _lib.ptr(out_data), _lib.ptr(out_cols), _lib.ptr(indptr), _lib.ptr(ws), ws.numel(),
        _lib.stream_handle(data.device))
    if rc == _lib.FS_E_INVALID:  # a size the workgroup passes do not take
        return coo_to_csr_for_spmv(data, row, col, shape)
    _lib.check(rc, "fs_coo_to_csr_by_row")
    return out_data, out_cols, indptr


def flagsparse_spmm_coo(data, row, col, B, shape, block_n=None, block_nnz=256, out=None, return_time=False):
    """COO SpMM: C = A @ B (spmm_coo.py:696-723).  No op argument, like the
    reference.  Returns C, or (C, ms) with return_time."""
    if block_n is not None and block_n <= 0:
        raise ValueError("block_n must be positive when provided")
    if block_nnz is not None and block_nnz <= 0:
        raise ValueError("block_nnz must be positive when provided")
    data, row, col, B, n_rows, n_cols, n_dense = _prepare_spmm_coo_inputs(data, row, col, B, shape)
    if out is not None:
        _check_out(out, data.device, n_rows, n_dense, data.dtype)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    # float16 / bfloat16 values are sorted as float32, which holds them exactly
    half = data.dtype in (torch.float16, torch.bfloat16)
    d, c32, indptr = _rows_together(data.to(torch.float32) if half else data, row, col, (n_rows, n_cols))
    if half:
        d = d.to(data.dtype)
    plan = None
    if n_rows > 0:
        plan = _SpmmPlan(d, c32, indptr, n_rows, n_cols, csr=CsrPlan.from_sizes(d, c32, indptr, n_rows, n_cols))
    C = _hip_spmm(d, c32, indptr, B, n_rows, plan, data.dtype)
    torch.cuda.synchronize()
    elapsed_ms = (time.perf_counter() - t0) * 1000.0
    if out is not None:
        out.copy_(C)
        C = out
    if return_time:
        return C, elapsed_ms
    return C


__all__ = ["flagsparse_spmm_coo"]
