"""The COO SpMM's own sort and checks: entries grouped by row in input order
(fs_coo_to_csr_by_row, bit-exact with a stable argsort) and the native range
check (fs_coo_check_ranges)."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _lib
from flagsparse_amd import synthetic as S
from flagsparse_amd.spmm_coo import _rows_together
from tests._helpers import INDEX_DTYPES, INDEX_IDS, np_

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nnz", [1, 6143, 6144, 6145, 50001])
@pytest.mark.parametrize("n_rows", [1, 2, 2047, 2049, (1 << 20) + 3])
@pytest.mark.parametrize("index_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.complex64], ids=["f32", "f64", "c64"])
def test_rows_together_is_a_stable_sort(dtype, index_dtype, n_rows, nnz):
    g = torch.Generator(device=DEV)
    g.manual_seed(nnz)
    row = torch.randint(0, n_rows, (nnz,), device=DEV, generator=g).to(index_dtype)
    col = torch.randint(0, 3001, (nnz,), device=DEV, generator=g).to(index_dtype)
    data = S.vector(nnz, dtype, DEV, 3)
    d, c, p = _rows_together(data, row, col, (n_rows, 3001))
    order = np.argsort(np_(row), kind="stable")
    assert np.array_equal(np_(d), np_(data)[order])
    assert np.array_equal(np_(c), np_(col)[order].astype(np.int32))
    assert np.array_equal(np_(p), np.concatenate([[0], np.cumsum(np.bincount(np_(row), minlength=n_rows))]))


@pytest.mark.parametrize("index_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("n", [1, 5, 4097, 300001])
def test_range_check_sees_every_place(index_dtype, n, shift):
    flags = torch.zeros(4, dtype=torch.int32, pin_memory=True)

    def check(row, col):
        _lib.check(_lib.lib().fs_coo_check_ranges(_lib.index_code(index_dtype), 10, 20, n, row.data_ptr(),
                                                  col.data_ptr(), flags.data_ptr(), _lib.stream_handle(row.device)),
                   "fs_coo_check_ranges")
        return flags.tolist()[:2]

    row = torch.full((n + shift,), 9, dtype=index_dtype, device=DEV)[shift:]
    col = torch.full((n + shift,), 19, dtype=index_dtype, device=DEV)[shift:]
    assert check(row, col) == [0, 0]
    for at in sorted({0, n // 2, max(0, n - 2), n - 1}):
        for bad in (-1, 10):
            row[at] = bad
            assert check(row, col) == [1, 0]
        row[at] = 0
        col[at] = 20
        assert check(row, col) == [0, 1]
        col[at] = 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.complex128])
def test_duplicates_and_errors(dtype):
    row = torch.tensor([4, 0, 4, 4, 2, 0], device=DEV)
    col = torch.tensor([1, 1, 1, 0, 2, 0], device=DEV, dtype=torch.int32)
    data = torch.arange(1, 7, device=DEV).to(dtype)
    B = torch.arange(1, 13, device=DEV).reshape(3, 4).to(dtype)
    want = torch.zeros(5, 3, dtype=dtype, device=DEV).index_put((row, col.long()), data, accumulate=True).cpu() @ B.cpu()
    assert torch.equal(fs.flagsparse_spmm_coo(data, row, col, B, (5, 3)).cpu(), want)
    with pytest.raises(IndexError, match="row indices out of range for n_rows"):
        fs.flagsparse_spmm_coo(data, row, col + 9, B, (4, 3))
    with pytest.raises(IndexError, match="col indices out of range for n_cols"):
        fs.flagsparse_spmm_coo(data, row, col + 1, B, (5, 3))
