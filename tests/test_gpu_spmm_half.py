"""SpMM on float16 / bfloat16 as they are (spmm_half.hip): every lane width,
odd widths and strides, both index types, long rows, special values, against
64-bit sums rounded as the reference rounds (to float32, then to 16 bits)."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _lib
from flagsparse_amd import synthetic as S
from oracle import csr_oracle as O
from tests._helpers import INDEX_DTYPES, INDEX_IDS, np_

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF = [torch.float16, torch.bfloat16]


def _matrix(rows, cols, density, dtype, index_dtype, seed, **kw):
    d, i, p, sh = S.random_csr(rows, cols, density, torch.float32, index_dtype, DEV, seed=seed, **kw)
    return d.to(dtype), i, p, sh


def _check(C, d, i, p, sh, B, op="non"):
    """Within one unit in the last place of the 64-bit sum rounded the same
    way (sums whose order differs may fall on either side of a tie)."""
    wide = O.spmm_csr_wide(np_(d.double()), np_(i), np_(p), np_(B.double()), sh, op=op)
    want = torch.from_numpy(wide).float().to(C.dtype)
    ulp = 2.0 ** (-10 if C.dtype == torch.float16 else -7)
    diff = (C.cpu().double() - want.double()).abs()
    assert bool((diff <= want.double().abs() * ulp + 1e-7).all())
    assert float((diff > 0).double().mean()) < 1e-3


@pytest.mark.parametrize("n", [1, 7, 8, 9, 64, 65, 68, 100, 128, 136, 256, 258, 260, 520, 1040])
@pytest.mark.parametrize("index_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("dtype", HALF, ids=["f16", "bf16"])
def test_widths(dtype, index_dtype, n):
    d, i, p, sh = _matrix(601, 1300, 0.01, dtype, index_dtype, n, empty_row_every=9, long_rows=((5, 1250), (600, 700)))
    B = S.dense(1300, n, torch.float32, DEV, 3).to(dtype)
    C = fs.flagsparse_spmm_csr(d, i, p, B, sh)
    assert C.dtype == dtype and _lib.last_kernel() == "spmm_group_kernel"
    _check(C, d, i, p, sh, B)


@pytest.mark.parametrize("op", ["non", "trans", "conj"])
@pytest.mark.parametrize("dtype", HALF, ids=["f16", "bf16"])
def test_ops_and_layouts(dtype, op):
    d, i, p, sh = _matrix(300, 500, 0.03, dtype, torch.int32, 4)
    inner = sh[1] if op == "non" else sh[0]
    B = S.dense(inner, 48, torch.float32, DEV, 3).to(dtype)
    for Bv in (B, B.t().contiguous().t(), torch.cat([B, B], 1)[:, 3:51]):  # row-major, column-major, off 16 bytes
        _check(fs.flagsparse_spmm_csr(d, i, p, Bv, sh, op=op), d, i, p, sh, Bv, op)
    route = fs.prepare_spmm_csr_route(d, i, p, sh, op=op)
    C = fs.flagsparse_spmm_csr_run(route, B, dense_layout="col")
    assert C.stride(0) == 1 and C.dtype == dtype
    _check(C, d, i, p, sh, B, op)


# up to 64 columns in 16 bits, above through float32 (a column-major B)
@pytest.mark.parametrize("n", [1, 48, 64, 65, 128])
@pytest.mark.parametrize("dtype", HALF, ids=["f16", "bf16"])
def test_column_major_result_at_any_width(dtype, n):
    d, i, p, sh = _matrix(300, 500, 0.03, dtype, torch.int32, 4)
    B = S.dense(500, n, torch.float32, DEV, 3).to(dtype)
    route = fs.prepare_spmm_csr_route(d, i, p, sh)
    C, meta = fs.flagsparse_spmm_csr_run(route, B, dense_layout="col", return_meta=True)
    assert C.dtype == dtype and C.stride() == (1, 300) and meta["c_stride"] == (1, 300)
    if n > 1:
        assert meta["output_layout"] == "col"
    _check(C, d, i, p, sh, B)


@pytest.mark.parametrize("dtype", HALF, ids=["f16", "bf16"])
def test_stencil_keeps_its_copy(dtype):
    """A prepared stencil runs on its float32 SELL-64 copy; widths it does not
    take run in 16 bits."""
    d, i, p, sh = S.stencil27(52, torch.float32, torch.int32, DEV, seed=1)
    d = d.to(dtype)
    route = fs.prepare_spmm_csr_route(d, i, p, sh)
    for n, kernel in ((8, "spmm_sell_kernel"), (6, "spmm_group_kernel")):
        B = S.dense(sh[1], n, torch.float32, DEV, 3).to(dtype)
        C = fs.flagsparse_spmm_csr_run(route, B)
        assert _lib.last_kernel() == kernel
        want = fs.flagsparse_spmm_csr(d.float(), i, p, B.float(), sh).to(dtype)
        assert float((C != want).double().mean()) < 1e-3


@pytest.mark.parametrize("dtype", HALF, ids=["f16", "bf16"])
def test_special_values_and_rounding(dtype):
    p = torch.tensor([0, 2, 3, 4, 4, 6], dtype=torch.int32, device=DEV)
    i = torch.tensor([0, 1, 2, 0, 0, 1], dtype=torch.int32, device=DEV)
    d = torch.tensor([1, 1, 1, float("inf"), 60000.0, 60000.0], device=DEV).to(dtype)
    # 1 + 2^-9 and 1 + 3 * 2^-9 are ties of bfloat16, 2^-24 a subnormal of float16
    B = torch.tensor([[1.0, 0.0, 1.0, 1.0], [2.0**-9, 3 * 2.0**-9, 2.0**-24, 0.0], [float("nan"), -0.0, 2.0**-24, 3.0]],
                     device=DEV).to(dtype)
    C = fs.flagsparse_spmm_csr(d, i, p, B, (5, 3))
    want = torch.zeros(5, 4, dtype=torch.float64, device=DEV)
    row = torch.tensor([0, 0, 1, 2, 4, 4], device=DEV)
    for e in range(6):
        want[row[e]] += d[e].double() * B[i[e].long()].double()
    want = want.float().to(dtype)
    assert np.array_equal(np_(C.float()), np_(want.float()), equal_nan=True)


def test_empty_matrix():
    e = torch.empty(0, dtype=torch.bfloat16, device=DEV)
    p = torch.zeros(5, dtype=torch.int32, device=DEV)
    C = fs.flagsparse_spmm_csr(e, torch.empty(0, dtype=torch.int32, device=DEV), p, torch.ones(3, 4, device=DEV).bfloat16(),
                               (4, 3))
    assert C.dtype == torch.bfloat16 and not bool(C.any())
