"""The one-launch SpMV's uneven 64-row blocks: rows on both sides of 64 and
4096 entries in one block (16 lanes, a wave, the workgroup), and 16-bit
values through the same call, against the CPU oracle."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _lib
from flagsparse_amd import synthetic as S
from oracle import csr_oracle as O
from tests._helpers import INDEX_DTYPES, INDEX_IDS, REL_TOL, VALUE_DTYPES, VALUE_IDS, np_, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENGTHS = [0, 1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 4095, 4096, 4097, 9000] + [3] * 100 + [5000, 0, 0]


def _matrix(dtype, index_dtype, lengths=LENGTHS, n_cols=20011):
    g = np.random.default_rng(3)
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    cols = torch.tensor(g.integers(0, n_cols, ptr[-1]), device=DEV).to(index_dtype)
    return S.vector(int(ptr[-1]), dtype, DEV, 4), cols, torch.tensor(ptr, device=DEV).to(index_dtype), (len(lengths), n_cols)


@pytest.mark.parametrize("index_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_row_lengths(dtype, index_dtype):
    d, i, p, sh = _matrix(dtype, index_dtype)
    x = S.vector(sh[1], dtype, DEV, 5)
    y = fs.flagsparse_spmv_csr(d, i, p, x, sh)
    assert _lib.last_kernel() == "spmv_oneshot_kernel"
    assert rel_err(np_(y), O.spmv_csr_wide(np_(d), np_(i), np_(p), np_(x), sh)) <= REL_TOL[dtype]
    assert torch.equal(torch.view_as_real(y) if y.is_complex() else y,
                       (lambda z: torch.view_as_real(z) if z.is_complex() else z)(fs.flagsparse_spmv_csr(d, i, p, x, sh)))
    i[int(p[14]) + 4500] = sh[1]  # a stray column in the longest row
    with pytest.raises(IndexError, match="out of range for n_cols"):
        fs.flagsparse_spmv_csr(d, i, p, x, sh)


@pytest.mark.parametrize("op", ["non", "trans", "conj"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_half_values(dtype, op):
    d, i, p, sh = _matrix(torch.float32, torch.int32, [7, 0, 70, 300, 2] * 40, 900)
    d = d.to(dtype)
    x = S.vector(sh[1] if op == "non" else sh[0], torch.float32, DEV, 5).to(dtype)
    y = fs.flagsparse_spmv_csr(d, i, p, x, sh, op=op)
    assert y.dtype == dtype
    want = fs.flagsparse_spmv_csr(d.float(), i, p, x.float(), sh, op=op).to(dtype)
    assert torch.equal(y, want)
    with pytest.raises(TypeError, match="x dtype must match"):
        fs.flagsparse_spmv_csr(d, i, p, x.float(), sh, op=op)


@pytest.mark.parametrize("length", [1024, 2048, 4096])
@pytest.mark.parametrize("dtype", [torch.float64, torch.complex128], ids=["f64", "c128"])
def test_rows_of_a_wave_sum_in_256_chains(dtype, length):
    """1 + (length - 1) 2^-54: a chain that starts with the 1 loses each of its
    later terms, and the other chains' sums are whole multiples of 2^-52, so the
    result says how long a chain is."""
    lengths = [length] * 32 + [3] * 32
    _, i, p, sh = _matrix(torch.float64, torch.int32, lengths, 9000)
    d = torch.full((int(p[-1]),), 2.0**-54, dtype=dtype, device=DEV)
    d[p[:-1].long()] = 1.0
    y = fs.flagsparse_spmv_csr(d, i, p, torch.ones(9000, dtype=dtype, device=DEV), sh)
    assert _lib.last_kernel() == "spmv_oneshot_kernel"
    lost = (length - 1) * 2.0**-54 - (np_(y)[:32].real - 1.0)
    assert np.all(np.abs(lost) <= (length // 256 - 1) * 2.0**-54)


@pytest.mark.parametrize("rows,per_row,one_launch", [
    (16384, 16, True), (16384, 17, False), (4096, 64, True), (4096, 65, False), (4000, 65, False), (1, 65536, True),
    (1, 65537, False), (20, 12000, False), (1024, 64, True), (100, 655, True),
])
def test_half_values_of_long_rows_take_the_general_path(rows, per_row, one_launch):
    d, i, p, sh = _matrix(torch.float32, torch.int32, [per_row] * rows, 70001)
    d = d.bfloat16()
    x = S.vector(sh[1], torch.float32, DEV, 5).bfloat16()
    y, meta = fs.flagsparse_spmv_csr(d, i, p, x, sh, return_meta=True)
    assert (meta["kernel"] == "oneshot") == one_launch
    want = torch.from_numpy(O.spmv_csr_wide(np_(d.double()), np_(i), np_(p), np_(x.double()), sh)).float().bfloat16()
    # the same sums in another order may round to the next value
    assert bool(((y.cpu().double() - want.double()).abs() <= want.double().abs() * 2.0**-7).all())
