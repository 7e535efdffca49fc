"""The unprepared A^T x / A^H x and COO SpMV by scattered products
(fs_spmv_csr_scatter, fs_spmv_coo_scatter) against the CPU oracle: tile and
segment edges, output counts from one bucket to thousands, crowded outputs,
structure errors, special values and determinism."""

import math

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _lib, spmv_coo
from flagsparse_amd import synthetic as S
from oracle import csr_oracle as O
from tests._helpers import INDEX_DTYPES, INDEX_IDS, REL_TOL, VALUE_DTYPES, VALUE_IDS, np_, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _coo(nnz, n_rows, n_cols, dtype, row_dtype, col_dtype, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    row = torch.randint(0, n_rows, (nnz,), device=DEV, generator=g).to(row_dtype)
    col = torch.randint(0, n_cols, (nnz,), device=DEV, generator=g).to(col_dtype)
    return S.vector(nnz, dtype, DEV, seed + 1), row, col


def _wide(data, row, col, x, n_out):
    """Sum in 64-bit floats on the host, real and imaginary parts apart."""
    p = np_(data).astype(np.complex128) * np_(x).astype(np.complex128)[np_(col)]
    re = np.bincount(np_(row), weights=p.real, minlength=n_out)
    return re + 1j * np.bincount(np_(row), weights=p.imag, minlength=n_out)


def _cancelling(nnz, n_out, n_x, cplx, seed):
    """Entries whose products are exact in float64 (25-bit whole values times
    powers of two; a complex x is real or imaginary) and of mixed sign, with the
    exactly rounded sums, the sums of magnitudes and the entries per output."""
    g = np.random.default_rng(seed)

    def values(n):
        return g.integers(-(2**25), 2**25, n) * 2.0 ** g.integers(-8, 9, n)

    out, src = g.integers(0, n_out, nnz), g.integers(0, n_x, nnz)
    val, x = values(nnz), values(n_x)
    if cplx:
        val = val + 1j * values(nnz)
        x = np.where(np.arange(n_x) % 2 == 0, x + 0j, 1j * x)
    terms = val * x[src]
    order = np.argsort(out, kind="stable")
    count = np.bincount(out, minlength=n_out)
    parts = []
    for t in (terms.real, terms.imag) if cplx else (terms,):
        groups = np.split(t[order], np.cumsum(count)[:-1])
        parts.append((np.array([math.fsum(p) for p in groups]), np.bincount(out, weights=np.abs(t), minlength=n_out),
                      np.bincount(out, weights=t, minlength=n_out)))
    return val, out, src, x, count, parts


@pytest.mark.parametrize("n_out", [1, 3, 64, 2500, 300007])
@pytest.mark.parametrize("dtype", [torch.float64, torch.complex128], ids=["f64", "c128"])
def test_double_sums_are_compensated(dtype, n_out):
    """Two roundings (2 u |sum|, u = 2^-53) and the rounding of the compensation
    itself (at most n terms of u times the sum of magnitudes, added with another
    n u): crowded lanes, buckets of one and of many segments.  A plain sum of the
    same terms misses the bound."""
    val, out, src, x, count, parts = _cancelling(100_003, n_out, 40, dtype.is_complex, n_out)
    args = [torch.tensor(v, device=DEV) for v in (val, out, src, x)]
    y = np_(fs.flagsparse_spmv_coo(*args, (n_out, 40)))
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    missed = False
    for got, (ref, mag, plain) in zip((y.real, y.imag), parts):
        bound = 2.0**-52 * np.abs(ref) + (count * 2.0**-53) ** 2 * mag
        assert np.all(np.abs(got - ref) <= bound)
        missed |= bool(np.any(np.abs(plain - ref) > bound))
    assert missed or n_out > 2500  # (most outputs of 300,007 are one product)


# one tile is 6144 entries; 2^8 outputs to a bucket up to 2^18 of them, more beyond
@pytest.mark.parametrize("nnz", [1, 63, 6143, 6144, 6145, 100003])
@pytest.mark.parametrize("n_out", [1, 2, 255, 257, 2500, 300007, (1 << 20) + 1])
@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_coo_sizes(nnz, n_out, dtype):
    data, row, col = _coo(nnz, n_out, 501, dtype, torch.int64, torch.int32, nnz % 97)
    x = S.vector(501, dtype, DEV, 5)
    y = fs.flagsparse_spmv_coo(data, row, col, x, (n_out, 501))
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    # crowded outputs cancel: the bound is on the sum of magnitudes (64-bit sums of
    # nnz terms, one rounding to the output type)
    ref = _wide(data, row, col, x, n_out)
    mag = np.bincount(np_(row), weights=np.abs(np_(data)) * np.abs(np_(x))[np_(col)], minlength=n_out)
    eps = 2.0 ** -23 if dtype in (torch.float32, torch.complex64) else nnz * 2.0 ** -52
    assert np.all(np.abs(np_(y) - ref) <= eps * (np.abs(ref) + mag * 1e-9) + 4 * 2.0 ** -52 * nnz * mag)


@pytest.mark.parametrize("op", ["non", "trans", "conj"])
@pytest.mark.parametrize("index_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_ops_against_oracle(dtype, index_dtype, op):
    d, i, p, sh = S.random_csr(1501, 2203, 0.01, dtype, index_dtype, DEV, seed=3, empty_row_every=7,
                               long_rows=((11, 2100), (1499, 900)))
    x = S.vector(sh[1] if op == "non" else sh[0], dtype, DEV, 4)
    ref = O.spmv_csr_wide(np_(d), np_(i), np_(p), np_(x), sh, op=op)
    row = torch.repeat_interleave(torch.arange(sh[0], device=DEV), (p[1:] - p[:-1]).long())
    perm = torch.randperm(d.numel(), device=DEV)
    y = fs.flagsparse_spmv_coo(d[perm], row[perm].to(index_dtype), i[perm], x, sh, op=op)
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    assert rel_err(np_(y), ref) <= REL_TOL[dtype]
    if op != "non":
        y = fs.flagsparse_spmv_csr(d, i, p, x, sh, op=op)
        assert _lib.last_kernel() == "scatter_reduce_kernel"
        assert rel_err(np_(y), ref) <= REL_TOL[dtype]
        again = fs.flagsparse_spmv_csr(d, i, p, x, sh, op=op)
        assert torch.equal(torch.view_as_real(y) if y.is_complex() else y,
                           torch.view_as_real(again) if again.is_complex() else again)


@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_hub_columns_and_split_buckets(dtype):
    """A matrix whose bucket of low columns holds most entries (several
    segments, crowded lanes), against the transpose in 64 bits."""
    g = torch.Generator(device=DEV)
    g.manual_seed(9)
    n_rows, n_cols, per = 40000, 70001, 20
    col = (torch.rand(n_rows * per, device=DEV, generator=g, dtype=torch.float64) ** 8 * n_cols).long()
    p = torch.arange(n_rows + 1, device=DEV) * per
    d = S.vector(n_rows * per, dtype, DEV, 10)
    x = S.vector(n_rows, dtype, DEV, 11)
    y = fs.flagsparse_spmv_csr(d, col.int(), p, x, (n_rows, n_cols), op="trans")
    row = torch.arange(n_rows, device=DEV).repeat_interleave(per)
    ref = _wide(d, col, row, x, n_cols)
    assert rel_err(np_(y), ref) <= REL_TOL[dtype]


@pytest.mark.parametrize("run", [1, 2, 5, 6, 7, 8, 13, 20, 31, 32, 63, 64, 65, 200])
@pytest.mark.parametrize("nnz", [50, 64, 4001, 50000])
@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_groups_of_equal_outputs(dtype, nnz, run):
    """Runs of one output: groups of every size among a wave's lanes, alone and
    several at once.  Whole values, so that every order gives the same bits."""
    g = np.random.default_rng(run)
    out = np.repeat(g.integers(0, 300, -(-nnz // run)), run)[:nnz]
    src = g.integers(0, 40, nnz)
    val, x = g.integers(-9, 10, nnz), g.integers(-9, 10, 40)
    ref = np.bincount(out, weights=(val * x[src]).astype(np.float64), minlength=300)
    args = [torch.tensor(v, device=DEV) for v in (val, out, src, x)]
    y = fs.flagsparse_spmv_coo(args[0].to(dtype), args[1].int(), args[2], args[3].to(dtype), (300, 40))
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    assert np.array_equal(np_(y), ref.astype(np_(y).dtype))


@pytest.mark.parametrize("n_out", [1, 3, 64, 100, 300, 1025])
@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_buckets_of_many_segments(dtype, n_out):
    """Up to 1,024 segments in a bucket, most entries in the last one.  Whole
    values, so that every order gives the same bits."""
    g = np.random.default_rng(n_out)
    nnz = 2_200_001
    out = n_out - 1 - (g.random(nnz) ** 4 * n_out).astype(np.int64)
    src, val, x = g.integers(0, 40, nnz), g.integers(-2, 3, nnz), g.integers(-2, 3, 40)
    ref = np.bincount(out, weights=(val * x[src]).astype(np.float64), minlength=n_out)
    args = [torch.tensor(v, device=DEV) for v in (val, out, src, x)]
    y = fs.flagsparse_spmv_coo(args[0].to(dtype), args[1].int(), args[2].int(), args[3].to(dtype), (n_out, 40))
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    assert np.array_equal(np_(y), ref.astype(np_(y).dtype))


def test_largest_output_counts_take_or_leave_the_path():
    n = 1 << 23
    data, row, col = _coo(50000, n, 9, torch.float32, torch.int32, torch.int32, 1)
    x = S.vector(9, torch.float32, DEV, 2)
    y = fs.flagsparse_spmv_coo(data, row, col, x, (n, 9))
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    np.testing.assert_allclose(np_(y), _wide(data, row, col, x, n).real, rtol=1e-6, atol=1e-6)
    y2 = fs.flagsparse_spmv_coo(data, row, col, x, (n + 1, 9))
    assert _lib.last_kernel() != "scatter_reduce_kernel"
    assert torch.allclose(y2[:n], y, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("name,value", [("FLAGSPARSE_SPMV_KERNEL", "vector"), ("FLAGSPARSE_SPMV_ONESHOT", "0")])
def test_coo_call_follows_the_switches(monkeypatch, name, value):
    data, row, col = _coo(5000, 300, 200, torch.float64, torch.int32, torch.int32, 4)
    x = S.vector(200, torch.float64, DEV, 2)
    monkeypatch.delenv("FLAGSPARSE_SPMV_KERNEL", raising=False)
    y = fs.flagsparse_spmv_coo(data, row, col, x, (300, 200))
    assert _lib.last_kernel() == "scatter_reduce_kernel"
    monkeypatch.setenv(name, value)
    y2 = fs.flagsparse_spmv_coo(data, row, col, x, (300, 200))
    assert _lib.last_kernel() != "scatter_reduce_kernel"
    if value == "vector":
        assert _lib.last_kernel() == "spmv_vector_kernel"
    assert torch.allclose(y, y2, rtol=1e-12, atol=1e-12)


def test_structure_errors_keep_their_order():
    d, i, p, sh = S.random_csr(300, 200, 0.05, torch.float32, torch.int32, DEV, seed=3)
    x = S.vector(300, torch.float32, DEV, 4)
    bad_start, bad_end, bad_step, bad_col = p.clone(), p.clone(), p.clone(), i.clone()
    bad_start[0] = 1
    bad_end[-1] += 1
    bad_step[100] = bad_step[99] - 3
    bad_col[5] = 200

    def call(ii, pp):
        return fs.flagsparse_spmv_csr(d, ii, pp, x, sh, op="trans")

    with pytest.raises(ValueError, match="start at zero"):
        call(bad_col, bad_start)
    with pytest.raises(ValueError, match="equal nnz"):
        call(bad_col, bad_end)
    with pytest.raises(ValueError, match="non-decreasing"):
        call(bad_col, bad_step)
    with pytest.raises(IndexError, match="out of range for n_cols"):
        call(bad_col, p)
    row = torch.repeat_interleave(torch.arange(300, device=DEV), (p[1:] - p[:-1]).long())
    bad_row = row.clone()
    bad_row[7] = -1
    xr = S.vector(200, torch.float32, DEV, 4)
    for op, xx in (("non", xr), ("trans", x)):
        with pytest.raises(IndexError, match="row indices"):
            fs.flagsparse_spmv_coo(d, bad_row, bad_col, xx, sh, op=op)
        with pytest.raises(IndexError, match="col indices"):
            fs.flagsparse_spmv_coo(d, row, bad_col, xx, sh, op=op)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_infinities_and_unaligned_views(dtype):
    data, row, col = _coo(20000, 700, 300, dtype, torch.int32, torch.int32, 8)
    x = S.vector(300, dtype, DEV, 2)
    data[3], data[17] = float("inf"), float("nan")
    x[5] = float("-inf")
    # views that start off a 16-byte boundary
    args = [torch.cat([t[:1], t])[1:] for t in (data, row, col)]
    y = fs.flagsparse_spmv_coo(*args, x, (700, 300))
    ref = np.zeros(700)
    with np.errstate(invalid="ignore"):
        np.add.at(ref, np_(row), np_(data).astype(np.float64) * np_(x).astype(np.float64)[np_(col)])
    fin = np.isfinite(ref)
    assert np.array_equal(np_(y)[~fin].astype(np.float64), ref[~fin], equal_nan=True)
    np.testing.assert_allclose(np_(y)[fin], ref[fin], rtol=1e-6, atol=1e-5)


@pytest.mark.parametrize("n_cols", [200, (1 << 23) + 1], ids=["scatter", "transpose"])
@pytest.mark.parametrize("value", [2**63 - 1, 2**63 - 700, 2**40, -(2**63)])
def test_row_pointers_of_any_value_are_refused(value, n_cols):
    """64-bit row pointers near the largest value: the structure error, from both ways to A^T x."""
    d, i, p, _ = S.random_csr(300, 200, 0.05, torch.float32, torch.int64, DEV, seed=3)
    p = p.long().clone()
    p[100] = value
    with pytest.raises(ValueError, match="non-decreasing"):
        fs.flagsparse_spmv_csr(d, i, p, S.vector(300, torch.float32, DEV, 4), (300, n_cols), op="trans")


def test_coo_failed_int64_call_runs_again_on_int32_indices(monkeypatch):
    data, row, col = _coo(5000, 300, 200, torch.float64, torch.int64, torch.int64, 4)
    x = S.vector(200, torch.float64, DEV, 2)
    y = fs.flagsparse_spmv_coo(data, row, col, x, (300, 200))
    kernel, tried = spmv_coo._hip_spmv_coo_scatter, []

    def fails_on_int64(launch, x):
        tried.append(launch.row.dtype)
        if launch.row.dtype == torch.int64:
            raise RuntimeError("refused")
        return kernel(launch, x)

    monkeypatch.setattr(spmv_coo, "_hip_spmv_coo_scatter", fails_on_int64)
    assert torch.equal(fs.flagsparse_spmv_coo(data, row, col, x, (300, 200)), y)
    assert tried == [torch.int64, torch.int32]
    row[3] = 300
    with pytest.raises(IndexError, match="row indices"):
        fs.flagsparse_spmv_coo(data, row, col, x, (300, 200))
