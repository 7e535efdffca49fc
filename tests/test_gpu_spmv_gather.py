"""The two-phase gather SpMV of prepared matrices (fs_spmv_csr_gather): edges
of tiles, regions and column slices, long and empty rows, against the CPU
oracle and, bit for bit, the merge-path kernel whose sums it keeps."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
import flagsparse_amd.spmv_csr as spmv_mod
from flagsparse_amd import _lib
from flagsparse_amd import synthetic as S
from oracle import csr_oracle as O
from tests._helpers import INDEX_DTYPES, INDEX_IDS, REL_TOL, np_, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = [torch.float32, torch.float64, torch.complex64]


@pytest.fixture
def any_size(monkeypatch):
    """The path for every matrix whose type and sizes it takes."""
    for k in ("FLAGSPARSE_SPMV_SELL", "FLAGSPARSE_SPMV_KERNEL", "FLAGSPARSE_SPMV_PANELS"):
        monkeypatch.delenv(k, raising=False)
    monkeypatch.setattr(spmv_mod, "_GATHER_MIN_NNZ", 0)
    monkeypatch.setattr(spmv_mod, "_GATHER_MIN_NNZ_SMALL_X", 0)
    monkeypatch.setattr(spmv_mod, "_GATHER_LONG_ROWS", 1 << 40)
    monkeypatch.setattr(spmv_mod, "_GATHER_X_BYTES", {4: 0, 8: 0})
    monkeypatch.setattr(spmv_mod, "_GATHER_TOUCHED", {4: 0, 8: 0})


def _matrix(lengths, n_cols, dtype, index_dtype, ptr_dtype, seed):
    g = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    cols = g.integers(0, n_cols, ptr[-1])
    cols[:: 17] = n_cols - 1
    data = S.vector(int(ptr[-1]), dtype, DEV, seed)
    return (data, torch.tensor(cols, device=DEV).to(index_dtype), torch.tensor(ptr, device=DEV).to(ptr_dtype),
            (len(lengths), n_cols))


def _check(mat, monkeypatch, x=None):
    data, sh = mat[0], mat[3]
    x = S.vector(sh[1], data.dtype, DEV, 5) if x is None else x
    prep = fs.prepare_spmv_csr(*mat)
    y = fs.flagsparse_spmv_csr(x=x, prepared=prep)
    assert _lib.last_kernel() == "spmv_region_kernel"
    ref = O.spmv_csr_wide(np_(mat[0]), np_(mat[1]), np_(mat[2]), np_(x), sh)
    assert rel_err(np_(y), ref) <= REL_TOL[data.dtype]
    monkeypatch.setenv("FLAGSPARSE_SPMV_KERNEL", "merge")
    monkeypatch.setenv("FLAGSPARSE_SPMV_PANELS", "0")
    y0 = fs.flagsparse_spmv_csr(x=x, prepared=fs.prepare_spmv_csr(*mat))
    monkeypatch.delenv("FLAGSPARSE_SPMV_KERNEL")
    monkeypatch.delenv("FLAGSPARSE_SPMV_PANELS")
    assert _lib.last_kernel() != "spmv_region_kernel"
    assert torch.equal(torch.view_as_real(y) if y.is_complex() else y,
                       torch.view_as_real(y0) if y0.is_complex() else y0)
    return prep, x, y


# a tile is 512 rows + entries; a region 16 tiles of float32, 8 of the others
@pytest.mark.parametrize("lengths", [
    [1], [0, 0, 3], [511], [510], [512], [5] * 85 + [1], [0] * 600 + [9] + [0] * 600,
    [8191], [8193, 0, 1], [20000, 3, 0, 70000, 1], [7] * 1100, list(range(120)), [64] * 130 + [0] * 70,
], ids=lambda v: f"{len(v)}rows{sum(v)}nnz")
@pytest.mark.parametrize("ptr_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "f64", "c64"])
def test_tile_and_region_edges(any_size, monkeypatch, dtype, ptr_dtype, lengths):
    _check(_matrix(lengths, 40001, dtype, torch.int32, ptr_dtype, 3), monkeypatch)


# a slice is 32768 columns of float32, 16384 of the others; at most 256 slices
@pytest.mark.parametrize("n_cols", [1, 3, 16384, 16385, 32768, 32769, 65537, 1000003])
@pytest.mark.parametrize("index_dtype", INDEX_DTYPES, ids=INDEX_IDS)
@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "f64", "c64"])
def test_slice_edges(any_size, monkeypatch, dtype, index_dtype, n_cols):
    g = np.random.default_rng(n_cols)
    _check(_matrix(g.integers(0, 30, 3000), n_cols, dtype, index_dtype, torch.int32, 4), monkeypatch)


def test_limits_of_the_path(any_size):
    for dtype, n_cols, takes in ((torch.float32, 1 << 23, True), (torch.float32, (1 << 23) + 1, False),
                                 (torch.float64, 1 << 22, True), (torch.float64, (1 << 22) + 1, False),
                                 (torch.complex128, 1000, False)):
        mat = _matrix([40] * 200, n_cols, dtype, torch.int32, torch.int32, 6)
        x = S.vector(n_cols, dtype, DEV, 7)
        y = fs.flagsparse_spmv_csr(x=x, prepared=fs.prepare_spmv_csr(*mat))
        assert (_lib.last_kernel() == "spmv_region_kernel") == takes
        ref = O.spmv_csr_wide(np_(mat[0]), np_(mat[1]), np_(mat[2]), np_(x), mat[3])
        assert rel_err(np_(y), ref) <= REL_TOL[dtype]


def test_chosen_by_spread_of_columns(monkeypatch):
    """Large uniform columns take the path, a band of the same size does not,
    nor does a call without a prepared matrix."""
    monkeypatch.delenv("FLAGSPARSE_SPMV_KERNEL", raising=False)
    monkeypatch.delenv("FLAGSPARSE_SPMV_PANELS", raising=False)
    n = 1 << 21
    d, i, p, sh = S.uniform_rows(n, n, 8, torch.float32, torch.int32, DEV, seed=1)
    x = S.vector(n, torch.float32, DEV, 2)
    for op in ("non", "trans"):
        prep = fs.prepare_spmv_csr(d, i, p, sh, op=op)
        _, meta = fs.flagsparse_spmv_csr(x=x, prepared=prep, return_meta=True)
        assert _lib.last_kernel() == "spmv_region_kernel"
        assert meta["kernel"] == prep.kernel_name == "gather" and prep._panels is None
    fs.flagsparse_spmv_csr(d, i, p, x, sh)
    assert _lib.last_kernel() == "spmv_oneshot_kernel"
    band = ((torch.arange(n, device=DEV).repeat_interleave(8) + i.long() % 30011) % n).int()
    fs.flagsparse_spmv_csr(x=x, prepared=fs.prepare_spmv_csr(d, band, p, sh))
    assert _lib.last_kernel() != "spmv_region_kernel"


def test_shared_by_two_streams_unaligned_x_and_infinities(any_size, monkeypatch):
    g = np.random.default_rng(1)
    mat = _matrix(g.integers(0, 60, 20000), 90001, torch.float32, torch.int32, torch.int32, 8)
    whole = S.vector(90002, torch.float32, DEV, 9)
    prep, x, y = _check(mat, monkeypatch, x=whole[1:])
    xs = [S.vector(90001, torch.float32, DEV, 20 + k) for k in range(2)]
    want = [fs.flagsparse_spmv_csr(x=v, prepared=prep) for v in xs]
    streams = [torch.cuda.Stream() for _ in xs]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(10):
        for k, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[k].append(fs.flagsparse_spmv_csr(x=xs[k], prepared=prep))
    torch.cuda.synchronize()
    for k in range(2):
        assert all(torch.equal(want[k], v) for v in got[k])
    # an infinity reaches the rows that hold its column and no padding or neighbour
    x2 = xs[0].clone()
    x2[int(mat[1][5])] = float("inf")
    y2 = fs.flagsparse_spmv_csr(x=x2, prepared=prep)
    row = torch.repeat_interleave(torch.arange(20000, device=DEV), (mat[2][1:] - mat[2][:-1]).long())
    hit = torch.zeros(20000, dtype=torch.bool, device=DEV)
    hit[row[mat[1] == mat[1][5]]] = True
    assert torch.equal(~torch.isfinite(y2), hit)


def test_plan_out_of_memory_keeps_the_csr_kernels(any_size, monkeypatch):
    mat = _matrix([9] * 4000, 50000, torch.float32, torch.int32, torch.int32, 8)
    x = S.vector(50000, torch.float32, DEV, 9)
    want = fs.flagsparse_spmv_csr(x=x, prepared=fs.prepare_spmv_csr(*mat))

    def no_memory(*args, **kwargs):
        raise torch.OutOfMemoryError("injected")

    monkeypatch.setattr(spmv_mod.GatheredCsr, "build", no_memory)
    y = fs.flagsparse_spmv_csr(x=x, prepared=fs.prepare_spmv_csr(*mat))
    assert _lib.last_kernel() != "spmv_region_kernel"
    assert torch.allclose(y, want, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("lengths", [[9] * 4000, [5000] + [3] * 3000], ids=["stream", "merge"])
def test_call_without_room_for_its_workspace(any_size, monkeypatch, lengths):
    mat = _matrix(lengths, 50000, torch.float32, torch.int32, torch.int32, 8)
    x = S.vector(50000, torch.float32, DEV, 9)
    prep = fs.prepare_spmv_csr(*mat)
    want = fs.flagsparse_spmv_csr(x=x, prepared=prep)
    assert _lib.last_kernel() == "spmv_region_kernel"

    def no_memory(self, x, y):
        raise torch.OutOfMemoryError("injected")

    with monkeypatch.context() as m:
        m.setattr(spmv_mod.GatheredCsr, "spmv", no_memory)
        for _ in range(2):
            with pytest.warns(RuntimeWarning, match="no room"):
                y = fs.flagsparse_spmv_csr(x=x, prepared=prep)
            assert _lib.last_kernel() != "spmv_region_kernel"
            assert torch.allclose(y, want, rtol=1e-6, atol=1e-6)
    # one call's shortage is not the matrix's
    assert torch.equal(fs.flagsparse_spmv_csr(x=x, prepared=prep), want)
    assert _lib.last_kernel() == "spmv_region_kernel" and prep.kernel_name == "gather"


def test_replayed_from_a_graph(any_size):
    g = np.random.default_rng(2)
    mat = _matrix(g.integers(0, 40, 9000), 70001, torch.float32, torch.int32, torch.int32, 8)
    x = S.vector(70001, torch.float32, DEV, 9)
    prep = fs.prepare_spmv_csr(*mat)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fs.flagsparse_spmv_csr(x=x, prepared=prep)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = fs.flagsparse_spmv_csr(x=x, prepared=prep)
    for _ in range(3):
        x.mul_(1.5)
        want = fs.flagsparse_spmv_csr(x=x, prepared=prep)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
