"""The lane-group SpMM on matrices too small for 2048-item waves
(fs_spmm_tile_items_sized): sub-tiles down to 128 items a wave, rows crossing
many of them, against the CPU oracle."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _lib
from flagsparse_amd import synthetic as S
from oracle import csr_oracle as O
from tests._helpers import REL_TOL, VALUE_DTYPES, VALUE_IDS, np_, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n", [1, 4, 17, 32, 64, 130, 256])
@pytest.mark.parametrize("rows,long_rows", [(3, ()), (40, ((3, 1900),)), (1501, ((0, 2000), (900, 1999), (1500, 700)))])
@pytest.mark.parametrize("dtype", VALUE_DTYPES, ids=VALUE_IDS)
def test_small_matrices(dtype, rows, long_rows, n):
    d, i, p, sh = S.random_csr(rows, 2003, 0.004, dtype, torch.int32, DEV, seed=rows + n, empty_row_every=5,
                               long_rows=long_rows)
    B = S.dense(2003, n, dtype, DEV, 3)
    ref = O.spmm_csr_wide(np_(d), np_(i), np_(p), np_(B), sh)
    C = fs.flagsparse_spmm_csr(d, i, p, B, sh)
    assert _lib.last_kernel() == "spmm_group_kernel"
    assert rel_err(np_(C), ref) <= REL_TOL[dtype]
    Ct = fs.flagsparse_spmm_csr_run(fs.prepare_spmm_csr_route(d, i, p, sh), B)
    assert torch.equal(torch.view_as_real(C) if C.is_complex() else C, torch.view_as_real(Ct) if C.is_complex() else Ct)


# 32 items a sub-tile with 16 lanes a row: rows of 4096 entries cross about 128
# of them, where the fix-up goes from one wave to a workgroup
@pytest.mark.parametrize("lengths", [[5, 1000, 2], [1010] * 3, [1023, 1, 1024, 1025, 0, 1090],
                                     [4095, 1, 4096, 4097, 0, 4160], [0, 40000, 3, 0, 0, 33000, 7],
                                     [100000] + [2] * 500], ids=lambda v: f"{len(v)}rows{sum(v)}nnz")
@pytest.mark.parametrize("n", [1, 3, 17, 64, 65, 200])
@pytest.mark.parametrize("dtype", VALUE_DTYPES + [torch.bfloat16], ids=VALUE_IDS + ["bf16"])
def test_long_rows_of_many_fragments(dtype, n, lengths):
    """Whole values, so that every order of the sums gives the same bits."""
    g = np.random.default_rng(len(lengths))
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    cols = g.integers(0, 5000, ptr[-1])
    top = 1 if dtype == torch.bfloat16 else 4
    vals, B = g.integers(-top, top + 1, ptr[-1]), g.integers(-top, top + 1, (5000, n))
    ref = np.zeros((len(lengths), n))
    for r in range(len(lengths)):
        s = slice(ptr[r], ptr[r + 1])
        ref[r] = vals[s] @ B[cols[s]]
    args = [torch.tensor(vals, device=DEV).to(dtype), torch.tensor(cols, device=DEV).int(),
            torch.tensor(ptr, device=DEV).int()]
    Bt = torch.tensor(B, device=DEV).to(dtype)
    C = fs.flagsparse_spmm_csr(*args, Bt, (len(lengths), 5000))
    want = torch.tensor(ref, device=DEV).to(dtype)
    assert torch.equal(C, want)
    route = fs.prepare_spmm_csr_route(*args, (len(lengths), 5000))
    assert torch.equal(fs.flagsparse_spmm_csr_run(route, Bt), want)


def test_sizes_shrink_with_the_matrix_only():
    lib = _lib.lib()
    for n in (1, 32, 64, 128, 256):
        full = lib.fs_spmm_tile_items(_lib.FS_F32, n)
        sizes = [lib.fs_spmm_tile_items_sized(_lib.FS_F32, n, 10, nnz) for nnz in (10, 10**5, 10**6, 10**7, 10**8)]
        assert sizes == sorted(sizes) and sizes[-1] == full and sizes[0] < full
    # B rows of 512 bytes and more: one size for both kernels once skewed columns are looked for
    assert lib.fs_spmm_tile_items_sized(_lib.FS_F32, 128, 10, (1 << 20) - 1) < 512
    assert lib.fs_spmm_tile_items_sized(_lib.FS_F32, 128, 10, 1 << 20) == 512


def test_one_round_of_waves_is_not_halved():
    """Short rows, whole slices, 32 lanes a row (N = 64 in float32): 2048 to
    3072 waves stay (32 lanes: half of a wave's items are a sub-tile's)."""
    size = lambda t, n, rows, nnz: _lib.lib().fs_spmm_tile_items_sized(t, n, rows, nnz)  # noqa: E731
    assert size(_lib.FS_F32, 64, 400_000, 4_000_000) == 1024  # 2149 waves of 2048
    assert size(_lib.FS_F32, 64, 600_000, 6_000_000) == 512  # 3223: two rounds, halved
    assert size(_lib.FS_F32, 64, 100_000, 1_000_000) == 256  # 2149 waves of 512
    assert size(_lib.FS_F32, 33, 400_000, 4_000_000) == 512  # element loads
    assert size(_lib.FS_F32, 64, 90_000, 4_300_000) == 512  # rows of 48
    assert size(_lib.FS_C128, 16, 400_000, 4_000_000) == 1024
    assert size(_lib.FS_C128, 16, 200_000, 4_000_000) == 512  # rows of 20
    # 16 lanes a row (a sub-tile is a quarter of a wave's items): 1792 waves of longer rows, 2048 of short ones
    assert size(_lib.FS_F64, 16, 36_499, 3_649_900) == 512  # 1800 waves of 2048
    assert size(_lib.FS_F64, 16, 36_093, 3_609_300) == 256  # 1780
    assert size(_lib.FS_F64, 16, 9_124, 912_400) == 128  # 1800 of 512
    assert size(_lib.FS_F64, 16, 555_885, 3_335_310) == 256  # 1900, rows of 6
    assert size(_lib.FS_BF16, 16, 38_526, 3_852_600) == 256  # 1900, 16-bit values
    assert size(_lib.FS_F32, 64, 41_365, 4_136_500) == 256  # 2040, 32 lanes


def test_either_tile_size_is_taken():
    """A caller that sizes its partition by fs_spmm_tile_items is served as before."""
    d, i, p, sh = S.random_csr(500, 400, 0.03, torch.float32, torch.int32, DEV, seed=2)
    B = S.dense(400, 40, torch.float32, DEV, 3)
    route = fs.prepare_spmm_csr_route(d, i, p, sh)
    plan = route.hip_plan().csr
    lib = _lib.lib()
    for items in (lib.fs_spmm_tile_items(_lib.FS_F32, 40), lib.fs_spmm_tile_items_sized(_lib.FS_F32, 40, 500, d.numel())):
        part, tiles = plan.partition(p, items), plan.n_tiles(items)
        ws = _lib.workspace(lib.fs_spmm_workspace_bytes(_lib.FS_F32, tiles, 40), B.device)
        C = torch.empty(500, 40, device=DEV)
        _lib.check(lib.fs_spmm_csr(plan.plan, _lib.ptr(d), _lib.ptr(i), _lib.ptr(p), _lib.ptr(B), 40, _lib.ptr(C), 40,
                                   40, _lib.ptr(part), items, tiles, _lib.ptr(ws), ws.numel(),
                                   _lib.stream_handle(B.device)), "fs_spmm_csr")
        ref = O.spmm_csr_wide(np_(d), np_(i), np_(p), np_(B), sh)
        assert rel_err(np_(C), ref) <= REL_TOL[torch.float32]
    assert lib.fs_spmm_csr(plan.plan, _lib.ptr(d), _lib.ptr(i), _lib.ptr(p), _lib.ptr(B), 40, _lib.ptr(C), 40, 40,
                           _lib.ptr(part), 96, plan.n_tiles(96), _lib.ptr(ws), ws.numel(),
                           _lib.stream_handle(B.device)) == _lib.FS_E_INVALID
