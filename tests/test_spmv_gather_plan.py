"""Host side of the two-phase gather SpMV's plan, with the library and the
stream replaced by recorders (no GPU): what a call may rely on once
GatheredCsr.build has returned."""

import ctypes
from types import SimpleNamespace

import pytest
import torch

import flagsparse_amd.spmv_csr as spmv_mod
from flagsparse_amd import _lib

REGIONS, SLICES = 3, 2


@pytest.fixture
def recorded(monkeypatch):
    """(plan of a small matrix, the order of its device work)."""
    events = []

    def fill_ints(address, values):
        for k, v in enumerate(values):
            ctypes.c_int32.from_address(address + 4 * k).value = v

    def slices(val_t, n_rows, n_cols, nnz, regions):
        regions.value = REGIONS
        return SLICES

    def count(*args):  # two quads and one slice touched per region, three quads per slice
        events.append("count")
        fill_ints(args[7], [2] * REGIONS)
        fill_ints(args[8], [1] * REGIONS)
        fill_ints(args[9], [3] * SLICES)
        return 0

    lib = SimpleNamespace(
        fs_spmv_gather_slices=slices,
        fs_spmv_gather_plan_bytes=lambda *a: 64,
        fs_spmv_gather_workspace_bytes=lambda *a: 256,
        fs_spmv_gather_count=count,
        fs_spmv_gather_fill=lambda *a: events.append("fill") or 0,
        fs_spmv_csr_gather=lambda *a: events.append(f"call on {a[-1]}") or 0,
    )
    stream = SimpleNamespace(synchronize=lambda: events.append("synchronize"))
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    monkeypatch.setattr(_lib, "stream_handle", lambda device: 11)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: stream)
    csr = SimpleNamespace(plan=SimpleNamespace(tile_items=512), partition=lambda indptr, items: torch.zeros(4).long())
    plan = spmv_mod.GatheredCsr.build(
        torch.ones(5), torch.zeros(5, dtype=torch.int32), torch.tensor([0, 5], dtype=torch.int32), 1, 9, csr,
        lambda regions, touched: True)
    return plan, events


def test_build_returns_a_finished_plan(recorded):
    """A call on any stream stores at the places the fill wrote, so the fill
    has ended when the plan is handed out."""
    plan, events = recorded
    assert plan.n_quads == 6 and plan.max_region_quads == 2
    assert events == ["count", "fill", "synchronize"]


def test_a_call_on_another_stream_keeps_the_plan_alive(recorded, monkeypatch):
    plan, events = recorded
    x, y = torch.ones(9), torch.empty(1)
    kept = []

    class Tensor:
        def __init__(self, t):
            self.t = t

        def record_stream(self, stream):
            kept.append(self.t.data_ptr())

        def __getattr__(self, name):
            return getattr(self.t, name)

    names = ("part", "pos", "columns", "place", "slice_q", "region_q")
    for name in names:
        setattr(plan, name, Tensor(getattr(plan, name)))
    plan.spmv(x, y)
    assert kept == [] and events[-1] == "call on 11"
    monkeypatch.setattr(_lib, "stream_handle", lambda device: 12)
    plan.spmv(x, y)
    assert kept == [getattr(plan, name).data_ptr() for name in names] and events[-1] == "call on 12"
