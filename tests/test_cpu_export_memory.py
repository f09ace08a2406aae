"""Host side of the path export at its memory limits, on CPU tensors with the
native calls stubbed: where the masked export's rows do not fit (its masks are
held, and it emits rows below the gain floor too), the masks are released and
the per-cell export runs."""

from __future__ import annotations

import ctypes
import weakref
from types import SimpleNamespace

import pytest
import torch

from witwin.channel import _native
from witwin.channel.propagation import engine

KEPT = 3


@pytest.fixture
def export(monkeypatch):
    """export(masked rows, per-cell rows, name of the step without memory while the masks are held)."""
    state = SimpleNamespace(calls=[], mask=lambda: None)

    def run(masked_total, cell_total, starve=None):
        def call(name, *args):
            state.calls.append(name)
            if name.endswith("workspace_bytes"):
                return 4096 if "masks" in name else 16
            if name == "wc_paths_row_offsets":
                total = masked_total if "wc_paths_count_masked" in state.calls[-3:] else cell_total
                ctypes.c_int64.from_address(args[5]).value = total
            if name == "wc_paths_compact":
                (ctypes.c_int32 * KEPT).from_address(args[7])[:] = list(range(KEPT))
                ctypes.c_int64.from_address(args[8]).value = KEPT
            return 0

        empty = torch.empty

        def short(size, *args, **kwargs):
            emitted = any(c.startswith("wc_paths_emit") for c in state.calls)
            if state.mask() is not None and (starve == "rows" and not emitted and size == masked_total
                                             or starve == "list" and size == masked_total + 2):
                raise torch.OutOfMemoryError("no memory beside the masks")
            if starve == "compaction" and emitted and "wc_paths_count" not in state.calls and size == masked_total:
                raise torch.OutOfMemoryError("no memory beside the masked rows")
            out = empty(size, *args, **kwargs)
            if size == 4096:
                state.mask = weakref.ref(out)
            elif emitted:
                assert state.mask() is None, "the masks outlive the emit"
            return out

        monkeypatch.setattr(_native, "call", call)
        monkeypatch.setattr(_native, "stream_handle", lambda device=None: 0)
        monkeypatch.setattr(torch, "empty", short)
        dscene = SimpleNamespace(device=torch.device("cpu"), view=SimpleNamespace(edge_count=0, face_count=770), edge_count=0,
                                 ref=lambda: None)
        inputs = SimpleNamespace(total_cells=1, tile_count=1, tiles=torch.zeros(2, dtype=torch.int32),
                                 view=_native.WcSolve(), pair_cell=torch.zeros(1, dtype=torch.int32))
        rows = engine.export_rows(dscene, inputs, width=1)
        assert rows["tx_id"].shape == (KEPT,)
        return [c for c in state.calls if c.startswith(("wc_paths_count", "wc_paths_emit"))]

    return run


def test_masked_export_where_it_fits(export):
    assert export(7, 5) == ["wc_paths_count_masked", "wc_paths_emit_masked"]


@pytest.mark.parametrize("starve", ["rows", "list", "compaction"])
def test_out_of_memory_falls_back_to_the_per_cell_export(export, starve):
    calls = export(7, 5, starve)
    assert calls[0] == "wc_paths_count_masked" and calls[-2:] == ["wc_paths_count", "wc_paths_emit"]


def test_row_limit_falls_back_to_the_per_cell_export(export):
    assert export(2 ** 31, 5) == ["wc_paths_count_masked", "wc_paths_count", "wc_paths_emit"]


def test_row_limit_of_the_per_cell_export_is_refused(export):
    with pytest.raises(RuntimeError, match="int32 row index"):
        export(2 ** 31, 2 ** 31)
