"""The workspaces this layer keeps: growth, what happens to the buffer before, captures, and
a device without room (on the CPU: sizes and lifetimes only)."""

from __future__ import annotations

import gc
import weakref

import pytest
import torch

from sglang_restomod_amd.attention.mi355x import backend as backend_module
from sglang_restomod_amd.attention.mi355x import ops
from tests import fakes

CPU = torch.device("cpu")


@pytest.fixture
def pool(monkeypatch):
    monkeypatch.setattr(ops, "_WORKSPACES", {})
    monkeypatch.setattr(ops, "_OUTGROWN_WORKSPACES", [])
    return ops


def test_the_shared_buffer_grows_and_keeps_its_predecessors(pool):
    first = pool.workspace_buffer(CPU, 5, stream=7)
    assert first.numel() == 1 << 20
    assert pool.workspace_buffer(CPU, 1 << 20, stream=7) is first
    assert pool.workspace_buffer(CPU, 5, stream=8) is not first
    alive = weakref.ref(first)
    address = first.data_ptr()
    second = pool.workspace_buffer(CPU, (1 << 20) + 1, stream=7)
    del first
    gc.collect()
    # a graph captured with the first buffer's address still finds it
    assert alive() is not None and alive().data_ptr() == address
    assert second.numel() == 2 << 20  # half again as large, in whole MiB
    for n in range(2, 60):
        pool.workspace_buffer(CPU, n << 20, stream=7)
    kept = sum(b.numel() for b in pool._OUTGROWN_WORKSPACES)
    assert kept <= 2 * pool._WORKSPACES[("cpu", 7)].numel() + (len(pool._OUTGROWN_WORKSPACES) << 20)


def test_a_buffer_that_cannot_grow_stays(pool, monkeypatch):
    first = pool.workspace_buffer(CPU, 5, stream=7)

    def full(*args, **kwargs):
        raise torch.OutOfMemoryError("full")

    monkeypatch.setattr(ops.torch, "empty", full)
    with pytest.raises(torch.OutOfMemoryError):
        pool.workspace_buffer(CPU, 2 << 20, stream=7)
    assert pool.workspace_buffer(CPU, 5, stream=7) is first and not pool._OUTGROWN_WORKSPACES


class _Backend:
    """A backend on the CPU with a split-KV workspace of `nbytes`."""

    def __new__(cls, monkeypatch, nbytes):
        be = backend_module.MI355XAttnBackend(fakes.Engine("cpu", hq=32, hkv=8, head_dim=128).runner)
        ws = torch.empty(nbytes, dtype=torch.uint8)
        monkeypatch.setattr(be, "splitkv_workspace", lambda: ws)
        cls.capturing = False
        monkeypatch.setattr(backend_module.torch.cuda, "is_current_stream_capturing", lambda: cls.capturing)
        return be


def test_backend_extend_workspace_lives_on(monkeypatch):
    be = _Backend(monkeypatch, 1 << 20)
    small = be.splitkv_workspace()
    assert be._workspace_for("verify", 64, 32, 8, 4) is small
    assert be._workspace_for("extend", 1 << 15, 32, 8, 40) is small     # whole row tiles: the list fits
    _Backend.capturing = True
    assert be._workspace_for("extend", 64, 32, 8, 4) is small           # nothing is allocated in a capture
    with pytest.raises(RuntimeError, match="capture smaller batches"):
        be._workspace_for("extend", 1 << 23, 32, 8, 4)
    _Backend.capturing = False
    own = be._workspace_for("extend", 64, 32, 8, 4)                     # key pieces: a buffer of its own
    assert own.numel() >= ops.extend_split_workspace_bytes(64, 32, 8, 4, 128)
    _Backend.capturing = True
    assert be._workspace_for("extend", 900, 32, 8, 7) is own            # the same one, at any size, in a capture too
    _Backend.capturing = False
    assert be._workspace_for("extend", 1, 32, 8, 31) is own
    be._extend_ws = own[:2 << 20]                                       # as if it had been smaller
    assert be._workspace_for("extend", 64, 32, 8, 4).numel() > 2 << 20
    assert [b.numel() for b in be._outgrown_ws] == [2 << 20]            # the replaced one is kept


def test_backend_without_room_runs_whole_row_tiles(monkeypatch):
    be = _Backend(monkeypatch, 1 << 20)
    small = be.splitkv_workspace()
    empty = torch.empty

    def full(*args, **kwargs):
        if kwargs.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("full")
        return empty(*args, **kwargs)

    monkeypatch.setattr(backend_module.torch, "empty", full)
    assert be._workspace_for("extend", 64, 32, 8, 4) is small
    with pytest.raises(torch.OutOfMemoryError):
        be._workspace_for("extend", 1 << 23, 32, 8, 4)
