"""Residual lengths on the device: one buffer written in place, from any grad mode."""
from __future__ import annotations

import pytest
import torch

from logitfill_amd import _native
from logitfill_amd.packed.cache import _LayerStore


def _store():
    """A layer's length bookkeeping alone, on the CPU (the packed cache itself lives on the GPU)."""
    store = _LayerStore.__new__(_LayerStore)
    store.batch, store.device = 3, torch.device("cpu")
    store.tail_lens, store._tail_len_dev, store._tail_dirty = [0] * 3, None, True
    return store


def test_lengths_are_written_in_place():
    store = _store()
    first = store.tail_len_device()
    store.tail_lens, store._tail_dirty = [7] * 3, True
    again = store.tail_len_device()
    assert again.data_ptr() == first.data_ptr() and again.tolist() == [7, 7, 7]


@pytest.mark.parametrize("made", ["equal", "ragged"])
def test_lengths_made_under_inference_mode_change_outside_of_it(made):
    store = _store()
    with torch.inference_mode():
        if made == "equal":
            store.tail_len_device()
        else:  # (what an upload of differing lengths leaves there)
            store._tail_len_dev, store._tail_dirty = torch.tensor([1, 2, 3], dtype=torch.int32), False
    store.tail_lens, store._tail_dirty = [5] * 3, True
    assert store.tail_len_device().tolist() == [5, 5, 5]


@pytest.mark.parametrize("current", [0, 1])
def test_rows_are_written_with_the_stores_device_current(monkeypatch, current):
    """A commit of several tokens to a cache on another device than the current one launches there (on the
    CPU, with the device calls replaced)."""
    now, launches = [current], []

    class Device:
        def __init__(self, device):
            self.index = device.index

        def __enter__(self):
            self.before, now[0] = now[0], self.index

        def __exit__(self, *exc):
            now[0] = self.before

    class Library:
        def lf_fill_tail(self, *args):
            launches.append(now[0])
            return 0

    monkeypatch.setattr(torch.cuda, "current_device", lambda: now[0])
    monkeypatch.setattr(torch.cuda, "device", Device)
    monkeypatch.setattr(_native, "load", Library)
    monkeypatch.setattr(_native, "current_stream_ptr", lambda device: 0)
    store = _store()
    store.device, store.page_size, store.n_kv, store.head_dim = torch.device("cuda", 1), 4, 2, 8
    store._tail_k = store._tail_v = torch.zeros(3, 2, 4, 8)
    rows = torch.zeros(3, 2, 2, 8)
    store._fill_tail(rows, rows, [(0, 0, 0, 2)], True)
    assert launches == [1] and now == [current]
