"""Residual lengths on the device: one buffer written in place, from any grad mode."""
from __future__ import annotations

import pytest
import torch

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
