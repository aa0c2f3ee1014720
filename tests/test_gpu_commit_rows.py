"""Commits of several tokens: rows into residual pages (lf_fill_tail) and pages packed straight
from the source, against the oracle's store, for the forms of source and position they take."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from logitfill_amd import _native
from logitfill_amd.packed import PackedKVManager
from tests.helpers import assert_history_equal, f32, oracle_store

pytestmark = pytest.mark.gpu


def _source(form, B, H, T, D, dtype, g, gpu):
    x = torch.randn(B, H, T, D, generator=g).to(dtype).to(gpu)
    if form == "contiguous":
        return x
    if form == "token_major":                       # [B, T, H, D] viewed as [B, H, T, D]
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "offset":                            # rows that start off 16 bytes
        wide = torch.zeros(B, H, T, D + 3, dtype=dtype, device=gpu)
        wide[..., 1:D + 1] = x
        return wide[..., 1:D + 1]
    return x.transpose(2, 3).contiguous().transpose(2, 3)  # "channel_stride": not unit


@pytest.mark.parametrize("form", ["contiguous", "token_major", "offset", "channel_stride"])
@pytest.mark.parametrize("dtype,D,page", [(torch.bfloat16, 128, 128), (torch.float32, 64, 32), (torch.float16, 12, 16)])
@pytest.mark.parametrize("defer", [False, True])
def test_commits_of_every_length(gpu, form, dtype, D, page, defer):
    """Ragged and even commits that leave the residual page part full, fill it exactly, cross one and
    several page ends, from empty and from part-full pages; then the history and residual rows are
    the oracle's, bit for bit."""
    B, H = 3, 2
    g = torch.Generator().manual_seed(D)
    levels = np.random.default_rng(D).choice(4, size=(H, D), p=[0.5, 0.3, 0.15, 0.05])
    mgr = PackedKVManager([levels], H, H, D, page, page, D, 2, gpu, batch_size=B, defer_flush=defer)
    done_k, done_v = [[] for _ in range(B)], [[] for _ in range(B)]
    steps = [(5, None), (page - 5, None), (page, None), (2 * page + 3, [2 * page + 3, page, 0]),
             (3 * page, None), (page, [page - 3, page, 4]), (1, None)]
    for T, lens in steps:
        k, v = _source(form, B, H, T, D, dtype, g, gpu), _source("contiguous", B, H, T, D, dtype, g, gpu)
        mgr.commit(0, k, v, lens)
        for b in range(B):
            n = T if lens is None else lens[b]
            done_k[b].append(f32(k[b, :, :n]))
            done_v[b].append(f32(v[b, :, :n]))
    mgr.flush_pending()
    for b in range(B):
        store = oracle_store(levels, np.concatenate(done_k[b], 1), np.concatenate(done_v[b], 1), page, page, D)
        assert_history_equal(mgr.layers[0], b, store)


def test_fill_tail_many_segments(gpu):
    """More segments than one launch carries (160), the last ones single rows."""
    B, H, cap, D = 170, 1, 4, 8
    src = torch.randn(B, H, 3, D, device=gpu)
    tk, tv = torch.zeros(B, H, cap, D, device=gpu), torch.zeros(B, H, cap, D, device=gpu)
    segs = [(b, b % 2, 1 + b % 3, 1) for b in range(B)]
    strides = (ctypes.c_int64 * 3)(*src.stride()[:3])
    st = _native.load().lf_fill_tail(
        tk.data_ptr(), tv.data_ptr(), src.data_ptr(), src.data_ptr(), _native.dtype_code(src.dtype), strides, strides,
        cap, (ctypes.c_int32 * (4 * B))(*[x for s in segs for x in s]), B, 0, B, H, D,
        _native.current_stream_ptr(src.device))
    assert st == 0
    want = torch.zeros_like(tk)
    for b, tok, row, n in segs:
        want[b, :, row] = src[b, :, tok]
    assert torch.equal(tk, want) and torch.equal(tv, want)
