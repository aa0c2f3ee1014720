"""The dequantise kernel (dequant.hip) at the shapes its two forms and its run lengths can go wrong
at, exactly equal to the oracle's float32 dequantisation."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from logitfill_amd.packed import PackedKVManager
from tests.helpers import f32, oracle_store

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,page,kg,vg,bit_v,n_kv,pages", [
    (128, 64, 32, 64, 4, 2, 7),      # four channels a thread
    (64, 16, 8, 32, 8, 3, 5),        # Key groups shorter than a run
    (12, 16, 16, 6, 2, 1, 3),        # Value groups that four channels would straddle: one a thread
    (10, 8, 4, 5, 4, 2, 1),          # head_dim not a multiple of four, one page
    (96, 32, 32, 96, 16, 2, 4),      # fp16 Values, threads left over
    (1024, 16, 16, 128, 2, 1, 2),    # a token per workgroup pass (four channels: 256 threads)
    (128, 128, 128, 128, 2, 4, 40),  # runs of more than 8 tokens
])
def test_dequantise_exact(gpu, D, page, kg, vg, bit_v, n_kv, pages):
    rng = np.random.default_rng(D + pages)
    levels = rng.choice(4, size=(n_kv, D), p=[0.5, 0.25, 0.15, 0.1])
    g = torch.Generator().manual_seed(D)
    key = torch.randn(1, n_kv, pages * page, D, generator=g) * 5
    value = torch.randn(1, n_kv, pages * page, D, generator=g)
    mgr = PackedKVManager([levels], n_kv, n_kv, D, page, kg, vg, bit_v, gpu)
    mgr.commit(0, key.to(gpu), value.to(gpu))
    k, v = mgr.layers[0].dequantize(0)
    store = oracle_store(levels, f32(key[0]), f32(value[0]), page, kg, vg, bit_v)
    ref_k, ref_v = store.dequantize()
    assert np.array_equal(k.cpu().numpy(), ref_k) and np.array_equal(v.cpu().numpy(), ref_v)
