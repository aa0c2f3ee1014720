"""The merge of sequences with many split items (decode_reduce_many_kernel) against the same decode
in few items, at the item counts where its loops change."""
from __future__ import annotations

import pytest
import torch

from logitfill_amd import _native
from tests.test_gpu_tiled import _decode, _float64, _rel, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,vg,pages", [
    (128, 128, 33),        # the fewest items it takes
    (128, 128, 127),       # 8 groups x 16 loads, full with the residual's item
    (128, 128, 140),       # and items past them
    (64, 64, 300),         # 16 groups: past 256 items
    (256, 64, 70),         # 4 groups: past 64
    (64, 64, 2100),        # more items than the weights kept in LDS (2 048)
])
def test_many_items(gpu, D, vg, pages):
    """One page per item against a plan of few items, next to float64: a sum of a few hundred float32
    terms in another order (5e-6 bounds 2 100 roundings of 2^-24 that add up randomly, x 2).  The
    partials come from the general kernel, whose own error is about 1e-6 for either plan; that of
    decode_mfma.hip is 1e-5 to 1e-4 and depends on the plan."""
    page = 128 if D == 128 else 32
    mgr, _, _, q, kn, vn = _setup(gpu, D, page, page, vg, 6, 2, [pages * page + 5, 3 * page], 1, torch.float16)
    many = _decode(mgr, q, kn, vn, _native.KERNEL_VALU, 1)
    few = _decode(mgr, q, kn, vn, _native.KERNEL_VALU, pages)
    want = _float64(mgr, q, kn, vn)
    assert _rel(many, want) < _rel(few, want) + 5e-6
