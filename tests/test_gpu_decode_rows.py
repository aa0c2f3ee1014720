"""Decode with many query rows per kv head (decode_rows.hip) against float64 attention over the
device's own history, at the edges of its row tiles, K-steps and residual chunks."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from logitfill_amd import _native
from logitfill_amd.packed import PackedKVManager
from logitfill_amd.packed.reference import decode_into
from tests.helpers import decode_kernel
from tests.test_gpu_tiled import _decode, _float64, _rel, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_q,n_kv,lengths,q_len,dtype,tb,pps", [
    (14, 2, [250 * 128 + 40, 128, 60], 9, torch.bfloat16, 3.0, None),    # 63 rows: 64-row tile; no page
    (41, 1, [510 * 128 + 127], 1, torch.float16, 4.0, 100),              # the fewest rows, one token
    (64, 2, [140 * 128, 70 * 128 + 1], 2, torch.bfloat16, 2.5, None),    # exactly 64
    (40, 8, [45 * 128 + 127, 128], 13, torch.float16, 2.5, None),        # 65 rows: 128-row tile
    (28, 4, [6 * 128 + 17, 3 * 128], 130, torch.bfloat16, 3.0, None),    # 910 rows, residual of two chunks
    (8, 8, [12 * 128, 50], 300, torch.float16, 2.5, 1),                  # no GQA, three chunks, no tail / tail
    (64, 1, [520 * 128], 1, torch.bfloat16, 2.5, 520),                   # one long item
])
def test_many_rows(gpu, n_q, n_kv, lengths, q_len, dtype, tb, pps):
    """float32 output within 5e-6 of float64 in the 2-norm (it measures 0.2 to 1.1e-6; decode_mfma.hip,
    which these calls took before, 1 to 6e-5): fp16 hi + lo operands keep 22 bits (2.4e-7 a term) and
    the largest scores here are about 30."""
    mgr, _, _, q, kn, vn = _setup(gpu, 128, 128, 128, 128, n_q, n_kv, lengths, q_len, dtype, tb)
    want = _float64(mgr, q, kn, vn)
    rel = _rel(_decode(mgr, q, kn, vn, _native.KERNEL_AUTO, pps), want)
    print(f"rel {rel:.2e}")
    assert decode_kernel(mgr) == _native.KERNEL_ROWS
    assert rel < 5e-6


@pytest.mark.parametrize("level", [0, 1, 2])
def test_many_rows_single_tier(gpu, level):
    """Every channel in one tier (int8: 32 words a token, 8 K-steps)."""
    mgr, _, _, q, kn, vn = _setup(gpu, 128, 128, 128, 128, 72, 1, [340 * 128 + 3], 1, torch.bfloat16,
                                  levels=np.full((1, 128), level))
    assert _rel(_decode(mgr, q, kn, vn, _native.KERNEL_AUTO), _float64(mgr, q, kn, vn)) < 5e-6
    assert decode_kernel(mgr) == _native.KERNEL_ROWS


def test_many_rows_commit(gpu):
    """The folded commit: the new rows land in the tail, the device length advances, and the output is
    float64 attention's rounded to bf16 (half a unit of 2^-8: 2e-3 in the 2-norm at most)."""
    mgr, _, _, q, kn, vn = _setup(gpu, 128, 128, 128, 128, 28, 4, [80 * 128 + 17], 12, torch.bfloat16)
    layer = mgr.layers[0]
    out = torch.empty_like(q)
    want = _float64(mgr, q, kn, vn)
    assert decode_into(mgr, 0, q, kn, vn, 128 ** -0.5, out, commit=True)
    torch.cuda.synchronize()
    assert decode_kernel(mgr) == _native.KERNEL_ROWS
    assert _rel(out.double(), want) < 2e-3
    tk, tv = layer.tail_buffers()
    assert layer.tail_lens == [29] and layer.tail_len_device().tolist() == [29]
    assert torch.equal(tk[:, :, 17:29], kn) and torch.equal(tv[:, :, 17:29], vn)


# Eight channels of a tier of their own: (tier, Key sigma, q of every second row there, scaling).
RANGES = {
    "fp16_keys_1e-3": (3, 1e-3, 4e3, None),      # stored values below 2^-8
    "fp16_keys_1e-4": (3, 1e-4, 5e3, None),
    "fp16_large_q": (3, 1e-3, 3e4, None),
    "fp16_scaling_1": (3, 1e-2, 800.0, 1.0),
    "int8_large_q": (2, 2e3, 1500.0, None),      # |q| x scale about 65 000
    "int4_large_q": (1, 1e4, 60.0, None),        # ... 300 000
    "plain": (2, 1.0, 0.1, None),
}


@pytest.mark.parametrize("name", RANGES)
def test_many_rows_operand_range(gpu, name):
    """Small fp16-tier Keys keep their bits and large q stay finite, as in decode_mfma.hip: no row
    further from float64 than twice that kernel's furthest on the same call (both sum in float32, in
    another order), plus 2e-6 for the float32 spacing of the scores.  (An overflow leaves a row empty or
    NaN: a distance of 1 or none.)"""
    tier, sigma, level, scaling = RANGES[name]
    scaling = 128 ** -0.5 if scaling is None else scaling
    n_q, T = 48, 505 * 128 + 20
    rng = np.random.default_rng(11)
    levels = np.where(rng.random((1, 128)) < 0.3, 1, 0)
    special = rng.permutation(128)[:8]
    levels[0, special] = tier
    g = torch.Generator().manual_seed(11)
    key, value = (torch.randn(1, 1, T, 128, generator=g) for _ in range(2))
    key[..., special] *= sigma
    q = torch.randn(1, n_q, 1, 128, generator=g) * 128 ** -0.5
    q[:, ::2, :, special] = level * (0.5 + torch.rand(1, n_q // 2, 1, 8, generator=g))
    kn, vn = (torch.randn(1, 1, 1, 128, generator=g) for _ in range(2))
    key, value, q, kn, vn = (t.to(torch.float16).to(gpu) for t in (key, value, q, kn, vn))
    mgr = PackedKVManager([levels], n_q, 1, 128, 128, 128, 128, 2, gpu)
    mgr.commit(0, key, value)
    want = _float64(mgr, q.double() * (scaling * 128 ** 0.5), kn, vn)

    def furthest(kernel):
        out = torch.empty(q.shape, dtype=torch.float32, device=gpu)
        decode_into(mgr, 0, q, kn, vn, scaling, out, kernel=kernel)
        torch.cuda.synchronize()
        assert decode_kernel(mgr) == (_native.KERNEL_MFMA if kernel else _native.KERNEL_ROWS)
        return float(((out.double() - want).norm(dim=-1) / want.norm(dim=-1)).max())

    wide, narrow = furthest(_native.KERNEL_AUTO), furthest(_native.KERNEL_MFMA)
    print(f"{name}: many rows {wide:.2e} decode_mfma {narrow:.2e}")
    assert narrow < 1e-2 and wide < 2 * narrow + 2e-6


@pytest.mark.parametrize("tail,new,q_len,offset,taken", [
    (torch.float32, torch.bfloat16, 1, 0, _native.KERNEL_MFMA),    # residual pages of another type
    (torch.float16, torch.bfloat16, 6, 0, _native.KERNEL_TILED),   # ... and several tokens
    (torch.bfloat16, torch.bfloat16, 1, 1, _native.KERNEL_MFMA),   # q off 16 bytes
])
def test_calls_the_kernel_declines(gpu, tail, new, q_len, offset, taken):
    """Many rows over many pages that the many-row kernel does not take, on a plan for the one that does.
    decode_mfma.hip's sums carry its code offsets (error 1e-5 to 1e-4, by the plan): 2e-4."""
    mgr, _, _, q, kn, vn = _setup(gpu, 128, 128, 128, 128, 48 // q_len, 1, [510 * 128 + 40, 128], q_len, tail)
    q = torch.zeros(q.numel() + offset, dtype=new, device=gpu)[offset:].view_as(q).copy_(q)
    kn, vn = kn.to(new), vn.to(new)
    rel = _rel(_decode(mgr, q, kn, vn, _native.KERNEL_AUTO), _float64(mgr, q, kn, vn))
    assert decode_kernel(mgr) == taken and mgr.layers[0].decode_plan.n_work > 256 // 6
    print(f"rel {rel:.2e}")
    assert rel < (2e-5 if taken == _native.KERNEL_TILED else 2e-4)
