"""The matrix-core decode of layouts other than 128-token pages and groups (decode_tiled.hip),
against float64 attention over the oracle's dequantised history and against the general kernel."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from logitfill_amd import _native, synth
from logitfill_amd.packed import PackedKVManager
from logitfill_amd.packed.reference import decode_into
from tests.helpers import decode_kernel

pytestmark = pytest.mark.gpu


def _setup(gpu, D, page, kg, vg, n_q, n_kv, lengths, q_len, dtype, tb=3.0, seed=3, levels=None):
    B, T = len(lengths), max(lengths)
    g = torch.Generator().manual_seed(seed)
    levels = synth.sample_tier_levels(n_kv, D, tb, seed) if levels is None else levels
    sigma = synth.channel_sigma(n_kv, D, g)[None, :, None, :]
    key = (torch.randn(B, n_kv, T, D, generator=g) * sigma).to(dtype).to(gpu)
    value = torch.randn(B, n_kv, T, D, generator=g).to(dtype).to(gpu)
    q = (torch.randn(B, n_q, q_len, D, generator=g) * D ** -0.5).to(dtype).to(gpu)
    kn = (torch.randn(B, n_kv, q_len, D, generator=g) * sigma).to(dtype).to(gpu)
    vn = torch.randn(B, n_kv, q_len, D, generator=g).to(dtype).to(gpu)
    mgr = PackedKVManager([levels], n_q, n_kv, D, page, kg, vg, 2, gpu, batch_size=B)
    mgr.commit(0, key, value, lengths)
    return mgr, key, value, q, kn, vn


def _float64(mgr, q, kn, vn):
    """Float64 attention over the stored codes (dequantised on the device, exact to fp32)."""
    layer, outs = mgr.layers[0], []
    tk, tv = layer.tail_buffers()
    for b in range(layer.batch):
        k, v = (x.double() for x in layer.dequantize(b))
        tl = layer.tail_lens[b]
        k = torch.cat([k, tk[b, :, :tl].double(), kn[b].double()], 1)
        v = torch.cat([v, tv[b, :, :tl].double(), vn[b].double()], 1)
        n, total = q.shape[2], k.shape[1]
        hidden = torch.arange(total, device=k.device)[None] > torch.arange(n, device=k.device)[:, None] + total - n
        rep = mgr.n_q // mgr.n_kv
        row = []
        for i in range(mgr.n_q):
            s = (q[b, i].double() @ k[i // rep].t()) * mgr.head_dim ** -0.5
            row.append(torch.softmax(s.masked_fill(hidden, -np.inf), -1) @ v[i // rep])
        outs.append(torch.stack(row))
    return torch.stack(outs)


def _decode(mgr, q, kn, vn, kernel, pps=None):
    out = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    decode_into(mgr, 0, q, kn, vn, q.shape[-1] ** -0.5, out, kernel=kernel, pages_per_split=pps)
    torch.cuda.synchronize()
    return out.double()


def _rel(a, b):
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("D,page,kg,vg,n_q,n_kv,lengths,q_len,dtype,pps", [
    (128, 128, 32, 32, 28, 4, [5 * 128 + 17, 128, 60], 1, torch.bfloat16, None),   # one page, none
    (128, 128, 64, 16, 14, 2, [7 * 128, 3 * 128 + 127], 1, torch.float16, 2),      # one word a Value group
    (128, 256, 256, 128, 8, 8, [5 * 256 + 200, 256], 1, torch.float32, 1),         # group past the window
    (128, 96, 96, 64, 12, 2, [11 * 96 + 5, 96], 1, torch.bfloat16, 3),             # runs across groups
    (64, 64, 64, 64, 14, 2, [40 * 64 + 63, 64, 130], 1, torch.bfloat16, None),
    (64, 32, 32, 32, 40, 2, [33 * 32 + 31, 31], 1, torch.float16, 5),              # 20 rows: two tiles
    (256, 128, 128, 256, 8, 4, [4 * 128 + 9], 1, torch.bfloat16, None),
    (256, 64, 32, 64, 16, 1, [9 * 64 + 1, 64], 1, torch.float32, 2),               # 16 rows
    (128, 64, 32, 32, 28, 4, [6 * 64 + 50, 10], 5, torch.bfloat16, None),          # 35 rows, causal
    (64, 128, 128, 64, 14, 2, [2 * 128 + 127], 40, torch.float32, 1),              # residual past 128
    (128, 128, 128, 128, 28, 4, [3 * 128 + 100, 128], 3, torch.float32, None),     # float32 rows
])
def test_tiled_layouts(gpu, D, page, kg, vg, n_q, n_kv, lengths, q_len, dtype, pps):
    """float32 output within 2e-5 of float64 in the 2-norm (fp32 sums over the scores; the largest
    scores here are about 30, whose fp32 spacing alone is 2e-6) and no further off than twice
    the general kernel, which works in plain fp32."""
    mgr, _, _, q, kn, vn = _setup(gpu, D, page, kg, vg, n_q, n_kv, lengths, q_len, dtype)
    want = _float64(mgr, q, kn, vn)
    tiled = _rel(_decode(mgr, q, kn, vn, _native.KERNEL_AUTO, pps), want)
    assert decode_kernel(mgr) == _native.KERNEL_TILED
    plain = _rel(_decode(mgr, q, kn, vn, _native.KERNEL_VALU, pps), want)
    print(f"tiled {tiled:.2e} general {plain:.2e}")
    assert tiled < 2e-5 and tiled < 2 * plain + 1e-7


@pytest.mark.parametrize("level", [0, 1, 2, 3])
def test_tiled_single_tier(gpu, level):
    """Every channel in one tier: the other tiers' regions are empty."""
    levels = np.full((2, 64), level)
    mgr, _, _, q, kn, vn = _setup(gpu, 64, 64, 32, 32, 6, 2, [5 * 64 + 3, 64], 1, torch.bfloat16, levels=levels)
    want = _float64(mgr, q, kn, vn)
    assert _rel(_decode(mgr, q, kn, vn, _native.KERNEL_AUTO), want) < 2e-5
    assert decode_kernel(mgr) == _native.KERNEL_TILED


@pytest.mark.parametrize("D,page,kg,vg,q_len,tail,new,offset", [
    (64, 64, 32, 32, 1, torch.bfloat16, torch.float16, 0),
    (64, 64, 64, 64, 7, torch.float32, torch.float16, 0),
    (128, 128, 32, 32, 1, torch.float16, torch.float32, 0),
    (128, 128, 128, 128, 5, torch.float32, torch.bfloat16, 0),  # the default layout, several tokens
    (128, 64, 32, 64, 40, torch.bfloat16, torch.bfloat16, 1),   # new rows that start off 16 bytes
    (256, 64, 64, 256, 1, torch.bfloat16, torch.float32, 0),
    (256, 128, 64, 64, 6, torch.float16, torch.float16, 3),
])
def test_tiled_residual_rows_of_any_type(gpu, D, page, kg, vg, q_len, tail, new, offset):
    """Residual pages and new tokens of unlike types, or rows off 16 bytes: element by element, with the
    causal mask and, past the tail, rows that are clamped to stored ones."""
    mgr, _, _, q, kn, vn = _setup(gpu, D, page, kg, vg, 8, 2, [3 * page + 17, 2 * page + 1, page], q_len, tail)
    q = q.to(new)
    kn, vn = (torch.zeros(t.numel() + offset, dtype=new, device=gpu)[offset:].view_as(t).copy_(t) for t in (kn, vn))
    assert (kn.data_ptr() % 16 != 0) == (offset > 0)
    want = _float64(mgr, q, kn, vn)
    rel = _rel(_decode(mgr, q, kn, vn, _native.KERNEL_AUTO), want)
    assert decode_kernel(mgr) == _native.KERNEL_TILED
    print(f"rel {rel:.2e}")
    assert rel < 2e-5


def test_tiled_infinite_fp16_key(gpu):
    """A Key value past float16 is stored as an infinity: the scores are those of fp32 arithmetic
    (a token at minus infinity weighs nothing), as in the general kernel."""
    levels = np.zeros((1, 64), dtype=np.int64)
    levels[:, 5] = 3
    g = torch.Generator().manual_seed(1)
    key = torch.randn(1, 1, 128, 64, generator=g)
    key[0, 0, 70, 5] = -1e5
    mgr = PackedKVManager([levels], 1, 1, 64, 64, 64, 64, 2, gpu)
    mgr.commit(0, key.to(gpu), torch.randn(1, 1, 128, 64, generator=g).to(gpu))
    q = torch.rand(1, 1, 1, 64, generator=g).to(gpu) + 0.1
    kn, vn = (torch.randn(1, 1, 1, 64, generator=g).to(gpu) for _ in range(2))
    a, b = (_decode(mgr, q, kn, vn, k) for k in (_native.KERNEL_AUTO, _native.KERNEL_VALU))
    assert torch.isfinite(a).all() and _rel(a, b) < 2e-5
    _decode(mgr, q, kn, vn, _native.KERNEL_AUTO)
    assert decode_kernel(mgr) == _native.KERNEL_TILED


def test_general_kernel_group_of_one_and_a_half_chunks(gpu):
    """Key groups of 96 tokens, which the general kernel's 64-token chunks do not divide."""
    mgr, _, _, q, kn, vn = _setup(gpu, 128, 96, 96, 64, 12, 2, [11 * 96 + 5, 96], 1, torch.bfloat16)
    assert _rel(_decode(mgr, q, kn, vn, _native.KERNEL_VALU, 3), _float64(mgr, q, kn, vn)) < 2e-5
