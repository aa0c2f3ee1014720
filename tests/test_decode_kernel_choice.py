"""Which kernel a decode call takes (lf_decode_kernel, host code, no GPU) and the split plan's rule for
it: one choice, asked by the launch and by the planner."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from logitfill_amd import _native
from logitfill_amd.packed.layout import sm_page_elems
from logitfill_amd.packed.reference import choose_pages_per_split, fit_scratch, plan_rule

VALU, MFMA, ROWS, TILED = (_native.KERNEL_VALU, _native.KERNEL_MFMA, _native.KERNEL_ROWS, _native.KERNEL_TILED)
AT = 1 << 20  # an address (nothing reads it)


def _layer(D=128, page=128, kg=128, vg=128, widths=(72, 28, 20, 8), bit_v=2, n_kv=1):
    words = [-(-w // per) for w, per in zip(widths, (16, 8, 4))]
    L = _native.PackedLayer()
    for t in range(3):
        L.k_code[t], L.k_scale[t], L.k_min[t] = AT, AT, AT
        L.k_words[t] = words[t]
    for t in range(4):
        L.tier_index[t], L.tier_count[t] = AT, AT
        L.k_width[t] = widths[t]
    L.k_value16 = L.v_code = L.v_scale = L.v_min = L.v_value16 = AT
    if page == kg and sm_page_elems(words):
        L.k_sm_page = AT
    L.batch, L.n_kv, L.head_dim, L.page_size, L.k_group, L.v_group, L.bit_v = 1, n_kv, D, page, kg, vg, bit_v
    L.cap_tokens, L.cap_kgroups = 1024 * page, 1024 * page // kg
    L.v_words, L.v_groups = -(-D * bit_v // 32), D // vg
    return L


def _call(q="bf16", new="bf16", tail="bf16", n_q=7, q_len=1, kernel=0, q_at=AT, new_at=AT, page=128):
    code = {"bf16": _native.LF_BF16, "fp16": _native.LF_FP16, "fp32": _native.LF_FP32}
    a = _native.DecodeArgs()
    a.query, a.q_dtype, a.out_dtype = q_at, code[q], code[q]
    if new:
        a.k_new, a.v_new, a.new_dtype = new_at, new_at, code[new]
    if tail:
        a.tail_k, a.tail_v, a.tail_dtype, a.tail_cap = AT, AT, code[tail], page
    a.n_q, a.q_len, a.kernel, a.scaling = n_q, q_len, kernel, 0.1
    return a


@pytest.mark.parametrize("layer,call,pages,want", [
    ({}, {}, 500, MFMA),
    ({}, {"n_q": 40}, 5000, MFMA),                                # five tiles of 8 rows
    ({}, {"n_q": 41}, 500, ROWS),                                 # six, 3 000 page-tiles
    ({}, {"n_q": 41}, 499, MFMA),
    ({}, {"n_q": 8, "q_len": 6}, 500, ROWS),
    ({}, {"n_q": 48, "q": "fp16", "new": "fp16", "tail": "fp16"}, 500, ROWS),
    ({}, {"n_q": 48, "tail": "fp16"}, 500, MFMA),                 # rows of two types
    ({}, {"n_q": 48, "tail": "fp32"}, 500, MFMA),
    ({}, {"n_q": 8, "q_len": 6, "tail": "fp32"}, 500, TILED),     # ... of several tokens
    ({}, {"n_q": 48, "q": "fp32", "new": "fp32", "tail": "fp32"}, 500, MFMA),
    ({}, {"n_q": 48, "q_at": AT + 2}, 500, MFMA),                 # q off 16 bytes
    ({}, {"n_q": 48, "new_at": AT + 2}, 500, TILED),              # new rows off 16 bytes
    ({}, {"n_q": 48, "new": None, "tail": None}, 500, ROWS),
    ({"widths": (30, 4, 4, 90)}, {"n_q": 48}, 500, MFMA),         # fp16 tier of 90 channels
    ({"widths": (70, 100, 100, 2)}, {"n_q": 48}, 500, MFMA),       # over ten K-steps (heads of unlike tiers)
    ({}, {"n_q": 48, "kernel": 2}, 500, MFMA),
    ({}, {"kernel": 1}, 500, VALU),
    ({"kg": 32}, {}, 500, TILED),
    ({"kg": 32}, {"kernel": 2}, 500, _native.LF_E_UNSUPPORTED),
    ({"kg": 16}, {}, 500, VALU),
    ({"D": 64, "page": 64, "kg": 64, "vg": 64, "widths": (40, 12, 8, 4)}, {"page": 64}, 500, TILED),
    ({"D": 256, "page": 64, "kg": 32, "vg": 8, "widths": (160, 48, 32, 16)}, {"page": 64}, 500, VALU),
    ({"D": 32, "vg": 32, "widths": (20, 6, 4, 2)}, {}, 500, VALU),
    ({"bit_v": 4}, {}, 500, _native.LF_E_UNSUPPORTED),
])
def test_kernel_of_a_call(layer, call, pages, want):
    assert _native.load().lf_decode_kernel(_layer(**layer), _call(**call), pages) == want


def _rule(n_q, q_len, q_dtype, new_dtype, tail_dtype, pages, kernel=0, q_at=AT, **layer):
    struct = _layer(**layer)
    tail = None if tail_dtype is None else torch.empty(1, 1, struct.page_size, struct.head_dim, dtype=tail_dtype)
    store = SimpleNamespace(page_size=struct.page_size, head_dim=struct.head_dim, n_kv=1,
                            tail_buffers=lambda: (tail, tail), layer_struct=lambda: struct)
    manager = SimpleNamespace(n_q=n_q, n_kv=1)
    call = ((pages,), q_len, kernel, q_dtype, new_dtype)
    return plan_rule(manager, store, call, q_at, AT if new_dtype else 0, AT if new_dtype else 0)


def test_plan_follows_the_kernel():
    """The one-workgroup-per-CU plan is made only for calls that the many-row kernel takes."""
    bf, fp16, fp32 = torch.bfloat16, torch.float16, torch.float32
    rule = _rule(48, 1, bf, bf, bf, 500)
    assert rule.kernel == ROWS and rule.per_cu == 1 and rule.tiles == 1 and rule.residual(100, 1) == 2
    assert _rule(130, 1, bf, bf, bf, 500).tiles == 2 and not rule.dispatch_order
    for other in (_rule(48, 1, bf, bf, fp16, 500), _rule(48, 1, bf, bf, bf, 500, q_at=AT + 2),
                  _rule(48, 1, fp32, fp32, fp32, 500), _rule(48, 1, bf, bf, bf, 400),
                  _rule(48, 1, bf, bf, bf, 500, widths=(30, 4, 4, 90))):
        assert other.kernel == MFMA and other.per_cu == 2 and other.tiles == 6 and not other.one_round
    rule = _rule(8, 1, bf, bf, bf, 500)
    assert rule.kernel == MFMA and rule.dispatch_order and rule.residual(100, 1) == 4
    for n_q, tiles in ((8, 1), (16, 2), (20, 3), (32, 4), (36, 5)):
        rule = _rule(n_q, 1, bf, bf, bf, 100)
        assert rule.tiles == tiles and rule.one_round == (tiles in (1, 2, 4))
    rule = _rule(8, 6, bf, bf, fp32, 500)     # rows of two types, several tokens
    assert rule.kernel == TILED and rule.per_cu == 2 and not rule.one_round and not rule.dispatch_order
    assert _rule(8, 1, bf, bf, bf, 500, kg=32).kernel == TILED
    assert _rule(8, 1, bf, bf, bf, 500, kg=32, kernel=2).kernel == MFMA  # refused by the launch


@pytest.mark.parametrize("pages,n_q,q_len,layer,want", [
    # head_dim 32, 16-row tiles: two kv heads' worth of the work below runs as one-page items
    ([39, 25, 21, 34, 25, 20, 36, 24], 7, 1, {"D": 32, "vg": 32, "widths": (20, 6, 4, 2)}, 1),
    ([39, 25, 21, 34, 25, 20, 36, 24], 7, 3, {"D": 32, "vg": 32, "widths": (20, 6, 4, 2)}, 1),
    ([62, 35, 28, 53, 36, 25, 56, 32], 4, 1, {"D": 16, "page": 64, "kg": 64, "vg": 16, "widths": (10, 3, 2, 1)}, 1),
    ([187, 109, 173, 63], 7, 1, {"page": 16, "kg": 16, "vg": 32}, 1),
    ([600] * 8, 7, 1, {"page": 16, "kg": 16, "vg": 32}, 5),            # 4 800 pages: 1 024 slots once
])
def test_general_kernel_items_stay_small(pages, n_q, q_len, layer, want):
    """The general kernel's plan: small items, up to four workgroups per CU (with the matrix-core
    kernels' per-item cost it took items of 3 to 16 pages here, up to four times slower)."""
    bf = torch.bfloat16
    rule = _rule(n_q, q_len, bf, bf, bf, sum(pages), **layer)
    assert rule.kernel == VALU and rule.tiles == -(-n_q * q_len // 16)
    res = rule.residual(50 % rule.page_size, q_len)
    assert res == 1
    assert choose_pages_per_split(pages, rule.tiles, res, None, rule.page_elems, rule.per_cu, rule.one_round,
                                  rule.overhead) == want


def test_plan_of_a_call_that_allocates_nothing_fits_its_scratch():
    limit = _native.load().lf_noalloc_scratch_bytes()
    assert fit_scratch(1, [100] * 8, 1, limit // 1000) == 1
    assert fit_scratch(1, [100] * 8, 1, limit // 500) == 2
    assert fit_scratch(3, [100, 0, 40], 1, limit // 10) == 24           # 5 + 1 + 2 items
    assert fit_scratch(1, [100] * 8, 1, limit) >= 101                    # cannot fit: one item a sequence
