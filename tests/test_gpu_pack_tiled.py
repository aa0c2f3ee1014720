"""The tiled page packer (pack_tile_kernel) bit-exact against the oracle at the layouts where its
blocks, pieces and groups change, and for values at the ends of the quantiser's range."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from logitfill_amd import _native
from logitfill_amd.packed import PackedKVManager
from tests.helpers import assert_history_equal, f32, oracle_store, pack_kernel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,page,kg,vg,bit_v,dtype", [
    (64, 32, 32, 32, 2, torch.bfloat16),      # one 32-token block, units for half the threads
    (128, 64, 32, 64, 4, torch.float16),      # two groups a block
    (128, 128, 32, 32, 8, torch.bfloat16),    # two blocks a page
    (128, 192, 96, 128, 2, torch.bfloat16),   # groups of three pieces
    (256, 128, 128, 256, 2, torch.float16),   # four pieces a thread
    (64, 64, 64, 64, 2, torch.bfloat16),      # the page-major scale copy
    (128, 128, 128, 128, 16, torch.float16),  # fp16 Values
])
def test_tiled_pack_bit_exact(gpu, D, page, kg, vg, bit_v, dtype):
    rng = np.random.default_rng(D + kg + bit_v)
    levels = rng.choice(4, size=(2, D), p=[0.5, 0.25, 0.15, 0.1])
    levels[1] = np.sort(levels[1])            # (heads with other counts: padding slots)
    g = torch.Generator().manual_seed(page)
    x = torch.randn(2, 2, 2, 3 * page, D, generator=g)
    x[0, 0, :, :page] *= 1e-6                 # scales at the lower clamp
    x[:, 1, 0, page:2 * page] = 0.75          # constant groups
    x[:, 1, 1, :page] = torch.randint(-8, 9, (page, D), generator=g) * 0.25  # ties
    if dtype == torch.bfloat16:
        x[1, 1, 0, 5, 3] = 3e38               # a range past the upper clamp
        x[1, 0, 1, 7, 2] = -1e6
    key, value = x[0].to(dtype), x[1].to(dtype)
    mgr = PackedKVManager([levels], 2, 2, D, page, kg, vg, bit_v, gpu, batch_size=2)
    key_d, value_d = key.to(gpu), value.to(gpu)
    # (128-channel heads with pages and Key groups of 128 and fp16 Values are not the fast packer's)
    assert pack_kernel(mgr, key_d, value_d) == _native.PACK_TILED
    mgr.commit(0, key_d, value_d)
    for b in range(2):
        with np.errstate(over="ignore"):
            store = oracle_store(levels, f32(key[b]), f32(value[b]), page, kg, vg, bit_v)
        assert_history_equal(mgr.layers[0], b, store)


def _slot(tier, block, pos):
    """The tier slot at ``pos`` (0..7) of the tier's ``block`` of a page's scale/min copy."""
    r, odd = pos >> 1, pos & 1
    if tier == 0:
        return 16 * (4 * (block >> 3) + (block & 3)) + 4 * (block >> 2 & 1) + r + 8 * odd
    return 8 * block + r + 4 * odd if tier == 1 else 4 * (2 * block + (r >> 1)) + (r & 1) + 2 * odd


@pytest.mark.parametrize("D,page,vg", [(64, 64, 64), (128, 128, 64)])
def test_tiled_scale_copy(gpu, D, page, vg):
    """Where the Key group is the page, the page-major copy holds the reference arrays' scales and mins, each
    at its block and position, and (1, 0) at the positions of no channel."""
    levels = np.random.default_rng(5).choice(4, size=(2, D), p=[0.5, 0.25, 0.15, 0.1])
    levels[1, :D // 4] = 1                       # (heads with unlike tiers)
    mgr = PackedKVManager([levels], 2, 2, D, page, page, vg, 2, gpu)
    x = torch.randn(1, 2, 3 * page, D, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(gpu)
    assert pack_kernel(mgr, x, x) == _native.PACK_TILED
    mgr.commit(0, x, x)
    hist_k, _ = mgr.layers[0].export_reference(0)
    copy = mgr.layers[0].page_scale_copy(0).reshape(2, 3, -1, 2, 8).cpu().numpy()
    words = mgr.layers[0].words
    blocks = [8 * -(-words[0] // 4), 4 * -(-words[1] // 4), 4 * -(-words[2] // 8)]
    assert copy.shape[2] == sum(blocks)
    first = 0
    for t in range(3):
        scale, lo = (hist_k[t][name].cpu().numpy() for name in ("scale", "min"))
        for h in range(2):
            count = int((levels[h] == t).sum())
            for block in range(blocks[t]):
                for pos in range(8):
                    j = _slot(t, block, pos)
                    got = copy[h, :, first + block, :, pos]
                    want = np.stack([scale[h, j], lo[h, j]], 1) if j < count else np.array([[1, 0]] * 3, np.float16)
                    assert np.array_equal(got.view(np.uint16), want.view(np.uint16)), (t, h, block, pos)
        first += blocks[t]


def test_tiled_pack_channel_of_no_tier(gpu):
    """Tables that name fewer channels than the head has: the channel left out changes nothing else."""
    levels = np.random.default_rng(7).choice(4, size=(2, 64), p=[0.5, 0.25, 0.15, 0.1])
    x = torch.randn(1, 2, 128, 64, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(gpu)
    full, part = (PackedKVManager([levels], 2, 2, 64, 64, 32, 64, 2, gpu) for _ in range(2))
    for t in range(4):
        part.layers[0]._tables_dev[t]["count"].sub_(1)  # every tier's last channel
    assert pack_kernel(full, x, x) == _native.PACK_TILED
    for mgr in (full, part):
        mgr.commit(0, x, x)
    (want, want_v), (got, got_v) = (mgr.layers[0].history_views(0) for mgr in (full, part))
    for name in want_v:
        assert torch.equal(want_v[name], got_v[name])
    for t in range(3):
        for h in range(2):
            n = int((levels[h] == t).sum()) - 1
            for name, padding in (("scale", 1.0), ("min", 0.0)):
                assert torch.equal(want[t][name][h, :n], got[t][name][h, :n])
                assert bool((got[t][name][h, n].float() == padding).all())


@pytest.mark.parametrize("D,page,kg,vg,bit_v,dtype", [
    (64, 64, 32, 32, 2, torch.bfloat16),
    (128, 64, 64, 64, 4, torch.float16),
    (128, 96, 96, 32, 8, torch.bfloat16),
])
def test_tiled_pack_not_finite(gpu, D, page, kg, vg, bit_v, dtype):
    """Infinities and NaN: the bytes are those of the general packer, which float32 pages of the same
    values take."""
    levels = np.random.default_rng(D + kg).choice(4, size=(2, D), p=[0.4, 0.3, 0.2, 0.1])
    g = torch.Generator().manual_seed(kg)
    x = torch.randn(2, 1, 2, 3 * page, D, generator=g)
    inf, nan = float("inf"), float("nan")
    x[:, 0, 0, 3, ::3] = inf                 # one infinity in a group, of either sign
    x[:, 0, 0, 7, 1::3] = -inf
    x[:, 0, 0, page:page + kg, 5:40] = inf   # whole groups of one infinity
    x[:, 0, 1, page:page + kg, 5:40] = -inf
    x[:, 0, 1, 4, :] = nan                   # a NaN among finite values, among a large range, alone
    x[:, 0, 1, 5, ::2] = 6e4
    x[:, 0, 1, 6, ::2] = -6e4
    x[:, 0, 0, 2 * page:2 * page + kg, 2:36] = nan
    key, value = x[0].to(dtype).to(gpu), x[1].to(dtype).to(gpu)
    mgr, general = (PackedKVManager([levels], 2, 2, D, page, kg, vg, bit_v, gpu) for _ in range(2))
    assert pack_kernel(mgr, key, value) == _native.PACK_TILED
    assert pack_kernel(general, key.float(), value.float()) == _native.PACK_GENERAL
    mgr.commit(0, key, value)
    general.commit(0, key.float(), value.float())
    (hk, hv), (gk, gv) = (m.layers[0].export_reference(0) for m in (mgr, general))
    for t in range(4):
        for name in hk[t]:
            same = hk[t][name].view(torch.int16) == gk[t][name].view(torch.int16)
            if hk[t][name].dtype == torch.float16:  # (a NaN's payload may differ between the types)
                same |= hk[t][name].isnan() & gk[t][name].isnan()
            assert bool(same.all()), (t, name)
    for name in hv:
        same = hv[name].view(torch.int16) == gv[name].view(torch.int16)
        if hv[name].dtype == torch.float16:
            same |= hv[name].isnan() & gv[name].isnan()
        assert bool(same.all()), name
