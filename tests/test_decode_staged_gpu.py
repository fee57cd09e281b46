"""The decode attention that stages keys and values in LDS: every count of waves a block and share of the keys, at lengths around the
edges of tiles of 64 keys, shares and waves; and the rule that chooses them."""
import itertools

import pytest
import torch

DEV = "cuda:0"
LENGTHS = [1, 63, 64, 65, 128, 129, 255, 257, 513, 700]


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,hs,ps", [(3, 3, 32, 64), (4, 4, 64, 64), (4, 1, 64, 128), (3, 3, 80, 64), (4, 2, 80, 256), (2, 2, 96, 64),
                                            (2, 2, 128, 64), (6, 2, 128, 128), (34, 2, 64, 64), (2, 2, 64, 32), (2, 2, 112, 64)])
@pytest.mark.parametrize("window", [None, 100])
def test_waves_and_shares_agree(heads, kv, hs, ps, window):
    from test_kernels_gpu import _fill_cache_and_compare
    from transformers_neuronx_amd.kernels.hip import HipOps
    ctx, q, kp, vp, _ = _fill_cache_and_compare(torch.bfloat16, heads, kv, hs, ps, [1] * len(LENGTHS), [n - 1 for n in LENGTHS], window)
    view = ctx.groups["full"]
    plain = HipOps(torch.bfloat16, DEV)
    plain.force_plain_attention = True
    want = plain.attention(q, heads, kv, hs, ctx, view, kp, vp, window).float()
    for splits, waves in itertools.product((1, 3, 8), (2, 4, 8)):
        ops = HipOps(torch.bfloat16, DEV)
        ops._splits_for = lambda *a: (splits, waves)
        got = ops.attention(q, heads, kv, hs, ctx, view, kp, vp, window).float()
        # probabilities are rounded to bfloat16 (2^-9 of each, against a sum of the unrounded) and so is the result: as the other
        # ways of making it are compared
        torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("head_size", [64, 80, 128])
@pytest.mark.parametrize("window", [0, 1024])
def test_the_rule_gives_launches_that_exist(head_size, window):
    """(What it answers at the sizes that were measured: `test_decode_shapes.py`.)"""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps.__new__(HipOps)
    ops.compute_units = 256
    for pairs, longest, alike in itertools.product((1, 8, 32, 96, 128, 160, 256, 257, 288, 384, 512, 768, 2048), (1, 100, 256, 257, 700, 2048, 8192), (True, False)):
        fills = min(8, -(-longest // 256))
        splits, waves = ops._splits_for(longest, fills, alike, pairs, window, head_size)
        assert waves in ((2, 4) if head_size > 80 else (2, 4, 8)) and 1 <= splits <= 8
        # no share without keys of the longest request's, and no more shares than units where the pairs leave some idle
        assert splits <= max(1, fills) and (splits == 1 or splits * pairs <= 256 or pairs > 256)


@pytest.mark.gpu
@pytest.mark.parametrize("hs", [64, 128])
def test_pages_that_begin_anywhere(hs):
    """Pages of 64 keys that do not begin on 16 bytes: the keys and values go through registers, with the same results."""
    from test_kernels_gpu import _fill_cache_and_compare
    from transformers_neuronx_amd.kernels.hip import HipOps
    ctx, q, kp, vp, _ = _fill_cache_and_compare(torch.bfloat16, 2, 2, hs, 64, [1] * len(LENGTHS), [n - 1 for n in LENGTHS], None)

    def moved(pages):
        room = torch.empty(pages.numel() + 4, dtype=pages.dtype, device=DEV)
        return room[4:].view(pages.shape).copy_(pages)

    assert moved(kp).data_ptr() % 16 == 8
    ops = HipOps(torch.bfloat16, DEV)
    ops._splits_for = lambda *a: (2, 4)
    view = ctx.groups["full"]
    got = [ops.attention(q, 2, 2, hs, ctx, view, k, v).float() for k, v in ((kp, vp), (moved(kp), moved(vp)), (kp, moved(vp)))]
    # (the same products and sums in the same order)
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])
