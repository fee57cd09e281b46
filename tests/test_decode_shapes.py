"""How the keys of decoding requests are shared out and by how many waves they are read: what a recorded step is sized by."""
import itertools

import numpy as np
import pytest


def _rule(longest, fills, alike, pairs, window=0, head_size=64, staged=True):
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps.__new__(HipOps)
    ops.compute_units = 256
    return ops._splits_for(longest, fills, alike, pairs, window, head_size, staged)


@pytest.mark.parametrize("head_size,staged", [(32, True), (64, True), (80, True), (96, True), (128, True), (64, False), (112, False), (256, False)])
@pytest.mark.parametrize("window", [0, 300, 1024])
def test_growing_batches_meet_few_launches(head_size, staged, window):
    """Every launch that differs is a recording. A batch that grows from one token to the longest allowed meets two at most where
    lengths are unlike, and no more than shares of 256 keys where they are alike."""
    for blocks, n, longest in itertools.product((1, 2, 8, 12, 16, 32), range(1, 49), (100, 700, 2048, 8192)):
        unlike, alike = ({_rule(longest, f, a, n * blocks, window, head_size, staged) for f in range(1, min(8, -(-longest // 256)) + 1)} for a in (False, True))
        assert len(unlike) <= 2, (blocks, n, longest, unlike)
        assert len(alike) <= 8 and (n * blocks < 180 or len(alike) <= 3 or not staged), (blocks, n, longest, alike)


def test_answers_that_were_measured():
    """The launches that were the quickest of those measured, at 256 units."""
    for want, *args in [((1, 2), 2048, 1, True, 32), ((1, 4), 2048, 1, True, 32, 0, 80), ((1, 4), 2048, 1, True, 32, 0, 128), ((1, 2), 2048, 1, True, 768), ((8, 4), 2048, 8, True, 32), ((1, 8), 2048, 3, True, 160), ((1, 4), 2048, 2, True, 32),
                        ((4, 4), 2048, 8, True, 64, 0, 128), ((2, 4), 2048, 8, True, 96, 0, 128), ((1, 8), 2048, 4, True, 96),
                        ((4, 4), 2048, 8, True, 288), ((4, 2), 2048, 4, True, 288, 0, 128), ((1, 4), 2048, 8, False, 768),
                        ((1, 2), 2048, 2, False, 768), ((1, 2), 2048, 2, False, 768, 0, 80), ((1, 4), 2048, 6, False, 768, 0, 128),
                        ((1, 4), 2048, 8, True, 256), ((1, 4), 2048, 3, True, 288)]:
        assert _rule(*args) == want, args


def test_launches_that_do_not_stage():
    """Pages under 64 keys and other heads: no block of two waves (there is none), shares as before where keys are many, whole requests
    where they are few; and the launch that a recorded step is known by is the one it makes."""
    import torch
    from transformers_neuronx_amd.kernels.hip import HipOps
    for longest, fills, alike, pairs, window, head_size in itertools.product((100, 2048), range(1, 9), (True, False), (1, 32, 96, 160, 256, 288, 768), (0, 300),
                                                                             (16, 48, 64, 112, 128, 256)):
        splits, waves = _rule(longest, fills, alike, pairs, window, head_size, False)
        assert waves in ((4, 8) if head_size <= 128 else (4,)) and 1 <= splits <= 8
    for want, *args in [((8, 4), 2048, 8, True, 96, 0, 64), ((4, 4), 2048, 4, True, 288, 0, 64), ((4, 4), 2048, 4, True, 1056, 0, 64),
                        ((8, 4), 2048, 8, True, 160, 0, 112), ((2, 4), 2048, 2, True, 16, 0, 256), ((1, 4), 2048, 2, True, 288, 0, 80),
                        ((1, 8), 2048, 4, True, 160, 0, 80), ((1, 4), 2048, 8, False, 768, 0, 64), ((3, 4), 2048, 8, False, 96, 0, 64)]:
        assert _rule(*args, False) == want, args

    class Step:
        run_lens, plan_host, length_bound = np.ones(9, int), {"decode_shape": (4, True)}, 2048

    ops = HipOps.__new__(HipOps)
    ops.compute_units, ops.dtype = 256, torch.bfloat16
    for Step.page_size, shape in ((16, (4, 4)), (32, (4, 4)), (64, (1, 4)), (256, (1, 4))):
        assert ops.attention_launch_shape(Step, 32, None, 64) == ("decode", 32, 64) + shape
    Step.page_size = 64
    assert ops.attention_launch_shape(Step, 32, None, 48)[-2:] == (4, 4)
