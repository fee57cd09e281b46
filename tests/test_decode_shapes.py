"""How the keys of decoding requests are shared out and by how many waves they are read: what a recorded step is sized by."""
import itertools

import pytest


def _rule(longest, fills, alike, pairs, window=0, head_size=64):
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps.__new__(HipOps)
    ops.compute_units = 256
    return ops._splits_for(longest, fills, alike, pairs, window, head_size)


@pytest.mark.parametrize("head_size", [32, 64, 80, 96, 128])
@pytest.mark.parametrize("window", [0, 300, 1024])
def test_growing_batches_meet_few_launches(head_size, window):
    """Every launch that differs is a recording. A batch that grows from one token to the longest allowed meets two at most where
    lengths are unlike, and no more than shares of 256 keys where they are alike."""
    for blocks, n, longest in itertools.product((1, 2, 8, 12, 16, 32), range(1, 49), (100, 700, 2048, 8192)):
        unlike, alike = ({_rule(longest, f, a, n * blocks, window, head_size) for f in range(1, min(8, -(-longest // 256)) + 1)} for a in (False, True))
        assert len(unlike) <= 2, (blocks, n, longest, unlike)
        assert len(alike) <= 8 and (n * blocks < 180 or len(alike) <= 3), (blocks, n, longest, alike)


def test_answers_that_were_measured():
    """The launches that were the quickest of those measured, at 256 units."""
    for want, *args in [((1, 2), 2048, 1, True, 32), ((8, 4), 2048, 8, True, 32), ((1, 8), 2048, 3, True, 160), ((1, 4), 2048, 2, True, 32),
                        ((4, 4), 2048, 8, True, 64, 0, 128), ((2, 4), 2048, 8, True, 96, 0, 128), ((1, 8), 2048, 4, True, 96),
                        ((4, 4), 2048, 8, True, 288), ((4, 2), 2048, 4, True, 288, 0, 128), ((1, 4), 2048, 8, False, 768),
                        ((1, 2), 2048, 2, False, 768), ((1, 2), 2048, 2, False, 768, 0, 80), ((1, 4), 2048, 6, False, 768, 0, 128),
                        ((1, 4), 2048, 8, True, 256), ((1, 4), 2048, 3, True, 288)]:
        assert _rule(*args) == want, args
