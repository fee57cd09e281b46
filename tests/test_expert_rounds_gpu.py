"""The experts' products by tiles of 128 pairs where their tiles go round the units: whole rounds, and what is left over whole, in
halves and in quarters of a tile's columns."""
import pytest
import test_tiles_gpu as tiles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,on", [("silu", "input"), ("relu", "output")])
@pytest.mark.parametrize("width,f", [(1024, 1024), (960, 1088)])
@pytest.mark.parametrize("rounds", [0.1, 0.4, 0.8, 1.06, 1.2, 1.4, 1.6, 2.1])
def test_rounds_of_tiles_and_what_is_left(rounds, width, f, act, on):
    from transformers_neuronx_amd.kernels.hip import HipOps
    import torch
    across = -(-width // 256)          # tiles of the second product's columns
    count = max(3, int(rounds * HipOps(torch.bfloat16, tiles.DEV).compute_units) // across)
    one = (count - 1) // 2
    tiles.test_experts_by_tiles([128 * one, 0, 128 * (count - 1 - one) - 5, 77], width, f, act, on, 0, 128)
