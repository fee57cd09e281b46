"""What a mixture of experts leaves to the product behind it, against the sum made before that product."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("top", [2, 3, 4])
@pytest.mark.parametrize("t", [1, 5, 16])
@pytest.mark.parametrize("width,f,inner", [(128, 64, 128), (1040, 72, 640), (4096, 128, 256), (8192, 64, 128)])
@pytest.mark.parametrize("on", ["input", "output"])
def test_pairs_left_to_a_product(t, top, width, f, inner, on):
    from transformers_neuronx_amd.kernels.hip import HipOps, PairRows
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator(device=DEV).manual_seed(t + width + top)

    def some(*shape, std=1.0):
        return torch.randn(shape, device=DEV, generator=g) * std

    experts = 6
    chosen = torch.stack([torch.randperm(experts, device=DEV, generator=g)[:top] for _ in range(t)]).int()
    weights, h, x = some(t, top).abs(), some(t, width).bfloat16(), some(t, width)
    up, down = some(experts, 2 * f, width, std=width ** -0.5).bfloat16(), some(experts, width, f, std=f ** -0.5).bfloat16()
    w, z = ops.prepare_weight(some(width, inner, std=inner ** -0.5).bfloat16()), some(t, inner).bfloat16()
    args = (h, chosen, weights, up, down, "silu", on, x)
    left, whole = ops.expert_mixture(*args, before=w), ops.expert_mixture(*args)
    assert isinstance(left, PairRows)
    got, want = ops.linear(z, w, None, residual=left, out_f32=True), ops.linear(z, w, None, residual=whole, out_f32=True)
    assert torch.equal(got, want)            # the same sums in the same order
    assert torch.equal(ops._settled_pairs(ops.expert_mixture(*args, before=w)), whole)
