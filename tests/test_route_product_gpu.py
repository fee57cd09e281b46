"""The router's product and its choice in one launch, against the same in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tokens", [1, 7, 300])
@pytest.mark.parametrize("width", [8, 520, 2048, 4104])
@pytest.mark.parametrize("experts,top,groups", [(1, 1, None), (8, 2, None), (13, 5, None), (16, 4, (4, 2)), (16, 16, None)])
@pytest.mark.parametrize("score,renormalize,corrected,biased", [("sigmoid", False, False, False), ("softmax", True, False, True),
                                                               ("sigmoid", True, True, False)])
def test_route_product(tokens, width, experts, top, groups, score, renormalize, corrected, biased):
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator(device=DEV).manual_seed(tokens + width + experts)
    h = torch.randn(tokens, width, device=DEV, generator=g).bfloat16()
    w = (torch.randn(experts + 3, width, device=DEV, generator=g) * width ** -0.5).bfloat16()       # rows behind the router's
    bias = torch.randn(experts + 3, device=DEV, generator=g) if biased else None
    correction = torch.rand(experts, device=DEV, generator=g) if corrected else None
    ran = []
    call = ops._call
    ops._call = lambda module, name, *a, **k: (ran.append(name), call(module, name, *a, **k))[1]
    chosen, weights = ops.route_product(h, w, bias, experts, top, score, renormalize, correction, 1.5, groups)
    assert ran == ["tnx_route_product"]
    z = h.double() @ w[:experts].double().T + (bias[:experts].double() if biased else 0.0)
    s = torch.sigmoid(z) if score == "sigmoid" else torch.softmax(z, -1)
    ranked = s + correction.double() if corrected else z
    if groups:
        best = ranked.view(tokens, groups[0], -1).amax(-1)
        edge = torch.sort(best, descending=True).values
        sure = edge[:, groups[1] - 1] - edge[:, groups[1]] > 1e-4
        ranked = ranked.masked_fill((best < edge[:, groups[1] - 1:groups[1]]).repeat_interleave(experts // groups[0], 1), float("-inf"))
    else:
        sure = torch.ones(tokens, dtype=torch.bool, device=DEV)
    order = torch.sort(ranked, descending=True)
    gaps = torch.nn.functional.pad(order.values[:, :-1] - order.values[:, 1:], (0, 1), value=1.0)
    # (sums of `width` float32 products of size 1 / sqrt(width) are off by 2^-24 of a few units: 1e-4 apart is clear)
    sure &= (gaps[:, :top] > 1e-4).all(-1)
    assert sure.double().mean() > 0.8 or tokens < 300
    assert torch.equal(chosen.long()[sure], order.indices[sure][:, :top])
    want = s.gather(1, chosen.long())
    want = 1.5 * (want / want.sum(-1, keepdim=True) if renormalize else want)
    assert (weights.double() - want).abs().max() < 2e-5
