"""What a router's product refuses before it reads anything."""
import pytest
import torch


@pytest.mark.parametrize("experts", [0, 5, 20])
def test_experts_beyond_the_matrix_are_refused(experts):
    """Either side of the sizes that go out in one launch, by both backends: the kernel reads as many rows as there are experts."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    from transformers_neuronx_amd.kernels.reference import ReferenceOps
    h, w = torch.randn(3, 64).bfloat16(), torch.randn(4, 64).bfloat16()
    calls = []
    ops = HipOps.__new__(HipOps)
    ops.route = ops.linear = ops._call = lambda *a, **k: calls.append(a)
    for of in (ops, ReferenceOps(torch.bfloat16)):
        with pytest.raises(ValueError, match="4 rows"):
            of.route_product(h, w, None, experts, 1)
    assert not calls


@pytest.mark.parametrize("matrix", [torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(4, 64, 2, dtype=torch.bfloat16)])
def test_matrices_not_on_the_gpu_are_refused(matrix, monkeypatch):
    """Nor may one of other dimensions be read as if it had two."""
    from transformers_neuronx_amd.kernels import hip
    ops, h = hip.HipOps.__new__(hip.HipOps), torch.randn(3, 64).bfloat16()
    want, calls = hip._want, []
    monkeypatch.setattr(hip, "_want", lambda t, *a: t if t is h else want(t, *a))       # (as if the rows were there)
    ops._call = lambda *a, **k: calls.append(a)
    with pytest.raises(ValueError):
        ops.route_product(h, matrix, None, 4, 2)
    assert not calls
