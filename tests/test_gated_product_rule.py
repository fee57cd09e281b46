"""Which gated products make their gates themselves, and what these refuse."""
import pytest
import torch


def _ops():
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps.__new__(HipOps)
    ops.compute_units, ops.dtype = 256, torch.bfloat16
    return ops


def test_matrices_not_on_the_gpu_are_refused(monkeypatch):
    from transformers_neuronx_amd.kernels import hip
    ops, h = _ops(), torch.randn(200, 64).bfloat16()
    want, calls = hip._want, []
    monkeypatch.setattr(hip, "_want", lambda t, *a: t if t is h else want(t, *a))       # (as if the rows were there)
    ops._call = lambda *a, **k: calls.append(a)
    with pytest.raises(ValueError, match="on the GPU"):
        ops.gated_product(h, torch.zeros(2 * 8192, 64, dtype=torch.bfloat16), "silu")
    assert not calls
