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


def test_lines_of_the_rule():
    """Where it turns: 2^25 elements from 17 rows on, 33 to 128 rows, the part of the units by K, more tiles than units with K beyond 2,048,
    and sizes that the kernels do not take."""
    way = _ops()._gated_way
    for want, *args in [("skinny", 16, 8192, 4096, True), ("skinny", 17, 4080, 4096, True), (None, 17, 4096, 4096, True), ("skinny", 32, 4096, 2048, True),
                        (None, 16, 8192, 4096, False), (None, 16, 4104, 4096, True), (None, 16, 4096, 4160, True), (None, 33, 512, 256, True),
                        (None, 128, 8192, 2048, True), ("tiles", 129, 8192, 2048, True), (None, 200, 1920, 1024, True), ("tiles", 200, 1984, 1024, True),
                        (None, 256, 2048, 1088, True), (None, 300, 1408, 2048, True), ("tiles", 396, 1408, 2048, True), (None, 256, 4096, 2112, True),
                        (None, 256, 4096, 4096, True), ("tiles", 300, 2816, 2560, True), (None, 512, 2048, 4096, True), ("tiles", 560, 2048, 4096, True),
                        ("tiles", 1024, 4096, 4096, True), (None, 1025, 4096, 4096, True), ("tiles", 1025, 4096, 2048, True), (None, 200, 8224, 2048, True),
                        (None, 200, 8192, 2080, True)]:
        assert way(*args) == want, args
