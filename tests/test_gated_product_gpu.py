"""Gated products that make their gates themselves, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(ops, m, f, k, act, limit, entry):
    g = torch.Generator(device=DEV).manual_seed(m + f + k)
    h = torch.randn(m, k, device=DEV, generator=g).bfloat16()
    raw = (torch.randn(2 * f, k, device=DEV, generator=g) * k ** -0.5).bfloat16()
    w = ops.prepare_weight(raw)
    ran = []
    call = ops._call
    ops._call = lambda module, name, *a, **kw: (ran.append(name), call(module, name, *a, **kw))[1]
    got = ops.gated_product(h, w, act, limit)
    assert (ran == [entry] if entry else ran[-1] == "tnx_gated_activation") and got.shape == (m, f) and got.dtype == torch.bfloat16
    z = h.double() @ raw.double().T
    a, u = z[:, :f], z[:, f:]
    if act == "silu":
        want = a * torch.sigmoid(a) * u
    elif act == "gelu_new":
        want = torch.nn.functional.gelu(a, approximate="tanh") * u
    else:
        a, u = a.clamp(max=limit), u.clamp(-limit, limit)
        want = a * torch.sigmoid(1.702 * a) * (u + 1)
    # one rounding to bfloat16 (2^-9 of a value), and float32 sums of up to 4,160 terms beside it
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()


ACTS = [("silu", None), ("gelu_new", None), ("clamped_swiglu", 0.7)]


@pytest.mark.parametrize("act,limit", ACTS)
@pytest.mark.parametrize("m", [1, 7, 16, 17, 32])
@pytest.mark.parametrize("f,k", [(16, 128), (48, 256), (1040, 640), (512, 4096)])
def test_few_rows(m, f, k, act, limit):
    from transformers_neuronx_amd.kernels.hip import HipOps
    _check(HipOps(torch.bfloat16, DEV), m, f, k, act, limit, "tnx_gated_activation_skinny")


@pytest.mark.parametrize("act,limit", ACTS)
@pytest.mark.parametrize("m,f,k", [(129, 64, 64), (200, 192, 128), (255, 4160, 192), (300, 8256, 64), (511, 8192, 128), (1100, 4096, 320), (2049, 1088, 64)])
def test_tiles(m, f, k, act, limit):
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps(torch.bfloat16, DEV)
    ops.gated_tiles_share = 0
    _check(ops, m, f, k, act, limit, "tnx_gated_activation_tiles")


@pytest.mark.parametrize("m,f,k,entry", [
    (16, 4096, 4096, "skinny"), (32, 4096, 2048, "skinny"), (32, 4096, 4096, None),             # 2^25 elements, 17 rows and more
    (33, 512, 256, None), (128, 2048, 512, None), (129, 2048, 512, "tiles"),                    # the rows between
    (200, 1920, 192, None), (200, 1984, 192, "tiles"), (256, 2048, 64, "tiles"),                # a quarter of 256 units,
    (300, 1408, 2048, None), (396, 1408, 2048, "tiles"), (256, 4096, 2560, None), (300, 2816, 2560, "tiles"),       # a third, a half
    (1100, 4096, 2048, "tiles"), (1100, 4096, 2112, None), (1100, 3584, 2112, "tiles")])        # more than one a unit, and K
def test_either_side_of_the_lines(m, f, k, entry):
    """The rule as it stands, at sizes where it turns, and the general way beyond."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps(torch.bfloat16, DEV)
    ops.compute_units = 256
    _check(ops, m, f, k, "silu", None, entry and f"tnx_gated_activation_{entry}")
