"""Queries, keys and values of many tokens at once against the same tokens a few at a time (which `test_sunatar_gpu` holds
against 64-bit arithmetic): values of long runs go into their pages by tiles of 64 tokens and 64 elements from 48 tiles on, and
every number is made by the same operations either way."""
import numpy as np
import pytest
import torch

from test_sunatar_gpu import _ctx

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [32, 385, 1600, 1601])
@pytest.mark.parametrize("heads,groups,n,v,d,blended,behind", [
    (4, 2, 64, 64, 64, False, 0), (3, 3, 16, 20, 32, True, 0), (5, 5, 12, 14, 16, True, 5), (8, 5, 128, 128, 128, False, 64)])
def test_values_by_tiles(dtype, tokens, heads, groups, n, v, d, blended, behind):
    from transformers_neuronx_amd.kernels import make_ops
    ops = make_ops("hip", dtype, DEV)
    g = torch.Generator(device=DEV).manual_seed(tokens + n)
    total = heads * n + groups * (n + v) + behind
    ps = 128
    proj = torch.randn(tokens, total, generator=g, device=DEV)
    first = torch.randn(tokens, groups * v, generator=g, device=DEV) if blended else None
    mix = torch.tensor([0.3], device=DEV)
    qw, kw = (torch.rand(c * n, generator=g, device=DEV) + 0.5 for c in (heads, groups))
    freqs = torch.rand(n // 2, generator=g, device=DEV)
    table = np.array([[(7 * i + 3) % 16 for i in range(16)]], dtype=np.int32)
    made = []
    for portion in (tokens, 19):
        k_pages = torch.full((17, groups, ps, d), 7.0, dtype=dtype, device=DEV)
        v_pages = torch.full((17, groups, d, ps), 7.0, dtype=dtype, device=DEV)
        queries = []
        for a in range(0, tokens, portion):
            b = min(tokens, a + portion)
            ctx = _ctx([b - a], [a + 5], [0], {"g": table}, ps)
            queries.append(ops.qkv_prepare(proj[a:b], heads, groups, n, v, d, qw, kw, 1e-5, freqs, False, 0.37, mix,
                                           first[a:b] if blended else None, ctx, ctx.groups["g"], k_pages, v_pages))
        made.append((torch.cat(queries), k_pages, v_pages))
    for one, few in zip(*made):
        assert torch.equal(one, few)
    assert float(made[0][2][16].float().min()) == 7.0        # a page of no one is not touched
