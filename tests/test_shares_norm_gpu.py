"""The shares of a product's sums added by the launch of the norm behind it (`HipOps.onto`, `SharesLeft`): the same bits as the sum
and the norm by launches of their own."""
import pytest
import torch

from transformers_neuronx_amd.engine.batch import StepEntry

DEV = "cuda:0"
BF16, F32 = torch.bfloat16, torch.float32


def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("shares,tokens,width", [(2, 1, 4), (3, 17, 1020), (4, 5, 1024), (5, 3, 1028), (8, 24, 2048), (9, 7, 2052),
                                                 (16, 4, 2560), (2, 33, 3072), (7, 2, 3076), (13, 3, 4096), (8, 600, 512)])
def test_sizes(shares, tokens, width, dtype):
    from transformers_neuronx_amd.kernels.hip import HipOps, SharesLeft
    hip, g = HipOps(dtype, DEV), _gen(shares + tokens + width)
    parts = torch.randn(shares, tokens, width, device=DEV, generator=g)
    bias, weight, shift = (torch.randn(width, device=DEV, generator=g) for _ in "abc")
    residual = 3 + torch.randn(tokens, width, device=DEV, generator=g)
    for add, w, b, center in ((bias, weight, shift, True), (None, weight, None, False), (bias, None, None, True), (None, weight, shift, False)):
        def left():
            return SharesLeft(hip, parts, shares, add, residual, torch.full((tokens, width), float("nan"), device=DEV))
        whole = left()
        want = whole.settled()
        total = parts[0].clone()                     # the shares in their order, then bias, then residual
        for part in parts[1:]:
            total += part
        assert torch.equal(want, (total + add if add is not None else total) + residual)
        norm = hip.layernorm(want, w, b, 1e-5, dtype, False, True, center)[1]
        x, h = left().normed(w, b, 1e-5, dtype, center)
        assert torch.equal(x, want) and torch.equal(h, norm) and h.dtype == dtype
        x, h = left().normed(w, b, 1e-5, dtype, center, alone=True)
        assert torch.equal(x, hip.layernorm(want, w, b, 1e-5, dtype, True, False, center)[0]) and torch.equal(h, norm)
        x, h = left().normed(w, b, torch.tensor(1e-5), dtype, center)           # (any number, as the norm's own launch takes)
        assert torch.equal(x, want) and torch.equal(h, norm)
        x, h = whole.normed(w, b, 1e-5, dtype, center)                          # one that was added already
        assert x is want and torch.equal(h, norm)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,m,n,k", [(BF16, 17, 2560, 10240), (BF16, 48, 1024, 4096), (BF16, 333, 2048, 8192), (BF16, 200, 1024, 4096),
                                         (F32, 17, 1024, 4096), (F32, 600, 2048, 2048), (F32, 100, 768, 768),
                                         # refused: wider than the norm's registers, fewer rows, K whole
                                         (BF16, 32, 5120, 20480), (BF16, 3, 1024, 4096), (BF16, 700, 4096, 512)])
def test_products(dtype, m, n, k):
    """Every way a product shares K out, and results that are whole."""
    from transformers_neuronx_amd.kernels.hip import HipOps, SharesLeft
    hip, g = HipOps(dtype, DEV), _gen(m + n)
    hip._choose_left = lambda *a: None              # the same way with a sum of its own and without
    x = torch.randn(m, k, device=DEV, generator=g).to(dtype)
    w = hip.prepare_weight((torch.randn(n, k, device=DEV, generator=g) * 0.02).to(dtype))
    residual, bias, weight = torch.randn(m, n, device=DEV, generator=g), torch.randn(n, device=DEV, generator=g), torch.randn(n, device=DEV, generator=g)
    want = hip.linear(x, w, bias, residual=residual, out_f32=True)
    norm = hip.layernorm(want, weight, None, 1e-5, dtype, False, True)[1]
    out = hip.linear(x, w, bias, residual=hip.onto(residual), out_f32=True)
    if type(out) is SharesLeft:
        out, h = out.normed(weight, None, 1e-5, dtype, True)
    else:
        assert m <= 16 or k < 1024 or n * k >= 1 << 26
        h = hip.layernorm(out, weight, None, 1e-5, dtype, False, True)[1]
    # (the vendor library's algorithm of a size is one for both)
    assert torch.equal(out, want) and torch.equal(h, norm)
    for act, f32 in (("relu", True), (None, False)):              # sums that a norm may not add: made at once
        assert type(hip.linear(x, w, bias, act, residual=hip.onto(residual) if f32 else None, out_f32=f32)) is torch.Tensor


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,way", [(9, 1024, 4096, (0, 0, 8)), (16, 1024, 1024, None), (17, 1024, 1024, (0, 0, 4)), (32, 768, 768, (0, 0, 3)),
                                       (32, 512, 512, None), (48, 2560, 2560, (0, 0, 5)), (48, 2688, 2688, (0, 0, 5)), (48, 2752, 2688, None),
                                       (48, 3072, 3072, None), (49, 3072, 3072, (1, 1, 5)), (33, 4096, 4096, (1, 1, 4)), (64, 4096, 16384, None),
                                       (65, 1032, 1088, (1, 1, 4)), (256, 2048, 2048, (1, 1, 2)), (257, 2048, 2048, None), (768, 640, 512, (1, 1, 2)),
                                       (769, 640, 512, None), (8, 2048, 8192, None), (100, 4104, 4096, None)])
def test_ways(m, n, k, way):
    """The rule's lines at 256 units, and that the product is right wherever it sends one, for rows that fill no tile as well."""
    from transformers_neuronx_amd.kernels.hip import HipOps, SharesLeft
    hip, g = HipOps(BF16, DEV), _gen(m + n + k)
    x = torch.randn(m, k, device=DEV, generator=g).to(BF16)
    raw = (torch.randn(n, k, device=DEV, generator=g) * 0.02).to(BF16)
    w = hip.prepare_weight(raw)
    hip.compute_units = 256
    if n % 16 == 0 and k % 128 == 0:
        assert hip._choose_left(m, n, k, True) == way
    elif way is not None:
        assert w.tiles is None and hip._choose_left(m, n, k, False) == way
    residual, bias = torch.randn(m, n, device=DEV, generator=g), torch.randn(n, device=DEV, generator=g)
    out = hip.linear(x, w, bias, residual=hip.onto(residual), out_f32=True)
    assert way is None or type(out) is SharesLeft and out.count in (way[2], way[2] - 1)      # (whole steps a share: the last may be none)
    out = hip.settled(out).double()
    want = x.double() @ raw.double().t() + bias.double() + residual.double()
    bound = x.double().abs() @ raw.double().abs().t() + bias.double().abs() + residual.double().abs()
    # k + 2 float32 sums, each off by 2^-24 of at most the sum of the magnitudes
    assert bool(((out - want).abs() <= (k + 2) * 2.0 ** -24 * bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,before", [("bfloat16", True), ("float32", True), ("bfloat16", False), ("float32", False)])
def test_through_the_model(tmp_path, dtype, before):
    """Prompts, a step of both kinds and recorded decode steps: the same logits, bit for bit, and sums that are looked at are made."""
    from transformers_neuronx_amd import debug
    from transformers_neuronx_amd.config.engine_config import EngineConfig
    from transformers_neuronx_amd.engine.factory import runner_from_folder
    from transformers_neuronx_amd.opt.config import OPTConfig
    from transformers_neuronx_amd.weights import write_random_model
    raw = dict(architectures=["OPTForCausalLM"], model_type="opt", vocab_size=640, hidden_size=1024, num_hidden_layers=3, num_attention_heads=16,
               ffn_dim=4096, max_position_embeddings=512, word_embed_proj_dim=1024, do_layer_norm_before=before, activation_function="relu",
               enable_bias=True, layer_norm_elementwise_affine=True, init_std=0.04)
    write_random_model(OPTConfig.from_dict(raw), str(tmp_path), 3, dtype=dtype)
    logits, made = {}, []
    for fused in (True, False, "by the rule"):
        runner = runner_from_folder(str(tmp_path), EngineConfig(dtype=dtype, page_size=64, max_tokens=8192, max_num_seqs=48, device=DEV))
        runner.use_graphs = True
        if fused != "by the rule":
            runner.ops._choose_left = lambda *a: None
        if fused:
            call = runner.ops._call
            runner.ops._call = lambda lib, name, *a, **k: (made.append(name), call(lib, name, *a, **k))[1]
            looked_at = runner
        else:
            runner.ops.onto = lambda x: x
        assert all(layer.block.leaves_shares if before else layer.block.norms_shares for layer in runner.model.layers)
        n = 40
        runner.step([StepEntry(r, [5 + i + r for i in range(9)], []) for r in range(1, n)])
        steps = [[StepEntry(0, [5 + i % 600 for i in range(333)], [332])]]
        steps += [[StepEntry(r, [7 * turn + r], [0]) for r in range(n)] for turn in range(4)]
        steps += [[StepEntry(n, [5 + i for i in range(60)], [59])] + [StepEntry(r, [r], [0]) for r in range(n)]]
        logits[fused] = torch.cat([runner.step(step).float().cpu() for step in steps])
    assert torch.equal(logits[True], logits[False])
    # (sums in another order, rounded to bfloat16 between the products)
    assert float((logits["by the rule"] - logits[False]).norm() / logits[False].norm()) < (0.02 if dtype == "bfloat16" else 1e-6)
    assert "tnx_shares_norm" in made
    assert ("tnx_gemm_shares_sum" in made) == before             # (the last sum is the head's, which has a norm of its own)
    del made[:]
    with debug.debug_context() as kept:
        looked_at.step([StepEntry("more", [5 + i for i in range(60)], [59])])
    assert "tnx_shares_norm" not in made and sum("after_mixer" in name for name in kept) == 3


@pytest.mark.gpu
@pytest.mark.parametrize("m,switches", [(256, [("tile_products", False), ("library_rows", 0)]), (32, [("some_rows", False)])])
def test_switches_turn_for_sizes_seen_before(m, switches):
    """Products of 2,048 x 2,048 by tiles and by rows of some number: off and on again, whatever a size's way was the last time."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g, called = HipOps(BF16, DEV), _gen(m), []
    call = hip._call
    hip._call = lambda lib, name, *a, **k: (called.append(name), call(lib, name, *a, **k))[1]
    x, residual = torch.randn(m, 2048, device=DEV, generator=g).to(BF16), torch.randn(m, 2048, device=DEV, generator=g)
    w = hip.prepare_weight((torch.randn(2048, 2048, device=DEV, generator=g) * 0.02).to(BF16))

    def left():
        del called[:]
        hip.settled(hip.linear(x, w, None, residual=hip.onto(residual), out_f32=True))
        return "tnx_gemm_left" in called
    for name, value in switches:
        kept = getattr(hip, name)
        assert left()
        setattr(hip, name, value)
        assert not left() and (name != "library_rows" or called == ["tnx_gemm_bf16"])
        setattr(hip, name, kept)
        assert left()
        fresh = HipOps(BF16, DEV)
        setattr(fresh, name, value)
        assert fresh._way_to_leave(m, 2048, 2048, True) is None
