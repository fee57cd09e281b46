"""Layers of a decode step in one launch (`HipOps.decode_layers`) against plain 64-bit arithmetic over the same weights and
cached keys and values, and beside the launches that it stands for."""
import numpy as np
import pytest
import torch

from transformers_neuronx_amd.cache.manager import LayerCache
from transformers_neuronx_amd.engine.batch import StepEntry, build_context
from transformers_neuronx_amd.engine.model import _Layer
from transformers_neuronx_amd.kernels.attention_plan import attention_plan
from transformers_neuronx_amd.parts.base import Stream
from transformers_neuronx_amd.parts.spec import LayerSpec, PartSpec

DEV = "cuda:0"
HEAD = 64
BF16, F32 = torch.bfloat16, torch.float32


def _layer(ops, dtype, width, inner, block, act, bias, seed):
    norm = PartSpec("layer_norm", dict(width=width, eps=1e-5, affine=bias))
    layer = _Layer(LayerSpec(
        prefix="l.", block=block, mixer_norm=norm, feed_forward_norm=norm, mixer_name="a.", feed_forward_name="", mixer_norm_name="n1",
        feed_forward_norm_name="n2",
        mixer=PartSpec("attention", dict(width=width, num_heads=width // HEAD, head_size=HEAD, names=("q", "k", "v", "o"), bias=bias)),
        feed_forward=PartSpec("dense", dict(width=width, inner=inner, activation=act, bias=bias, up_name="up", down_name="down"))))
    gen = torch.Generator().manual_seed(seed)
    tensors = {}
    for d in layer.param_decls():
        t = torch.randn(d.shape, generator=gen) * (1.5 / d.shape[-1] ** 0.5 if d.role == "matrix" else 0.2)
        if d.role != "matrix" and d.init == "around_one":
            t += 1.0
        tensors[d.name] = t.to(DEV).to(dtype if d.role == "matrix" else F32).contiguous()
    layer.load(tensors, ops, dtype)
    return layer, tensors


def _step(ops, dtype, held, width, page_size, seed, layer=0):
    """Requests with `held` cached tokens each, pages dealt out of order (the same for every layer) and some elements apart: (context,
    cache, their plain keys and values)."""
    heads, rows = width // HEAD, len(held)
    pages_of = [n // page_size + 1 for n in held]
    count = sum(pages_of) + 3
    rng = np.random.default_rng(seed)
    order = rng.permutation(count)
    table = np.full((rows, max(pages_of)), -1, dtype=np.int32)
    at = 0
    for i, n in enumerate(pages_of):
        table[i, :n] = order[at:at + n]
        at += n
    gen = torch.Generator().manual_seed(seed + 1 + 1000 * layer)
    pad = 16
    stores = [torch.full((count, heads * page_size * HEAD + pad), float("nan"), dtype=dtype, device=DEV) for _ in range(2)]
    k_pages = stores[0][:, :-pad].view(count, heads, page_size, HEAD)
    v_pages = stores[1][:, :-pad].view(count, heads, HEAD, page_size)
    plain = []
    for i, n in enumerate(held):
        k, v = (torch.randn(n, heads, HEAD, generator=gen).to(dtype) for _ in range(2))
        plain.append((k.double(), v.double()))
        for t in range(n):
            k_pages[table[i, t // page_size], :, t % page_size] = k[t].to(DEV)
            v_pages[table[i, t // page_size], :, :, t % page_size] = v[t].to(DEV)
    entries = [StepEntry(i, [0], [0]) for i in range(rows)]
    ctx = build_context(entries, list(held), list(range(rows)), {"full": table}, page_size, DEV, planners={"attention": attention_plan})
    ctx.memo = {}
    return ctx, LayerCache(0, "full", True, {"k": k_pages, "v": v_pages}), plain


def _norm(v, tensors, name):
    v = v - v.mean(-1, keepdim=True)
    v = v / torch.sqrt(v.square().mean(-1, keepdim=True) + 1e-5)
    if f"l.{name}.weight" not in tensors:
        return v
    return v * tensors[f"l.{name}.weight"].double().cpu() + tensors[f"l.{name}.bias"].double().cpu()


def _exact(tensors, x, plain, width, block, act, before):
    """The layer in 64 bits. `before`: the tensors whose norm stands behind the sum that `x` is (post-norm layers)."""
    def w(name):
        t = tensors.get("l." + name)
        return None if t is None else t.double().cpu()

    def norm(v, name):
        return _norm(v, tensors, name)

    def linear(v, name):
        y = v @ w(name + ".weight").T
        return y if w(name + ".bias") is None else y + w(name + ".bias")

    def part(h):
        q, k, v = (linear(h, "a." + n).view(len(h), -1, HEAD) for n in "qkv")
        rows = []
        for i, (ks, vs) in enumerate(plain):
            ks, vs = torch.cat([ks, k[i:i + 1]]), torch.cat([vs, v[i:i + 1]])
            p = torch.softmax(torch.einsum("hd,thd->ht", q[i], ks) / HEAD ** 0.5, dim=-1)
            rows.append(torch.einsum("ht,thd->hd", p, vs).reshape(-1))
        return linear(torch.stack(rows), "a.o")

    acts = {"relu": torch.relu, "gelu": torch.nn.functional.gelu, "gelu_new": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}
    x = x.double().cpu()
    if block == "pre_norm":
        x = x + part(norm(x, "n1"))
        return x + linear(acts[act](linear(norm(x, "n2"), "up")), "down")
    if before is not None:
        x = _norm(x, before, "n2")
    x = norm(x + part(x), "n1")
    return x + linear(acts[act](linear(x, "up")), "down")


# widths and inner widths: a tile a block and fewer, tiles that not every block has, K that some waves have no step of, K in chunks;
# requests: none cached, the edges of a tile of 64 keys, a page's end, keys cut over blocks (up to eight, some rows and not others)
CASES = [
    (BF16, 512, 256, [5]), (BF16, 512, 128, [0, 1, 63, 64]), (BF16, 640, 1152, [100, 127, 128]), (BF16, 1024, 4096, [100]),
    (BF16, 1024, 4096, [2047]), (BF16, 1024, 4096, [700, 30, 1300, 0]), (BF16, 1024, 4096, [65] * 8), (BF16, 896, 3584, [300, 20]),
    (BF16, 1024, 4096, [1, 900, 64, 129, 513, 63, 10, 200]), (BF16, 512, 2048, [1200, 3, 64, 512]),
    (F32, 512, 256, [5]), (F32, 512, 128, [0, 1, 31, 64]), (F32, 640, 1152, [100, 127, 128]), (F32, 1024, 4096, [60, 61, 62]),
    (F32, 1024, 4096, [1500]), (F32, 1024, 4096, [65, 0, 33, 32, 700, 31, 1, 96]), (F32, 896, 3584, [300, 20]),
    (F32, 1024, 4096, [40] * 5), (F32, 512, 2048, [600, 3, 64, 900]),
]


def _chain(ops, layers, stream, steps):
    for layer, (ctx, cache, _) in zip(layers, steps):
        stream = layer.block.forward(stream, ctx, cache)
    return stream


def _in_one(ops, layers, stream, steps):
    blocks = [layer.block for layer in layers]
    x, first, residual_normed = blocks[0].into_one(stream)
    norms = [(first, blocks[0].norms_in_one(blocks[0])[1])] + [b.norms_in_one(a) for a, b in zip(blocks, blocks[1:])]
    ctx = steps[0][0]
    y = ops.decode_layers([b.in_one for b in blocks], x, norms, residual_normed, ctx, ctx.groups["full"], [cache for _, cache, _ in steps])
    assert y is not None
    return blocks[-1].out_of_one(y)


@pytest.mark.gpu
@pytest.mark.parametrize("block", ["pre_norm", "post_norm", "post_norm behind another"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_layers_in_one_launch(case, block):
    """Three layers. Errors are those of the roundings: float32 sums of up to 8,192 products; bfloat16 operands (2^-9 each, five
    products a layer one after another), which the launches apart have as well: half as much again as theirs is allowed."""
    from transformers_neuronx_amd.kernels.hip import HipOps, NormBetween
    dtype, width, inner, held = CASES[case]
    normed, kind = block.endswith("another"), block.split()[0]
    act, bias = [("relu", True), ("gelu", False), ("gelu_new", True)][case % 3]
    ops = HipOps(dtype, DEV)
    print(f"layers {dtype} {width} {inner} {held} {block}", flush=True)
    made = [_layer(ops, dtype, width, inner, kind, act, bias, 10 + 100 * i + case) for i in range(3)]
    layers = [layer for layer, _ in made]
    assert all(layer.block.in_one is not None for layer in layers)
    norm = layers[-1].block.feed_forward_norm
    weight, vector, center, eps = norm.fused_form()
    x = (torch.randn(len(held), width, generator=torch.Generator().manual_seed(case)) * 2.0 + 0.3).to(DEV)
    results, pages = {}, {}
    for one in (True, False):
        for page_size in (64, 128):
            steps = [_step(ops, dtype, held, width, page_size, 30 + case, i) for i in range(3)]
            if normed:
                n = NormBetween(ops, x, weight, vector, eps, dtype, center)
                stream = Stream(n, n) if one or dtype == BF16 else Stream(*ops.layernorm(x, weight, vector, eps, dtype, True, True))
            else:
                stream = Stream(x, x.to(dtype))
            stream = (_in_one if one else _chain)(ops, layers, stream, steps)
            y = ops.settled(stream.x)
            results[one, page_size] = y.double().cpu()
            pages[one, page_size] = [p.clone() for _, cache, _ in steps for p in (cache.k_pages, cache.v_pages)]
    ops.raise_if_lost()
    exact = x
    tables = [t for _, t in made]
    steps = [_step(ops, dtype, held, width, 64, 30 + case, i) for i in range(3)]
    for i, (tensors, (_, _, plain)) in enumerate(zip(tables, steps)):
        before = tables[i - 1] if i or normed else None
        exact = _exact(tensors, exact, plain, width, kind, act, before if kind == "post_norm" else None)
    if kind == "post_norm":
        exact = _norm(exact, tables[-1], "n2")
    for page_size in (64, 128):
        errors = {one: float((results[one, page_size] - exact).norm() / exact.norm()) for one in (True, False)}
        print(errors, flush=True)
        assert errors[True] <= (1.5 * errors[False] if dtype == F32 else max(1.5 * errors[False], 1e-3)), errors
        for a, b in zip(pages[True, page_size], pages[False, page_size]):
            assert torch.equal(torch.isnan(a), torch.isnan(b))          # the same places are written, and no others
            a, b = (torch.nan_to_num(t.double()) for t in (a, b))
            # (a token's keys and values: each of the two as far from 64 bits as the rows they come from, 0.005 at most, and rounded)
            assert float((a - b).norm() / b.norm()) <= (2e-6 if dtype == F32 else 2 * 0.005 + 2 ** -9)


def _ready(dtype, width, inner, held, seed, layers=3, page_size=64, block="pre_norm"):
    """Layers, and a function that runs them in one launch over caches that no launch has written: (result, pages)."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps(dtype, DEV)
    made = [_layer(ops, dtype, width, inner, block, "relu", True, seed + i)[0] for i in range(layers)]
    x = (torch.randn(len(held), width, generator=torch.Generator().manual_seed(seed)) * 2.0).to(DEV)
    steps = [_step(ops, dtype, held, width, page_size, seed, i) for i in range(layers)]
    return ops, lambda: ops.settled(_in_one(ops, made, Stream(x, x.to(dtype)), steps).x), [p for _, c, _ in steps for p in (c.k_pages, c.v_pages)]


@pytest.mark.gpu
@pytest.mark.parametrize("joined", [1, 5, 16, 40, 127])
@pytest.mark.parametrize("dtype,width,inner,held", [(BF16, 1024, 4096, [1, 900, 64, 129, 513, 63, 10, 200]), (BF16, 640, 1152, [700, 3]),
                                                    (F32, 1024, 4096, [65, 0, 33, 32, 300, 31, 1, 96]), (F32, 896, 3584, [300, 20])])
def test_fewer_blocks_do_the_same(dtype, width, inner, held, joined):
    """A launch of which only some blocks found room: tiles in several groups, K in chunks for each, several (row, head, share) a block.
    The sums are the same ones in the same order: the same bits, in the result and in every layer's pages."""
    ops, run, pages = _ready(dtype, width, inner, held, 7)
    print(f"fewer {dtype} {width} {inner} {held} {joined}", flush=True)
    want = run().clone()
    kept = [p.clone() for p in pages]
    ops.layer_join_most = joined
    got = run()
    ops.raise_if_lost()
    assert torch.equal(got, want) and bool(torch.isfinite(want).all())
    assert all(torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)) for a, b in zip(pages, kept))


@pytest.mark.gpu
@pytest.mark.parametrize("page_size", [256, 1024])
@pytest.mark.parametrize("dtype,width,inner,held", [(BF16, 1024, 4096, [2047, 255, 256]), (F32, 640, 1152, [700, 0, 1023, 1024])])
def test_larger_pages_do_the_same(dtype, width, inner, held, page_size):
    """Where keys lie changes no sum: the bits of pages of 64."""
    print(f"pages {dtype} {width} {inner} {held} {page_size}", flush=True)
    results = []
    for size in (64, page_size):
        ops, run, _ = _ready(dtype, width, inner, held, 11, page_size=size)
        results.append(run())
        ops.raise_if_lost()
    assert torch.equal(*results) and bool(torch.isfinite(results[0]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("block", ["pre_norm", "post_norm"])
@pytest.mark.parametrize("dtype,held", [(BF16, [70, 700, 3]), (F32, [70, 300, 3]), (F32, [1, 12, 3, 40, 65])])
def test_rows_that_are_no_numbers(dtype, held, block):
    """Infinities and NaN (with the bits that stand for "not yet" as well) in one request's stream, keys or values: that row is finite
    where it is by launches apart, and the others keep their bits."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    print(f"no numbers {dtype} {held} {block}", flush=True)
    ops, width, inf = HipOps(dtype, DEV), 1024, float("inf")
    layers = [_layer(ops, dtype, width, 1024, block, "relu", True, 50 + i)[0] for i in range(2)]
    clean = (torch.randn(len(held), width, generator=torch.Generator().manual_seed(5)) * 2.0).to(DEV)
    ones = torch.full((1,), -1, dtype=torch.int32, device=DEV).view(F32)

    def run(how, where, value):
        steps, x = [_step(ops, dtype, held, width, 64, 60, i) for i in range(2)], clean.clone()
        ctx, cache, _ = steps[0]
        page = int(ctx.groups["full"].block_table[1, 0])
        if where == "x":
            x[1, 77] = value
        elif where == "keys":
            cache.k_pages[page, 3, 10, 5] = value
        elif where == "values":
            cache.v_pages[page, 3, 5, 10] = value
        return ops.settled(how(ops, layers, Stream(x, x.to(dtype)), steps).x).clone()
    want = run(_in_one, None, None)
    assert bool(torch.isfinite(want).all())
    others = [r for r in range(len(held)) if r != 1]
    for where in ("x", "keys", "values"):
        for value in (inf, -inf, float("nan"), ones[0]):
            got, apart = run(_in_one, where, value), run(_chain, where, value)
            ops.raise_if_lost()
            assert torch.equal(got[others], want[others]), (where, value)
            assert torch.equal(torch.isfinite(got[1]), torch.isfinite(apart[1])), (where, value)


@pytest.mark.gpu
@pytest.mark.parametrize("dtypes", [(F32,) * 6, (BF16,) * 8, (F32, BF16) * 4])
def test_many_launches_at_a_time(dtypes):
    """More launches on streams of their own than have room together, each with its own engine: every one gives what it gives alone."""
    engines = [_ready(dtype, 1024, 4096, [40 + i, 3, 65 * (i % 2)], 20 + i) for i, dtype in enumerate(dtypes)]
    print(f"at a time {dtypes}", flush=True)
    alone = [run().clone() for _, run, _ in engines]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in engines]
    results = []
    for _ in range(12):
        for (_, run, _), stream in zip(engines, streams):
            with torch.cuda.stream(stream):
                results.append(run())
    torch.cuda.synchronize()
    for i, got in enumerate(results):
        assert torch.equal(got, alone[i % len(engines)]), i
    for ops, _, _ in engines:
        ops.raise_if_lost()


@pytest.mark.gpu
def test_layers_in_one_launch_through_the_model(tmp_path):
    """A model of such layers: recorded steps (the launch replayed, other steps between) give what the launches apart give, bit for bit
    the same at every replay of the same step; and a wait that was given up is raised by the next step."""
    from transformers_neuronx_amd.config.engine_config import EngineConfig
    from transformers_neuronx_amd.engine.factory import runner_from_folder
    from transformers_neuronx_amd.opt.config import OPTConfig
    from transformers_neuronx_amd.weights import write_random_model
    raw = dict(architectures=["OPTForCausalLM"], model_type="opt", vocab_size=640, hidden_size=512, num_hidden_layers=3, num_attention_heads=8,
               ffn_dim=1024, max_position_embeddings=256, word_embed_proj_dim=512, do_layer_norm_before=True, activation_function="relu",
               enable_bias=True, layer_norm_elementwise_affine=True, init_std=0.04)
    write_random_model(OPTConfig.from_dict(raw), str(tmp_path), 3, dtype="bfloat16")
    logits = {}
    for one in (True, False):
        runner = runner_from_folder(str(tmp_path), EngineConfig(dtype="bfloat16", page_size=64, max_tokens=1024, max_num_seqs=4, device=DEV))
        runner.use_graphs = True
        runner.ops.layer_in_one = one
        assert runner.model.layers_in_one == {0: 3}
        runner.step([StepEntry(r, [5 + i + r for i in range(40 + 30 * r)], []) for r in range(3)])
        out = []
        for turn in range(4):
            out.append(runner.step([StepEntry(r, [7 * turn + r], [0]) for r in range(3)]).float().cpu())
            out.append(runner.step([StepEntry(1, [9], [0])]).float().cpu())
        logits[one] = torch.cat(out)
        runner.ops.raise_if_lost()
    assert float((logits[True] - logits[False]).norm() / logits[False].norm()) < 0.02
    assert runner.ops._lost is None or not int(runner.ops._lost[0][0])
    runner.ops._lost = (torch.ones(1, dtype=torch.int32), None)
    with pytest.raises(RuntimeError, match="waited in vain"):
        runner.step([StepEntry(1, [9], [0])])


@pytest.mark.gpu
@pytest.mark.parametrize("run_ahead", [True, False])
@pytest.mark.parametrize("graphs", [True, False])
def test_a_wait_that_was_given_up(tmp_path, run_ahead, graphs):
    """Waits of one question: the launch ends, says that it is void before a token of its step is handed out, and the engine goes on
    with launches apart."""
    from transformers_neuronx_amd.config.engine_config import EngineConfig
    from transformers_neuronx_amd.engine.engine import LLMEngine
    from transformers_neuronx_amd.engine.factory import runner_from_folder
    from transformers_neuronx_amd.kernels import LostStep
    from transformers_neuronx_amd.opt.config import OPTConfig
    from transformers_neuronx_amd.sampling import SamplingParams
    from transformers_neuronx_amd.weights import write_random_model
    raw = dict(architectures=["OPTForCausalLM"], model_type="opt", vocab_size=640, hidden_size=512, num_hidden_layers=3, num_attention_heads=8,
               ffn_dim=1024, max_position_embeddings=256, word_embed_proj_dim=512, do_layer_norm_before=True, activation_function="relu",
               enable_bias=True, layer_norm_elementwise_affine=True, init_std=0.2)
    write_random_model(OPTConfig.from_dict(raw), str(tmp_path), 3, dtype="float32")
    config = EngineConfig(dtype="float32", page_size=64, max_tokens=1024, max_num_seqs=4, device=DEV)
    prompts, params = [[5, 6, 7, 8], [9, 10]], SamplingParams(max_new_tokens=5, do_sample=False)

    def engine():
        made = LLMEngine(runner_from_folder(str(tmp_path), config), config)
        made.run_ahead, made.runner.use_graphs = run_ahead, graphs
        return made

    want = engine().generate(prompts, params)
    void = engine()
    void.runner.ops.layer_wait_most = 1
    handed = []
    with pytest.raises(LostStep, match="waited in vain"):
        for p in prompts:
            void.add_request(p, params)
        void.run(lambda out: handed.append(out.token))
    # the prompts' own tokens, launches apart, at most: a step ahead of their being read may be void by then
    assert handed in ([w[0] for w in want], []) and (run_ahead or handed) and not void.has_work
    assert not void.runner.ops.layer_in_one
    assert void.generate(prompts, params) == want


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("blocks,runs", [(["post", "pre", "post", "post"], {0: 1, 1: 2, 2: 4}), (["pre", "pre", "post"], {0: 2, 2: 3}),
                                         (["pre"] * 33, {0: 30, 30: 33}), (["post"] * 32, {0: 30, 30: 32})])
def test_several_launches_of_layers(blocks, runs, dtype):
    """Models whose layers are several such launches one behind the other: another arrangement, or more layers than one takes."""
    import toy_parts
    from transformers_neuronx_amd.cache import CacheManager
    from transformers_neuronx_amd.engine import DecoderModel, ModelRunner
    from transformers_neuronx_amd.kernels.hip import HipOps
    from transformers_neuronx_amd.weights import TensorDict, random_tensors
    spec = toy_parts.toy_spec_blocks([b + "_norm" for b in blocks], 512)
    logits = {}
    for one in (True, False):
        model, ops = DecoderModel(spec), HipOps(dtype, DEV)
        model.load(TensorDict(random_tensors(model.param_decls(), spec.init_std, 3, dtype)), ops, dtype, DEV)
        ops.layer_in_one, called = one, []
        call = ops._call
        ops._call = lambda lib, name, *a, **k: (called.append(name), call(lib, name, *a, **k))[1]
        assert model.layers_in_one == runs
        runner = ModelRunner(model, CacheManager(model.cache_needs(), 64, 12, 4, dtype, DEV), ops)
        runner.step([StepEntry(r, [5 + i + r for i in range(40 + 30 * r)], []) for r in range(3)])
        del called[:]
        logits[one] = torch.cat([runner.step([StepEntry(r, [7 * turn + r], [0]) for r in range(3)]).float().cpu() for turn in range(3)])
        assert called.count("tnx_decode_layers") == 3 * one * len(runs)
    # float32 sums in another order; in bfloat16 their roundings through up to 33 layers
    assert float((logits[True] - logits[False]).norm() / logits[False].norm()) < (0.03 if dtype == BF16 else 1e-5)
