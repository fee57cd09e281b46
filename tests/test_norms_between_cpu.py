"""What a post-norm block hands to its parts in steps of few rows, with a backend that leaves a norm behind a sum to the products
next to it: parts that say they take that get it, every other part, norm and arrangement gets tensors as in longer steps."""
import pytest
import torch

import toy_parts
from transformers_neuronx_amd.kernels.reference import ReferenceOps
from transformers_neuronx_amd.parts import FeedForward, Mixer, Stream
from transformers_neuronx_amd.parts.block import PostNormBlock, PreNormBlock
from transformers_neuronx_amd.parts.feed_forward import DenseFeedForward
from transformers_neuronx_amd.parts.base import residual_to_product
from transformers_neuronx_amd.parts.norm import LayerNorm, RMSNorm

WIDTH, ROWS = 32, 5


class Unmade:
    """Stands for (float32, compute dtype) of a norm: nothing that a tensor can do."""

    def __init__(self, made):
        self.made = made


class LateOps(ReferenceOps):
    """Leaves the norms of up to eight rows to `linear`, as the HIP backend does."""

    norm_beside_rows = 8

    def __init__(self):
        super().__init__(torch.float32, "cpu")
        self.left = 0

    def norm_between(self, x, weight, bias, eps, dtype, center=True):
        made = self.layernorm(x, weight, bias, eps, dtype, True, True, center)
        if x.shape[0] > self.norm_beside_rows:
            return made
        self.left += 1
        return (Unmade(made),) * 2

    def linear(self, x, w, bias=None, act=None, residual=None, **more):
        x = x.made[1] if isinstance(x, Unmade) else x
        residual = residual.made[0] if isinstance(residual, Unmade) else residual
        return super().linear(x, w, bias, act=act, residual=residual, **more)

    @staticmethod
    def settled(x):
        return x.made[0] if isinstance(x, Unmade) else x


class Multiplies(Mixer):
    def __init__(self, seed):
        self.w = torch.randn(WIDTH, WIDTH, generator=torch.Generator().manual_seed(seed)) / WIDTH ** 0.5

    def first_weight(self):
        return self.w

    @residual_to_product
    def forward(self, h, ctx, cache, residual):
        return self.ops.linear(self.ops.linear(h, self.w), self.w, None, residual=residual, out_f32=True)


class AddsItself(Multiplies):
    """Has a `first_weight` and adds the stream by itself."""

    def forward(self, h, ctx, cache, residual):
        return residual + self.ops.linear(self.ops.linear(h, self.w), self.w, None, out_f32=True)


class DenseThatAdds(DenseFeedForward):
    def forward(self, h, ctx, residual):
        return residual * 1.0 + super().forward(h, ctx, None)


class Counting(PostNormBlock):
    """An arrangement of its own that looks at the stream."""

    def forward(self, stream, ctx, cache):
        self.seen = float(stream.x.sum())
        return super().forward(stream, ctx, cache)


class _Ctx:
    num_tokens = ROWS


def _dense(cls):
    ff = cls(WIDTH, 48, "relu", "up", "down")
    g = torch.Generator().manual_seed(3)
    return ff, {"up.weight": torch.randn(48, WIDTH, generator=g) / 6, "up.bias": torch.randn(48, generator=g),
                "down.weight": torch.randn(WIDTH, 48, generator=g) / 7, "down.bias": torch.randn(WIDTH, generator=g)}


def _run(ops, mixer, ff, norm=LayerNorm, arrangement=PostNormBlock, layers=2):
    g = torch.Generator().manual_seed(5)
    stream, blocks = Stream(torch.randn(ROWS, WIDTH, generator=g)), []
    for layer in range(layers):
        m, (f, tensors), norms = mixer(layer), _dense(ff), [norm(WIDTH, 1e-5) for _ in "ab"]
        for part, t in [(m, {}), (f, tensors)] + [(n, {".weight": 1 + torch.randn(WIDTH, generator=g) / 9,
                                                      ".bias": torch.randn(WIDTH, generator=g)}) for n in norms]:
            part.load(t, "", ops, torch.float32)
        block = arrangement(m, f, *norms)
        block.load({}, "", ops, torch.float32)
        block.after_load()
        blocks.append(block)
        if not block.norms_between:
            stream = Stream(ops.settled(stream.x), None)
        stream = block.forward(stream, _Ctx(), None)
    return ops.settled(stream.x), blocks


@pytest.mark.parametrize("mixer,ff,arrangement,left", [
    (Multiplies, DenseFeedForward, PostNormBlock, True), (AddsItself, DenseFeedForward, PostNormBlock, False),
    (Multiplies, DenseThatAdds, PostNormBlock, False), (Multiplies, DenseFeedForward, Counting, False)])
def test_parts_that_take_a_norm_left_to_them(mixer, ff, arrangement, left):
    want, _ = _run(ReferenceOps(torch.float32, "cpu"), mixer, ff, arrangement=arrangement)
    ops = LateOps()
    got, blocks = _run(ops, mixer, ff, arrangement=arrangement)
    assert [b.norms_between for b in blocks] == [left] * 2 and (ops.left > 0) == left
    assert torch.equal(got, want)


class Doubled(LayerNorm):
    def forward(self, x, want_f32, want_compute):
        return tuple(None if y is None else 2 * y for y in super().forward(x, want_f32, want_compute))


class Renamed(RMSNorm):
    pass


@pytest.mark.parametrize("norm,left", [(LayerNorm, True), (RMSNorm, True), (Renamed, True), (Doubled, False)])
def test_norms_with_a_forward_of_their_own_are_run(norm, left):
    want, _ = _run(ReferenceOps(torch.float32, "cpu"), Multiplies, DenseFeedForward, norm=norm)
    ops = LateOps()
    got, _ = _run(ops, Multiplies, DenseFeedForward, norm=norm)
    assert (ops.left > 0) == left and torch.equal(got, want)


@pytest.mark.parametrize("norm", [LayerNorm, RMSNorm])
def test_deferred_without_the_classes_own_fold_into(norm):
    """A subclass that folds in a way of its own and inherits `deferred`."""
    class Folding(norm):
        def fold_into(self, w):
            return self.ops.fold_norm(w, self.weight, None)

    class FoldingOps(ReferenceOps):
        def fold_norm(self, w, weight, bias, center=True):
            return True

        def layernorm_deferred(self, x, *more, **named):
            return "left to the product"

    n = Folding(WIDTH, 1e-5)
    n.load({".weight": torch.ones(WIDTH), ".bias": torch.zeros(WIDTH)}, "", FoldingOps(torch.float32, "cpu"), torch.float32)
    assert n.fold_into(None) and n.deferred(torch.zeros(3, WIDTH)) == "left to the product"


@pytest.mark.parametrize("tokens,asked", [(4, True), (5, False)])
def test_longer_steps_ask_nothing_of_a_norm_left_to_a_product(tokens, asked):
    """The pre-norm block compares the step's tokens with what the norm said at load, once a norm."""
    class Few(LayerNorm):
        calls = 0

        def fold_into(self, w):
            self.defer_rows = 4
            return True

        def deferred(self, x):
            self.calls += 1
            return self.forward(x, False, True)[1]

    class Step(_Ctx):
        num_tokens = tokens

    ops, norms = ReferenceOps(torch.float32, "cpu"), [Few(WIDTH, 1e-5, affine=False) for _ in "ab"]
    mixer, (ff, tensors) = Multiplies(1), _dense(DenseFeedForward)
    for part, t in [(mixer, {}), (ff, tensors)] + [(n, {}) for n in norms]:
        part.load(t, "", ops, torch.float32)
    block = PreNormBlock(mixer, ff, *norms)
    block.after_load()
    block.forward(Stream(torch.randn(tokens, WIDTH)), Step(), None)
    assert [n.calls for n in norms] == [int(asked)] * 2


class InOneOps(LateOps):
    """Asks for layers in one launch as well, and takes none of them."""

    layer_rows, layers_most = 8, 30

    def __init__(self):
        super().__init__()
        self.asked = []

    def layer_parts(self, attention, feed_forward):
        return attention, feed_forward

    def layers_fit(self, ctx):
        return True

    def layers_alike(self, first, block, before):
        return True

    def decode_layers(self, layers, x, norms, residual_normed, ctx, view, caches):
        assert type(x) is torch.Tensor
        self.asked.append(len(layers))


@pytest.mark.parametrize("kinds,runs", [("post pre", [1, 1]), ("pre post post", [1, 2]), ("post post pre pre post", [2, 2, 1])])
def test_runs_of_layers_behind_another_kind(kinds, runs):
    """Layers of one launch behind a block whose last sum's norm has been left to them, where they take none: the norm is made."""
    from transformers_neuronx_amd.engine.model import DecoderModel
    from transformers_neuronx_amd.engine.runner import ModelRunner
    from transformers_neuronx_amd.cache import CacheManager
    from transformers_neuronx_amd.engine import StepEntry
    from transformers_neuronx_amd.weights import TensorDict, random_tensors
    spec = toy_parts.toy_spec_blocks([k + "_norm" for k in kinds.split()], 128)
    logits = {}
    for ops in (ReferenceOps(torch.float32, "cpu"), InOneOps()):
        model = DecoderModel(spec)
        model.load(TensorDict(random_tensors(model.param_decls(), spec.init_std, 3, torch.float32)), ops, torch.float32, "cpu")
        runner = ModelRunner(model, CacheManager(model.cache_needs(), 16, 12, 4, torch.float32, "cpu"), ops)
        runner.step([StepEntry(r, [5 + i + r for i in range(9)], []) for r in range(3)])
        logits[type(ops)] = runner.step([StepEntry(r, [7 + r], [0]) for r in range(3)])
    assert ops.asked == runs and ops.left > 0
    assert torch.equal(logits[ReferenceOps], logits[InOneOps])


def test_built_in_parts_say_so():
    from transformers_neuronx_amd.parts.mixer import Attention
    for part in (Attention, DenseFeedForward):
        assert part.forward.residual_to_product
    assert not getattr(FeedForward.forward, "residual_to_product", False) and not getattr(Mixer.forward, "residual_to_product", False)


class Unadded:
    """A product's result that a norm is to read next, as the HIP backend leaves it; as `onto` makes it, a residual."""

    def __init__(self, ops, x):
        self.ops, self.x = ops, x

    def settled(self):
        return self.x

    def normed(self, weight, bias, eps, dtype, center, alone=False):
        y, h = self.ops.layernorm(self.x, weight, bias, eps, dtype, True, True, center)
        return (y if alone else self.x), h


class SharingOps(InOneOps):
    """Leaves sums to the norms behind them too."""

    def onto(self, x):
        return Unadded(self, x)

    def linear(self, x, w, bias=None, act=None, residual=None, **more):
        leave = isinstance(residual, Unadded)
        y = super().linear(x, w, bias, act=act, residual=residual.x if leave else residual, **more)
        return Unadded(self, y) if leave else y

    @staticmethod
    def settled(x):
        return x.x if isinstance(x, Unadded) else LateOps.settled(x)

    def decode_layers(self, layers, *more):
        super().decode_layers(layers, *more)
        self.layers = layers


def _toy_runner(kind, ops):
    from transformers_neuronx_amd.engine.model import DecoderModel
    from transformers_neuronx_amd.engine.runner import ModelRunner
    from transformers_neuronx_amd.cache import CacheManager
    from transformers_neuronx_amd.weights import TensorDict, random_tensors
    spec = toy_parts.toy_spec_blocks([kind] * 3, 128)
    model = DecoderModel(spec)
    model.load(TensorDict(random_tensors(model.param_decls(), spec.init_std, 3, torch.float32)), ops, torch.float32, "cpu")
    return ModelRunner(model, CacheManager(model.cache_needs(), 16, 12, 4, torch.float32, "cpu"), ops)


def _steps(runner):
    """A step of more rows than few, and one of few."""
    from transformers_neuronx_amd.engine import StepEntry
    return torch.cat([runner.step([StepEntry(r, [5 + i + r for i in range(9)], [8]) for r in range(3)]),
                      runner.step([StepEntry(r, [7 + r], [0]) for r in range(3)])])


@pytest.mark.parametrize("part", ["", "mixer", "feed_forward", "mixer_norm", "feed_forward_norm"])
@pytest.mark.parametrize("kind", ["pre_norm", "post_norm"])
@pytest.mark.parametrize("dressed", [True, False])
def test_a_forward_put_on_an_object_is_called(kind, part, dressed):
    """Put there after loading, on a block, a part or a norm: called in every step, with tensors; and not once it is taken away."""
    import functools
    want = _steps(_toy_runner(kind, ReferenceOps(torch.float32, "cpu")))
    ops = SharingOps()
    runner = _toy_runner(kind, ops)
    assert torch.equal(_steps(runner), want) and ops.asked == [3]
    block, calls = runner.model.layers[1].block, []
    of = getattr(block, part) if part else block
    inner = of.forward

    def forward(*args, **named):
        for a in (args[0].x if not part else args[0], *(args[-1:] if part in ("mixer", "feed_forward") else ())):
            assert type(a) is torch.Tensor
        out = inner(*args, **named)
        assert not isinstance(out.x if not part else out, Unadded)
        calls.append(1)
        return out
    of.forward = functools.wraps(inner)(forward) if dressed else forward
    runner.cache.reset()
    assert torch.equal(_steps(runner), want) and len(calls) == 2 and ops.asked == [3]
    del of.forward
    runner.cache.reset()
    assert torch.equal(_steps(runner), want) and len(calls) == 2 and ops.asked == [3, 3]


@pytest.mark.parametrize("name", ["mixer", "feed_forward"])
def test_a_forward_put_on_a_class_before_loading_is_called(monkeypatch, name):
    import functools
    from transformers_neuronx_amd.parts.mixer import Attention
    cls, calls = {"mixer": Attention, "feed_forward": DenseFeedForward}[name], []
    inner = cls.forward

    @functools.wraps(inner)
    def forward(self, *args):
        assert type(args[-1]) is torch.Tensor
        calls.append(1)
        return inner(self, *args)
    monkeypatch.setattr(cls, "forward", forward)
    ops = SharingOps()
    _steps(_toy_runner("pre_norm", ops))
    assert len(calls) == 6 and not ops.asked


def test_layers_in_one_launch_take_the_tensors_of_the_step():
    """Another matrix in a part's place, as `forward` would read it."""
    ops = SharingOps()
    runner = _toy_runner("pre_norm", ops)
    _steps(runner)
    mixer, ff = runner.model.layers[1].block.mixer, runner.model.layers[2].block.feed_forward
    mixer.w_out, ff.b1, mixer.scale = mixer.w_out * 2, ff.b1 + 1, 0.5
    runner.cache.reset()
    _steps(runner)
    assert ops.layers[1][0][2] is mixer.w_out and ops.layers[1][0][5] == 0.5 and ops.layers[2][1][1] is ff.b1
