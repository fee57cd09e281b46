"""The decoder, put together from a `ModelSpec`.

It owns the parts and their tensors and runs them in the order the spec lists.
What takes the place of the reference's graph owner
(`DecoderLmHeadForSamplingNoEmbedding`, decoder.py:43-1115, with its 26 named
weight slots per layer, :1275-1312) is this loop over parts that launch kernels.
"""
from typing import Dict, List, Optional

import torch

from ..parts.base import BLOCKS, EMBEDDINGS, FEED_FORWARDS, HEADS, MIXERS, NORMS, CacheNeed, Stream
from ..parts.spec import LayerSpec, ModelSpec, ParamDecl
from ..weights.loader import load_tensors
from .. import debug


class _Layer:
    def __init__(self, spec: LayerSpec):
        self.spec = spec
        self.mixer = MIXERS.build(spec.mixer)
        self.feed_forward = FEED_FORWARDS.build(spec.feed_forward)
        self.mixer_norm = NORMS.build(spec.mixer_norm)
        self.feed_forward_norm = NORMS.build(spec.feed_forward_norm)
        self.block = BLOCKS.build(
            _spec_of(spec.block), self.mixer, self.feed_forward, self.mixer_norm, self.feed_forward_norm)

    def _named(self):
        s = self.spec
        return [(self.mixer, s.prefix + s.mixer_name), (self.feed_forward, s.prefix + s.feed_forward_name),
                (self.mixer_norm, s.prefix + s.mixer_norm_name),
                (self.feed_forward_norm, s.prefix + s.feed_forward_norm_name),
                (self.block, s.prefix)]          # what the arrangement itself reads

    def param_decls(self) -> List[ParamDecl]:
        return [d for part, prefix in self._named() for d in part.param_decls(prefix)]

    def load(self, tensors, ops, dtype, finish=True):
        for part, prefix in self._named():
            part.load(tensors, prefix, ops, dtype)
        if finish:
            self.block.after_load()


def _spec_of(kind):
    from ..parts.spec import PartSpec
    return kind if isinstance(kind, PartSpec) else PartSpec(kind)


class DecoderModel:
    def __init__(self, spec: ModelSpec):
        self.spec = spec
        self.embedding = EMBEDDINGS.build(spec.embedding)
        self.layers = [_Layer(ls) for ls in spec.layers]
        self.head = HEADS.build(spec.head)
        self.schedule = spec.resolved_schedule()
        written = set()
        for layer, cid, writes in self.schedule:
            if writes:
                written.add(cid)
            elif cid not in written:
                raise ValueError(f"layer {layer} reads cache {cid} before the call that writes it")
        # parts other than mixers that keep something per request get a cache of their own, numbered after
        # the run order's: the embedding, and every call's block (a layer named twice keeps two)
        nxt = max((cid for _, cid, _ in self.schedule), default=-1) + 1
        self.part_state_needs: Dict[int, CacheNeed] = {}
        self.input_state_id = None
        if self.embedding.state_need() is not None:
            self.input_state_id = nxt
            self.part_state_needs[nxt] = self.embedding.state_need()
            nxt += 1
        self.call_state_ids: List[Optional[int]] = []
        for layer, _, _ in self.schedule:
            need = self.layers[layer].block.state_need()
            self.call_state_ids.append(nxt if need is not None else None)
            if need is not None:
                self.part_state_needs[nxt] = need
                nxt += 1
        self.loaded = False
        self.layers_in_one: Dict[int, int] = {}       # runs of calls that are one launch in decode steps of few rows
        parts = [self.embedding, self.embedding.position, self.head] + ([self.head.norm] if self.head.norm else [])
        for l in self.layers:
            parts += [l.block, l.mixer, l.feed_forward, l.mixer_norm, l.feed_forward_norm]
        self.recordable = all(getattr(p, "recordable", False) for p in parts)
        self.parts = [p for p in parts if p is not None]

    # ---------------------------------------------------------------- declarations

    def param_decls(self) -> List[ParamDecl]:
        decls, seen = [], set()
        for d in (self.embedding.param_decls() + [d for l in self.layers for d in l.param_decls()]
                  + self.head.param_decls()):
            if d.name not in seen:
                seen.add(d.name)
                decls.append(d)
        return decls

    def cache_needs(self) -> Dict[int, Optional[CacheNeed]]:
        """{cache id: need} of the calls that write a cache, and of the parts that keep state of their own."""
        needs = {cid: self.layers[layer].mixer.cache_need() for layer, cid, writes in self.schedule if writes}
        needs.update(self.part_state_needs)
        return needs

    def step_planners(self) -> Dict[str, object]:
        """The step planners that the parts bring with them."""
        out: Dict[str, object] = {}
        for part in self.parts:
            out.update(part.step_planners())
        return out

    def launch_shape(self, step) -> tuple:
        """What the parts' launches of a decode step are sized by, beyond its layout (`Part.launch_shape`)."""
        shapes = []
        for part in self.parts:
            shape = part.launch_shape(step)
            if shape is not None and shape not in shapes:
                shapes.append(shape)
        return tuple(shapes)

    # ---------------------------------------------------------------- accounting (for measurements)

    def step_flops(self, tokens: float, keys: float, wanted: float) -> float:
        """Multiply-adds times two of a step of `tokens` tokens that see `keys` cached tokens each on
        average (a whole prompt of T tokens: (T + 1) / 2) and ask for `wanted` rows of logits."""
        per_token = self.embedding.flops_per_token(keys)
        for layer, _, _ in self.schedule:
            l = self.layers[layer]
            per_token += sum(p.flops_per_token(keys) for p in (l.mixer, l.feed_forward, l.mixer_norm, l.feed_forward_norm,
                                                               l.block))
        return tokens * per_token + wanted * self.head.flops_per_token(keys)

    def cache_bytes_read(self, keys: float, dtype: torch.dtype, page_size: int = 1) -> float:
        """Bytes of its request's cache that one decoded token reads at a context of `keys` tokens: every call
        of the run order reads the cache it names (a windowed one up to its window)."""
        needs = {cid: self.layers[layer].mixer.cache_need() for layer, cid, writes in self.schedule if writes}
        total = 0.0
        for _, cid, _ in self.schedule:
            need = needs.get(cid)
            if need is None or need.kind != "paged":
                continue
            from ..cache.manager import CacheManager
            per_token = CacheManager.bytes_per_page({0: need}, page_size, dtype) / page_size
            total += per_token * (min(keys, need.window) if need.window else keys)
        return total

    # ---------------------------------------------------------------- weights

    def load(self, source, ops, dtype: torch.dtype, device, cast_float32: bool = False,
             finish: bool = True) -> "DecoderModel":
        """`finish=False` leaves out what the blocks do once their parts have their tensors (`finish_load`
        does it later: the caller has something to do to the weights in between)."""
        tensors = load_tensors(self.param_decls(), source, dtype, device, self.spec.base_model_prefix, cast_float32,
                               self.spec.unread)
        self.embedding.load(tensors, "", ops, dtype)
        for layer in self.layers:
            layer.load(tensors, ops, dtype, finish)
        self.head.load(tensors, "", ops, dtype)
        self.ops, self.dtype, self.device = ops, dtype, device
        self.weight_bytes = sum(t.numel() * t.element_size() for t in {id(t): t for t in tensors.values()}.values())
        self.loaded = True
        if finish:
            self.layers_in_one = self._layers_in_one() if hasattr(ops, "layers_most") else {}
        return self

    def finish_load(self) -> None:
        for layer in self.layers:
            layer.block.after_load()
        self.layers_in_one = self._layers_in_one() if hasattr(self.ops, "layers_most") else {}

    # ---------------------------------------------------------------- one step

    def forward(self, ctx, caches) -> torch.Tensor:
        """Logits float32 `[len(ctx.logits_rows), vocab]` for the step `ctx` describes."""
        first_block = self.layers[self.schedule[0][0]].block if self.schedule else None
        want_compute = bool(getattr(first_block, "reads_compute_copy", False))
        ctx.memo = {}
        ctx.input_state = caches[self.input_state_id] if self.input_state_id is not None else None
        stream: Stream = self.embedding.forward(ctx, want_compute)
        debug.tap("embedding", stream.x)
        # in steps of few rows, what the last block left may be a norm that the next products do (`norms_between`)
        few, between = ctx.num_tokens <= getattr(self.ops, "norm_beside_rows", 0), False
        left = False                    # and in steps of more, shares of a sum that the next norm adds (`leaves_shares`)
        in_one = self.layers_in_one if ctx.num_tokens <= getattr(self.ops, "layer_rows", 0) and self.ops.layers_fit(ctx) else {}
        done = 0
        for call, (layer, cid, writes) in enumerate(self.schedule):
            if call < done:
                continue
            block = self.layers[layer].block
            leaves = getattr(block, "leaves_shares", False)
            if (left and (call in in_one or not leaves)
                    or between and not getattr(block, "norms_between", False)):
                stream, left, between = self._settled(stream), False, False
            if call in in_one:
                behind = self._run_in_one(stream, call, in_one[call], ctx, caches)
                if behind is not None:
                    stream, done = behind, in_one[call]
                    between = few and getattr(self.layers[self.schedule[done - 1][0]].block, "norms_between", False)
                    continue
            cache = caches[cid] if writes else caches[cid].reader()
            state_id = self.call_state_ids[call]
            ctx.call_state = caches[state_id] if state_id is not None else None
            stream = block.forward(stream, ctx, cache)
            between = few and getattr(block, "norms_between", False)
            left = leaves
            debug.tap(f"call{call}.layer{layer}", stream.x)
        if between or left:
            stream = self._settled(stream)
        if stream.copies is not None and (stream.x is None or stream.pending is not None):
            # an arrangement that keeps several copies of the stream: their sum is what the head reads
            stream = Stream(self.ops.hyper_sum(stream.copies, stream.pending))
        return debug.tap("logits", self.head.forward(stream, ctx))


    def _layers_in_one(self) -> Dict[int, int]:
        """{first call: the call behind the last} of the runs of calls whose blocks can be one launch (`Block.in_one`)."""
        out, call, n = {}, 0, len(self.schedule)
        layers = [self.layers[layer] for layer, _, _ in self.schedule]

        def joins(call, end):
            first, before, this = layers[call], layers[end - 1], layers[end]
            return (type(this.block) is type(first.block) and this.mixer.cache_need().group_key() == first.mixer.cache_need().group_key()
                    and self.ops.layers_alike(first.block, this.block, before.block))
        while call < n:
            end = call
            while (end < n and end - call < self.ops.layers_most and layers[end].block.in_one is not None and self.schedule[end][2]
                   and (end == call or joins(call, end))):
                end += 1
            if end > call:
                out[call] = end
            call = max(end, call + 1)
        return out

    def _run_in_one(self, stream: Stream, begin: int, end: int, ctx, caches):
        """The stream behind the calls from `begin` to `end`, run as one launch; None where the backend does not take the step, or a
        block no longer is what a launch runs."""
        blocks = [self.layers[layer].block for layer, _, _ in self.schedule[begin:end]]
        parts = [b.in_one for b in blocks]
        if any(p is None for p in parts):
            return None
        of_calls = [caches[cid] for _, cid, _ in self.schedule[begin:end]]
        x, first, residual_normed = blocks[0].into_one(stream)
        norms = [(first, blocks[0].norms_in_one(blocks[0])[1])] + [b.norms_in_one(before) for before, b in zip(blocks, blocks[1:])]
        y = self.ops.decode_layers(parts, x, norms, residual_normed, ctx, ctx.groups[of_calls[0].group], of_calls)
        return None if y is None else blocks[-1].out_of_one(y)

    def _settled(self, stream: Stream) -> Stream:
        x = self.ops.settled(stream.x)
        return stream if x is stream.x else Stream(x, None)


def model_param_decls(spec: ModelSpec) -> List[ParamDecl]:
    return DecoderModel(spec).param_decls()
