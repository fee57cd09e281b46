"""The calls by which this engine's speed is judged: what a program that serves or scores with it has it do.

Two designs stand for all: OPT (the family the engine is first of all for, at the sizes of its published models) and
Sunatar (attention over a window, a matrix memory, a mixture of experts), as 4 layers at two published widths. Kinds:

  decode   one token each for a number of live sequences (the continuous-batching form of `model(ids, positions,
           sequences)`); the tokens are given, as when a text is scored or a trace is run again
  prompt   whole prompts, up to their first token's logits (`model(ids)`, rows padded on the left where they differ)
  mixed    a portion of a prompt beside sequences that decode, in one step of the runner (chunked prefill)
  serve    requests of unlike lengths through the engine from their prompts to their last token, greedily
  sample   `model.sample`, top-k sampling

Weights are drawn on the device from the seed, with the names of the checkpoints; `exact` reads the same tensors.
"""
import math
import random

import torch

VOCAB = 50272
#            width, layers, heads, inner, width of the token table, norm before the part
OPT_SIZES = {"350m": (1024, 24, 16, 4096, 512, False), "1.3b": (2048, 24, 32, 8192, 2048, True),
             "2.7b": (2560, 32, 32, 10240, 2560, True), "6.7b": (4096, 32, 32, 16384, 4096, True)}
#                width, heads, head, inner
SUNATAR_SIZES = {"sunatar-2048": (2048, 32, 64, 8192), "sunatar-4096": (4096, 32, 128, 16384)}
SUNATAR_LAYERS = 4
SUNATAR_WINDOW = 1024
SUNATAR_MEMORY_HEAD = 64
EXPERTS, CHOSEN = 8, 2
PAGE = 64


def listed():
    return [
        # one user at a small model, a short conversation: the launches and the gaps between them count
        dict(name="decode 350m 1x100", kind="decode", model="350m", dtype="bf16", rows=1, context=100, turns=400, ragged=False),
        # a larger batch of unlike lengths; a head size that is no power of two
        dict(name="decode 2.7b 32x700", kind="decode", model="2.7b", dtype="bf16", rows=32, context=700, turns=400, ragged=True),
        # the headline: 8 requests at the full context of the 6.7b model
        dict(name="decode 6.7b 8x2048", kind="decode", model="6.7b", dtype="bf16", rows=8, context=2048, turns=512, ragged=False),
        # the mixture of experts and the matrix memory, decoding
        dict(name="decode sunatar 8x1500", kind="decode", model="sunatar-2048", dtype="bf16", rows=8, context=1500, turns=512,
             ragged=False),
        # time to the first token of a short question of odd length
        dict(name="prompt 1.3b 1x333", kind="prompt", model="1.3b", dtype="bf16", rows=1, context=333, ragged=False),
        # the headline's other half: a prompt that fills the context, in one step
        dict(name="prompt 6.7b 1x2048", kind="prompt", model="6.7b", dtype="bf16", rows=1, context=2048, ragged=False),
        # prompts over experts, a memory carried through the whole run
        dict(name="prompt sunatar 1x2048", kind="prompt", model="sunatar-4096", dtype="bf16", rows=1, context=2048, ragged=False),
        # a few short rows of unlike lengths together
        dict(name="prompt sunatar 3x210", kind="prompt", model="sunatar-2048", dtype="bf16", rows=3, context=210, ragged=True),
        # the float32 engine: prompts scored without any rounding to 16 bits
        dict(name="prompt 1.3b f32 2x300", kind="prompt", model="1.3b", dtype="f32", rows=2, context=300, ragged=True),
        # a step of a loaded server: part of a new prompt beside the sequences that are decoding
        dict(name="mixed 1.3b 40x500+600", kind="mixed", model="1.3b", dtype="bf16", rows=40, context=500, turns=400,
             portion=600, ragged=True),
        # a small server's burst, whole: prompts come in, every request decodes to its end
        dict(name="serve 1.3b 24x400", kind="serve", model="1.3b", dtype="bf16", rows=24, context=400, new=24, ragged=True),
        # sampling from the float32 engine
        dict(name="sample 350m f32 3x60", kind="sample", model="350m", dtype="f32", rows=3, context=60, new=16, ragged=False),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "serve", "sample"])
    dtype = "bf16"
    if kind in ("decode", "prompt"):
        model = rng.choice(["350m", "1.3b", "2.7b", "6.7b", "sunatar-2048", "sunatar-4096"])
        if model in ("350m", "1.3b") and rng.random() < 0.25:
            dtype = "f32"
    else:
        model = rng.choice(["350m", "1.3b", "2.7b"])
    if kind == "decode":
        rows = _log_int(rng, 1, 8 if dtype == "f32" else 64)
        context = _log_int(rng, 32, min(2048, (2048 if dtype == "f32" else 24576) // rows))
        return dict(kind=kind, model=model, dtype=dtype, rows=rows, context=context, turns=512, ragged=rng.random() < 0.5)
    if kind == "prompt":
        rows = _log_int(rng, 1, 4)
        context = _log_int(rng, 17, (700 if dtype == "f32" else 2048) // rows)
        return dict(kind=kind, model=model, dtype=dtype, rows=rows, context=context, ragged=rows > 1 and rng.random() < 0.5)
    if kind == "mixed":
        rows = _log_int(rng, 3, 48)
        return dict(kind=kind, model=model, dtype=dtype, rows=rows, context=_log_int(rng, 48, min(1024, 16384 // rows)), turns=400,
                    portion=_log_int(rng, 33, 1024), ragged=True)
    if kind == "serve":
        return dict(kind=kind, model=model, dtype=dtype, rows=_log_int(rng, 3, 32), context=_log_int(rng, 24, 500),
                    new=_log_int(rng, 6, 32), ragged=True)
    return dict(kind=kind, model="350m", dtype="f32", rows=rng.randint(1, 4), context=_log_int(rng, 20, 150),
                new=rng.randint(8, 20), ragged=False)


def _lengths(case):
    """Tokens of each row before the pass: all `context`, or spread over its last three quarters."""
    n, most = case["rows"], case["context"]
    if not case["ragged"] or n == 1:
        return [most] * n
    rng = random.Random(n * 4099 + most)
    return [most] + [rng.randint(max(2, most // 4), most) for _ in range(n - 1)]


# ---------------------------------------------------------------- weights and configurations

def _normal(gen, std, *shape, mean=0.0):
    return torch.randn(shape, generator=gen, device=gen.device, dtype=torch.float32).mul_(std).add_(mean)


def _opt_weights(case, seed):
    """Matrices of 0.02 as the family's initialisation has them; what ends in the residual sum drawn smaller by the depth.
    For requests that generate greedily the token table is wide, so that the first choice is a clear one, as a trained
    model's mostly is."""
    width, layers, _, inner, table, pre = OPT_SIZES[case["model"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    store = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    w = {}

    def matrix(name, n, k, std=0.02):
        w[name] = _normal(gen, std, n, k).to(store)

    def vector(name, n, mean=0.0):
        w[name] = _normal(gen, 0.02, n, mean=mean)

    def norm(name):
        vector(name + ".weight", width, 1.0)
        vector(name + ".bias", width)

    p = "model.decoder."
    matrix(p + "embed_tokens.weight", VOCAB, table, 0.5 if case["kind"] == "serve" else 0.02)
    matrix(p + "embed_positions.weight", _positions(case) + 2, width)
    if table != width:
        matrix(p + "project_in.weight", width, table)
        matrix(p + "project_out.weight", table, width)
    end = 0.02 / math.sqrt(2 * layers)
    for i in range(layers):
        q = f"{p}layers.{i}."
        for name in ("q", "k", "v"):
            matrix(f"{q}self_attn.{name}_proj.weight", width, width)
            vector(f"{q}self_attn.{name}_proj.bias", width)
        matrix(q + "self_attn.out_proj.weight", width, width, end)
        vector(q + "self_attn.out_proj.bias", width)
        matrix(q + "fc1.weight", inner, width)
        vector(q + "fc1.bias", inner)
        matrix(q + "fc2.weight", width, inner, end)
        vector(q + "fc2.bias", width)
        norm(q + "self_attn_layer_norm")
        norm(q + "final_layer_norm")
    if pre:
        norm(p + "final_layer_norm")
    return w


def _sunatar_weights(case, seed):
    """Every token has two experts that it prefers (some experts more often than others) along directions that its row of
    the table carries and the routers read: which experts a token meets is then as clear as trained routers make it."""
    width, heads, head, inner = SUNATAR_SIZES[case["model"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    store = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    w = {}

    def matrix(name, n, k, std=0.02):
        w[name] = _normal(gen, std, n, k).to(store)

    def vector(name, n, mean=0.0):
        w[name] = _normal(gen, 0.02, n, mean=mean)

    ways = torch.linalg.qr(_normal(gen, 1.0, width, EXPERTS))[0].T.contiguous()         # [experts, width], orthonormal
    first = (torch.rand(VOCAB, generator=gen, device="cuda").pow(1.5) * EXPERTS).long().clamp_(max=EXPERTS - 1)
    second = (first + 1 + (torch.rand(VOCAB, generator=gen, device="cuda") * (EXPERTS - 1)).long().clamp_(max=EXPERTS - 2)) % EXPERTS
    liking = 0.3 * math.sqrt(width)
    w["embed"] = (_normal(gen, 1.0, VOCAB, width) + liking * (ways[first] + ways[second])).to(store)
    end = 0.02 / math.sqrt(SUNATAR_LAYERS)
    for i in range(SUNATAR_LAYERS):
        p = f"l{i}.mix."
        vector(f"l{i}.norm1", width, 1.0)
        if i % 4 == 1:
            matrix(p + "q", heads * SUNATAR_MEMORY_HEAD, width)
            matrix(p + "k", heads * SUNATAR_MEMORY_HEAD, width)
            matrix(p + "v", heads * head, width)
            matrix(p + "g", heads * head, width)
            matrix(p + "i", heads, width)
            matrix(p + "f", heads, width)
            vector(p + "i.b", heads)
            vector(p + "f.b", heads, 3.0)
            vector(p + "norm", heads * head, 1.0)
        else:
            for name, n in (("q", heads * head), ("k", heads // 4 * head), ("v", heads // 4 * head)):
                matrix(p + name, n, width)
                vector(p + name + ".b", n)
            vector(p + "q.norm", heads * head, 1.0)
            vector(p + "k.norm", heads // 4 * head, 1.0)
            if i > 0:
                w[p + "vmix"] = _normal(gen, 0.02, mean=0.5)
        matrix(p + "o", width, heads * head, end)
        p = f"l{i}.mlp."
        w[p + "router"] = (ways * (8.0 / liking) + _normal(gen, 0.005, EXPERTS, width)).to(store)
        for e, ff in [(f"e{j}", inner // 4) for j in range(EXPERTS)] + [("shared", inner // 2)]:
            matrix(f"{p}{e}.gate", ff, width)
            matrix(f"{p}{e}.up", ff, width)
            matrix(f"{p}{e}.down", width, ff, end)
    vector("final.norm", width, 1.0)
    matrix("head", VOCAB, width)
    return w


def _weights(case, seed):
    return (_sunatar_weights if case["model"] in SUNATAR_SIZES else _opt_weights)(case, seed)


def _positions(case):
    return case["context"] + case.get("turns", 0) + case.get("new", 0) + 1


def _raw_config(case):
    if case["model"] in SUNATAR_SIZES:
        width, heads, head, inner = SUNATAR_SIZES[case["model"]]
        attention = dict(heads=heads, kv_heads=heads // 4, dim=head, vdim=head, scale=head ** -0.5, v_mix=True,
                         mask=dict(size=SUNATAR_WINDOW),
                         rot=dict(base=500000.0, dims=head // 2, scaling=dict(factor=8.0, low=1.0, high=4.0, original=8192)))
        memory = dict(heads=heads, dim=SUNATAR_MEMORY_HEAD, vdim=head, gate_cap=15.0)
        mlp = dict(kind="moe", router=dict(experts=EXPERTS, top=CHOSEN), expert=dict(ff=inner // 4), shared=dict(ff=inner // 2))
        return dict(architecture="Sunatar", vocab=VOCAB, width=width, norm=dict(eps=1e-5), embedding=dict(scale=1.0), init_std=0.02,
                    max_positions=4096,
                    layers=[dict(type="mlstm", mixer=memory, mlp=mlp) if i % 4 == 1 else
                            dict(type="attention", mixer=attention, mlp=mlp) for i in range(SUNATAR_LAYERS)])
    width, layers, heads, inner, table, pre = OPT_SIZES[case["model"]]
    return dict(architectures=["OPTForCausalLM"], model_type="opt", vocab_size=VOCAB, max_position_embeddings=_positions(case),
                do_layer_norm_before=pre, activation_function="relu", enable_bias=True, layer_norm_elementwise_affine=True,
                init_std=0.02, torch_dtype="bfloat16" if case["dtype"] == "bf16" else "float32", hidden_size=width,
                num_hidden_layers=layers, num_attention_heads=heads, ffn_dim=inner, word_embed_proj_dim=table)


# ---------------------------------------------------------------- states and passes

def _tokens(case, seed):
    """The prompts, the tokens that follow them turn by turn `[turns][rows]`, and the prompt that a mixed step takes part of."""
    rng = torch.Generator().manual_seed(seed)

    def some(*shape):
        return torch.randint(3, VOCAB, shape, generator=rng)

    prompts = [some(n).tolist() for n in _lengths(case)]
    return prompts, some(case.get("turns", 0), case["rows"]), some(case.get("portion", 0)).tolist()


def _sequences(case, prompts):
    """Every row's prompt into the cache, a call a length."""
    return [([i], prompts[i:i + 1]) for i in range(len(prompts))] if case["ragged"] else [(list(range(len(prompts))), prompts)]


def _begin(state):
    """The conversations start: their prompts go into the cache. After `turns` passes they are over, and others start."""
    model, case = state["model"], state["case"]
    model.reset()
    for rows, prompts in _sequences(case, state["prompts"]):
        ids = torch.tensor(prompts)
        model(ids, torch.arange(ids.shape[1]).expand(len(rows), -1), torch.tensor(rows))
    state["turn"] = 0


def prepare(case, seed):
    from transformers_neuronx_amd import NeuronConfig, OPTForSampling, SunatarForSampling
    from transformers_neuronx_amd.config.registry import resolve
    from transformers_neuronx_amd.weights import TensorDict
    raw = _raw_config(case)
    config = resolve(raw).config_class.from_dict(raw)
    rows = case["rows"] + (1 if case["kind"] == "mixed" else 0)
    kind = SunatarForSampling if case["model"] in SUNATAR_SIZES else OPTForSampling
    live = case["kind"] in ("decode", "mixed")
    longest = max(_positions(case), case.get("portion", 0) + 1)
    model = kind.from_config(config, TensorDict(_weights(case, seed)), batch_size=rows, amp=case["dtype"],
                             n_positions=_positions(case), page_size=PAGE, num_pages=rows * -(-longest // PAGE),
                             neuron_config=NeuronConfig(continuous_batching=dict(max_num_seqs=rows)) if live else None)
    model.load()
    prompts, turns, portion = _tokens(case, seed)
    state = dict(case=case, model=model, prompts=prompts, turns=turns, portion=portion, lengths=_lengths(case), turn=0)
    if live:
        _begin(state)
    elif case["kind"] == "prompt" or case["kind"] == "sample":
        width = max(len(p) for p in prompts)
        state["ids"] = torch.tensor([[1] * (width - len(p)) + p for p in prompts])
        state["starts"] = torch.tensor([width - len(p) for p in prompts]) if case["ragged"] else None
    return state


def run(state):
    return {"decode": _decode, "prompt": _prompt, "mixed": _mixed, "serve": _serve, "sample": _sample}[state["case"]["kind"]](state)


def _next_turn(state):
    if state["turn"] >= state["case"]["turns"]:
        _begin(state)
    turn = state["turn"]
    state["turn"] += 1
    return turn, state["turns"][turn]


def _decode(state):
    turn, ids = _next_turn(state)
    places = torch.tensor(state["lengths"]).add_(turn)
    return state["model"](ids.unsqueeze(1), places.unsqueeze(1), torch.arange(len(places)))


def _prompt(state):
    return state["model"](state["ids"], start_ids=state["starts"])


def _mixed(state):
    from transformers_neuronx_amd.engine.batch import StepEntry
    _, ids = _next_turn(state)
    runner = state["model"].engine.runner
    entries = [StepEntry("new", state["portion"], [len(state["portion"]) - 1])]
    entries += [StepEntry(("seq", i), [t], [0]) for i, t in enumerate(ids.tolist())]
    logits = runner.step(entries)
    runner.finish("new")
    return logits


def _serve(state):
    from transformers_neuronx_amd import SamplingParams
    engine, case = state["model"].engine, state["case"]
    first = {}

    def keep(requests, logits):         # the log-odds of every request's first token, as a client may ask for them
        for i, q in enumerate(requests):
            if not q.output:
                first[q.req_id] = logits[i].clone()

    engine.reset()
    engine.logits_hook = keep
    try:
        ids = [engine.add_request(p, SamplingParams(max_new_tokens=case["new"], do_sample=False)) for p in state["prompts"]]
        engine.run()
        tokens = [engine.pop_request(i).output for i in ids]
    finally:
        engine.logits_hook = None
    return {"logits": torch.stack([first[i] for i in ids]), "tokens": torch.tensor(tokens)}


def _sample(state):
    model, case, last = state["model"], state["case"], {}

    def keep(requests, logits):
        last["logits"] = logits

    model.engine.logits_hook = keep
    try:
        tokens = model.sample(state["ids"], sequence_length=case["context"] + case["new"], top_k=50, temperature=0.8, top_p=0.95)
    finally:
        model.engine.logits_hook = None
    return {"logits": last["logits"], "tokens": tokens}


# ---------------------------------------------------------------- what a pass cannot do without

def _sizes(case):
    """(weights that every pass reads, weights of one expert of all layers, weights a token meets, multiply-adds a pair of a
    token and a key it sees, numbers cached a token, numbers of fixed state a sequence, window), all over the whole depth;
    the head and the token table apart."""
    if case["model"] in SUNATAR_SIZES:
        width, heads, head, inner = SUNATAR_SIZES[case["model"]]
        n = SUNATAR_MEMORY_HEAD
        attending = SUNATAR_LAYERS - 1
        memory = (2 * heads * n + 3 * heads * head + 2 * heads) * width
        attention = (2 * heads * head + 2 * (heads // 4) * head) * width
        expert = 3 * width * (inner // 4)
        always = attending * attention + memory + SUNATAR_LAYERS * (3 * width * (inner // 2) + EXPERTS * width)
        state = heads * n * (head + 1)
        return (always, SUNATAR_LAYERS * expert, always + SUNATAR_LAYERS * CHOSEN * expert, 2 * attending * heads * head,
                2 * attending * (heads // 4) * head, state, SUNATAR_WINDOW)
    width, layers, _, inner, table, _ = OPT_SIZES[case["model"]]
    always = layers * (4 * width * width + 2 * width * inner) + (2 * table * width if table != width else 0)
    return always, 0, always, 2 * layers * width, 2 * layers * width, 0, None


def _step_work(case, runs, wanted):
    """(bytes, flops) of one step over runs of (tokens already cached, new tokens) with `wanted` rows of logits."""
    always, expert, meets, pair, cached, fixed, window = _sizes(case)
    item = 2 if case["dtype"] == "bf16" else 4
    table = OPT_SIZES[case["model"]][4] if case["model"] in OPT_SIZES else SUNATAR_SIZES[case["model"]][0]
    tokens = sum(new for _, new in runs)
    met = EXPERTS * (1.0 - (1.0 - CHOSEN / EXPERTS) ** tokens)
    weights = always + met * expert + VOCAB * table
    read = sum(min(have, window) if window else have for have, _ in runs) * cached
    seen = sum(sum(min(have + i + 1, window) if window else have + i + 1 for i in range(new)) for have, new in runs)
    nbytes = item * (weights + read + tokens * (cached + table)) + 8 * fixed * len(runs) + 4 * wanted * VOCAB
    return nbytes, 2.0 * (tokens * meets + seen * pair + wanted * VOCAB * table)


def work(case):
    lens = _lengths(case)
    steps = []
    if case["kind"] == "decode":
        steps = [([(n, 1) for n in lens], len(lens))]
    elif case["kind"] == "prompt":
        steps = [([(0, n) for n in lens], len(lens))]
    elif case["kind"] == "mixed":
        steps = [([(n, 1) for n in lens] + [(0, case["portion"])], len(lens) + 1)]
    else:
        steps = [([(0, n) for n in lens], len(lens))]
        steps += [([(n + i, 1) for n in lens], len(lens)) for i in range(case["new"] - 1)]
    each = [_step_work(case, *s) for s in steps]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}


def tolerance(case):
    """About four times the error against `exact` that was measured: 2e-6 in float32, 0.003 to 0.0056 in bfloat16 (the
    stream stays in float32, every product rounds its operands to 8 bits)."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    return {"rel": 0.02, "max": 0.15, "differ": 0.01}


# ---------------------------------------------------------------- 64 bits

def exact(case, seed):
    """The logits of `run`'s first pass by plain arithmetic in 64 bits over whole sequences; nothing for the tokens (they are
    whole numbers) nor for logits after drawn tokens."""
    if case["kind"] == "sample":
        return None
    prompts, turns, portion = _tokens(case, seed)
    if case["kind"] in ("decode", "mixed"):
        prompts = [p + [int(t)] for p, t in zip(prompts, turns[0])]
    if case["kind"] == "mixed":
        prompts = [portion] + prompts
    w = _weights(case, seed)
    with torch.no_grad():
        logits = (_sunatar_exact if case["model"] in SUNATAR_SIZES else _opt_exact)(case, w, prompts)
    return {"logits": logits, "tokens": None} if case["kind"] == "serve" else logits


def _layer_norm(x, weight, bias=None, eps=1e-5):
    x = x - x.mean(-1, keepdim=True)
    x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * weight
    return x if bias is None else x + bias


def _unit_rms(x, eps=1e-5):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _attend(q, k, v, window=None):
    """q `[T, H, n]`, k and v `[T, G, n]` -> `[T, H n]`, a group of heads at a time."""
    t, heads, _ = q.shape
    per = heads // k.shape[1]
    far = torch.arange(t, device=q.device)
    far = far[:, None] - far[None, :]
    hidden = (far < 0) if window is None else (far < 0) | (far >= window)
    out = []
    for h in range(heads):
        s = (q[:, h].contiguous() @ k[:, h // per].T.contiguous()).masked_fill_(hidden, float("-inf"))
        out.append(torch.softmax(s, dim=-1) @ v[:, h // per].contiguous())
    return torch.stack(out, 1).reshape(t, -1)


def _opt_exact(case, w, prompts):
    _, layers, heads, _, table, pre = OPT_SIZES[case["model"]]

    def get(name):
        return w["model.decoder." + name].double()

    def norm(x, name):
        return _layer_norm(x, get(name + ".weight"), get(name + ".bias"))

    embed, places = w["model.decoder.embed_tokens.weight"], w["model.decoder.embed_positions.weight"]
    xs = []
    for p in prompts:
        x = embed[torch.tensor(p, device="cuda")].double()
        if "model.decoder.project_in.weight" in w:
            x = x @ get("project_in.weight").T
        xs.append(x + places[2:2 + len(p)].double())
    for i in range(layers):
        q = f"layers.{i}."
        m = {n: (get(f"{q}{n}.weight"), get(f"{q}{n}.bias")) for n in
             ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.out_proj", "fc1", "fc2")}
        for j, x in enumerate(xs):
            def linear(name, y):
                return torch.addmm(m[name][1], y, m[name][0].T)

            def attention(y):
                a = [linear(f"self_attn.{n}_proj", y).view(len(y), heads, -1) for n in "qkv"]
                return linear("self_attn.out_proj", _attend(a[0] * a[0].shape[-1] ** -0.5, a[1], a[2]))

            n1, n2 = q + "self_attn_layer_norm", q + "final_layer_norm"
            if pre:
                x = x + attention(norm(x, n1))
                x = x + linear("fc2", torch.relu(linear("fc1", norm(x, n2))))
            else:
                x = norm(x + attention(x), n1)
                x = norm(x + linear("fc2", torch.relu(linear("fc1", x))), n2)
            xs[j] = x
    x = torch.stack([x[-1] for x in xs])
    if pre:
        x = norm(x, "final_layer_norm")
    if "model.decoder.project_out.weight" in w:
        x = x @ get("project_out.weight").T
    return x @ embed.double().T


def _turned(x):
    """Positions turned into the first half of every head, `[T, heads, head]`; frequencies as the configuration scales them."""
    t, _, head = x.shape
    dims, half = head // 2, head // 4
    freqs = []
    for i in range(half):
        f = 500000.0 ** (-2.0 * i / dims)
        length = 2.0 * math.pi / f
        s = min(1.0, max(0.0, (8192 / length - 1.0) / (4.0 - 1.0)))
        freqs.append((1.0 - s) * f / 8.0 + s * f)
    angle = torch.arange(t, device="cuda").double()[:, None, None] * torch.tensor(freqs, dtype=torch.float64, device="cuda")
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin(), x[..., dims:]], -1)


def _memory(w, p, hs, heads, head):
    """The matrix memory over several sequences side by side (the shorter ones filled up at their end)."""
    t, n = max(len(h) for h in hs), SUNATAR_MEMORY_HEAD
    h = torch.stack([torch.nn.functional.pad(x, (0, 0, 0, t - len(x))) for x in hs], 1)                # [T, rows, width]

    def many(name, size):
        return (h @ w(p + name).T).view(t, len(hs), heads, size)

    q, k, v = many("q", n) * n ** -0.5, many("k", n), many("v", head)
    gi = 15.0 * torch.tanh((h @ w(p + "i").T + w(p + "i.b")) / 15.0)
    gf = torch.nn.functional.logsigmoid(15.0 * torch.tanh((h @ w(p + "f").T + w(p + "f.b")) / 15.0))
    v = torch.cat([v, torch.ones_like(v[..., :1])], -1)                 # the last column is the normaliser
    held = torch.zeros(len(hs), heads, n, head + 1, dtype=torch.float64, device="cuda")
    peak = torch.zeros(len(hs), heads, dtype=torch.float64, device="cuda")
    out = []
    for s in range(t):
        new = torch.maximum(gf[s] + peak, gi[s])
        keep, take = torch.exp(gf[s] + peak - new), torch.exp(gi[s] - new)
        held = keep[..., None, None] * held + (take[..., None] * k[s])[..., None] * v[s][..., None, :]
        peak = new
        o = (held * q[s][..., None]).sum(-2)
        out.append(o[..., :-1] / (torch.maximum(o[..., -1].abs(), torch.exp(-peak)) + 1e-6)[..., None])
    y = _unit_rms(torch.stack(out)).reshape(t, len(hs), -1) * w(p + "norm") * torch.sigmoid(h @ w(p + "g").T)
    y = y @ w(p + "o").T
    return [y[:len(x), j] for j, x in enumerate(hs)]


def _sunatar_exact(case, tensors, prompts):
    _, heads, head, _ = SUNATAR_SIZES[case["model"]]

    def w(name):
        return tensors[name].double()

    def attention(p, h, first):
        def project(name, count):
            return h @ w(p + name).T + w(p + name + ".b"), count
        q, k, own = (project(n, c)[0] for n, c in (("q", heads), ("k", heads // 4), ("v", heads // 4)))
        q = _turned((_unit_rms(q) * w(p + "q.norm")).view(len(h), heads, head))
        k = _turned((_unit_rms(k) * w(p + "k.norm")).view(len(h), heads // 4, head))
        own = own.view(len(h), heads // 4, head)
        v = own if first is None else (1.0 - w(p + "vmix")) * own + w(p + "vmix") * first
        return _attend(q * head ** -0.5, k, v, SUNATAR_WINDOW) @ w(p + "o").T, own

    def expert(p, x):
        return (torch.nn.functional.silu(x @ w(p + "gate").T) * (x @ w(p + "up").T)) @ w(p + "down").T

    xs = [tensors["embed"][torch.tensor(p, device="cuda")].double() for p in prompts]
    first = [None] * len(xs)
    for i in range(SUNATAR_LAYERS):
        hs = [_layer_norm(x, w(f"l{i}.norm1")) for x in xs]
        if i % 4 == 1:
            ys = _memory(w, f"l{i}.mix.", hs, heads, head)
        else:
            ys = []
            for j, h in enumerate(hs):
                y, own = attention(f"l{i}.mix.", h, first[j])
                first[j] = own if first[j] is None else first[j]
                ys.append(y)
        h, p = torch.cat(hs), f"l{i}.mlp."
        score, chosen = torch.topk(torch.sigmoid(h @ w(p + "router").T), CHOSEN, dim=-1)
        out = expert(p + "shared.", h)
        for e in range(EXPERTS):
            rows, place = torch.nonzero(chosen == e, as_tuple=True)
            out[rows] += expert(f"{p}e{e}.", score[rows, place][:, None] * h[rows])
        for j, o in enumerate(torch.split(out, [len(x) for x in xs])):
            xs[j] = xs[j] + ys[j] + o
    return _layer_norm(torch.stack([x[-1] for x in xs]), w("final.norm")) @ w("head").T
