"""Products by tiles of 64 and 128 rows against 64-bit arithmetic: the experts' over many pairs each, at the edges of tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _apart(got, want):
    return float((got.double() - want).norm() / want.norm())


def _act(name, g, u, limit):
    if name == "silu":
        return torch.nn.functional.silu(g) * u
    if name == "gelu_new":
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    if name == "clamped_swiglu":
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(1.702 * g) * (u + 1)
    return {"relu": torch.relu, "relu2": lambda x: torch.relu(x) ** 2}[name](g)


@pytest.mark.parametrize("counts", [[64, 0, 65, 127], [1, 128, 129, 300], [200, 31, 0, 1], [700, 513, 5, 64]])
@pytest.mark.parametrize("width,f", [(64, 64), (192, 320), (256, 128)])
@pytest.mark.parametrize("act,on,identity", [("silu", "input", 0), ("gelu_new", "output", 0), ("clamped_swiglu", "output", 2),
                                             ("relu2", "output", 0), ("relu", "output", 1)])
@pytest.mark.parametrize("rows", [64, 128])
def test_experts_by_tiles(counts, width, f, act, on, identity, rows):
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops = HipOps(torch.bfloat16, DEV)
    ops.expert_grouped_rows = 1
    ops.expert_wide_tiles = 1 if rows == 128 else 1 << 30
    g = torch.Generator(device=DEV).manual_seed(sum(counts) + width)
    experts, gated = len(counts), act not in ("relu", "relu2")
    flat = torch.repeat_interleave(torch.arange(experts, device=DEV), torch.tensor(counts, device=DEV))
    flat = flat[torch.randperm(flat.numel(), device=DEV, generator=g)]
    tokens = -(-flat.numel() // 2)
    # the places left over: experts without tensors where there are some, else the first again
    fill = torch.full((2 * tokens - flat.numel(),), experts if identity else 0, device=DEV)
    chosen = torch.cat([flat, fill]).view(tokens, 2)
    if identity:
        chosen[::7, 1] = experts + identity - 1
    weights = torch.rand(tokens, 2, device=DEV, generator=g) + 0.1
    h = torch.randn(tokens, width, device=DEV, generator=g).bfloat16()
    up = (torch.randn(experts, (2 if gated else 1) * f, width, device=DEV, generator=g) * width ** -0.5).bfloat16()
    down = (torch.randn(experts, width, f, device=DEV, generator=g) * f ** -0.5).bfloat16()
    residual = torch.randn(tokens, width, device=DEV, generator=g)
    want = torch.zeros(tokens, width, dtype=torch.float64, device=DEV)
    for c in range(2):
        for e in range(experts):
            at = (chosen[:, c] == e).nonzero().flatten()
            x, s = h[at].double(), weights[at, c].double()[:, None]
            z = (x * s if on == "input" else x) @ up[e].double().T
            y = _act(act, z[:, :f], z[:, f:], 1.5) @ down[e].double().T
            want[at] += y if on == "input" else s * y
        same = chosen[:, c] >= experts
        want[same] += weights[same, c].double()[:, None] * h[same].double()
    for r in (residual, None):
        got = ops.expert_mixture(h, chosen.int().contiguous(), weights, up, down, act, on, r,
                                 limit=1.5 if act == "clamped_swiglu" else None, identity=identity)
        # the inner values are rounded to bfloat16 (by 2^-8 of themselves at most), everything else is summed in float32
        assert _apart(got - (r if r is not None else 0), want) < 2.0 ** -8


@pytest.mark.parametrize("tokens,experts,top,width,f", [(16, 1, 1, 32768, 32768), (32768, 8, 8, 64, 8192), (65536, 1, 1, 32768, 64)])
def test_experts_beyond_the_reach_of_tiles(tokens, experts, top, width, f):
    """A matrix, the pairs' inner rows or the tokens' rows of 4 GB: more than the tiles can count, so the step goes the other way."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops, g = HipOps(torch.bfloat16, DEV), torch.Generator(device=DEV).manual_seed(width)
    assert not ops._tiles_reach(tokens, experts, top, width, f, 128) and ops._tiles_reach(tokens // 2, experts, top, width, f // 2, 128)

    def some(*shape, std=1.0):
        return torch.empty(shape, device=DEV, dtype=torch.bfloat16).normal_(0.0, std, generator=g)

    h, up, down = some(tokens, width), some(experts, f, width, std=width ** -0.5), some(experts, width, f, std=f ** -0.5)
    chosen = torch.arange(top, device=DEV, dtype=torch.int32).expand(tokens, top).contiguous()
    weights = torch.rand(tokens, top, device=DEV, generator=g) + 0.1
    got = ops.expert_mixture(h, chosen, weights, up, down, "relu", "output", None)
    rows = torch.arange(tokens, device=DEV) if tokens < 64 else torch.cat([torch.arange(32, device=DEV), torch.arange(tokens - 32, tokens, device=DEV)])
    want = torch.zeros(len(rows), width, device=DEV)
    for e in range(top):        # (in float32, whose error is none beside the inner values' rounding to bfloat16)
        want += weights[rows, e, None] * (torch.relu(h[rows].float() @ up[e].float().T) @ down[e].float().T)
    assert _apart(got[rows], want.double()) < 2.0 ** -8


@pytest.mark.parametrize("m,n,k", [(17, 64, 64), (33, 200, 64), (64, 72, 320), (65, 2048, 2048), (128, 136, 8192), (129, 128, 512),
                                   (333, 264, 2048), (700, 520, 2112)])
@pytest.mark.parametrize("tile,shares", [(1, 1), (1, 3), (2, 1), (2, 5)])
def test_product_by_tiles(m, n, k, tile, shares):
    """Every tile with and without shares of K, at sizes that end inside a tile."""
    from transformers_neuronx_amd.kernels.hip import HipOps, _ptr, _stream
    ops, g = HipOps(torch.bfloat16, DEV), torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = torch.randn(m, k, device=DEV, generator=g).bfloat16(), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).bfloat16()
    bias, res = torch.randn(n, device=DEV, generator=g), torch.randn(m, n, device=DEV, generator=g)
    exact = x.double() @ w.double().T
    space = torch.empty(shares * m * n, device=DEV)
    magnitude = x.double().abs() @ w.double().abs().T + bias.abs() + res.abs()
    for b, r, act, dtype in ((bias, None, 1, torch.bfloat16), (bias, res, 0, torch.float32), (None, None, 0, torch.float32)):
        out = torch.full((m, n), float("nan"), device=DEV, dtype=dtype)
        ops.call("gemm", "tnx_gemm_bf16_tiles", _ptr(x), _ptr(w), _ptr(b), _ptr(r), _ptr(out), int(dtype == torch.bfloat16), act,
                 m, n, k, _ptr(space), space.numel(), tile, shares, _stream())
        want = exact + (b.double() if b is not None else 0)
        want = want.relu() if act else want
        want = want + (r.double() if r is not None else 0)
        # products of bfloat16 are exact in float32; a sum of k of them is off by k 2^-24 of the magnitudes at most, and a
        # bfloat16 result (8 bits) by half a place, 2^-8 of it at most, more
        bound = 2 * (k + 4) * 2.0 ** -24 * magnitude + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
        assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k", [(40, 2048, 2048), (100, 6144, 2048), (333, 2048, 8192), (512, 2048, 2048), (640, 6144, 2048), (640, 3072, 1024)])
def test_products_that_the_tiles_take(m, n, k):
    """`linear` takes the tiles there, with what the library's way gives up to the rounding of the result."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops, lib = HipOps(torch.bfloat16, DEV), HipOps(torch.bfloat16, DEV)
    lib.tile_products = False
    g = torch.Generator(device=DEV).manual_seed(n)
    x, w = torch.randn(m, k, device=DEV, generator=g).bfloat16(), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).bfloat16()
    bias, res = torch.randn(n, device=DEV, generator=g), torch.randn(m, n, device=DEV, generator=g)
    assert ops._tiles_room(m, n, k, x, w, None, False, False) >= 0
    for kw in (dict(bias=bias, act="relu"), dict(bias=bias, act="gelu"), dict(residual=res, out_f32=True), dict()):
        torch.testing.assert_close(ops.linear(x, w, **kw).float(), lib.linear(x, w, **kw).float(), rtol=1e-2, atol=2e-2)


@pytest.mark.parametrize("m,n,k", [(64, 12288, 4096), (40, 16384, 4096), (600, 4096, 16384), (640, 4096, 16384), (700, 3072, 12288),
                                   (705, 2048, 8192), (768, 5120, 20480), (768, 2048, 2048), (513, 2048, 2048), (640, 3072, 2048),
                                   (700, 1536, 2048)])
def test_products_that_the_tiles_leave_alone(m, n, k):
    """Products that bound a step by their own time, at sizes where the library was measured to be quicker."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops, x, w = HipOps(torch.bfloat16, DEV), torch.empty(m, k, device=DEV, dtype=torch.bfloat16), torch.empty(n, k, device=DEV, dtype=torch.bfloat16)
    assert ops._tiles_room(m, n, k, x, w, None, False, False) == -1


@pytest.mark.parametrize("n,k,few", [(6144, 2048, True), (8192, 2048, True), (7680, 2560, False), (8320, 2048, False), (4096, 4096, True),
                                     (2048, 8192, False), (1024, 16384, False), (16384, 1024, True), (20480, 768, False), (2048, 4096, True),
                                     (512, 16384, True)])
def test_few_rows_with_a_rounded_result(n, k, few):
    """17 to 24 rows go to the few-rows kernel up to 2^24 elements of the matrix, 2^23 where K is short or long."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops, w = HipOps(torch.bfloat16, DEV), torch.empty(n, k, device=DEV, dtype=torch.bfloat16)
    for m in (17, 24):
        assert ops._library_product(m, n, k, w, False, plain=True) != few


@pytest.mark.parametrize("m,n,k,few", [(17, 6144, 2048, True), (32, 4608, 4096, True), (24, 2688, 7168, True), (17, 1536, 8192, False),
                                       (32, 1024, 8192, True), (24, 18432, 1024, True), (25, 18432, 1024, False), (24, 12288, 4096, False)])
def test_few_rows_of_queries_keys_and_values(m, n, k, few):
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops, w = HipOps(torch.bfloat16, DEV), torch.empty(n, k, device=DEV, dtype=torch.bfloat16)
    assert ops._library_product(m, n, k, w, False, True) != few


@pytest.mark.parametrize("tokens,top", [(1, 2), (3, 3), (8, 2), (9, 7), (32, 2), (33, 2), (16, 4)])
@pytest.mark.parametrize("experts,width,f", [(4, 1024, 1040), (8, 200, 1288), (40, 1032, 72), (1, 1088, 40), (300, 72, 48)])
@pytest.mark.parametrize("act,on", [("silu", "input"), ("relu2", "output")])
def test_experts_of_few_pairs(tokens, top, experts, width, f, act, on):
    """Up to 64 pairs (the blocks find theirs) and beyond, one set of waves or two, experts with no pair and with all."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    if top > experts:
        pytest.skip("more choices than experts")
    ops, g = HipOps(torch.bfloat16, DEV), torch.Generator(device=DEV).manual_seed(tokens * top + experts)
    gated = act == "silu"
    chosen = torch.stack([torch.randperm(experts, device=DEV, generator=g)[:top] for _ in range(tokens)])
    chosen[:, 0] = experts - 1                      # one expert that every token has (perhaps twice: its rows are then added)
    weights = torch.rand(tokens, top, device=DEV, generator=g) + 0.1
    h = torch.randn(tokens, width, device=DEV, generator=g).bfloat16()
    up = (torch.randn(experts, (2 if gated else 1) * f, width, device=DEV, generator=g) * width ** -0.5).bfloat16()
    down = (torch.randn(experts, width, f, device=DEV, generator=g) * f ** -0.5).bfloat16()
    residual = torch.randn(tokens, width, device=DEV, generator=g)
    want = torch.zeros(tokens, width, dtype=torch.float64, device=DEV)
    for t in range(tokens):
        for c in range(top):
            e, s, x = int(chosen[t, c]), weights[t, c].double(), h[t].double()
            z = up[e].double() @ (x * s if on == "input" else x)
            y = down[e].double() @ _act(act, z[:f], z[f:], None)
            want[t] += y if on == "input" else s * y
    got = ops.expert_mixture(h, chosen.int().contiguous(), weights, up, down, act, on, residual)
    assert _apart(got - residual, want) < 2.0 ** -8
