"""Products of 9 to 48 rows by blocks of two to four waves with K whole, at the edges of their rows, columns and steps of K, against
64 bits. Bound: n 2^-24 of the sum of magnitudes for float32 sums of n exact products (first order; 2 covers the rest), and the
result's rounding to bfloat16."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


@pytest.mark.parametrize("waves", [0, 2, 3, 4])
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (9, 48, 256), (16, 80, 384), (17, 208, 512), (32, 1040, 640), (33, 64, 1152), (48, 112, 2048),
                                   (48, 96, 128)])
def test_sizes(m, n, k, waves):
    from transformers_neuronx_amd.kernels.hip import HipOps, tile_order
    hip, g = HipOps(torch.bfloat16, DEV), _gen(m + n + k + waves)
    x = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
    w = torch.randn(n, k, device=DEV, generator=g).to(torch.bfloat16)
    tiles, bias = tile_order(w), torch.randn(n, device=DEV, generator=g)
    exact = x.double() @ w.double().T + bias.double()
    sizes = x.double().abs() @ w.double().abs().T + bias.abs()
    for dtype, act, code in ((torch.bfloat16, 1, 1), (torch.float32, 0, 0)):
        out = torch.full((m + 1, n), 7.0, device=DEV, dtype=dtype)         # (a row behind the last stays)
        hip.call("gemm", "tnx_gemm_bf16_whole", x.data_ptr(), tiles.data_ptr(), bias.data_ptr(), out.data_ptr(), code, act, m, n, k, waves,
                 hip.stream())
        want = exact.relu() if act else exact
        off = 2 * (k + 2) * 2.0 ** -24 * sizes + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
        assert bool(((out[:m].double() - want).abs() <= off).all()) and bool((out[m] == 7).all())


@pytest.mark.parametrize("m", [9, 17, 33, 48])
def test_folded_and_plain_copies_of_their_sizes(m):
    """`linear` takes them where a step has so many rows, from a folded copy and from a plain one."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g, k, n = HipOps(torch.bfloat16, DEV), _gen(m), 2048, 6144
    assert hip._whole_product(m, n, k) and not hip._whole_product(8, n, k) and not hip._whole_product(49, n, k)
    t = torch.randn(m, k, device=DEV, generator=g) + 1
    gamma, beta = 1 + 0.1 * torch.randn(k, device=DEV, generator=g), torch.randn(k, device=DEV, generator=g)
    w, bias = (torch.randn(n, k, device=DEV, generator=g) * 0.05).to(torch.bfloat16), torch.randn(n, device=DEV, generator=g)
    y = (t - t.mean(-1, keepdim=True)).double()
    y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-5) * gamma + beta
    want = (y @ w.double().T + bias).relu()
    plain, folded = hip.prepare_weight(w), hip.prepare_weight(w.clone())
    assert hip.fold_norm(folded, gamma, beta)
    for pw in (plain, folded):
        got = hip.linear(hip.layernorm_deferred(t, gamma, beta, 1e-5, torch.bfloat16), pw, bias, act="relu")
        # three roundings to bfloat16 (the weight's with its factor, the operand's, the result's), independent of one another
        assert (got.double() - want).norm() <= 3 * 2.0 ** -9 * want.norm()


@pytest.mark.parametrize("m,n,k,linear,placed", [
    (16, 3072, 16384, False, False), (24, 4096, 4096, False, False), (48, 4096, 16384, False, False), (9, 6144, 4096, False, False),
    (16, 8192, 8192, False, False), (16, 16384, 4096, False, False), (17, 16384, 4096, True, True), (16, 12288, 4096, True, True),
    (16, 15360, 5120, True, True), (16, 8192, 2048, True, True), (24, 6144, 4096, True, True), (32, 6144, 4096, False, True),
    (33, 6144, 4096, True, True), (48, 15360, 5120, False, True), (48, 16384, 4096, True, True), (48, 16384, 1024, False, True), (48, 12288, 2048, True, True), (32, 16384, 1024, True, True),
    (40, 5632, 4096, False, False), (40, 16400, 4096, False, False), (40, 8192, 1024, False, False)])
def test_the_rule_on_sizes(m, n, k, linear, placed):
    """The lines of the rule at 256 units, by what lies on either side of each, and that a step goes where the rule says."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip = HipOps(torch.bfloat16, DEV)
    hip.compute_units = 256
    assert (hip._whole_product(m, n, k), hip._whole_product(m, n, k, placed=True)) == (linear, placed)
    called = []
    hip._linear_whole = lambda *a: called.append(a)
    hip.linear(torch.zeros(m, k, device=DEV, dtype=torch.bfloat16), hip.prepare_weight(torch.zeros(n, k, device=DEV, dtype=torch.bfloat16)))
    assert bool(called) == (linear and n % 16 == 0)


@pytest.mark.parametrize("m,heads,kv,hs,k,turned", [(9, 32, 32, 64, 2048, False), (40, 32, 32, 64, 2048, True), (24, 32, 32, 80, 2560, False),
                                                       (9, 320, 40, 18, 1024, True)])       # heads that do not come in fours
def test_queries_keys_and_values(m, heads, kv, hs, k, turned):
    """The same places hold what the few-rows kernel, or the product and the launch behind it, leave there."""
    from test_float32_gpu import _step
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g, page = HipOps(torch.bfloat16, DEV), _gen(m + heads + k), 16
    ctx, pages = _step([1] * m, [3 + 7 * (i % 9) for i in range(m)], page, seed=m)
    view, total = ctx.groups["full"], (heads + 2 * kv) * hs
    h = torch.randn(m, k, device=DEV, generator=g).to(torch.bfloat16)
    w = hip.prepare_weight((torch.randn(total, k, device=DEV, generator=g) * 0.05).to(torch.bfloat16))
    bias = torch.randn(total, device=DEV, generator=g)
    turn = tuple(torch.randn(128, hs, device=DEV, generator=g) for _ in "ab") if turned else None
    left = []
    for rows in (0, HipOps.whole_rows):
        hip.whole_rows = rows
        kp = torch.zeros(pages, kv, page, hs, device=DEV, dtype=torch.bfloat16)
        vp = torch.zeros(pages, kv, hs, page, device=DEV, dtype=torch.bfloat16)
        q = hip.qkv_project(h, w, bias, heads, kv, hs, 0.125, ctx, view, kp, vp, turn=turn)
        left.append((q.float(), kp.float(), vp.float()))
    for a, b in zip(*left):
        # sums in another order: a result in a hundred falls to the other side of a rounding, 2^-8 of it
        assert bool((b != 0).equal(a != 0)) and (a - b).norm() <= 2.0 ** -8 * a.norm()
