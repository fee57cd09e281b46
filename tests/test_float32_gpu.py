"""The float32 engine's kernels on the matrix instructions and for single tokens, against 64-bit arithmetic, at the edges of
their tiles. Bounds: a sum of n float32 products in any order is off by at most n 2^-24 times the sum of their magnitudes
(first order; 2 covers the rest)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


@pytest.mark.parametrize("m,n,k", [(1, 5, 4), (1, 1000, 1028), (2, 64, 260), (3, 1024, 4096), (4, 20000, 512), (8, 100, 2052),
                                   (16, 20000, 260), (17, 48, 32), (64, 64, 64), (65, 100, 96), (101, 2048, 2048),
                                   (129, 50, 512), (180, 1024, 4096), (401, 2048, 1024), (513, 4100, 320), (40, 7, 1056)])
def test_float32_product(m, n, k):
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g = HipOps(torch.float32, DEV), _gen(m + n + k)
    x = torch.randn(m, k, device=DEV, generator=g)
    w = torch.randn(n, k, device=DEV, generator=g)
    bias, res = torch.randn(n, device=DEV, generator=g), torch.randn(m, n, device=DEV, generator=g)
    exact = x.double() @ w.double().T
    bound = 2 * (k + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + bias.abs() + res.abs())
    for b, r, act in ((None, None, None), (bias, None, "relu"), (bias, res, None)):
        got = hip.linear(x, w, b, act=act, residual=r, out_f32=True).double()
        want = exact + (b.double() if b is not None else 0)
        want = want.relu() if act else want
        want = want + (r.double() if r is not None else 0)
        assert bool(((got - want).abs() <= bound).all())
    # a row that is not finite is its own alone
    x[m // 2, k // 2] = float("inf")
    got = hip.linear(x, w, out_f32=True)
    assert not bool(torch.isfinite(got[m // 2]).any())
    rest = torch.arange(m, device=DEV) != m // 2
    assert bool(torch.isfinite(got[rest]).all())


@pytest.mark.parametrize("m,n,k", [(17, 64, 32), (64, 132, 96), (65, 2048, 224), (128, 129, 1024), (180, 3072, 1024), (401, 512, 2048),
                                   (401, 2048, 2048), (401, 8192, 2048), (401, 8190, 2048)])
def test_float32_product_by_parts(m, n, k):
    """Products of more than 16 rows are made of the operands' bfloat16 parts: operands over twenty powers of two, whose lower
    parts count, and numbers that have no parts. An element's error is at most one rounding of a running sum for each 16 of K
    (h h; 16 exact products join it), one for the five other products' sums (2^-8 of the magnitudes, 5 roundings for each 16 of K),
    what is left out (2^-24) and the shares' sum: together less than (k / 16 + 8) 2^-23 of the sum of magnitudes. (A lost part of a
    long sum hides in that: `test_every_part_reaches_the_result` has results of one product each.)"""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g = HipOps(torch.float32, DEV), _gen(m + n + k)

    def some(*shape):
        x = torch.randn(*shape, device=DEV, generator=g)
        return x * torch.exp2(torch.randint(-10, 10, shape, device=DEV, generator=g).float())

    x, w = some(m, k), some(n, k)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    got = hip.linear(x, w, out_f32=True).double()
    assert bool(((got - want).abs() <= (k / 16 + 8) * 2.0 ** -23 * size).all())
    # infinities meet weights that one part holds whole (the others are 0), and numbers that round to an infinity
    w[0], w[1] = 1.0, -0.5
    x[0, 3], x[1, k - 1], x[2, 5], x[2, 6] = float("inf"), float("-inf"), float("inf"), float("-inf")
    x[3], x[4], x[4, 7] = 0.0, 0.0, float("nan")
    x[3, 1], w[2] = 3.4e38, 0.25
    got = hip.linear(x, w, out_f32=True)
    assert got[0, 0].item() == float("inf") and got[0, 1].item() == float("-inf")
    assert got[1, 0].item() == float("-inf") and got[1, 1].item() == float("inf")
    assert bool(got[2, :2].isnan().all()) and bool(got[4].isnan().all())
    assert got[3, 2].item() == x[3, 1].item() * 0.25 and got[3, 1].item() == x[3, 1].item() * -0.5
    assert bool(torch.isfinite(got[5:]).all())


def _full(shape, g, least, most):
    """Numbers with all 24 bits of a mantissa, from 2^least to 2^(most + 1), of either sign."""
    bits = torch.randint(0, 1 << 23, shape, device=DEV, generator=g).double() / (1 << 23)
    power = torch.randint(least, most + 1, shape, device=DEV, generator=g).double()
    sign = torch.randint(0, 2, shape, device=DEV, generator=g).double() * 2 - 1
    return (sign * (1 + bits) * torch.exp2(power)).float()


def _by_parts(x, w, tile, shares):
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, (m, k), n = HipOps(torch.float32, DEV), x.shape, w.shape[0]
    out, space = torch.full((m + 1, n), 7.0, device=DEV), torch.empty(shares * m * n, device=DEV)
    hip.call("gemm", "tnx_gemm_f32_parts", x.data_ptr(), w.data_ptr(), None, None, out.data_ptr(), 0, 0, m, n, k, tile, shares,
             space.data_ptr(), space.numel(), hip.stream())
    assert bool((out[m] == 7).all())              # (a row behind the last stays)
    return out[:m].double()


def _one_a_row(m, k):
    """A place of K for every row, over all steps of 32 and the places in them."""
    row, steps = torch.arange(m, device=DEV), k // 32
    return row, 32 * (row % steps) + (11 * row + row // steps) % 32


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("m,n,k,shares", [(130, 129, 32 * steps, 1) for steps in range(1, 9)] +
                         [(17, 66, 416, 1), (65, 64, 512, 16), (257, 132, 1184, 4), (401, 260, 2048, 8), (128, 128, 2048, 1)])
def test_every_part_reaches_the_result(m, n, k, shares, tile):
    """One number in a row of x, so that a result is one product of two numbers of 24 bits. What is left out is 2^-24 of it
    (l m and m l, 2^-17 and 2^-8 of the operands at most) and 2^-34 (l l), the sum of the other five parts rounds below 2^-30, and
    that joins the h h with one rounding, 2^-24: together under 2.05 of those, on every
    tile, at every number of steps, in every share. The smallest part made, a product of an h with an l, is up to 2^-17."""
    g = _gen(m + n + k + tile)
    row, place = _one_a_row(m, k)
    x, w = torch.zeros(m, k, device=DEV), _full((n, k), g, -9, 9)
    x[row, place] = _full((m,), g, -9, 9)
    want = x[row, place].double()[:, None] * w[:, place].double().T
    assert bool(((_by_parts(x, w, tile, shares) - want).abs() <= 2.05 * 2.0 ** -24 * want.abs()).all())


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("least,most", [(-113, -105), (-126, -114), (-136, -127)])
def test_operands_whose_parts_are_too_small_for_numbers(least, most, tile):
    """Lower parts end at 2^-133, the smallest bfloat16 number: an operand under 2^-110 is off by up to half of that, no more."""
    m, n, k = 130, 128, 256
    g = _gen(least + tile)
    row, place = _one_a_row(m, k)
    x, w = torch.zeros(m, k, device=DEV), _full((n, k), g, 95, 100)
    x[row, place] = _full((m,), g, least, most)
    assert bool((x[row, place] != 0).all())
    want = x[row, place].double()[:, None] * w[:, place].double().T
    off = 2.05 * 2.0 ** -24 * want.abs() + 2.0 ** -134 * w[:, place].double().abs().T
    assert bool(((_by_parts(x, w, tile, 1) - want).abs() <= off).all())


@pytest.mark.parametrize("m,n,k,shares", [(17, 1024, 1024, 16), (64, 1024, 1024, 11), (31, 132, 4096, 16), (33, 2304, 768, 6), (128, 512, 4096, 16),
                                          (129, 512, 4096, 8)])
def test_shares_of_few_rows(m, n, k, shares):
    """K shared out over up to sixteen blocks at 128 rows, eight beyond; every share's sums go out by themselves, and what is not
    finite in one is made again in it. Bound: as `test_float32_product_by_parts`, and the shares' sum."""
    from transformers_neuronx_amd.kernels.hip import HipOps, library
    hip, g = HipOps(torch.float32, DEV), _gen(m + n + k)
    if hip.compute_units == 256:
        assert library("gemm").tnx_gemm_f32_workspace(m, n, k) == shares * m * n
    x, w = torch.randn(m, k, device=DEV, generator=g), torch.randn(n, k, device=DEV, generator=g)
    bias, residual = torch.randn(n, device=DEV, generator=g), torch.randn(m, n, device=DEV, generator=g)
    want = (x.double() @ w.double().T + bias).relu() + residual
    size = x.double().abs() @ w.double().abs().T + bias.abs() + residual.abs()
    got = hip.linear(x, w, bias, act="relu", residual=residual, out_f32=True)
    assert bool(((got.double() - want).abs() <= (k / 16 + 8 + 16) * 2.0 ** -23 * size).all())
    w[3] = w[3].abs()
    x[0, 5], x[1, k - 1], x[m - 1, k // 2] = float("inf"), float("nan"), 3.4e38
    w[:, k // 2] = 0.25
    got = hip.linear(x, w, None, out_f32=True)
    assert got[0, 3].item() == float("inf") and bool(got[1].isnan().all())
    assert bool((got[m - 1] == x[m - 1, k // 2] * 0.25).all()) and bool(torch.isfinite(got[2:]).all())


def _step(runs, cached, page, seed):
    from transformers_neuronx_amd.engine.batch import StepEntry, build_context
    from transformers_neuronx_amd.kernels.attention_plan import attention_plan
    width = max(-(-(c + r) // page) for c, r in zip(cached, runs))
    order = torch.randperm(len(runs) * width, generator=torch.Generator().manual_seed(seed)).view(len(runs), width)
    table = order.to(torch.int32).numpy()
    entries = [StepEntry(i, [0] * r, [r - 1]) for i, r in enumerate(runs)]
    return build_context(entries, list(cached), list(range(len(runs))), {"full": table}, page, DEV,
                         {"attention": attention_plan}), len(runs) * width


@pytest.mark.parametrize("heads,kv,hs", [(4, 4, 64), (8, 2, 80), (2, 1, 128), (3, 3, 16), (4, 2, 48)])
@pytest.mark.parametrize("page", [16, 48, 64])
@pytest.mark.parametrize("window", [None, 37])
def test_float32_attention(heads, kv, hs, page, window):
    """Portions of prompts behind a cache, single tokens, whole short prompts, in one step; what lies behind a request's last
    token in its pages is not a number."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g = HipOps(torch.float32, DEV), _gen(heads * hs + page)
    runs, cached = [70, 1, 33, 1, 2, 1, 129], [45, 0, 0, 700, 31, 64, 0]
    ctx, pages = _step(runs, cached, page, seed=hs)
    view = ctx.groups["full"]
    kp = torch.full((pages, kv, page, hs), float("nan"), device=DEV)
    vp = torch.full((pages, kv, hs, page), float("nan"), device=DEV)
    q = torch.randn(sum(runs), heads * hs, device=DEV, generator=g) * hs ** -0.5
    want, bound, at = torch.empty(sum(runs), heads, hs, dtype=torch.float64, device=DEV), None, 0
    for r, (n, c) in enumerate(zip(runs, cached)):
        total = c + n
        keys = torch.randn(kv, total, hs, device=DEV, generator=g)
        vals = torch.randn(kv, total, hs, device=DEV, generator=g)
        for b in range(-(-total // page)):
            p, rows = int(view.block_table[r, b]), slice(b * page, min(total, (b + 1) * page))
            kp[p, :, :rows.stop - rows.start] = keys[:, rows]
            vp[p, :, :, :rows.stop - rows.start] = vals[:, rows].transpose(1, 2)
        qr = q[at:at + n].double().view(n, heads, hs).transpose(0, 1)
        s = qr @ keys.double().repeat_interleave(heads // kv, 0).transpose(1, 2)
        i, j = torch.arange(c, total, device=DEV)[:, None], torch.arange(total, device=DEV)[None]
        hidden = (j > i) | ((i - j >= window) if window else (j > i))
        want[at:at + n] = (torch.softmax(s.masked_fill(hidden, float("-inf")), -1)
                           @ vals.double().repeat_interleave(heads // kv, 0)).transpose(0, 1)
        at += n
    got = hip.attention(q, heads, kv, hs, ctx, view, kp, vp, window)
    # weights of scores up to 8 or so: off by their scores' error (hs + 2 roundings of at most 8) and their sums' (760 keys)
    torch.testing.assert_close(got.double(), want.reshape(sum(runs), -1), rtol=0, atol=5 * (8 * hs + 760) * 2.0 ** -24)


def test_float32_attention_keeps_a_value_that_is_no_number_to_its_readers():
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g = HipOps(torch.float32, DEV), _gen(3)
    heads, hs, page, n = 2, 64, 64, 50
    ctx, pages = _step([n], [0], page, seed=1)
    kp = torch.randn(pages, heads, page, hs, device=DEV, generator=g)
    vp = torch.randn(pages, heads, hs, page, device=DEV, generator=g)
    q = torch.randn(n, heads * hs, device=DEV, generator=g) * 0.1
    clean = hip.attention(q, heads, heads, hs, ctx, ctx.groups["full"], kp, vp)
    vp[int(ctx.groups["full"].block_table[0, 0]), 1, 5, 21] = float("inf")
    got = hip.attention(q, heads, heads, hs, ctx, ctx.groups["full"], kp, vp).view(n, heads, hs)
    clean = clean.view(n, heads, hs).clone()
    assert bool(torch.isinf(got[21:, 1, 5]).all())
    got[21:, 1, 5] = clean[21:, 1, 5] = 0
    torch.testing.assert_close(got, clean, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("runs,cached", [([2], [0]), ([16], [0]), ([17], [0]), ([24], [0]), ([25], [0]), ([5, 1, 3], [11, 15, 0]), ([16, 16], [0, 0])])
@pytest.mark.parametrize("heads,kv,hs", [(4, 2, 64), (32, 8, 128), (40, 40, 16)])
def test_float32_attention_of_short_steps(runs, cached, heads, kv, hs):
    """Either side of the lengths up to which a wave takes a query alone, beside the kernel that always does."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, plain, g, page, n = HipOps(torch.float32, DEV), HipOps(torch.float32, DEV), _gen(hs), 32, sum(runs)
    plain.force_plain_attention = True
    ctx, pages = _step(runs, cached, page, seed=3)
    few = max(r + c for r, c in zip(runs, cached)) <= (24 if hs > 96 else 16) and n * heads <= 1024
    assert hip._few_scores(ctx, heads, hs) == few
    kp = torch.randn(pages, kv, page, hs, device=DEV, generator=g)
    vp = torch.randn(pages, kv, hs, page, device=DEV, generator=g)
    q = torch.randn(n, heads * hs, device=DEV, generator=g) * hs ** -0.5
    got, want = (x.attention(q, heads, kv, hs, ctx, ctx.groups["full"], kp, vp) for x in (hip, plain))
    # (the bound of `test_float32_attention`)
    torch.testing.assert_close(got, want, rtol=0, atol=5 * (8 * hs + 760) * 2.0 ** -24)


@pytest.mark.parametrize("runs,cached,first,last", [([160], [0], 32, 63), ([300], [0], 0, 31), ([33], [0], 32, 32), ([20], [90], 64, 95),
                                                    ([1], [200], 64, 127), ([1], [128], 128, 128), ([1], [700], 0, 63), ([1, 1], [63, 448], 0, 511)])
@pytest.mark.parametrize("window", [None, 37])
@pytest.mark.parametrize("heads,kv,hs", [(4, 2, 64), (3, 3, 80)])
def test_float32_attention_of_keys_that_are_no_numbers(runs, cached, first, last, window, heads, kv, hs):
    """Keys `first` to `last`, the whole share of one wave or of several, are no numbers: nor is the result of a query that sees
    one of them, and the others are as without. Keys infinitely far from a query weigh nothing."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g, page, n = HipOps(torch.float32, DEV), _gen(first + hs), 64, sum(runs)
    ctx, pages = _step(runs, cached, page, seed=hs)
    view = ctx.groups["full"]
    clean = torch.randn(pages, kv, page, hs, device=DEV, generator=g)
    vp = torch.randn(pages, kv, hs, page, device=DEV, generator=g)
    q = torch.randn(n, heads * hs, device=DEV, generator=g) * hs ** -0.5
    q.view(n, heads, hs)[..., 0] = 0.1
    for spoil in (float("nan"), -float("inf")):
        kp, want, sees = clean.clone(), [], []
        for r, (count, c) in enumerate(zip(runs, cached)):
            at = torch.arange(c + count, device=DEV)
            table = view.block_table[r].long()[at // page]
            own = (at >= first) & (at <= last)
            kp[table[own], :, at[own] % page, 0] = spoil
            keys, vals = (x.double().transpose(0, 1).repeat_interleave(heads // kv, 0)
                          for x in (kp[table, :, at % page], vp[table, :, :, at % page]))
            i = torch.arange(c, c + count, device=DEV)[:, None]
            hidden = (at > i) | ((i - at >= window) if window else (at > i))
            s = q[sum(runs[:r]):][:count].double().view(count, heads, hs).transpose(0, 1) @ keys.transpose(1, 2)
            want.append((torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ vals).transpose(0, 1))
            sees.append((own & ~hidden).any(1))
        want, sees = torch.cat(want).reshape(n, -1), torch.cat(sees)
        if spoil != spoil:
            assert torch.equal(torch.isnan(want).any(1), sees) and torch.equal(torch.isnan(want).all(1), sees)
        got = hip.attention(q, heads, kv, hs, ctx, view, kp, vp, window).double()
        # (the bound of `test_float32_attention`: nothing here is longer)
        torch.testing.assert_close(got, want, rtol=0, atol=5 * (8 * hs + 760) * 2.0 ** -24, equal_nan=True)


@pytest.mark.parametrize("runs,cached", [([1], [0]), ([1, 1, 1], [63, 64, 200]), ([5, 1], [0, 30]), ([16], [120]), ([17], [7])])
@pytest.mark.parametrize("heads,kv,hs,page,width", [(4, 4, 16, 16, 68), (6, 2, 48, 32, 1280), (16, 16, 64, 64, 1024), (3, 1, 80, 64, 2052),
                                                    (64, 0, 64, 16, 516)])
@pytest.mark.parametrize("turned", [False, True])
def test_float32_projections_go_where_they_belong(runs, cached, heads, kv, hs, page, width, turned):
    """From the few-rows product straight into queries, keys and values, against the product and the scatter apart: the same
    operations on every number."""
    from test_kernels_gpu import _make_step
    from transformers_neuronx_amd.kernels.hip import HipOps
    pages = sum(-(-(r + c) // page) for r, c in zip(runs, cached)) + 2
    ctx = _make_step(runs, cached, page, pages, seed=hs)
    g = _gen(hs + width)
    total = (heads + 2 * kv) * hs
    h = torch.randn(ctx.num_tokens, width, device=DEV, generator=g)
    w, bias = torch.randn(total, width, device=DEV, generator=g), torch.randn(total, device=DEV, generator=g)
    turn = tuple(torch.randn(300, hs, device=DEV, generator=g) for _ in range(2)) if turned else None
    made = []
    for rows in (16, 0):
        ops = HipOps(torch.float32, DEV)
        ops.f32_scatter_rows = rows
        for b in (bias, None):
            kp = torch.full((pages, kv, page, hs), 7.0, device=DEV) if kv else None
            vp = torch.full((pages, kv, hs, page), 7.0, device=DEV) if kv else None
            q = ops.qkv_project(h, w, b, heads, kv, hs, 0.3, ctx, ctx.groups["full"], kp, vp, turn=turn)
            made.append([q] + ([kp, vp] if kv else []))
    for fused, apart in zip(made[:2], made[2:]):
        for one, other in zip(fused, apart):
            # (a multiplication and an addition may be one rounding here and two there)
            assert torch.equal(one, other) or (turned and float((one - other).abs().max()) <= 2.0 ** -21 * float(other.abs().max()))
