"""Products of few rows that norm the rows beside them, as their operand and as the residual they add, against 64 bits and
against the norm's own kernel. Bounds: n 2^-24 of the sum of magnitudes for float32 sums of n products (first order; 2 covers the
rest), and one rounding of the normed operand to bfloat16 (2^-8 of the magnitudes)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normed(t, weight, bias, eps, center):
    t = t.double()
    mean = t.mean(-1, keepdim=True) if center else torch.zeros_like(t[:, :1])
    y = (t - mean) / torch.sqrt(((t - mean) ** 2).mean(-1, keepdim=True) + eps)
    y = y * weight.double() if weight is not None else y
    return y + bias.double() if bias is not None else y


@pytest.mark.parametrize("m,k,n", [(1, 1024, 4096), (5, 128, 48), (8, 1024, 1024), (8, 2048, 8192), (2, 1152, 12288), (4, 2048, 64)])
@pytest.mark.parametrize("affine,center", [(True, True), (True, False), (False, True)])
def test_operand_and_residual(m, k, n, affine, center):
    from transformers_neuronx_amd.kernels.hip import HipOps, NormBetween
    dt = torch.bfloat16
    hip, g = HipOps(dt, DEV), _gen(m + k + n)
    t = torch.randn(m, k, device=DEV, generator=g) * 3 + torch.randn(m, 1, device=DEV, generator=g) * 5
    gamma = 1 + 0.1 * torch.randn(k, device=DEV, generator=g) if affine else None
    beta = torch.randn(k, device=DEV, generator=g) if affine and center else None
    w = hip.prepare_weight((torch.randn(n, k, device=DEV, generator=g)).to(dt))
    bias = torch.randn(n, device=DEV, generator=g)
    y = _normed(t, gamma, beta, 1e-5, center)
    sizes = y.abs() @ w.tensor.double().abs().T + bias.abs()

    # the operand
    d, same = hip.norm_between(t, gamma, beta, 1e-5, dt, center)
    assert isinstance(d, NormBetween) and same is d
    want = y @ w.tensor.double().T + bias
    for act in (None, "relu"):
        got = hip.linear(d, w, bias, act=act, out_f32=True)
        assert d.done is None                                    # the norm's own kernel has not run
        exact = want.relu() if act else want
        assert bool(((got.double() - exact).abs() <= (2 * (k + 8) * 2.0 ** -24 + 2.0 ** -8) * sizes).all())
    rounded = hip.linear(d, w, bias)
    assert rounded.dtype == dt and torch.allclose(rounded.float(), hip.linear(d, w, bias, out_f32=True), rtol=2.0 ** -8, atol=0)

    # the residual: rows of k beside a product of k columns
    inner = torch.randn(m, 1024, device=DEV, generator=g).to(dt)
    w2 = hip.prepare_weight((torch.randn(k, 1024, device=DEV, generator=g) * 0.02).to(dt))
    got = hip.linear(inner, w2, None, residual=d, out_f32=True)
    assert d.done is None
    product = inner.double() @ w2.tensor.double().T
    bound = 2 * (1024 + 8) * 2.0 ** -24 * (inner.double().abs() @ w2.tensor.double().abs().T + y.abs() + 1)
    assert bool(((got.double() - (product + y)).abs() <= bound).all())

    # settled, it is what the norm's kernel gives, and the products take that
    x32, x = d.settled()
    assert bool(((x32.double() - y).abs() <= 32 * 2.0 ** -24 * (y.abs() + 1)).all()) and x.dtype == dt
    assert torch.equal(hip.linear(inner, w2, None, residual=d, out_f32=True), hip.linear(inner, w2, None, residual=x32, out_f32=True))
    assert torch.equal(hip.linear(d, w, bias, out_f32=True), hip.linear(x, w, bias, out_f32=True))


@pytest.mark.parametrize("dtype,m,width", [(torch.bfloat16, 9, 1024), (torch.bfloat16, 1, 2176), (torch.bfloat16, 1, 1000), (torch.float32, 1, 1024)])
def test_other_sizes_go_to_the_norms_kernel(dtype, m, width):
    from transformers_neuronx_amd.kernels.hip import HipOps
    x, h = HipOps(dtype, DEV).norm_between(torch.randn(m, width, device=DEV), None, None, 1e-5, dtype)
    assert isinstance(x, torch.Tensor) and x.dtype == torch.float32 and h.dtype == dtype


@pytest.mark.parametrize("m,heads,kv,hs,k", [(8, 16, 16, 64, 1024), (1, 8, 2, 80, 256), (3, 32, 32, 64, 2048)])
def test_queries_keys_and_values(m, heads, kv, hs, k):
    """The same places hold what the norm's kernel and the projection of its result leave there."""
    from test_float32_gpu import _step
    from transformers_neuronx_amd.kernels.hip import HipOps
    dt = torch.bfloat16
    hip, g, page = HipOps(dt, DEV), _gen(m + heads + k), 16
    ctx, pages = _step([1] * m, [3 + 7 * i for i in range(m)], page, seed=m)
    view, total = ctx.groups["full"], (heads + 2 * kv) * hs
    t, gamma = torch.randn(m, k, device=DEV, generator=g) + 1, 1 + 0.1 * torch.randn(k, device=DEV, generator=g)
    beta, bias = torch.randn(k, device=DEV, generator=g), torch.randn(total, device=DEV, generator=g)
    w = hip.prepare_weight((torch.randn(total, k, device=DEV, generator=g) * 0.05).to(dt))
    left = []
    for settled in (True, False):
        d = hip.norm_between(t, gamma, beta, 1e-5, dt)[0]
        kp, vp = torch.zeros(pages, kv, page, hs, device=DEV, dtype=dt), torch.zeros(pages, kv, hs, page, device=DEV, dtype=dt)
        q = hip.qkv_project(d.settled()[1] if settled else d, w, bias, heads, kv, hs, 0.125, ctx, view, kp, vp)
        assert (d.done is None) != settled
        left.append((q.float(), kp.float(), vp.float()))
    for a, b in zip(*left):
        # sums in another order, of operands whose rounding may fall the other way
        assert bool((b != 0).equal(a != 0)) and (a - b).norm() <= 8e-3 * a.norm()


@pytest.mark.parametrize("m,k,n", [(1, 256, 48), (8, 1024, 4096), (5, 2176, 6144), (8, 3072, 1040), (4, 2560, 10240), (8, 4096, 4096), (8, 3200, 4096)])
def test_folded_copies(m, k, n):
    """A folded copy's product, of the widths that layers fold (beyond 3,072) and of others, from shifted rows and behind the norm's kernel."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g = HipOps(torch.bfloat16, DEV), _gen(m + k + n)
    t = torch.randn(m, k, device=DEV, generator=g) * 3 + torch.randn(m, 1, device=DEV, generator=g) * 5
    gamma, beta = 1 + 0.1 * torch.randn(k, device=DEV, generator=g), torch.randn(k, device=DEV, generator=g)
    w = torch.randn(n, k, device=DEV, generator=g).to(torch.bfloat16)
    pw, bias = hip.prepare_weight(w), torch.randn(n, device=DEV, generator=g)
    assert hip.fold_norm(pw, gamma, beta)
    got = hip.linear(hip.layernorm_deferred(t, gamma, beta, 1e-5, torch.bfloat16), pw, bias, act="relu")
    y, bare = _normed(t, gamma, beta, 1e-5, True), _normed(t, None, None, 1e-5, True)
    exact = y @ w.double().T + bias
    # the folded weight, the operand (or its shifted row, as large) and the result are each rounded once
    sizes = (bare.abs() + 2) @ (w.double() * gamma).abs().T + (w.double() @ beta.double()).abs() + bias.abs()
    assert bool(((got.double() - exact.relu()).abs() <= 3 * 2.0 ** -8 * sizes).all())


@pytest.mark.parametrize("m,k,n", [(1, 256, 48), (8, 2048, 6144), (5, 3072, 1040), (8, 3072, 12288), (9, 2048, 6144), (3, 3200, 96)])
@pytest.mark.parametrize("center", [True, False])
def test_deferred_norms_of_plain_copies(m, k, n, center):
    """A layer's norm before its matrix: rows of up to 3,072 leave the matrix as it is."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g = HipOps(torch.bfloat16, DEV), _gen(m + k + n)
    t = torch.randn(m, k, device=DEV, generator=g) * 3 + 1
    gamma, beta = 1 + 0.1 * torch.randn(k, device=DEV, generator=g), torch.randn(k, device=DEV, generator=g)
    w = torch.randn(n, k, device=DEV, generator=g).to(torch.bfloat16)
    pw, bias = hip.prepare_weight(w), torch.randn(n, device=DEV, generator=g)
    assert hip.defer_norm(pw, gamma, beta, center) and (pw.folded is None) == (k <= 3072)
    got = hip.linear(hip.layernorm_deferred(t, gamma, beta, 1e-5, torch.bfloat16, center), pw, bias)
    y = _normed(t, gamma, beta, 1e-5, center)
    want = y @ w.double().T + bias
    # independent roundings to bfloat16: the operand's and the result's, and a folded weight's
    assert (got.double() - want).norm() <= 2.5 * 2.0 ** -9 * want.norm()


@pytest.mark.parametrize("m,k", [(4, 256), (8, 2048), (12, 1024)])
def test_rows_and_vectors_that_no_norm_takes(m, k):
    """Refused as the norm's own kernel refuses them, before a product is handed their addresses."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    dt = torch.bfloat16
    hip = HipOps(dt, DEV)
    x, weight = torch.randn(m, k, device=DEV), torch.ones(k, device=DEV)
    w = hip.prepare_weight(torch.randn(64, k, device=DEV).to(dt))
    assert hip.defer_norm(w, weight, None)
    wide = torch.randn(m, 2 * k, device=DEV)
    for rows, vector, error in ((wide[:, :k], weight, ValueError), (x[:1].expand(m, k), weight, ValueError),
                                (torch.randn(k, m, device=DEV).t(), weight, ValueError), (x.to(dt), weight, TypeError),
                                (x, weight[:k // 2], ValueError), (x, weight.to(dt), TypeError)):
        for make in (lambda: hip.layernorm_deferred(rows, vector, None, 1e-5, dt), lambda: hip.norm_between(rows, vector, None, 1e-5, dt)[1]):
            with pytest.raises(error):
                hip.linear(make(), w)


@pytest.mark.parametrize("m,k,n,beside", [(8, 3072, 12288, True), (1, 3072, 12304, False), (4, 2048, 40960, True), (5, 2048, 16384, True),
                                          (5, 2048, 16400, False), (8, 1024, 40960, True)])
def test_very_many_columns_read_the_norms_kernel(m, k, n, beside):
    """The line at 256 units, for norms before a matrix and behind a sum; the results are of one norm either way."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    hip, g, dt = HipOps(torch.bfloat16, DEV), _gen(m + k + n), torch.bfloat16
    hip.compute_units = 256
    t, gamma = torch.randn(m, k, device=DEV, generator=g) * 3 + 1, 1 + 0.1 * torch.randn(k, device=DEV, generator=g)
    w = hip.prepare_weight((torch.randn(n, k, device=DEV, generator=g) * 0.05).to(dt))
    assert hip.defer_norm(w, gamma, None)
    want = _normed(t, gamma, None, 1e-5, True) @ w.tensor.double().T
    way, made = [], hip._linear_beside_norm
    hip._linear_beside_norm = lambda *a: way.append(a) or made(*a)
    d = hip.layernorm_deferred(t, gamma, None, 1e-5, dt)
    # (independent roundings to bfloat16: the operand's and the result's)
    assert (hip.linear(d, w).double() - want).norm() <= 2.0 * 2.0 ** -9 * want.norm() and bool(way) == beside
    if k <= hip.norm_between_width:
        d = hip.norm_between(t, gamma, None, 1e-5, dt)[0]
        assert (hip.linear(d, w, out_f32=True).double() - want).norm() <= 2.0 ** -9 * 1.5 * want.norm() and (d.done is None) == beside
