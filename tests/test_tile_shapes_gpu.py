"""Products by tiles of 64 x 128 and 96 x 128, and the rule that chooses among the tiles."""
import pytest
import torch

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(33, 72, 64), (96, 128, 320), (97, 136, 512), (192, 96, 2048), (193, 264, 2112), (700, 520, 8192)])
@pytest.mark.parametrize("tile", [3, 4])
@pytest.mark.parametrize("shares", [1, 3])
def test_product_by_tiles(m, n, k, tile, shares):
    """At sizes that end on a tile's edge, one past it, and inside."""
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


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(34, 3072, 1024), (100, 5120, 4096), (150, 2560, 2560), (200, 8192, 2048), (257, 4096, 4096), (333, 2048, 8192),
                                   (450, 7680, 2560), (704, 1024, 4096)])
def test_products_that_the_rule_takes(m, n, k):
    """`linear` with the tile and the shares of the rule against the other way, up to the rounding of the result."""
    from transformers_neuronx_amd.kernels.hip import HipOps
    ops, other = HipOps(torch.bfloat16, DEV), HipOps(torch.bfloat16, DEV)
    other.tile_products = False
    g = torch.Generator(device=DEV).manual_seed(n)
    x, w = torch.randn(m, k, device=DEV, generator=g).bfloat16(), (torch.randn(n, k, device=DEV, generator=g) * k ** -0.5).bfloat16()
    bias, res = torch.randn(n, device=DEV, generator=g), torch.randn(m, n, device=DEV, generator=g)
    assert ops._tiles_room(m, n, k, x, w, None, False, False) >= 0
    for kw in (dict(bias=bias, act="relu"), dict(bias=bias, act="gelu"), dict(residual=res, out_f32=True), dict()):
        torch.testing.assert_close(ops.linear(x, w, **kw).float(), other.linear(x, w, **kw).float(), rtol=1e-2, atol=2e-2)


def test_the_rule_asks_for_what_it_uses():
    """The workspace is the shares' sums, and sizes beyond the tiles' reach are refused. A share has as many steps of K as come to each,
    rounded up, eight at least; the last one has what is left, one at least (64 steps in seven shares: six of ten and one of four)."""
    from transformers_neuronx_amd.kernels.hip import library
    room = library("gemm").tnx_gemm_bf16_tiles_workspace
    for m in (33, 64, 65, 96, 100, 128, 129, 200, 333, 512, 576, 640, 705, 768):
        for n in (8, 64, 1000, 1024, 2048, 3072, 6144, 10240, 50272):
            for k in (64, 128, 1024, 2048, 2560, 4096, 8192, 16384):
                r = room(m, n, k)
                assert r == -1 or r % (m * n) == 0
                if r > 0:
                    shares, steps = r // (m * n), k // 64
                    each = -(-steps // shares)
                    assert 2 <= shares <= 8 and each >= 8 and 1 <= steps - (shares - 1) * each <= each
    for m, n, k in ((32, 1024, 1024), (769, 1024, 1024), (100, 1001, 1024), (100, 1024, 1000), (0, 64, 64)):
        assert room(m, n, k) == -1


@pytest.mark.parametrize("m", [49, 52, 56, 64])
def test_few_rows_of_a_matrix_that_widens_are_one_launch(m):
    """No norm stands behind such a product to add its shares, and a prompt of so few rows waits for the host's launches."""
    from transformers_neuronx_amd.kernels.hip import library
    room = library("gemm").tnx_gemm_bf16_tiles_workspace
    assert room(m, 6144, 2048) == 0 and room(m, 8192, 2048) == 0
    assert room(m, 2048, 8192) > 0 and room(m, 2048, 2048) > 0
