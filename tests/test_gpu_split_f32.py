"""Float32 products on the bfloat16 matrix cores (every number as the sum of three): against 64 bits, infinities and NaN against
float32's own, and the rule that chooses them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(DEV)


def bound(x, w):
    """The six products of parts leave 2^-22 of each product out; its sums are rounded once for sixteen numbers, and the small ones'
    five times, 2^-7 of it; the two accumulators (and groups) are added in the end."""
    K = x.shape[1]
    return (2.0 ** -22 + (K / 16 + 4) * 2.0 ** -23) * (x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("rows,n,k", [(1, 1, 64), (33, 37, 64), (64, 64, 128), (65, 130, 192), (128, 192, 256), (129, 193, 320),
                                      (200, 260, 512), (300, 100, 2048)])
def test_linear_split(rows, n, k, tile):
    """Tiles that are whole and not, one to thirty-two stages and more, reductions that start at a stage of their own and not."""
    from inferx_amd import ops
    x, w = rnd(rows, k), rnd(n, k, seed=1, scale=0.02)
    x[0] *= 1e-20  # (parts far below one)
    buf = torch.full((rows * n + 16,), 7.0, device=DEV)
    out = buf[8:-8].view(rows, n)
    ops.linear_split(x, w, out, tile)
    assert (buf[:8] == 7).all() and (buf[-8:] == 7).all()
    assert ((out.double() - x.double() @ w.double().T).abs() <= bound(x, w)).all()
    again = torch.empty_like(out)
    ops.linear_split(x, w, again, tile, ops.split_rows(x))
    assert torch.equal(out, again)


def test_split_rows_are_the_numbers():
    from inferx_amd import ops
    x = rnd(5, 96)
    x[0, :4] = torch.tensor([1.0, -3.4028234e38, 1.1754944e-38, 0.0])
    parts = ops.split_rows(x).float()
    assert torch.equal(parts.sum(2).view(5, 96), x)  # (any order of three such numbers gives the sum exactly)
    assert (parts[:, :, 1].abs() <= 2 ** -7 * parts[:, :, 0].abs()).all() and (parts[:, :, 2].abs() <= 2 ** -15 * parts[:, :, 0].abs()).all()


@pytest.mark.parametrize("tile", [0, 1, 2])
def test_linear_split_of_infinities(tile):
    from inferx_amd import ops
    x, w = rnd(70, 128), rnd(100, 128, seed=1)
    x[3, 5], x[4, 7], x[6, 1], x[7, :2] = float("inf"), float("nan"), 3.4e38, torch.tensor([float("inf"), float("-inf")], device=DEV)
    w[9, 11], w[12, 0], w[13] = float("-inf"), float("nan"), 2.0 ** -130
    out = torch.empty(70, 100, device=DEV)
    ops.linear_split(x, w, out, tile)
    want = x @ w.t()
    assert torch.equal(torch.isnan(out), torch.isnan(want)) and torch.equal(out[torch.isinf(want)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(out), ok)
    exact = x.double() @ w.double().T
    assert ((out.double() - exact).abs()[ok] <= bound(x, w)[ok] + 2.0 ** -133).all()  # (below 2^-126 parts may be lost)


def test_the_rule_and_the_runtime():
    from inferx_amd import ops
    from inferx_amd.engine.runtime import Runtime
    assert ops.linear_split_tile(511, 11264, 2048) >= 0 and ops.linear_split_tile(64, 2048, 2048) < 0
    assert ops.linear_split_tile(511, 11264, 2080) < 0 and ops.linear_split_tile(0, 11264, 2048) < 0
    rt = Runtime("float32", DEV)
    for rows, n, k in ((511, 4096, 2048), (700, 3000, 1088), (511, 4096, 2040), (40, 300, 128)):
        x, w = rnd(rows, k), rnd(n, k, seed=1, scale=0.02)
        for got in (rt.linear(x, w), rt.linear_f32(x, w)):
            assert got.dtype == torch.float32
            assert ((got.double() - x.double() @ w.double().T).abs() <= bound(x, w) * 4).all()  # (the library rounds once for four)
    place = torch.empty(511, 4096, device=DEV)
    assert rt.linear_f32(rnd(511, 2048), rnd(4096, 2048, seed=1), place) is place
