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


def grouped(counts, seed=1):
    """offsets, rows, tile map of experts with so many rows, the rows in any order."""
    from inferx_amd import ops
    E, A, R = len(counts), sum(counts), ops.MOE_TILED_F32_ROWS
    g = torch.Generator().manual_seed(seed)
    topk_e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(A, generator=g)].to(torch.int32)[:, None].to(DEV)
    offsets, rows, dest = (torch.empty(n, dtype=torch.int32, device=DEV) for n in (E + 1, A, A))
    tile_map = torch.empty(2 * ops.moe_max_tiles(A, E, R) + 1, dtype=torch.int32, device=DEV)
    ops.moe_dispatch(topk_e, offsets, rows, dest, E, R, tile_map)
    return offsets, rows, tile_map


@pytest.mark.parametrize("epilogue", [0, 1, 2])
@pytest.mark.parametrize("K,n", [(32, 7), (64, 64), (96, 130), (128, 200), (256, 72), (512, 1028), (2048, 96)])
def test_grouped_split(K, n, epilogue):
    """Tiles of one and two blocks of rows, whole and not, experts of none, one and several tiles; one to sixty-four stages."""
    from inferx_amd import ops
    counts = [1, 32, 33, 64, 65, 0, 130, 5]
    offsets, rows, tile_map = grouped(counts)
    A = sum(counts)
    x, w = rnd(A, K), rnd(len(counts), (2 if epilogue == 1 else 1) * n, K, seed=1, scale=K ** -0.5)
    buf = torch.full((A * n + 16,), 7.0, device=DEV)
    out = buf[8:-8].view(A, n)
    ops.moe_grouped_split(x, ops.split_rows(x), w, out, offsets, rows, tile_map, epilogue)
    assert (buf[:8] == 7).all() and (buf[-8:] == 7).all()
    for e, (lo, hi) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        xe = x[rows[lo:hi].long()]
        z, err = xe.double() @ w[e].double().T, bound(xe, w[e])
        if epilogue == 1:  # silu has slopes up to 1.1
            want = torch.nn.functional.silu(z[:, :n]) * z[:, n:]
            err = 1.1 * err[:, :n] * z[:, n:].abs() + z[:, :n].abs() * err[:, n:] + 1.1 * err[:, :n] * err[:, n:]
        else:
            want = z.clamp(min=0) ** 2 if epilogue == 2 else z
            err = 2 * z.abs() * err + err ** 2 if epilogue == 2 else err
        assert ((out[lo:hi].double() - want).abs() <= err + 8 * 2.0 ** -24 * want.abs() + 1e-37).all()
    again = torch.empty_like(out)
    ops.moe_grouped_split(x, ops.split_rows(x), w, again, offsets, rows, tile_map, epilogue)
    assert torch.equal(out, again)
    gathered = x[rows.long()].contiguous()
    ops.moe_grouped_split(gathered, ops.split_rows(gathered), w, again, offsets, None, tile_map, epilogue)
    assert torch.equal(out, again)


@pytest.mark.parametrize("gate_up", [False, True])
def test_grouped_split_of_infinities(gate_up):
    from inferx_amd import ops
    counts = [3, 40]
    offsets, rows, tile_map = grouped(counts)
    x, w = rnd(43, 64), rnd(2, 24, 64, seed=1)
    x[3, 5], x[4, 7], x[6, 1] = float("inf"), float("nan"), 3.4e38
    w[1, 9, 11], w[0, 12, 0] = float("-inf"), float("nan")
    out = torch.empty(43, 12 if gate_up else 24, device=DEV)
    ops.moe_grouped_split(x, ops.split_rows(x), w, out, offsets, rows, tile_map, gate_up)
    for e, (lo, hi) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        z = x[rows[lo:hi].long()] @ w[e].t()
        want = z[:, :12] / (1 + torch.exp(-z[:, :12])) * z[:, 12:] if gate_up else z
        assert torch.equal(torch.isnan(out[lo:hi]), torch.isnan(want))
        assert torch.equal(out[lo:hi][torch.isinf(want)], want[torch.isinf(want)])
        ok = torch.isfinite(want)
        assert torch.allclose(out[lo:hi][ok], want[ok], rtol=1e-4, atol=1e-4)
