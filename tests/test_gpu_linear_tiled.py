"""Dense products in tiles for a few dozen to some hundred rows against float64, and which products they take."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = [(32, 32), (32, 64), (64, 64), (64, 96), (64, 128), (96, 128), (128, 128), (128, 192), (128, 64)]  # weight x activation rows


def operands(T, N, K, off=0):
    g = torch.Generator().manual_seed(T * 7 + N + K)
    def make(n, k, scale):
        t = torch.full((n * k + off + 64,), float("nan"), dtype=torch.bfloat16, device=DEV)  # (what lies around reaches no result)
        t[off:off + n * k] = (torch.randn(n * k, generator=g) * scale).to(torch.bfloat16).to(DEV)
        return t[off:off + n * k].view(n, k)
    return make(T, K, 1.0), make(N, K, K ** -0.5)


@pytest.mark.parametrize("tile", range(9))
@pytest.mark.parametrize("f32", [False, True])
def test_every_tile(tile, f32):
    """Rows and features one less, as many and one more than a tile's, several tiles; one to a ring's depth and more stages, the
    last one whole or not; results that are no whole pieces."""
    from inferx_amd import ops
    W, X = TILES[tile]
    for T, N, K in ((1, 1, 8), (X - 1, W + 1, 64), (X, W, 72), (X + 1, 2 * W - 8, 200), (3 * X - 5, 3 * W + 8, 512), (X, 9 * W, 640),
                    (2 * X, W + 4, 704), (33, 40, 1096)):
        x, w = operands(T, N, K)
        buf = torch.full((T * N + 32,), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device=DEV)
        for off in (0, 4, 1):
            out = buf[off:off + T * N].view(T, N)
            assert ops.linear_tiled(x, w, out, tile)
            want = x.double() @ w.double().T
            # float32 sums of K products, and one rounding of a bfloat16 result
            bound = K * 2.0 ** -24 * float((x.double().abs() @ w.double().abs().T).max()) + (0 if f32 else 2.0 ** -8 * float(want.abs().max()))
            assert float((out.double() - want).abs().max()) <= bound, (T, N, K, off)
            assert (buf[:off] == 7).all() and (buf[off + T * N:] == 7).all()
            buf.fill_(7.0)


@pytest.mark.parametrize("T,N,K,taken", [
    (33, 2048, 2048, True), (17, 6144, 2048, True), (850, 6144, 2048, True), (1400, 2048, 5632, False), (2048, 6144, 2048, False),
    (64, 32768, 256, True), (65, 70000, 64, False), (850, 3584, 3584, False), (40, 100, 8, True),
    (3000, 700, 64, False), (3000, 700, 256, True)])
def test_which_products_are_taken(T, N, K, taken):
    from inferx_amd import ops
    x, w = operands(T, N, K)
    out = torch.full((T, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert ops.linear_tiled(x, w, out) == taken
    if taken:
        want = x.float() @ w.float().T
        assert float((out.float() - want).norm() / want.norm()) < 4e-3  # one rounding to bfloat16
    else:
        assert torch.isnan(out).all()


def test_the_runtime_falls_back_where_tiles_do_not_go():
    """Operands off 16-byte boundaries, odd reductions and strided rows go through the products before, no features through none here."""
    from inferx_amd.engine.runtime import Runtime
    rt = Runtime("bfloat16")
    x, w = operands(40, 264, 136)
    xo, wo = operands(40, 264, 136, off=1)
    xo.copy_(x), wo.copy_(w)
    want = x.float() @ w.float().T
    close = lambda got: float((got.float() - want).norm() / want.norm()) < 4e-3
    assert rt._tiled(x, w, torch.bfloat16) is not None and close(rt.linear(x, w)) and close(rt.linear_f32(x, w))
    for a, b in ((xo, w), (x, wo)):
        assert rt._tiled(a, b, torch.bfloat16) is None and close(rt.linear(a, b)) and close(rt.linear_f32(a, b))
    wide = torch.zeros(40, 272, dtype=torch.bfloat16, device=DEV)
    wide[:, :136] = x
    assert rt._tiled(wide[:, :136], w, torch.bfloat16) is None and close(rt.linear(wide[:, :136], w))
    x7, w7 = x[:, :133].contiguous(), w[:, :133].contiguous()
    assert rt._tiled(x7, w7, torch.bfloat16) is None and rt.linear(x7, w7).shape == (40, 264)
    assert rt._tiled(x, w[:0].contiguous(), torch.bfloat16) is None
