"""Which dense products go through the streaming kernel for few rows, on the CPU."""
import pytest
import torch

from inferx_amd.engine.runtime import Runtime


@pytest.mark.parametrize("dtype,rows,features,reduction,off,streamed", [
    (torch.float32, 1, 8, 8, 0, True), (torch.float32, 32, 8, 8, 0, True), (torch.float32, 33, 8, 8, 0, False),
    (torch.float32, 4, 8, 6, 0, False), (torch.float32, 4, 8, 8, 1, False), (torch.float32, 4, 8, 8, 4, True),
    (torch.float32, 4, 0, 8, 0, False), (torch.float32, 4, 8, 0, 0, False), (torch.float32, 0, 8, 8, 0, False),
    (torch.bfloat16, 9, 8, 8, 0, True), (torch.bfloat16, 32, 8, 16, 0, True), (torch.bfloat16, 33, 8, 16, 0, False),
    (torch.bfloat16, 4, 8, 12, 0, False)])
def test_products_of_few_rows(dtype, rows, features, reduction, off, streamed):
    rt = Runtime.__new__(Runtime)  # (a whole one needs the HIP library)
    x = torch.zeros(off + rows * reduction, dtype=dtype)[off:].view(rows, reduction)
    w = torch.zeros(features, reduction, dtype=dtype)
    assert rt._skinny_ok(x, w) == streamed
    assert not rt._skinny_ok(x, w.to(torch.float64))


@pytest.mark.parametrize("dtype,rows,features,reduction,pairs", [
    (torch.bfloat16, 1, 8, 8, True), (torch.bfloat16, 16, 8, 8, True), (torch.bfloat16, 17, 8, 8, False), (torch.bfloat16, 4, 8, 12, False),
    (torch.float32, 4, 8, 8, False), (torch.bfloat16, 1, (1 << 24) - 1, 8, True), (torch.bfloat16, 1, 1 << 24, 8, False)])
def test_products_that_may_share_a_launch(dtype, rows, features, reduction, pairs):
    """Sizes that the launch of two refuses go through launches of their own."""
    rt = Runtime.__new__(Runtime)
    x, w = torch.empty(rows, reduction, dtype=dtype, device="meta"), torch.empty(features, reduction, dtype=dtype, device="meta")
    assert rt.pairs_ok(x, w) == pairs


@pytest.mark.parametrize("dtype,heads,dim,rot,vdim,rank,gate,uk,uv", [
    (torch.bfloat16, 4, 64, 32, 48, 96, False, True, True), (torch.float32, 4, 64, 32, 48, 96, False, False, False),
    (torch.bfloat16, 4, 48, 32, 48, 96, False, False, True),   # a reduction of 48
    (torch.bfloat16, 4, 64, 32, 40, 96, False, True, False),   # values of 40
    (torch.bfloat16, 4, 64, 32, 48, 80, False, True, False),   # a rank of 80: rows of weights, but no reduction
    (torch.bfloat16, 4, 64, 36, 48, 96, False, False, True),   # heads of 100 numbers
    (torch.bfloat16, 5, 64, 32, 4, 96, True, False, False),    # rows of 20 numbers more: q does not lie on 16 bytes
    (torch.bfloat16, 4, 64, 0, 48, 70, False, True, True)])    # brought to 96
def test_latent_attention_keeps_weights_twice_only_where_few_tokens_use_them(dtype, heads, dim, rot, vdim, rank, gate, uk, uv):
    from inferx_amd.parts.latent_attention import LatentAttention
    rt = Runtime.__new__(Runtime)
    rt.dtype = dtype
    part = LatentAttention(64, heads, dim, rot, vdim, rank, gate=gate)
    part.bind({p.name: torch.randn(p.shape).to(dtype) for p in part.param_specs()}, rt)
    assert ((part.w_uk_rows is not None), (part.w_uv_rows is not None)) == (uk, uv)
    if uk:
        assert torch.equal(part.w_uk_rows.transpose(1, 2), part.w_uk)
    if uv:
        assert torch.equal(part.w_uv_rows.transpose(1, 2), part.w_uv_t)


@pytest.mark.parametrize("pieces,width,tokens,along", [
    (4, 1408, 33, True), (4, 1408, 1535, True), (4, 1408, 1536, False), (0, 1408, 33, False),
    (32, 40000, 1535, True), (32, 48000, 767, True), (32, 48000, 1355, True), (32, 48000, 1356, False)])  # 2^31 numbers
def test_shared_expert_rides_along_as_far_as_the_products_reach(pieces, width, tokens, along):
    from inferx_amd.parts.moe import MoeFeedForward
    part = MoeFeedForward(64, 4, 1, width, pieces * width)
    assert part._shared_rides_along(tokens) == along


@pytest.mark.parametrize("hidden,pieces,tokens,whole", [
    (2048, 4, 1535, False), (2048, 4, 1536, True), (2048, 8, 2112, True), (2048, 4, 2113, False), (2048, 9, 1536, False),
    (2048, 0, 1536, False), (2040, 4, 1536, False)])
def test_shared_expert_whole_in_the_launches(hidden, pieces, tokens, whole):
    from inferx_amd.parts.moe import MoeFeedForward
    part = MoeFeedForward(hidden, 4, 1, 1408, pieces * 1408)
    assert part._shared_in_the_launches(tokens) == whole and not (whole and part._shared_rides_along(tokens))


@pytest.mark.parametrize("hidden,shared,tokens,wide", [
    (2048, 5632, 33, True), (2048, 5632, 2112, True), (2048, 5632, 2113, False), (2048, 0, 9000, True), (2048, 1000, 33, False),
    (2040, 5632, 33, False), (2040, 0, 33, False), (3072, 5632, 2113, True), (3072, 1000, 33, True)])
def test_wide_expert_products(hidden, shared, tokens, wide):
    """From a width of 3,072 on always, from 2,048 on where the shared expert is not a product of its own."""
    from inferx_amd.parts.moe import MoeFeedForward
    part = MoeFeedForward(hidden, 4, 1, 1408, shared)
    assert part._wide(tokens) == wide


@pytest.mark.parametrize("experts,top,width,shared,tokens,wide", [
    (60, 4, 1408, 5632, 64, True), (60, 4, 1408, 5632, 255, True), (60, 4, 1408, 0, 479, False),
    (60, 4, 1408, 0, 480, True), (60, 4, 1408, 5632, 2112, True), (8, 6, 768, 0, 203, False), (8, 2, 1408, 1408, 1500, False),
    (8, 2, 2816, 0, 9000, True), (128, 8, 768, 0, 60, False)])
def test_wide_expert_products_take_many_workgroups_and_rows(experts, top, width, shared, tokens, wide):
    """At a width of 2,048 the narrow form stays where the wide one would leave compute units without work, or waits for weights."""
    from types import SimpleNamespace
    from inferx_amd import ops
    from inferx_amd.parts.moe import MoeFeedForward
    part = MoeFeedForward(2048, experts, top, width, shared)
    part.w13 = part.w2 = torch.empty(0, dtype=torch.bfloat16)
    x = torch.empty(tokens, 2048, dtype=torch.bfloat16)
    assert part._wide(tokens) and part._tile_rows(SimpleNamespace(rt=SimpleNamespace(SKINNY_ROWS=32)), x) == ops.moe_tiled_rows(wide)


def test_products_that_tiles_do_not_take_are_allocated_once(monkeypatch):
    from inferx_amd import ops
    rt = Runtime.__new__(Runtime)
    made = []
    monkeypatch.setattr(rt, "empty", lambda shape, dtype=None: made.append(shape) or torch.empty(shape, dtype=dtype or torch.bfloat16), raising=False)
    monkeypatch.setattr(ops, "gemm_bf16", lambda x, w, out: True)
    monkeypatch.setattr(ops, "linear_tiled", lambda x, w, out, tile=-1: tile >= 0)
    for rows, tiled in ((2048, False), (40, True)):
        x, w = torch.zeros(rows, 2048, dtype=torch.bfloat16), torch.zeros(6144, 2048, dtype=torch.bfloat16)
        assert (ops.linear_tiled_tile(rows, 6144, 2048) >= 0) == tiled
        for product in (rt.linear, rt.linear_f32):
            made.clear()
            product(x, w)
            assert made == [(rows, 6144)]


@pytest.mark.parametrize("rows,features,width,tile", [
    # a long reduction in up to 128 tiles of 32 x 32, in more, up to 5,120; the same of 32 x 64
    (40, 512, 20480, -1), (66, 192, 8704, -1), (64, 2048, 5128, -1), (66, 192, 5120, 0), (64, 2080, 5128, 0), (64, 3584, 18944, 0),
    (64, 8192, 20480, 1),
    # results of no whole fours a row from 64 x 96 on; longer reductions in 64 x 128 for few units; what was left to the library before
    (240, 3510, 480, 2), (240, 5118, 480, -1), (240, 5120, 480, 3), (780, 6355, 480, -1), (500, 3840, 4104, 4), (640, 2400, 4096, 4), (640, 2400, 4104, -1),
    (500, 3838, 4096, -1), (3000, 700, 64, -1), (3000, 700, 256, 5), (850, 3584, 3584, -1), (2048, 6144, 2048, -1),
    # up to 64 rows that do not fit otherwise
    (33, 151936, 2048, 8), (46, 43637, 2056, 8), (64, 151936, 20480, 8), (65, 151936, 2048, -1),
    # sizes that the kernel does not take
    (40, 512, 100, -1), (0, 512, 64, -1), (1 << 20, 64, 4096, -1), (40, 1 << 31, 64, -1)])
def test_tiles_of_dense_products(rows, features, width, tile):
    from inferx_amd import ops
    assert ops.linear_tiled_tile(rows, features, width) == tile


@pytest.mark.parametrize("units,longest,span,head_dim,slices,loads", [
    (16, 517, 0, 128, 16, 1), (16, 65, 0, 128, 1, 1), (4, 128, 0, 128, 1, 1), (4, 129, 0, 128, 4, 1),   # one request
    (4, 64, 0, 128, 1, 2), (32, 40, 0, 128, 1, 2), (33, 40, 0, 128, 1, 1), (2048, 64, 0, 128, 1, 2), (2048, 65, 0, 128, 1, 1),
    (128, 2048, 0, 128, 16, 1), (1024, 2048, 0, 128, 4, 1), (1024, 2048, 0, 64, 4, 1), (128, 4096, 1024, 128, 8, 1),
    (2048, 1000, 0, 64, 1, 1), (2048, 1025, 0, 64, 2, 1), (2048, 4096, 1024, 64, 1, 1), (2048, 4096, 1024, 128, 2, 1), (2048, 1000, 0, 128, 2, 1), (4096, 16000, 0, 128, 4, 1)])
def test_slices_and_loads_of_decoding(units, longest, span, head_dim, slices, loads):
    """Up to 128 keys stay whole; whole contexts that are two wavefronts a SIMD already are cut by their bytes; half lines for
    few or very many wavefronts on up to 64 keys.  As a captured step rounds its longest context."""
    from inferx_amd.parts.attention import decode_loads, decode_slices
    rounded = 1 << (longest - 1).bit_length()
    for n in (longest, rounded):
        assert (decode_slices(units, n, span, head_dim), decode_loads(units, n)) == (slices, loads)
