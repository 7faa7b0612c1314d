"""The mixture-of-experts kernels alone against PyTorch references: router, grouping,
grouped products (plain and matrix-core), combine.  Properties follow the reference's
tests/kernel/moe_test.cc (lines cited per test)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(*shape, seed=0, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def rel_err(got, want):
    want = want.double().cpu()
    return float((got.double().cpu() - want).abs().max()) / max(float(want.abs().max()), 1e-30)


def route_reference(x, wr, k, renorm, scale=1.0):
    p = torch.softmax(x.double().cpu() @ wr.double().cpu().T, -1)
    w, e = torch.topk(p, k, dim=-1)
    if renorm:
        w = w / w.sum(-1, keepdim=True)
    return w * scale, e


@pytest.mark.parametrize("T,H,E,k,renorm", [(24, 64, 8, 2, False), (7, 200, 60, 4, True), (130, 72, 5, 1, False),
                                            (3, 2048, 64, 8, True), (50, 96, 32, 32, True),
                                            (300, 136, 60, 4, True), (203, 40, 70, 6, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_route(T, H, E, k, renorm, dtype):
    # reference: moe_test.cc:170-246 (router equals host to 1e-5, renormalised sums to 1, un-normalised below)
    from inferx_amd import ops
    x, wr, wsg = rnd(T, H, dtype=dtype), rnd(E, H, seed=1, dtype=dtype, scale=0.3), rnd(1, H, seed=2, dtype=dtype, scale=0.1)
    topk_w = torch.empty(T, k, dtype=torch.float32, device=DEV)
    topk_e = torch.empty(T, k, dtype=torch.int32, device=DEV)
    gate = torch.empty(T, dtype=torch.float32, device=DEV)
    ops.moe_route(x, wr, wsg, topk_w, topk_e, gate, renorm, 1.0)
    want_w, want_e = route_reference(x, wr, k, renorm)
    assert torch.equal(topk_e.cpu().long(), want_e)
    assert rel_err(topk_w, want_w) < 1e-5
    assert rel_err(gate, torch.sigmoid(x.double().cpu() @ wsg.double().cpu().T)[:, 0]) < 1e-5
    sums = topk_w.sum(-1).cpu()
    if renorm:
        assert torch.allclose(sums, torch.ones(T), atol=1e-5)
    elif k < E:
        assert (sums < 0.9999).all()


@pytest.mark.parametrize("T,E", [(129, 32), (129, 33), (2048, 32), (2049, 32), (2049, 4), (300, 4)])
def test_route_of_few_experts_and_many(T, E):
    """float32 tokens on both sides of the lines between one kernel per token and the scores as a product with 64-bit sums."""
    from inferx_amd import ops
    H, k = 60, 3
    x, wr = rnd(T, H), rnd(E, H, seed=1, scale=0.3)
    topk_w, topk_e = torch.empty(T, k, device=DEV), torch.empty(T, k, dtype=torch.int32, device=DEV)
    ops.moe_route(x, wr, None, topk_w, topk_e, None, True, 1.0)
    want_w, want_e = route_reference(x, wr, k, True)
    margin = torch.topk(x.double().cpu() @ wr.double().cpu().T, k + 1, dim=-1).values
    sure = (margin[:, :-1] - margin[:, 1:]).min(-1).values > 1e-5  # (float32 sums of 60 numbers: 1e-6 of scores up to 10)
    assert int(sure.sum()) > 0.99 * T and torch.equal(topk_e.cpu().long()[sure], want_e[sure])
    assert rel_err(topk_w[sure.to(DEV)], want_w[sure]) < 1e-5


def test_route_refuses_what_it_cannot_do():
    from inferx_amd import ops
    x, wr = rnd(4, 96), rnd(40, 96, seed=1)
    with pytest.raises(ops.KernelError, match="top_k"):
        ops.moe_route(x, wr, None, torch.empty(4, 33, device=DEV), torch.empty(4, 33, dtype=torch.int32, device=DEV),
                      None, False, 1.0)


def test_route_equal_logits_take_the_lowest_indices():
    # reference vector: moe_test.cc:248-273
    from inferx_amd import ops
    T, H, E, k = 5, 16, 32, 2
    x = torch.ones(T, H, device=DEV)
    wr = torch.full((E, H), 0.25 / H, device=DEV)
    topk_w = torch.empty(T, k, device=DEV)
    topk_e = torch.empty(T, k, dtype=torch.int32, device=DEV)
    ops.moe_route(x, wr, None, topk_w, topk_e, None, False, 1.0)
    assert topk_e.cpu().tolist() == [[0, 1]] * T
    assert torch.allclose(topk_w.cpu(), torch.full((T, k), 1 / 32))


def dispatch(topk_e, E, tile_rows=0):
    from inferx_amd import ops
    T, k = topk_e.shape
    A = T * k
    offsets = torch.empty(E + 1, dtype=torch.int32, device=DEV)
    rows = torch.empty(A, dtype=torch.int32, device=DEV)
    dest = torch.empty(A, dtype=torch.int32, device=DEV)
    tile_map = None
    if tile_rows:
        tile_map = torch.full((2 * ops.moe_max_tiles(A, E, tile_rows) + 1,), -7, dtype=torch.int32, device=DEV)
    ops.moe_dispatch(topk_e, offsets, rows, dest, E, tile_rows, tile_map)
    return offsets, rows, dest, tile_map


@pytest.mark.parametrize("T,E,k,tile_rows", [(24, 8, 2, 16), (300, 60, 4, 32), (1, 4, 2, 16), (1000, 7, 3, 64),
                                             (40, 64, 1, 0), (2048, 60, 4, 160), (3000, 60, 4, 160), (500, 200, 3, 32),
                                             (600, 1024, 2, 16), (4100, 3, 2, 0)])
def test_dispatch_is_a_stable_bijection(T, E, k, tile_rows):
    # reference: moe_test.cc:277-350
    g = torch.Generator().manual_seed(T)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32)
    if E > 3:
        topk_e[topk_e == 2] = 3  # expert 2 stays empty (an assignment may then repeat expert 3; fine for grouping)
    offsets, rows, dest, tile_map = dispatch(topk_e.to(DEV), E, tile_rows)
    offsets, rows, dest = offsets.cpu(), rows.cpu(), dest.cpu()
    flat = topk_e.flatten()
    A = T * k
    assert offsets[0] == 0 and offsets[E] == A
    assert sorted(dest.tolist()) == list(range(A))  # every assignment exactly once
    for a in range(A):
        e = int(flat[a])
        assert offsets[e] <= dest[a] < offsets[e + 1]      # in its expert's range
        assert rows[dest[a]] == a // k                      # rows and dest are inverse
    if E > 3:
        assert offsets[2] == offsets[3]                     # an empty expert has an empty range
    for e in range(E):
        mine = [int(dest[a]) for a in range(A) if int(flat[a]) == e]
        assert mine == sorted(mine)                         # stable: assignment order is kept
    if tile_rows:
        mt = (tile_map.numel() - 1) // 2
        n = int(tile_map[2 * mt])
        te, tr = tile_map[:n].cpu().tolist(), tile_map[mt:mt + n].cpu().tolist()
        covered = []
        for e_, r0 in zip(te, tr):
            assert offsets[e_] <= r0 < offsets[e_ + 1]
            covered += list(range(r0, min(r0 + tile_rows, int(offsets[e_ + 1]))))
        assert covered == list(range(A))  # tiles cover every row once, in order


@pytest.mark.parametrize("A", [1, 1024, 1025, 4095, 4096, 4097, 8192, 8193, 20000])
@pytest.mark.parametrize("E", [1, 5, 600])
def test_dispatch_of_few_and_many_assignments(A, E):
    """Around the sizes at which the kernel's sweeps end and change their form."""
    topk_e = torch.randint(0, E, (A, 1), generator=torch.Generator().manual_seed(A)).to(torch.int32)
    offsets, rows, dest, _ = dispatch(topk_e.to(DEV), E)
    order = torch.sort(topk_e.flatten(), stable=True).indices
    counts = torch.bincount(topk_e.flatten(), minlength=E)
    assert torch.equal(offsets.cpu(), torch.cat([torch.zeros(1), counts.cumsum(0)]).to(torch.int32))
    assert torch.equal(rows.cpu().long(), order) and torch.equal(dest.cpu().long()[order], torch.arange(A))


@pytest.mark.parametrize("T,H,E,k,renorm,tile_rows", [(1, 64, 4, 2, False, 16), (8, 2048, 60, 4, False, 16),
                                                       (11, 96, 8, 3, True, 32), (16, 72, 5, 1, False, 0),
                                                       (16, 200, 256, 32, True, 16), (16, 136, 60, 4, True, 16),
                                                       (5, 88, 7, 3, False, 0), (13, 200, 256, 8, True, 16),
                                                       # at most 64 assignments: experts with more rows than a tile; 256 experts
                                                       (16, 64, 3, 2, False, 4), (4, 200, 256, 8, True, 16), (7, 80, 130, 9, False, 2),
                                                       # one token, also with 64 and 65 router rows and a wide row
                                                       (1, 2048, 60, 4, False, 16), (1, 200, 63, 8, True, 16), (1, 96, 64, 3, False, 16),
                                                       (1, 4104, 17, 5, True, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_route_and_dispatch_for_few_tokens(T, H, E, k, renorm, tile_rows, dtype):
    """Scores, selection and grouping in one launch (up to 16 tokens) give exactly what the separate kernels give."""
    from inferx_amd import ops
    x, wr, wsg = rnd(T, H, dtype=dtype), rnd(E, H, seed=1, dtype=dtype, scale=0.3), rnd(1, H, seed=2, dtype=dtype, scale=0.1)
    A = T * k
    mk = lambda *shape, dt=torch.int32: torch.full(shape, -9, dtype=dt, device=DEV)
    w1, e1, g1 = mk(T, k, dt=torch.float32), mk(T, k), mk(T, dt=torch.float32)
    ops.moe_route(x, wr, wsg, w1, e1, g1, renorm, 1.0)
    o1, r1, d1, tm1 = dispatch(e1, E, tile_rows)
    w2, e2, g2 = mk(T, k, dt=torch.float32), mk(T, k), mk(T, dt=torch.float32)
    o2, r2, d2 = mk(E + 1), mk(A), mk(A)
    tm2 = mk(2 * ops.moe_max_tiles(A, E, tile_rows) + 1) if tile_rows else None
    ops.moe_route_dispatch(x, wr, wsg, w2, e2, g2, renorm, 1.0, o2, r2, d2, tile_rows, tm2)
    assert torch.equal(e1, e2) and torch.equal(o1, o2) and torch.equal(r1, r2) and torch.equal(d1, d2)
    assert rel_err(w2, w1) < 1e-6 and rel_err(g2, g1) < 1e-6
    if tile_rows:
        mt = (tm1.numel() - 1) // 2
        n = int(tm1[2 * mt])
        assert int(tm2[2 * mt]) == n and torch.equal(tm1[:n], tm2[:n]) and torch.equal(tm1[mt:mt + n], tm2[mt:mt + n])


def test_route_in_one_launch_again_and_again():
    """The one-launch router counts its workgroups off on a counter that every launch leaves at zero, and its
    last workgroup reads what workgroups on other dies wrote: many launches of changing sizes one after the
    other, without waiting, all agree with the separate kernels."""
    from inferx_amd import ops
    mk = lambda *shape, dt=torch.int32: torch.full(shape, -9, dtype=dt, device=DEV)
    cases, got = [(3, 2048, 60, 4), (16, 136, 60, 4), (1, 64, 4, 2), (9, 200, 256, 8), (8, 2048, 60, 4)] * 40, []
    for i, (T, H, E, k) in enumerate(cases):
        x, wr, wsg = (rnd(T, H, seed=i, dtype=torch.bfloat16), rnd(E, H, seed=100 + i, dtype=torch.bfloat16, scale=0.3),
                      rnd(1, H, seed=200 + i, dtype=torch.bfloat16, scale=0.1))
        w2, e2, g2 = mk(T, k, dt=torch.float32), mk(T, k), mk(T, dt=torch.float32)
        o2, r2, d2 = mk(E + 1), mk(T * k), mk(T * k)
        ops.moe_route_dispatch(x, wr, wsg, w2, e2, g2, True, 1.0, o2, r2, d2, 0, None)
        got.append((x, wr, wsg, w2, e2, g2, o2, r2, d2))
    for (T, H, E, k), (x, wr, wsg, w2, e2, g2, o2, r2, d2) in zip(cases, got):
        w1, e1, g1 = mk(T, k, dt=torch.float32), mk(T, k), mk(T, dt=torch.float32)
        ops.moe_route(x, wr, wsg, w1, e1, g1, True, 1.0)
        o1, r1, d1, _ = dispatch(e1, E, 0)
        assert torch.equal(e1, e2) and torch.equal(o1, o2) and torch.equal(r1, r2) and torch.equal(d1, d2)
        assert rel_err(w2, w1) < 1e-6 and rel_err(g2, g1) < 1e-6


def grouped_reference(a, w, offsets, rows, gate_up):
    a, w = a.double().cpu(), w.double().cpu()
    E = w.shape[0]
    A = int(offsets[E])
    n = w.shape[1] // 2 if gate_up else w.shape[1]
    out = torch.zeros(A, n, dtype=torch.float64)
    for e in range(E):
        for r in range(int(offsets[e]), int(offsets[e + 1])):
            x = a[int(rows[r])] if rows is not None else a[r]
            z = w[e] @ x
            out[r] = torch.nn.functional.silu(z[:n]) * z[n:] if gate_up else z
    return out


GROUPED = [(24, 64, 8, 2, 32), (300, 96, 8, 3, 48), (9, 72, 5, 1, 40), (700, 256, 60, 4, 176), (3, 2048, 60, 4, 1408),
           (20, 1160, 5, 2, 200)]


@pytest.mark.parametrize("T,H,E,k,mi", GROUPED)
@pytest.mark.parametrize("dtype,wdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                          (torch.bfloat16, torch.float32)])
def test_grouped_plain(T, H, E, k, mi, dtype, wdtype):
    from inferx_amd import ops
    if T * mi * H > 300 * 96 * 48 * 40:
        pytest.skip("large for the plain kernel's test")
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, rows, dest, _ = dispatch(topk_e, E)
    x = rnd(T, H, dtype=dtype)
    w13, w2 = rnd(E, 2 * mi, H, seed=2, dtype=wdtype, scale=H ** -0.5), rnd(E, H, mi, seed=3, dtype=wdtype, scale=mi ** -0.5)
    act = torch.empty(T * k, mi, dtype=dtype, device=DEV)
    ops.moe_grouped_plain(x, w13, act, offsets, rows, True)
    tol = 1e-5 if dtype == torch.float32 else 1.5e-2
    assert rel_err(act, grouped_reference(x, w13, offsets.cpu(), rows.cpu(), True)) < tol
    y = torch.empty(T * k, H, dtype=dtype, device=DEV)
    ops.moe_grouped_plain(act, w2, y, offsets, None, False)
    assert rel_err(y, grouped_reference(act, w2, offsets.cpu(), None, False)) < tol


@pytest.mark.parametrize("T,H,E,k,mi", GROUPED)
@pytest.mark.parametrize("tile_rows", [16, 32, 64])
@pytest.mark.parametrize("k_split", [1, 4])
def test_grouped_mfma(T, H, E, k, mi, tile_rows, k_split):
    from inferx_amd import ops
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, E, tile_rows)
    x = rnd(T, H, dtype=torch.bfloat16)
    w13 = rnd(E, 2 * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    w2 = rnd(E, H, mi, seed=3, dtype=torch.bfloat16, scale=mi ** -0.5)
    act = torch.full((T * k, mi), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_mfma(x, w13, act, offsets, rows, tile_map, tile_rows, True, k_split)
    assert rel_err(act, grouped_reference(x, w13, offsets.cpu(), rows.cpu(), True)) < 1.5e-2
    y = torch.full((T * k, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_mfma(act, w2, y, offsets, None, tile_map, tile_rows, False, k_split)
    assert rel_err(y, grouped_reference(act, w2, offsets.cpu(), None, False)) < 1.5e-2
    # bitwise repeatable (reference: moe_test.cc:972-1046)
    y2 = torch.empty_like(y)
    ops.moe_grouped_mfma(act, w2, y2, offsets, None, tile_map, tile_rows, False, k_split)
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("T,H,E,k,mi", GROUPED + [(900, 136, 6, 2, 88), (2048, 512, 12, 4, 352)])
def test_grouped_tiled(T, H, E, k, mi, wide):
    """Experts with a handful of rows, with about one tile of them, and with several tiles (the last one partial);
    128 and 256 weight rows per workgroup, which give the same bits."""
    from inferx_amd import ops
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, E, ops.moe_tiled_rows(wide))  # tiles of 160 rows, wide 192
    x = rnd(T, H, dtype=torch.bfloat16)
    w13 = rnd(E, 2 * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    w2 = rnd(E, H, mi, seed=3, dtype=torch.bfloat16, scale=mi ** -0.5)
    act = torch.full((T * k, mi), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_tiled(x, w13, act, offsets, rows, tile_map, True, wide)
    y = torch.full((T * k, H), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_tiled(act, w2, y, offsets, None, tile_map, False, wide)
    if wide:
        _, _, _, narrow_map = dispatch(topk_e, E, ops.moe_tiled_rows(False))
        act_n, y_n = torch.empty_like(act), torch.empty_like(y)
        ops.moe_grouped_tiled(x, w13, act_n, offsets, rows, narrow_map, True, False)
        ops.moe_grouped_tiled(act, w2, y_n, offsets, None, narrow_map, False, False)
        if H % 512 and mi % 512:
            # the same sums in the same order (rows of a multiple of 1,024 bytes start the reduction at a stage
            # that depends on the tile, and the two forms cut tiles differently)
            assert torch.equal(act.view(torch.int16), act_n.view(torch.int16))
            assert torch.equal(y.view(torch.int16), y_n.view(torch.int16))
        else:
            assert rel_err(act, act_n) < 1e-2 and rel_err(y, y_n) < 1e-2
    if T <= 900:
        assert rel_err(act, grouped_reference(x, w13, offsets.cpu(), rows.cpu(), True)) < 1.5e-2
        assert rel_err(y, grouped_reference(act, w2, offsets.cpu(), None, False)) < 1.5e-2
    else:  # large: against the wavefront-level kernel, which the small cases pin to the reference
        act2, y2 = torch.empty_like(act), torch.empty_like(y)
        _, _, _, map64 = dispatch(topk_e, E, 64)
        ops.moe_grouped_mfma(x, w13, act2, offsets, rows, map64, 64, True, 1)
        ops.moe_grouped_mfma(act, w2, y2, offsets, None, map64, 64, False, 1)
        assert rel_err(act, act2) < 1e-2 and rel_err(y, y2) < 1e-2


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("mi", [8, 72, 76, 264])
def test_grouped_tiled_rows_read_once_and_results_at_any_place(mi, wide):
    """Experts of 64 and 65 rows (the most whose weights go past the caches, and one more), of one row, none, a whole tile and
    one more; results on and off 16-byte boundaries, rows of them whole 16-byte pieces or not: the same bits."""
    from inferx_amd import ops
    R, H = ops.moe_tiled_rows(wide), 136
    counts = [64, 65, 1, 0, R, R + 1]
    topk_e = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, len(counts), R)
    T = sum(counts)
    x = rnd(T, H, dtype=torch.bfloat16)
    w = rnd(len(counts), 2 * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    got = []
    for off in (0, 4):  # (the buffer's numbers before and behind the result must stay)
        buf = torch.full((T * mi + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.moe_grouped_tiled(x, w, buf[off:off + T * mi].view(T, mi), offsets, rows, tile_map, True, wide)
        assert (buf[:off] == 7).all() and (buf[off + T * mi:] == 7).all()
        got.append(buf[off:off + T * mi].view(T, mi).clone())
    assert torch.equal(got[0].view(torch.int16), got[1].view(torch.int16))
    assert rel_err(got[0], grouped_reference(x, w, offsets.cpu(), rows.cpu(), True)) < 1.5e-2


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("H", [8, 64, 72, 128, 200, 256, 320, 328, 512])
def test_grouped_tiled_rings_of_every_depth(H, wide):
    """One to eight stages of the reduction, the last one whole or not, through the rings of every tile height (one to six
    pairs of sixteens of rows); operands off 16-byte boundaries, which go through registers, give the same bits."""
    from inferx_amd import ops
    R, mi = ops.moe_tiled_rows(wide), 136
    counts = [n for n in (1, 33, 70, 128, 129, 161, R) if n <= R] + [R + 40]
    topk_e = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, len(counts), R)
    T = sum(counts)
    x = rnd(T, H, dtype=torch.bfloat16)
    w = rnd(len(counts), mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)

    def off_by(t, n):
        buf = torch.empty(t.numel() + n, dtype=t.dtype, device=DEV)
        buf[n:] = t.reshape(-1)
        return buf[n:].view(t.shape)

    out = []
    for a, b in ((x, w), (off_by(x, 1), w), (x, off_by(w, 4))):
        out.append(torch.full((T, mi), float("nan"), dtype=torch.bfloat16, device=DEV))
        ops.moe_grouped_tiled(a, b, out[-1], offsets, rows, tile_map, False, wide)
    want = torch.cat([x[rows.long()][lo:hi].double() @ w[e].double().T
                      for e, (lo, hi) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:]))])
    # one rounding of the result and float32 sums of H products
    assert float((out[0].double() - want).abs().max()) <= 2 ** -8 * float(want.abs().max()) + 1e-5
    assert all(torch.equal(out[0].view(torch.int16), o.view(torch.int16)) for o in out[1:])


@pytest.mark.parametrize("gate_up", [False, True])
@pytest.mark.parametrize("H", [8, 64, 72, 128, 192, 256, 264, 320, 384, 448, 512, 584, 1024])
def test_grouped_tiled_of_few_and_many_workgroups(H, gate_up):
    """The narrow form with all of a compute unit's LDS, and with half where (further, empty) experts make many workgroups: float64's
    results, and the same bits.  Tiles of all heights, one to sixteen stages through rings of two to six buffers."""
    from inferx_amd import ops
    R, mi = ops.moe_tiled_rows(False), 136
    counts = [1, 33, 70, 128, 129, R, R + 40]
    E, T = len(counts), sum(counts)
    topk_e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    x = rnd(T, H, dtype=torch.bfloat16)
    few = rnd(E, (2 if gate_up else 1) * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    many = torch.cat([few, torch.full((300 - E,) + few.shape[1:], float("nan"), dtype=torch.bfloat16, device=DEV)])
    out = []
    for w in (few, many):
        assert (ops.moe_tiled_tiles(T, w.shape[0], at_most=True) * ops.moe_tiled_columns(mi, gate_up) <= ops.MOE_TILED_ALONE) == (w is few)
        offsets, rows, dest, tile_map = dispatch(topk_e, w.shape[0], R)
        out.append(torch.full((T, mi), float("nan"), dtype=torch.bfloat16, device=DEV))
        ops.moe_grouped_tiled(x, w, out[-1], offsets, rows, tile_map, gate_up)
    z = torch.cat([x[rows.long()][lo:hi].double() @ few[e].double().T
                   for e, (lo, hi) in enumerate(zip(offsets.tolist()[:E], offsets.tolist()[1:E + 1]))])
    want = torch.nn.functional.silu(z[:, :mi]) * z[:, mi:] if gate_up else z
    # one rounding of the result and float32 sums of H products
    assert float((out[0].double() - want).abs().max()) <= 2 ** -8 * float(want.abs().max()) + 1e-5
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("last", [1, 3, 7, 8, 1000])
def test_grouped_tiled_order_of_the_last_tiles(last, wide):
    """Working the last tiles of the map spread among the others changes no bit, whatever their number."""
    from inferx_amd import ops
    T, H, E, k, mi = 400, 136, 6, 2, 88
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, E, ops.moe_tiled_rows(wide))
    x, w = rnd(T, H, dtype=torch.bfloat16), rnd(E, 2 * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    out = [torch.full((T * k, mi), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    for o, n in zip(out, (0, last)):
        ops.moe_grouped_tiled(x, w, o, offsets, rows, tile_map, True, wide, last_tiles=n)
    assert torch.isfinite(out[0]).all() and torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("T,E,mi", [(30, 12, 160), (330, 5, 520), (500, 9, 72)])
@pytest.mark.parametrize("pieces", [1, 2, 4])
def test_grouped_tiled_last_tiles_of_one_expert_together(T, E, mi, pieces, wide):
    """The last experts hold every row (one to four tiles each); their tiles, worked expert by expert and spread over the
    dies, with more and with fewer tiles than the others have, change no bit.  Reductions of 1 to 9 stages of 64, whole
    and not."""
    from inferx_amd import ops
    g = torch.Generator().manual_seed(1)
    top = torch.stack([torch.randperm(E, generator=g)[:1] for _ in range(T)])
    always = torch.arange(E, E + pieces).expand(T, pieces)
    topk_e = torch.cat([top, always], 1).to(torch.int32).to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, E + pieces, ops.moe_tiled_rows(wide))
    each = -(-T // ops.moe_tiled_rows(wide))
    for H in (64, 200, 256, 320, 512, 576):
        x = rnd(T, H, dtype=torch.bfloat16)
        w = rnd(E + pieces, mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
        out = [torch.full((topk_e.numel(), mi), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        ops.moe_grouped_tiled(x, w, out[0], offsets, rows, tile_map, False, wide)
        ops.moe_grouped_tiled(x, w, out[1], offsets, rows, tile_map, False, wide, last_tiles=pieces * each, last_each=each)
        assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
        for t in (0, T // 2, T - 1):
            for c in range(1 + pieces):
                want = x[t].double().cpu() @ w[int(topk_e[t, c])].double().cpu().T
                got = out[0][int(dest[t * (1 + pieces) + c])].double().cpu()
                assert float((got - want).abs().max()) <= 2 ** -8 * float(want.abs().max()) + 1e-5, (H, t, c)


@pytest.mark.parametrize("gate_up", [False, True])
@pytest.mark.parametrize("rows,n,k", [(1, 8, 8), (192, 128, 200), (193, 264, 576), (400, 1000, 1160), (600, 44, 64)])
def test_grouped_tiled_with_a_second_product(rows, n, k, gate_up):
    """A dense product in the launch of a grouped one, with longer, equal and shorter reductions, one and more row tiles, fewer and
    more of them than the grouped product has: its results, and the grouped product's bits as without it."""
    from inferx_amd import ops
    T, E, top, mi = 300, 6, 2, 136
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, order, dest, tile_map = dispatch(topk_e, E, ops.MOE_TILED_ROWS_WIDE)
    a2 = rnd(rows, k, seed=3, dtype=torch.bfloat16)
    w2 = rnd((2 if gate_up else 1) * n, k, seed=4, dtype=torch.bfloat16, scale=k ** -0.5)
    for H in (72, 200, 576):
        x = rnd(T, H, dtype=torch.bfloat16)
        w = rnd(E, (2 if gate_up else 1) * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
        out = [torch.full((T * top, mi), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        buf = torch.full((rows * n + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.moe_grouped_tiled(x, w, out[0], offsets, order, tile_map, gate_up, True)
        ops.moe_grouped_tiled(x, w, out[1], offsets, order, tile_map, gate_up, True, second=(a2, w2, buf[8:-8].view(rows, n)))
        assert torch.isfinite(out[0]).all() and torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
        assert (buf[:8] == 7).all() and (buf[-8:] == 7).all()
        want = a2.double() @ w2.double().T
        if gate_up:
            want = torch.nn.functional.silu(want[:, :n]) * want[:, n:]
        assert float((buf[8:-8].view(rows, n).double() - want).abs().max()) <= 2 ** -8 * float(want.abs().max()) + 1e-5
    with pytest.raises(ops.KernelError):  # (last tiles beside it)
        ops.moe_grouped_tiled(x, w, out[1], offsets, order, tile_map, gate_up, True, last_tiles=1, second=(a2, w2, buf[8:-8].view(rows, n)))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("last", [0, 1, 2, 3, 4, 6])
def test_grouped_tiled_experts_of_several_tiles_beside_the_last_ones(last, wide):
    """Experts of six, one, five and three tiles, which go together up to four at a time; the last ones of the map, worked
    spread among the others, are some or all of the last expert's, or of the one before it, too: every row is formed."""
    from inferx_amd import ops
    R, H, mi = ops.moe_tiled_rows(wide), 72, 1100
    counts = [5 * R + 3, 2, 5 * R, 2 * R + 1]
    topk_e = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    offsets, rows, dest, tile_map = dispatch(topk_e, len(counts), R)
    x, w = rnd(sum(counts), H, dtype=torch.bfloat16), rnd(len(counts), mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    out = torch.full((sum(counts), mi), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_tiled(x, w, out, offsets, rows, tile_map, False, wide, last_tiles=last)
    assert rel_err(out, grouped_reference(x, w, offsets.cpu(), rows.cpu(), False)) < 1e-2


def with_queue(topk_e, E):
    """`dispatch` for the wide form's tiles, most rows first, with a queue."""
    from inferx_amd import ops
    A, R = topk_e.numel(), ops.MOE_TILED_ROWS_WIDE
    offsets, rows, dest = (torch.empty(n, dtype=torch.int32, device=DEV) for n in (E + 1, A, A))
    tile_map = torch.full((2 * ops.moe_max_tiles(A, E, R) + 1,), -7, dtype=torch.int32, device=DEV)
    mt = ops.moe_max_tiles(A, E, R)
    queues = torch.full((ops.moe_queues_size(mt),), -7, dtype=torch.int32, device=DEV)
    ops.moe_dispatch(topk_e, offsets, rows, dest, E, R, tile_map, queues)
    counts = (offsets[1:] - offsets[:-1]).tolist()
    tiles = [(e, i) for e in sorted(range(E), key=lambda e: (-counts[e], e)) for i in range(-(-counts[e] // R))]
    start = [int(offsets[e]) + R * i for e, i in tiles]
    assert int(tile_map[2 * mt]) == len(tiles)
    assert list(zip(tile_map[:len(tiles)].tolist(), tile_map[mt:mt + len(tiles)].tolist())) == [(e, r) for (e, _), r in zip(tiles, start)]
    heavy = sum(-(-n // R) for n in counts if n > 128)
    want = ([0] * 8 + [heavy]) * 2
    for (e, i), r in zip(tiles, start):
        of = -(-counts[e] // R)
        want += [r, min(R, counts[e] - R * i) | e << 8 | i % 4 << 19 | min(4, of - i // 4 * 4) - 1 << 21 | (of == 1) << 23]
    assert queues.tolist() == want + [-7] * (queues.numel() - len(want))
    return offsets, rows, tile_map, queues


@pytest.mark.parametrize("epilogue", [False, True, 2])
@pytest.mark.parametrize("H,mi,few", [(256, 1544, False), (320, 1544, False), (512, 1536, False), (1024, 520, False), (640, 264, True),
                                      (192, 1544, False), (264, 1544, False), (256, 1540, False)])
def test_grouped_tiled_by_workgroups_that_stay(H, mi, few, epilogue):
    """The bits of a workgroup for each tile: tiles of all heights one after the other on a place (and no more tiles than places),
    four and more stages, column blocks that are whole and not; the shapes that do not go there leave the queue alone."""
    from inferx_amd import ops
    counts = [1, 33, 70, 97, 129, 161, 192, 193, 400, 0, 16, 64] * (1 if few else 3)
    E, T = len(counts), sum(counts)
    g = torch.Generator().manual_seed(1)
    topk_e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)].to(torch.int32)[:, None].to(DEV)
    offsets, rows, tile_map, queues = with_queue(topk_e, E)
    x = rnd(T, H, dtype=torch.bfloat16)
    w = rnd(E, (2 if epilogue == 1 else 1) * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    want = torch.full((T, mi), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_tiled(x, w, want, offsets, rows, tile_map, epilogue, True)
    assert torch.isfinite(want).all()
    buf = torch.full((T * mi + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.moe_grouped_tiled(x, w, buf[8:-8].view(T, mi), offsets, rows, tile_map, epilogue, True, queues=queues, nth=1)
    assert torch.equal(buf[8:-8].view(T, mi).view(torch.int16), want.view(torch.int16))
    assert (buf[:8] == 7).all() and (buf[-8:] == 7).all()
    assert (int(queues[9:17].sum()) > 0) == (H % 64 == 0 and H >= 256 and mi % 8 == 0)


@pytest.mark.parametrize("gate_up", [False, True])
@pytest.mark.parametrize("rows,n,k", [(1, 8, 256), (193, 264, 576), (700, 2000, 2048), (600, 2000, 320), (400, 1000, 192)])
def test_grouped_tiled_with_a_second_product_by_workgroups_that_stay(rows, n, k, gate_up):
    """A second product of shorter, equal and longer reductions among the tiles: the bits of both as by a workgroup for each."""
    from inferx_amd import ops
    T, E, top, mi, H = 900, 20, 3, 1160, 576
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, order, tile_map, queues = with_queue(topk_e, E)
    x, a2 = rnd(T, H, dtype=torch.bfloat16), rnd(rows, k, seed=3, dtype=torch.bfloat16)
    w = rnd(E, (2 if gate_up else 1) * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    w2 = rnd((2 if gate_up else 1) * n, k, seed=4, dtype=torch.bfloat16, scale=k ** -0.5)
    out = [torch.full((T * top, mi), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    out2 = [torch.full((rows, n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    for i in (0, 1):
        ops.moe_grouped_tiled(x, w, out[i], offsets, order, tile_map, gate_up, True, second=(a2, w2, out2[i]), queues=queues if i else None)
    assert (int(queues[:8].sum()) > 0) == (k >= 256)
    for a, b in (out, out2):
        assert torch.isfinite(a).all() and torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("kind", ["unit", "few rows", "few rows of experts", "tiles", "wide tiles", "staying"])
def test_gates_at_the_ends_of_their_range(kind):
    """The gated unit where the exponential's sum is largest, past the largest and not a number: what the division of 32-bit numbers
    gives, up to the exponential's own error and one rounding to bfloat16."""
    from inferx_amd import ops
    bf, H, T = torch.bfloat16, 256, 64
    gates = [float("-inf"), float("nan"), float("inf"), -3e38, -1e30, -100.0, -88.5, -88.0, -87.5, -87.0, -30.0, -0.0, 1e-3, 90.0, 3e38]
    g = torch.tensor(gates).repeat_interleave(3).to(bf)
    u = torch.tensor([1.0, -1e30, 0.5]).repeat(len(gates)).to(bf)
    n = -(-len(g) // 8) * 8
    g, u = (torch.cat([t, t.new_ones(n - len(t))]) for t in (g, u))
    w = torch.zeros(2 * n, H, dtype=bf)
    w[:, 0] = torch.cat([g, u])
    x = torch.zeros(T, H, dtype=bf, device=DEV)
    x[:, 0] = 1
    w = w.to(DEV)
    if kind == "unit":
        out = torch.empty(T, n, dtype=bf, device=DEV)
        ops.silu_mul(torch.cat([g, u]).to(DEV)[None].repeat(T, 1), out)
    elif kind == "few rows":
        out = torch.empty(8, n, dtype=bf, device=DEV)
        ops.linear_skinny(x[:8], w, out, True)
    else:
        topk_e = torch.zeros(T, 1, dtype=torch.int32, device=DEV)
        out = torch.empty(T, n, dtype=bf, device=DEV)
        if kind in ("wide tiles", "staying"):
            offsets, rows, tile_map, queues = with_queue(topk_e, 1)
            ops.moe_grouped_tiled(x, w[None], out, offsets, rows, tile_map, True, True, queues=queues if kind == "staying" else None)
        else:
            R = 16 if kind == "few rows of experts" else ops.MOE_TILED_ROWS
            offsets, rows, dest = (torch.empty(m, dtype=torch.int32, device=DEV) for m in (2, T, T))
            tile_map = torch.empty(2 * ops.moe_max_tiles(T, 1, R) + 1, dtype=torch.int32, device=DEV)
            ops.moe_dispatch(topk_e, offsets, rows, dest, 1, R, tile_map)
            if R == 16:
                ops.moe_grouped_mfma(x, w[None], out, offsets, rows, tile_map, R, True, 4)
            else:
                ops.moe_grouped_tiled(x, w[None], out, offsets, rows, tile_map, True, False)
    want = (g.float() / (1 + torch.exp(-g.float())) * u.float()).to(bf).float().expand(out.shape)
    got = out.cpu().float()
    ends = ~torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[ends].nan_to_num(), want[ends].nan_to_num())
    assert ((got - want).abs()[~ends] <= 2.0 ** -7 * want.abs()[~ends]).all()


@pytest.mark.parametrize("counts", [[193, 400, 70, 1, 64, 0, 130] * 3, [5, 200]])  # more pairs than places, and fewer
def test_workgroups_that_stay_can_be_launched_again(counts):
    """A launch leaves its counters at their start: the same product again, and another of another number of pairs, by the same queue."""
    from inferx_amd import ops
    E, T, H, mi = len(counts), sum(counts), 256, 1544
    topk_e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    offsets, rows, tile_map, queues = with_queue(topk_e, E)
    x = rnd(T, H, dtype=torch.bfloat16)
    for epilogue, n in ((True, mi), (True, mi), (False, 520), (False, 520)):
        w = rnd(E, (2 if epilogue else 1) * n, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
        got, want = (torch.full((T, n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ops.moe_grouped_tiled(x, w, want, offsets, rows, tile_map, epilogue, True)
        ops.moe_grouped_tiled(x, w, got, offsets, rows, tile_map, epilogue, True, queues=queues)
        assert torch.isfinite(want).all() and torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 8, 17, 64])
# at most 256 blocks of sixteen, and more; at most 128 (both halves of an even reduction in one block for up to eight rows)
@pytest.mark.parametrize("N,K", [(33, 8), (4096, 1160), (4100, 264), (2048, 1040), (37, 16), (43, 2064), (5637, 72)])
@pytest.mark.parametrize("form", [None, 0.0, 1.5, -1.0])  # a plain product; gate|up rows by the unit's limit
@pytest.mark.parametrize("biased", [False, True])
def test_dense_products_of_few_rows(dtype, T, N, K, form, biased):
    """x . w^T in one launch with the gated unit and the biases behind it, against float64.  The bound is the result's own
    rounding (half of a bfloat16's last place, at most 2^-8 of the number) and that of K float32 sums on both of a unit's sides."""
    from inferx_amd import ops
    rows = N if form is None else 2 * N
    x, w = rnd(T, K, dtype=dtype), rnd(rows, K, seed=1, dtype=dtype, scale=K ** -0.5)
    bias = rnd(rows, seed=2, dtype=dtype) if biased else None
    out = torch.full((T, N), float("nan"), dtype=dtype, device=DEV)
    ops.linear_skinny(x, w, out, form is not None, form or 0.0, bias)
    want = x.double() @ w.double().T + (bias.double() if biased else 0.0)
    if form is not None:
        g, u = want[:, :N], want[:, N:]
        if form > 0:
            g, u = g.clamp(max=form), u.clamp(-form, form) + 1.0
            want = g * torch.sigmoid(1.702 * g) * u
        elif form < 0:
            want = torch.nn.functional.gelu(g, approximate="tanh") * u
        else:
            want = torch.nn.functional.silu(g) * u
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22
    err = (out.double() - want).abs()
    assert float((err - eps * want.abs()).max()) <= 4e-5, float(err.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N", [4096, 4097, 6137, 6144, 6145])  # 256 blocks of sixteen, 257 and 384 (eights), 385
@pytest.mark.parametrize("T", [1, 8, 9])
def test_gated_products_in_sixteens_and_eights(dtype, T, N):
    """On both sides of the line the features' sums have one order: a column that both have, alone on its side of it."""
    from inferx_amd import ops
    K = 264
    x, w = rnd(T, K, dtype=dtype), rnd(2 * N, K, seed=1, dtype=dtype, scale=K ** -0.5)
    out, other = (torch.full((T, n), float("nan"), dtype=dtype, device=DEV) for n in (N, 7168))
    ops.linear_skinny(x, w, out, True)
    gate, up = (torch.cat([part, part.new_zeros(7168 - N, K)]) for part in (w[:N], w[N:]))
    ops.linear_skinny(x, torch.cat([gate, up]), other, True)
    want = torch.nn.functional.silu(x.double() @ w[:N].double().T) * (x.double() @ w[N:].double().T)
    assert rel_err(out, want) < (1e-2 if dtype == torch.bfloat16 else 1e-5)
    if N > 4096:  # (up to 256 blocks eight wavefronts share the reduction, from there on four)
        assert torch.equal(out, other[:, :N])


@pytest.mark.parametrize("which", ["bfloat16", "float32", "q/k/v"])
def test_streaming_products_of_very_long_rows(which):
    """Weight rows so long that the sixteenth starts 2^32 bytes behind the first: every row's own first and last number
    meet the activations' (all others are zero, the sums are small whole numbers)."""
    from inferx_amd import ops
    dtype = torch.float32 if which == "float32" else torch.bfloat16
    K = (1 << 32) // 15 // (4 if which == "float32" else 2) // 16 * 16 + 16
    T, N = (9 if which == "bfloat16" else 1), (96 if which == "q/k/v" else 16)
    x, w = torch.zeros(T, K, dtype=dtype, device=DEV), torch.zeros(N, K, dtype=dtype, device=DEV)
    row = torch.arange(N, device=DEV)
    x[:, 0], x[:, -1] = 64, 1
    w[:, 0], w[:, -1] = 1, (row + 1).to(dtype)
    if which == "q/k/v":
        q = torch.full((1, 1, 32), float("nan"), dtype=dtype, device=DEV)
        kc, vc = torch.zeros(1, 1, 16, 32, dtype=dtype, device=DEV), torch.zeros(1, 1, 32, 16, dtype=dtype, device=DEV)
        ops.qkv_rope_skinny(x, w, None, None, torch.zeros(1, dtype=torch.int32, device=DEV), q, kc, vc, 1, 1, 32)
        out = torch.cat([q[0, 0], kc[0, 0, 0], vc[0, 0, :, 0]])[None]
    else:
        out = torch.full((T, N), float("nan"), dtype=dtype, device=DEV)
        ops.linear_skinny(x, w, out)
    want = (65 + row).float().expand(T, N)
    del x, w
    torch.cuda.empty_cache()
    assert torch.equal(out.float(), want), (out.float() - want).nonzero()[:4].tolist()


@pytest.mark.parametrize("T,N,K", [(3, 40, 264), (16, 33, 1160), (2, 16, 8), (5, 48, 520)])
def test_streaming_kernels_read_nothing_past_their_operands(T, N, K):
    """Reduction widths that leave a wavefront a ragged last round: what lies behind the last row of the weights
    and of the activations (here NaN) must not reach a result, not even multiplied by zero."""
    from inferx_amd import ops
    xbuf = torch.full((T + 1, K), float("nan"), dtype=torch.bfloat16, device=DEV)
    wbuf = torch.full((2 * N + 1, K), float("nan"), dtype=torch.bfloat16, device=DEV)
    xbuf[:T] = rnd(T, K, dtype=torch.bfloat16)
    wbuf[:2 * N] = rnd(2 * N, K, seed=1, dtype=torch.bfloat16, scale=K ** -0.5)
    x, w = xbuf[:T], wbuf[:N]
    out = torch.full((T, N), float("nan"), device=DEV)
    ops.linear_skinny_f32(x, w, out)
    want = x.double().cpu() @ w.double().cpu().t()
    assert torch.isfinite(out).all() and rel_err(out, want) < 1e-5
    # the grouped product, one expert: gate|up over both halves of the weights, then a plain product
    offsets = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    tile_map = torch.tensor([0, 0, 0, 0, 1], dtype=torch.int32, device=DEV)  # one tile of expert 0 from row 0
    for k_split in (1, 4):
        act = torch.full((T, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.moe_grouped_mfma(x, wbuf[:2 * N].unsqueeze(0), act, offsets, None, tile_map, 16, True, k_split)
        z = x.double().cpu() @ wbuf[:2 * N].double().cpu().t()
        assert torch.isfinite(act).all()
        assert rel_err(act, torch.nn.functional.silu(z[:, :N]) * z[:, N:]) < 1.5e-2
        y = torch.full((T, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.moe_grouped_mfma(x, w.unsqueeze(0), y, offsets, None, tile_map, 16, False, k_split)
        assert torch.isfinite(y).all() and rel_err(y, want) < 1.5e-2


@pytest.mark.parametrize("T,N,K", [(1, 301, 72), (8, 151936, 2048), (16, 384, 96), (33, 1000, 64), (64, 256, 40)])
def test_linear_skinny_f32(T, N, K):
    from inferx_amd import ops
    x, w = rnd(T, K, dtype=torch.bfloat16), rnd(N, K, seed=1, dtype=torch.bfloat16, scale=K ** -0.5)
    out = torch.full((T, N), float("nan"), device=DEV)
    ops.linear_skinny_f32(x, w, out)
    assert rel_err(out, x.double().cpu() @ w.double().cpu().T) < 1e-5  # float32 accumulation of exact products


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gather_then_combine_is_the_identity(dtype):
    # reference: moe_test.cc:352-411 (weights 0.25 / 0.75)
    from inferx_amd import ops
    T, H, E, k = 24, 64, 8, 2
    g = torch.Generator().manual_seed(2)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    offsets, rows, dest, _ = dispatch(topk_e, E)
    x = rnd(T, H, dtype=dtype)
    y = x[rows.long()]  # what an identity expert would produce
    topk_w = torch.tensor([[0.25, 0.75]] * T, device=DEV)
    out = torch.empty_like(x)
    ops.moe_combine(y, dest, topk_w, None, None, out)
    assert rel_err(out, x) < (1e-6 if dtype == torch.float32 else 1e-2)
    shared, gate = rnd(T, H, seed=5, dtype=dtype), torch.rand(T, device=DEV)
    ops.moe_combine(y, dest, topk_w, shared, gate, out)
    assert rel_err(out, x.double() + gate.double()[:, None] * shared.double()) < (1e-6 if dtype == torch.float32 else 1e-2)
    ops.moe_combine(y, dest, topk_w, shared, None, out)  # an ungated shared expert adds exactly its output
    assert rel_err(out, x.double() + shared.double()) < (1e-6 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("T,H,E,k", [(1, 64, 4, 2), (8, 2048, 60, 4), (16, 136, 60, 4), (5, 88, 7, 3), (13, 200, 256, 8),
                                     (1, 2048, 60, 4), (1, 200, 63, 8), (1, 96, 64, 3), (1, 4104, 17, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_norm_route_and_dispatch_in_one_launch(T, H, E, k, dtype):
    """The norm before the feed-forward as part of the one-launch router: the residual stream is brought up to
    date exactly, the normalised rows are those of the separate norm kernel up to the rounding of one sum, and
    the routing is exactly that of the separate kernels on the rows it wrote."""
    from inferx_amd import ops
    mk = lambda *shape, dt=torch.int32: torch.full(shape, -9, dtype=dt, device=DEV)
    h0, delta = rnd(T, H, seed=3, dtype=torch.float32, scale=2.0), rnd(T, H, seed=4, dtype=dtype)
    gamma = (1.0 + rnd(H, seed=5, dtype=torch.float32, scale=0.2)).to(dtype)
    wr, wsg = rnd(E, H, seed=1, dtype=dtype, scale=0.3), rnd(1, H, seed=2, dtype=dtype, scale=0.1)
    eps = 1e-5
    h1, x1 = h0.clone(), torch.empty(T, H, dtype=dtype, device=DEV)
    ops.add_rmsnorm(h1, delta, gamma, x1, eps)
    for tile_rows in (0, 16):
        h2, x2 = h0.clone(), torch.full((T, H), 7.0, dtype=dtype, device=DEV)
        w2, e2, g2 = mk(T, k, dt=torch.float32), mk(T, k), mk(T, dt=torch.float32)
        o2, r2, d2 = mk(E + 1), mk(T * k), mk(T * k)
        tm2 = mk(2 * ops.moe_max_tiles(T * k, E, tile_rows) + 1) if tile_rows else None
        ops.moe_route_dispatch(None, wr, wsg, w2, e2, g2, True, 1.0, o2, r2, d2, tile_rows, tm2,
                               norm=(h2, delta, gamma, eps, x2))
        assert torch.equal(h2, h1)
        ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -21
        assert ((x2.float() - x1.float()).abs() <= ulp * x1.float().abs() + 1e-30).all()
        w1, e1, g1 = mk(T, k, dt=torch.float32), mk(T, k), mk(T, dt=torch.float32)
        ops.moe_route(x2, wr, wsg, w1, e1, g1, True, 1.0)
        o1, r1, d1, tm1 = dispatch(e1, E, tile_rows)
        assert torch.equal(e1, e2) and torch.equal(o1, o2) and torch.equal(r1, r2) and torch.equal(d1, d2)
        assert rel_err(w2, w1) < 1e-6 and rel_err(g2, g1) < 1e-6


@pytest.mark.parametrize("T,H,E,k,mi,S", [(1, 64, 4, 2, 32, 48), (8, 2048, 60, 4, 1408, 5632), (16, 136, 60, 4, 40, 24),
                                          (21, 96, 8, 3, 48, 80), (40, 72, 5, 1, 40, 200), (64, 264, 7, 2, 88, 1000)])
def test_routed_and_shared_experts_in_one_launch(T, H, E, k, mi, S):
    """The launch that holds the routed experts' product and the shared expert's: the routed part is bit for bit
    the routed launch's, the shared part is the product of all tokens with the shared weights; both products
    (gate|up with SwiGLU, down), every tile height that takes the token count."""
    from inferx_amd import ops
    g = torch.Generator().manual_seed(1)
    topk_e = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    x = rnd(T, H, dtype=torch.bfloat16)
    w13 = rnd(E, 2 * mi, H, seed=2, dtype=torch.bfloat16, scale=H ** -0.5)
    w2 = rnd(E, H, mi, seed=3, dtype=torch.bfloat16, scale=mi ** -0.5)
    ws13 = rnd(2 * S, H, seed=4, dtype=torch.bfloat16, scale=H ** -0.5)
    ws2 = rnd(H, S, seed=5, dtype=torch.bfloat16, scale=S ** -0.5)
    nan = lambda *shape: torch.full(shape, float("nan"), dtype=torch.bfloat16, device=DEV)
    for tile_rows in (16, 32, 64):
        offsets, rows, dest, tile_map = dispatch(topk_e, E, tile_rows)
        act1, act2, sact = nan(T * k, mi), nan(T * k, mi), nan(T, S)
        ops.moe_grouped_mfma(x, w13, act1, offsets, rows, tile_map, tile_rows, True, 4)
        ops.moe_grouped_dual(x, w13, act2, offsets, rows, tile_map, tile_rows, x, ws13, sact, True)
        assert torch.equal(act1.view(torch.int16), act2.view(torch.int16))
        want = torch.nn.functional.silu(x.double() @ ws13[:S].double().T) * (x.double() @ ws13[S:].double().T)
        assert rel_err(sact, want) < 1.5e-2
        y1, y2, sout = nan(T * k, H), nan(T * k, H), nan(T, H)
        ops.moe_grouped_mfma(act1, w2, y1, offsets, None, tile_map, tile_rows, False, 4)
        ops.moe_grouped_dual(act2, w2, y2, offsets, None, tile_map, tile_rows, sact, ws2, sout, False)
        assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
        assert rel_err(sout, sact.double() @ ws2.double().T) < 1.5e-2
        assert rel_err(y2, grouped_reference(act2, w2, offsets.cpu(), None, False)) < 1.5e-2


@pytest.mark.parametrize("T,H,k,A", [(1, 64, 2, 2), (8, 2048, 4, 32), (21, 96, 3, 70), (5, 1000, 1, 5), (130, 72, 8, 1040),
                                      (4, 2052, 9, 40), (3, 4100, 12, 40), (3, 8196, 2, 9)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("with_shared,gated", [(False, False), (True, False), (True, True)])
def test_expert_sum_add_and_norm_in_one_pass(T, H, k, A, dtype, with_shared, gated):
    """h += sum_s w[t, s] y[dest[t, s]] + gate[t] shared[t]; out = rmsnorm(h) * weight: against the two kernels one
    after the other (the sum rounded to the run's type in between, as they leave it) and against float64; with
    picked rows the stream is left alone."""
    from inferx_amd import ops
    g = torch.Generator().manual_seed(5)
    y = rnd(A, H, seed=1, dtype=dtype)
    dest = torch.stack([torch.randperm(A, generator=g)[:k] for _ in range(T)]).to(torch.int32).to(DEV)
    topk_w = torch.rand(T, k, generator=g).to(DEV)
    shared = rnd(T, H, seed=2, dtype=dtype) if with_shared else None
    gate = torch.rand(T, generator=g).to(DEV) if gated else None
    weight = (1.0 + rnd(H, seed=3, scale=0.2)).to(dtype)
    h0 = rnd(T, H, seed=4, scale=2.0)
    eps = 1e-5
    total = (topk_w.double()[:, :, None] * y.double()[dest.long()]).sum(1)
    if with_shared:
        total = total + (gate.double()[:, None] if gated else 1.0) * shared.double()
    h_want = h0.double() + total
    x_want = h_want * torch.rsqrt((h_want ** 2).mean(-1, keepdim=True) + eps) * weight.double()
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    h1, out1 = h0.clone(), torch.empty(T, H, dtype=dtype, device=DEV)
    ops.moe_combine_add_rmsnorm(h1, y, dest, topk_w, shared, gate, weight, out1, eps)
    assert rel_err(h1, h_want) < (1e-6 if dtype == torch.float32 else 4e-3) and rel_err(out1, x_want) < tol
    summed, h2, out2 = torch.empty(T, H, dtype=dtype, device=DEV), h0.clone(), torch.empty(T, H, dtype=dtype, device=DEV)
    ops.moe_combine(y, dest, topk_w, shared, gate, summed)
    ops.add_rmsnorm(h2, summed, weight, out2, eps)
    assert rel_err(h1, h2) < (1e-6 if dtype == torch.float32 else 4e-3) and rel_err(out1, out2) < tol
    rows = torch.tensor([T - 1, 0, T // 2, T // 2], dtype=torch.int32, device=DEV)
    h3, picked = h0.clone(), torch.empty(4, H, dtype=dtype, device=DEV)
    ops.moe_combine_add_rmsnorm(h3, y, dest, topk_w, shared, gate, weight, picked, eps, rows)
    assert torch.equal(h3, h0) and rel_err(picked, x_want[rows.long()]) < tol


# rows of the experts (around the sixteens of a tile and its 64 rows), reduction width (no multiple of a stage of 32; rows
# of a multiple of 1,024 bytes), columns (no multiple of a workgroup's, of four)
F32_PRODUCTS = [([1, 0, 16, 17], 36, 40), ([63, 64, 65], 100, 33), ([130, 5], 256, 64), ([31, 33, 48, 49], 2048, 100),
                ([2, 200], 4, 4)]


@pytest.mark.parametrize("counts,K,n", F32_PRODUCTS)
@pytest.mark.parametrize("kind", ["tiled", "streaming", "dual"])
@pytest.mark.parametrize("gate_up,limit", [(0, 0.0), (1, 0.0), (1, 7.0), (2, 0.0)])
def test_grouped_products_in_float32(counts, K, n, kind, gate_up, limit):
    """The matrix-core products in float32 against float64: every product and sum is 32-bit, so a result is off by at
    most K roundings of 2^-24 of the sum of magnitudes, here (normal numbers) under 1e-5 of the largest result.  What
    lies behind the operands (NaN) reaches no result."""
    from inferx_amd import ops
    E, A, T = len(counts), sum(counts), 50
    if kind == "dual" and gate_up == 2:
        pytest.skip("the shared expert is gated")
    wn = 2 * n if gate_up == 1 else n
    buf = lambda rows, seed: torch.cat([rnd(rows, K, seed=seed, scale=K ** -0.25), torch.full((1, K), float("nan"), device=DEV)])
    x, w = buf(T, 0)[:T], buf(E * wn, 1)[:E * wn].view(E, wn, K)
    offsets = torch.tensor([sum(counts[:e]) for e in range(E + 1)], dtype=torch.int32, device=DEV)
    rows = torch.randint(0, T, (A,), generator=torch.Generator().manual_seed(2)).to(torch.int32).to(DEV)
    tr = ops.MOE_TILED_F32_ROWS if kind == "tiled" else 16
    mt = ops.moe_max_tiles(A, E, tr)
    tiles = [(e, int(offsets[e]) + r) for e in range(E) for r in range(0, counts[e], tr)]
    tile_map = torch.zeros(2 * mt + 1, dtype=torch.int32)
    for i, (e, r) in enumerate(tiles):
        tile_map[i], tile_map[mt + i] = e, r
    tile_map[2 * mt] = len(tiles)
    tile_map = tile_map.to(DEV)
    out = torch.full((A, n), float("nan"), device=DEV)
    if kind == "tiled":
        ops.moe_grouped_tiled_f32(x, w, out, offsets, rows, tile_map, gate_up, limit)
    elif kind == "streaming":
        ops.moe_grouped_mfma(x, w, out, offsets, rows, tile_map, tr, gate_up, 4, limit)
    else:
        shared = torch.full((T, n), float("nan"), device=DEV)
        ops.moe_grouped_dual(x, w, out, offsets, rows, tile_map, tr, x, w[0], shared, gate_up == 1, limit, limit)

    def want(z):
        if gate_up == 0:
            return z
        if gate_up == 2:
            return torch.relu(z) ** 2
        g, u = z[:, :n], z[:, n:]
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            return g * torch.sigmoid(1.702 * g) * (u + 1)
        return torch.nn.functional.silu(g) * u

    xd, wd = x.double().cpu(), w.double().cpu()
    expect = torch.cat([want(xd[rows.cpu().long()[sum(counts[:e]):sum(counts[:e + 1])]] @ wd[e].T) for e in range(E)])
    assert torch.isfinite(out).all() and rel_err(out, expect) < 1e-5
    if kind == "dual":
        assert torch.isfinite(shared).all() and rel_err(shared, want(xd @ wd[0].T)) < 1e-5


@pytest.mark.parametrize("counts", [[5, 64, 17, 1, 0, 40, 33, 130, 16, 48, 49, 32], [1] * 40 + [70] * 30 + [20] * 30, [2] * 511 + [65]])
@pytest.mark.parametrize("K", [32, 64, 68, 96, 128, 160, 256])
def test_grouped_tiled_in_float32_worked_by_their_rows(counts, K):
    """Tiles of all heights in any order of the map, up to 64, some more and over 512 of them: each is formed, whichever the
    order in which they are worked; one to eight stages of the reduction through the rings."""
    from inferx_amd import ops
    E, A, T, n = len(counts), sum(counts), 70, 132
    topk_e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    offsets, _, _, tile_map = dispatch(topk_e, E, ops.MOE_TILED_F32_ROWS)
    rows = torch.randint(0, T, (A,), generator=torch.Generator().manual_seed(2)).to(torch.int32).to(DEV)
    x, w = rnd(T, K, scale=K ** -0.25), rnd(E, n, K, seed=1, scale=K ** -0.25)
    out = torch.full((A, n), float("nan"), device=DEV)
    ops.moe_grouped_tiled_f32(x, w, out, offsets, rows, tile_map, False)
    want = torch.cat([x[rows.long()][lo:hi].double() @ w[e].double().T
                      for e, (lo, hi) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:]))])
    assert rel_err(out, want) < 1e-5  # (every product and sum is 32-bit)


@pytest.mark.parametrize("gate_up", [0, 1, 2])
@pytest.mark.parametrize("K", [4, 32, 68, 96, 128, 160, 196, 256, 512, 1024, 1280])
def test_grouped_tiled_in_float32_of_few_and_many_workgroups(K, gate_up):
    """One block of weight rows a workgroup, and two where (further, empty) experts make many workgroups: float64's results, and the
    same bits.  Tiles of all heights, one to forty stages through rings of three to six buffers, columns past the last block."""
    from inferx_amd import ops
    counts, T, n = [5, 64, 17, 1, 0, 40, 33, 130], 70, 388  # (four blocks of 128 and more: 52 workgroups at least, 1,160)
    E, A = len(counts), sum(counts)
    topk_e = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32)[:, None].to(DEV)
    rows = torch.randint(0, T, (A,), generator=torch.Generator().manual_seed(2)).to(torch.int32).to(DEV)
    x, few = rnd(T, K, scale=K ** -0.25), rnd(E, (2 if gate_up == 1 else 1) * n, K, seed=1, scale=K ** -0.25)
    many = torch.cat([few, torch.full((300 - E,) + few.shape[1:], float("nan"), device=DEV)])
    out = []
    for w in (few, many):
        offsets, _, _, tile_map = dispatch(topk_e, w.shape[0], ops.MOE_TILED_F32_ROWS)
        out.append(torch.full((A, n), float("nan"), device=DEV))
        ops.moe_grouped_tiled_f32(x, w, out[-1], offsets, rows, tile_map, gate_up)
    z = torch.cat([x[rows.long()][lo:hi].double() @ few[e].double().T
                   for e, (lo, hi) in enumerate(zip(offsets.tolist()[:E], offsets.tolist()[1:E + 1]))])
    want = z if gate_up == 0 else torch.relu(z) ** 2 if gate_up == 2 else torch.nn.functional.silu(z[:, :n]) * z[:, n:]
    assert rel_err(out[0], want) < 1e-5 and torch.equal(*out)  # (every product and sum is 32-bit)


@pytest.mark.parametrize("T,N,K", [(1, 301, 36), (16, 33, 2048), (17, 384, 100), (32, 70, 4), (64, 1000, 260)])
def test_linear_skinny_in_float32(T, N, K):
    from inferx_amd import ops
    x, w = rnd(T, K), rnd(N, K, seed=1, scale=K ** -0.5)
    out = torch.full((T, N), float("nan"), device=DEV)
    ops.linear_skinny_f32(x, w, out)
    assert rel_err(out, x.double().cpu() @ w.double().cpu().T) < 1e-5
