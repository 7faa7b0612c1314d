"""Bibevik's mechanisms one by one, each kernel against a slow float64 function written from the equations (here
or in `plain_bibevik.py`): the recurrence with a matrix of state (per token and in chunks, with and without the
correction, carried over steps and slots), attention over the compressed cache (plain and on the matrix cores, for
prompt portions, mixed steps and single tokens whose keys are cut into slices; one key made to stand out far back, at a
page border and at the last visible place), the router with groups scored by their two best, the clamped gated unit,
the norm with one number."""
import math

import numpy as np
import pytest
import torch

import plain_bibevik as pb

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(shape, seed, scale=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


# ---- the recurrence ---------------------------------------------------------------------------------------------------
def plain_recurrence(r, k, v, w, a, b, state):
    """S <- diag(w_t) S - a_t (b_t^T S) + k_t v_t^T; o_t = S^T r_t, float64.  r, k, w, a, b [T, H, D]; v [T, H, V];
    state [H, D, V] (changed in place)."""
    T, H, _ = r.shape
    out = torch.zeros(T, H, v.shape[2], dtype=torch.float64)
    for t in range(T):
        for h in range(H):
            S = state[h]
            read = b[t, h] @ S
            S = w[t, h][:, None] * S - torch.outer(a[t, h], read) + torch.outer(k[t, h], v[t, h])
            state[h] = S
            out[t, h] = S.T @ r[t, h]
    return out


def step_rows(lengths, slots):
    from inferx_amd import ops
    q_start = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    seq = np.repeat(np.arange(len(lengths)), lengths).astype(np.int32)
    return ops.StepRows(torch.from_numpy(seq).to(DEV), torch.from_numpy(q_start).to(DEV),
                        torch.tensor(slots, dtype=torch.int32, device=DEV))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("corrected", [True, False])
@pytest.mark.parametrize("H,D,V", [(2, 16, 24), (3, 20, 12), (1, 32, 40), (2, 64, 64), (2, 128, 80), (1, 192, 16), (32, 128, 128)])
def test_recurrence_over_steps_and_slots(H, D, V, corrected, dtype):
    """Three requests in slots that are not in order: a step of unequal portions (several chunks, a chunk's edge, one
    row), then steps of one row each, then a portion of two rows, then portions around the longest chunk's length:
    outputs and the state that is left against the float64 loop over the rows."""
    from inferx_amd import ops
    silu = not corrected
    steps = [(33, 16, 1), (1, 1, 1), (1, 1, 1), (2, 17, 5)]
    if H <= 3:  # portions longer than the longest chunk: two whole chunks and two rows, a whole chunk, a chunk and a row
        steps.append((130, 64, 65))
    slots = [4, 0, 2]
    state = torch.zeros(6, H * D * V + 8, dtype=torch.float32, device=DEV)
    state[1] = float("nan")  # a slot that nobody owns
    plain_state = [torch.zeros(H, D, V, dtype=torch.float64) for _ in slots]
    tol = 2e-5 if dtype == torch.float32 else 2e-2
    for n, lengths in enumerate(steps):
        T = sum(lengths)
        r, k = rnd((T, H * D), 10 * n + 1, 0.7, dtype), rnd((T, H * D), 10 * n + 2, 0.7, dtype)
        v = rnd((T, H * V), 10 * n + 3, 1.0, dtype)
        if corrected:
            w = torch.exp(-0.6 * torch.sigmoid(rnd((T, H * D), 10 * n + 4)))
            u = rnd((T, H, D), 10 * n + 5)
            u = (u / u.norm(dim=2, keepdim=True)).reshape(T, H * D).contiguous()
            a = (u * torch.sigmoid(rnd((T, H * D), 10 * n + 6))).contiguous()
            w_head = None
        else:
            w_head = torch.tensor(([0.97, 0.6, 1.0] * H)[:H], dtype=torch.float32)
        out = torch.empty(T, H, V, dtype=torch.float32, device=DEV)
        ops.linear_state(r.to(DEV), k.to(DEV), v.to(DEV), state, step_rows(lengths, slots), out, H, D, V,
                         w_rows=w.to(DEV) if corrected else None, w_head=None if corrected else w_head.to(DEV),
                         a_rows=a.to(DEV) if corrected else None, b_rows=u.to(DEV) if corrected else None, silu=silu)
        act = (lambda x: x * torch.sigmoid(x)) if silu else (lambda x: x)
        r64, k64, v64 = (act(x.double()) for x in (r, k, v))
        at = 0
        for i, L in enumerate(lengths):
            rows = slice(at, at + L)
            if corrected:
                w64, a64, b64 = (x.double()[rows].view(L, H, D) for x in (w, a, u))
            else:
                w64 = w_head.double()[None, :, None].expand(L, H, D)
                a64 = b64 = torch.zeros(L, H, D, dtype=torch.float64)
            want = plain_recurrence(r64[rows].view(L, H, D), k64[rows].view(L, H, D), v64[rows].view(L, H, V), w64, a64,
                                    b64, plain_state[i])
            got = out[rows].cpu().double()
            scale = float(want.abs().max()) + 1e-9
            assert float((got - want).abs().max()) <= tol * scale, f"step {n} request {i}"
            at += L
    for i, slot in enumerate(slots):  # the state is kept [head][column][row]
        got = state[slot, :H * D * V].cpu().double().view(H, V, D).transpose(1, 2)
        scale = float(plain_state[i].abs().max())
        assert float((got - plain_state[i]).abs().max()) <= tol * scale
    assert bool(torch.isnan(state[1]).all()), "a slot of no request was written"


# rows of the requests of a step (one of them without any), around chunks of 64 and the sixteens within them
@pytest.mark.parametrize("lengths", [[1, 15, 0, 16], [17, 64, 63], [65, 130]])
@pytest.mark.parametrize("H,D,V", [(3, 32, 48), (2, 64, 64), (1, 128, 144)])
@pytest.mark.parametrize("decay,same_key", [(0.6, False), (1.0, False), (1e-3, False), (0.6, True)])
def test_generalized_delta_rule_in_chunks(lengths, H, D, V, decay, same_key):
    """The chunked form against the float64 recurrence, from a state that is not zero, its last state too; in one call and
    cut into slices of two chunks; with the strongest decays that it takes (e^-1 a row), hardly any, and one unit key
    for all rows.  float32 sums of at most D + 64 products of numbers up to the results' size: 1e-5 of the largest."""
    from inferx_amd import ops
    T, S = sum(lengths), len(lengths)
    strided = rnd((T, 3 * H * (D + 1)), 1, 0.7, torch.bfloat16)  # rows neither dense nor on 16-byte boundaries
    r, k = strided[:, 1:1 + H * D], strided[:, H * (D + 1):H * (D + 1) + H * D]
    v = rnd((T, H * V), 3, 1.0, torch.bfloat16)
    logit = rnd((T, H * D), 4, 3.0)
    w = torch.exp(-decay * (torch.ones_like(logit) if decay == 1.0 else torch.sigmoid(logit)))
    u = rnd((1 if same_key else T, H, D), 5).expand(T, H, D)
    u = (u / u.norm(dim=2, keepdim=True)).reshape(T, H * D).contiguous()
    a = (u * torch.sigmoid(rnd((T, H * D), 6))).contiguous()
    before = rnd((S + 1, H * D * V + 4), 7, 0.3)
    starts = [sum(lengths[:s]) for s in range(S + 1)]
    row0 = [(s, starts[s] + at, min(64, n - at)) for s, n in enumerate(lengths) for at in range(0, n, 64)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    slots = i32([S - s for s in range(S)])
    on = strided.to(DEV)
    r_dev, k_dev = on[:, 1:1 + H * D], on[:, H * (D + 1):H * (D + 1) + H * D]
    for most in (1000, 2):
        state = before.to(DEV)
        out = torch.full((T, H, V), float("nan"), device=DEV)
        for first in range(0, len(row0), most):
            part = row0[first:first + most]
            live = sorted({s for s, _, _ in part})
            ops.general_delta_chunks(r_dev, k_dev, v.to(DEV), state, slots,
                                     i32([[x[1] for x in part], [x[2] for x in part]]),
                                     i32([live, [[x[0] for x in part].index(s) for s in live],
                                          [sum(x[0] == s for x in part) for s in live]]),
                                     out, H, D, V, w.to(DEV), a.to(DEV), u.to(DEV))
        for s, n in enumerate(lengths):
            slot, at = S - s, slice(starts[s], starts[s] + n)
            if n == 0:
                assert torch.equal(state[slot].cpu(), before[slot])
                continue
            M = before[slot, :H * D * V].double().view(H, V, D).transpose(1, 2).clone()
            rows = [x[at].double().view(n, H, -1) for x in (r, k, v, w, a, u)]
            want = plain_recurrence(*rows, M)
            assert float((out[at].cpu().double() - want).abs().max()) <= 1e-5 * float(want.abs().max()), f"request {s}"
            left = state[slot, :H * D * V].cpu().double().view(H, V, D).transpose(1, 2)
            assert float((left - M).abs().max()) <= 1e-5 * float(M.abs().max()), f"state of request {s}"
            assert torch.equal(state[slot, H * D * V:].cpu(), before[slot, H * D * V:])


def test_delta_operands_and_the_plain_mixer_agree():
    """decay, removal and unit key as the kernel makes them against the plain mixer's formulas."""
    from inferx_amd import ops
    T, H, D = 7, 3, 20
    wl, al, k = rnd((T, H * D), 1, 2.0), rnd((T, H * D), 2, 2.0), rnd((T, H * D), 3)
    w0, ab = rnd((H * D,), 4), rnd((H * D,), 5)
    w, a, u = (torch.empty(T, H * D, dtype=torch.float32, device=DEV) for _ in range(3))
    ops.delta_operands(wl.to(DEV), w0.to(DEV), al.to(DEV), ab.to(DEV), k.to(DEV), w, a, u, H, D, math.exp(-0.5), 1e-6)
    k3 = k.double().view(T, H, D)
    unit = (k3 / torch.sqrt((k3 * k3).sum(dim=2, keepdim=True) + 1e-6)).view(T, H * D)
    assert torch.allclose(w.cpu().double(), torch.exp(-math.exp(-0.5) * torch.sigmoid(wl.double() + w0.double())), atol=1e-6)
    assert torch.allclose(u.cpu().double(), unit, atol=1e-6)
    assert torch.allclose(a.cpu().double(), unit * torch.sigmoid(al.double() + ab.double()), atol=1e-6)


# ---- attention over the compressed cache ------------------------------------------------------------------------------
def plain_latent_scores(q_lat, q_rot, rows, positions, scale):
    """out[t, h] = softmax over j <= pos(t) of (q_lat[t, h] . c[j] + q_rot[t, h] . kr[j]) * scale, times c; float64.
    rows [n, rank + rot] are the request's cached rows."""
    rank = q_lat.shape[2]
    c, kr = rows[:, :rank], rows[:, rank:]
    out = torch.zeros_like(q_lat)
    for t, p in enumerate(positions):
        s = (q_lat[t] @ c[:p + 1].T + q_rot[t] @ kr[:p + 1].T) * scale
        out[t] = torch.softmax(s, dim=1) @ c[:p + 1]
    return out


class Paged:
    """Requests with contexts in a paged cache whose pages are dealt out of order."""

    def __init__(self, contexts, width, page_size, dtype, seed):
        self.page_size, self.width = page_size, width
        pages_of = [-(-n // page_size) for n in contexts]
        total = sum(pages_of) + 3
        order = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).tolist()
        self.cache = torch.full((total, 1, page_size, width), float("nan"), dtype=dtype)
        self.table = torch.zeros(len(contexts), max(pages_of), dtype=torch.int32)
        self.rows = []
        for i, n in enumerate(contexts):
            rows = rnd((n, width), seed + 10 + i, 1.0, dtype)
            self.rows.append(rows)
            for p in range(pages_of[i]):
                page = order.pop()
                self.table[i, p] = page
                part = rows[p * page_size:(p + 1) * page_size]
                self.cache[page, 0, :part.shape[0]] = part


def run_latent(paged, lengths, contexts, H, rank, rot, scale, dtype, mfma, q_scale=1.0, standout=None):
    """The last `lengths[i]` positions of request i (its context is contexts[i]) as one step's rows; returns the
    kernel's result and the float64 one, [T, H, rank] each.  standout = (request, key): that key's row and every
    query of the request are made to match, so that this key takes nearly all the weight."""
    from inferx_amd import ops
    T = sum(lengths)
    seq = np.repeat(np.arange(len(lengths)), lengths).astype(np.int32)
    pos = np.concatenate([np.arange(c - n, c) for c, n in zip(contexts, lengths)]).astype(np.int32)
    q_lat, q_rot = rnd((T, H, rank), 77, q_scale, dtype), rnd((T, H, max(rot, 8)), 78, q_scale, dtype)[:, :, :rot]
    if standout is not None:
        i, key = standout
        direction = paged.rows[i][key].float()
        direction = direction / direction.norm()
        for t in np.nonzero(seq == i)[0]:
            q_lat[t] += (12.0 / scale * direction[:rank] / direction.norm()).to(dtype)
    full = torch.zeros(T, H, rank + 64, dtype=dtype)  # queries as views with strides, as the mixer hands them over
    full[:, :, :rank] = q_lat
    dq = full.to(DEV)
    qr = q_rot.contiguous().to(DEV)
    out = torch.empty(H, T, rank, dtype=dtype, device=DEV).transpose(0, 1)
    one_each = all(n == 1 for n in lengths)
    args = (dq[:, :, :rank], qr, paged.cache.to(DEV), paged.table.to(DEV), torch.from_numpy(seq).to(DEV),
            torch.from_numpy(pos).to(DEV))
    if mfma:
        assert ops.latent_mfma_fits(dq[:, :, :rank], qr, out, rank, rot)
        splits, work = 1, None
        if one_each:
            out = torch.empty(T, H, rank, dtype=dtype, device=DEV)
            splits = ops.latent_mfma_splits(T, H)
            work = (torch.empty(T * H * splits, rank, dtype=torch.float32, device=DEV),
                    torch.empty(T * H * splits, 2, dtype=torch.float32, device=DEV))
        ops.latent_attention_mfma(*args, out, rank, rot, scale, one_each, splits, work)
    else:
        ops.latent_attention_plain(*args, out, rank, rot, scale)
    want = torch.zeros(T, H, rank, dtype=torch.float64)
    at = 0
    for i, n in enumerate(lengths):
        rows = slice(at, at + n)
        want[rows] = plain_latent_scores(q_lat[rows].double(), q_rot[rows].double(), paged.rows[i].double(),
                                         pos[rows].tolist(), scale)
        at += n
    return out.cpu().double(), want


SIZES = [(2, 64, 32, 16), (5, 96, 64, 8), (16, 128, 64, 16), (3, 256, 64, 48), (4, 512, 64, 16), (70, 32, 32, 16)]


@pytest.mark.parametrize("H,rank,rot,page", SIZES)
def test_latent_attention_on_the_matrix_cores(H, rank, rot, page):
    """Prompt portions of unequal requests in one step (one of them from position 0, one row alone between two
    portions, a portion that ends on a tile's edge), then one token per request with the keys cut into slices."""
    contexts = [70, 33, 1, 150, 48]
    paged = Paged(contexts, rank + rot, page, torch.bfloat16, seed=3)
    scale = (rank + rot) ** -0.5
    for lengths in ([70, 20, 1, 9, 16], [1, 1, 1, 1, 1], [3, 1, 1, 2, 1]):
        got, want = run_latent(paged, lengths, contexts, H, rank, rot, scale, torch.bfloat16, True)
        err = float((got - want).abs().max()) / float(want.abs().max())
        assert err <= 2e-2, f"{lengths}: {err:.2e}"


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 2e-2)])
def test_latent_attention_plain_kernel(dtype, tol):
    contexts = [40, 300, 7]
    for H, rank, rot, page in [(3, 40, 8, 16), (2, 24, 0, 8), (1, 64, 32, 48)]:
        paged = Paged(contexts, rank + rot, page, dtype, seed=5)
        for lengths in ([40, 5, 1], [1, 1, 1]):
            got, want = run_latent(paged, lengths, contexts, H, rank, rot, 0.2, dtype, False)
            assert float((got - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("mfma", [False, True])
@pytest.mark.parametrize("key", [0, 15, 16, 255, 256, 600, 1021, 1022])
def test_one_key_that_stands_out(mfma, key):
    """1,023 keys of which one takes nearly all the weight: the first, the last two, both sides of a page's and of a
    slice's border, one far back.  The queries: a portion of 40 rows, then the last token alone (slices of its keys)."""
    H, rank, rot, page = 4, 64, 32, 16
    n = 1023
    paged = Paged([n], rank + rot, page, torch.bfloat16, seed=9)
    for lengths in ([40], [1]):
        got, want = run_latent(paged, lengths, [n], H, rank, rot, 0.1, torch.bfloat16, mfma, q_scale=0.2, standout=(0, key))
        visible = [t for t in range(lengths[0]) if n - lengths[0] + t >= key]
        assert visible
        c = paged.rows[0][key, :rank].double()
        for t in visible:  # the result is that key's latent, nearly
            assert float((want[t] - c).abs().max()) < 0.2 * float(c.abs().max()), "the test's key does not stand out"
        assert float((got - want).abs().max()) <= 2e-2 * float(want.abs().max())


# ---- router, gated unit, norm -------------------------------------------------------------------------------------------
@pytest.mark.parametrize("E,top,groups,keep", [(8, 2, 2, 1), (6, 2, 3, 2), (16, 4, 8, 3), (5, 1, 1, 1), (12, 3, 4, 4), (6, 2, 6, 3)])
def test_router_with_groups_scored_by_their_two_best(E, top, groups, keep):
    from inferx_amd import ops
    T, W = 37, 48
    x, w = rnd((T, W), 1), rnd((E, W), 2, 0.5)
    topk_w = torch.empty(T, top, dtype=torch.float32, device=DEV)
    topk_e = torch.empty(T, top, dtype=torch.int32, device=DEV)
    ops.moe_route(x.to(DEV), w.to(DEV), None, topk_w, topk_e, None, False, 2.5, 0, groups, keep, True, True)
    scores = torch.sigmoid(x.double() @ w.double().T)
    want = pb.choose_experts(scores, top, groups, keep)
    for t in range(T):
        assert set(topk_e[t].tolist()) == set(want[t].tolist()), f"token {t}"
        for e, wt in zip(topk_e[t].tolist(), topk_w[t].tolist()):
            assert abs(wt - 2.5 * float(scores[t, e])) < 1e-5


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.bfloat16, 1e-2)])
@pytest.mark.parametrize("limit", [0.7, 7.0])
def test_clamped_gated_unit_with_biases(dtype, tol, limit):
    from inferx_amd import ops
    T, n = 9, 40
    gate_up, bias = rnd((T, 2 * n), 1, 3.0, dtype), rnd((2 * n,), 2, 1.0, dtype)
    act = torch.empty(T, n, dtype=dtype, device=DEV)
    ops.glu_bias(gate_up.to(DEV), bias.to(DEV), act, limit)
    z = gate_up.double() + bias.double()
    g, u = z[:, :n].clamp(max=limit), z[:, n:].clamp(-limit, limit)
    want = g * torch.sigmoid(1.702 * g) * (u + 1)
    assert float((act.cpu().double() - want).abs().max()) <= tol * float(want.abs().max())


@pytest.mark.parametrize("T", [1, 8, 16])
@pytest.mark.parametrize("H,n,width", [(16, 512, 128), (3, 16, 32), (5, 48, 160), (2, 128, 512), (1, 80, 1056)])
def test_product_of_every_head(T, H, n, width):
    """Rows with strides of their own on both sides, what lies between and behind them not-a-number.  The bound is the
    result's own rounding and that of `width` float32 sums."""
    from inferx_amd import ops
    x = torch.full((T, H, width + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    x[:, :, :width] = rnd((T, H, width), 1, 1.0, torch.bfloat16).to(DEV)
    w = rnd((H, n, width), 2, width ** -0.5, torch.bfloat16).to(DEV)
    out = torch.full((H, T, n), float("nan"), dtype=torch.bfloat16, device=DEV).transpose(0, 1)
    assert ops.heads_product_fits(x[:, :, :width], w)
    ops.heads_product(x[:, :, :width], w, out)
    want = (w.double()[None] * x[:, :, None, :width].double()).sum(-1)
    assert float(((out.double() - want).abs() - 2.0 ** -8 * want.abs()).max()) <= 4e-5


@pytest.mark.parametrize("bias", ["bfloat16", "float32", "bfloat16 off a boundary"])
def test_clamped_gated_unit_of_many_rows(bias):
    """More rows than lines of workgroups (512), a width of 257 pieces of eight; a bias of either type, also one that does
    not lie on 16 bytes."""
    from inferx_amd import ops
    T, n, limit = 600, 2056, 7.0
    gate_up = rnd((T, 2 * n), 1, 3.0, torch.bfloat16)
    b = rnd((2 * n + 1,), 2, 1.0, torch.float32 if bias == "float32" else torch.bfloat16)
    dev = b.to(DEV)
    b, dev = (b[1:], dev[1:]) if bias.endswith("boundary") else (b[:-1], dev[:-1])
    act = torch.empty(T, n, dtype=torch.bfloat16, device=DEV)
    ops.glu_bias(gate_up.to(DEV), dev, act, limit)
    z = gate_up.double() + b.double()
    g, u = z[:, :n].clamp(max=limit), z[:, n:].clamp(-limit, limit)
    want = g * torch.sigmoid(1.702 * g) * (u + 1)
    assert float((act.cpu().double() - want).abs().max()) <= 1e-2 * float(want.abs().max())


@pytest.mark.parametrize("T,n", [(1, 8), (7000, 8), (131, 136), (20000, 264), (9, 1368), (3, 2040), (2049, 2048)])
@pytest.mark.parametrize("biased", [False, True])
def test_gated_unit_of_narrow_rows(T, n, biased):
    """Several rows a workgroup (32 of 8 columns, one of 1,368), a last one with fewer, one to three turns of rows a thread;
    what lies behind the result stays."""
    from inferx_amd import ops
    gate_up = rnd((T, 2 * n), 1, 3.0, torch.bfloat16).to(DEV)
    b = rnd((2 * n,), 2, 1.0, torch.bfloat16).to(DEV) if biased else None
    buf = torch.full((T + 3, n), 9.0, dtype=torch.bfloat16, device=DEV)
    ops.glu_bias(gate_up, b, buf[:T])
    z = gate_up.double() + (b.double() if biased else 0.0)
    want = torch.nn.functional.silu(z[:, :n]) * z[:, n:]
    assert float((buf[:T].double() - want).abs().max()) <= 1e-2 * float(want.abs().max()) and (buf[T:] == 9.0).all()


def test_norm_with_one_number():
    x = rnd((5, 24), 1).double()
    g = torch.tensor(1.3, dtype=torch.float64)
    want = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-5) * g
    assert torch.allclose(pb.scalar_norm(x, g, 1e-5), want)
    from inferx_amd import ops
    out = torch.empty(5, 24, dtype=torch.float32, device=DEV)
    h = x.float().to(DEV)
    ops.add_rmsnorm(h, None, torch.full((24,), 1.3, dtype=torch.float32, device=DEV), out, 1e-5, None)
    assert torch.allclose(out.cpu().double(), want, atol=1e-5)


# head groups that are not full, pages that eight keys do not share, all numbers of a row in its first 64 pieces or not
@pytest.mark.parametrize("H,rank,rot,page", [(1, 512, 64, 16), (7, 512, 64, 12), (4, 256, 0, 8), (9, 480, 64, 16), (3, 16, 16, 4),
                                             (16, 512, 32, 32)])
@pytest.mark.parametrize("window,gated", [(0, False), (40, True)])
def test_latent_attention_of_prompts(H, rank, rot, page, window, gated):
    """Portions long enough for several rounds of 32 keys and both buffers, requests that share a tile of rows, portions on
    contexts; against the plain kernel in float32 on the same numbers.  Weights and results are bfloat16: 2e-2."""
    from inferx_amd import ops
    contexts, lengths = [200, 33, 64, 97], [200, 20, 1, 40]
    paged = Paged(contexts, rank + rot, page, torch.bfloat16, seed=5)
    T, scale = sum(lengths), (rank + rot) ** -0.5
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    seq = i32(np.repeat(np.arange(4), lengths).tolist())
    pos = i32(np.concatenate([np.arange(c - n, c) for c, n in zip(contexts, lengths)]).tolist())
    q = rnd((T, H, rank + 64), 6, 2.0, torch.bfloat16).to(DEV)
    qr = rnd((T, H, max(rot, 8)), 7, 2.0, torch.bfloat16).to(DEV)[:, :, :rot] if rot else q
    gate = rnd((T, H + 8), 8, 1.0, torch.bfloat16).to(DEV)[:, :H] if gated else None
    cache, table = paged.cache.to(DEV), paged.table.to(DEV)
    out = torch.full((H, T, rank), float("nan"), dtype=torch.bfloat16, device=DEV).transpose(0, 1)
    assert ops.latent_mfma_fits(q[:, :, :rank], qr, out, rank, rot)
    ops.latent_attention_mfma(q[:, :, :rank], qr, cache, table, seq, pos, out, rank, rot, scale, False, 1, None, window, gate)
    want = torch.empty(T, H, rank, device=DEV)
    f32 = lambda t: None if t is None else t.float().contiguous()
    ops.latent_attention_plain(f32(q[:, :, :rank]), f32(qr), f32(cache), table, seq, pos, want, rank, rot, scale, window, f32(gate))
    err = float((out.float() - want).abs().max()) / float(want.abs().max())
    assert torch.isfinite(out).all() and err <= 2e-2, f"{err:.2e}"


@pytest.mark.parametrize("T,H,dim,rot,rank", [(1, 1, 32, 0, 16), (8, 16, 128, 64, 512), (16, 3, 160, 32, 96)])
@pytest.mark.parametrize("halves", [False, True])
def test_latent_rows_and_the_queries_way_to_them_in_one_launch(T, H, dim, rot, rank, halves):
    """The same numbers as in two launches."""
    from inferx_amd import ops
    q = rnd((T, H * (dim + rot) + rank + rot), 1, 1.0, torch.bfloat16).to(DEV)
    w, norm = rnd((H, rank, dim), 2, 0.1, torch.bfloat16).to(DEV), rnd((rank,), 3, 1.0, torch.bfloat16).to(DEV)
    angles = rnd((T, rot // 2, 1), 4, 3.0) if rot else None
    table = torch.cat([angles.cos(), angles.sin()], 2).float().contiguous().to(DEV) if rot else None
    slots = torch.arange(T, dtype=torch.int32, device=DEV).flip(0)
    got = []
    for fused in (False, True):
        mine, cache = q.clone(), torch.zeros((2, 1, 16, rank + rot), dtype=torch.bfloat16, device=DEV)
        out = torch.full((T, H, rank), float("nan"), dtype=torch.bfloat16, device=DEV)
        rows, d = mine[:, :H * (dim + rot)], mine[:, H * (dim + rot):]
        ops.latent_prepare(rows, d, norm, 1e-6, table, slots, cache, H, rot, rank, halves, None, (w, out) if fused else None)
        if not fused:
            ops.heads_product(rows.unflatten(1, (H, dim + rot))[:, :, :dim], w, out)
        got.append((mine, cache, out))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,H,rank,n,splits", [(1, 1, 32, 16, 2), (8, 16, 512, 128, 32), (16, 3, 96, 144, 9), (2, 5, 264, 40, 70)])
@pytest.mark.parametrize("gated", [False, True])
def test_slices_of_latents_merged_and_multiplied_in_one_launch(T, H, rank, n, splits, gated):
    """Some tokens have keys in the first slices only, and NaN where the others' parts would be.  Against float64 on the same
    numbers: float32 sums of `rank` terms and a result rounded to bfloat16."""
    from inferx_amd import ops
    o, m = rnd((T, H, splits, rank), 1, 1.0), rnd((T, H, splits), 2, 3.0)
    l = rnd((T, H, splits), 3, 1.0).abs() + 0.1
    for t in range(T):
        used = 1 + (t * 5) % splits
        o[t, :, used:], m[t, :, used:], l[t, :, used:] = float("nan"), float("-inf"), 0.0
    w, gate = rnd((H, n, rank), 4, 0.1, torch.bfloat16), rnd((T, H + 3), 5, 1.0, torch.bfloat16)
    work = (o.float().contiguous().to(DEV), torch.stack([m, l], 3).float().contiguous().to(DEV))
    wide = torch.full((T, H * n + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = wide[:, :H * n].unflatten(1, (H, n))
    ops.latent_merge_product(work, splits, w.to(DEV), out, gate.to(DEV)[:, 3:] if gated else None)
    f = torch.exp2(m.double() - m.double().amax(2, keepdim=True))
    x = (f[..., None] * o.double().nan_to_num()).sum(2) / (f * l.double()).sum(2)[..., None]
    if gated:
        x = x * torch.sigmoid(gate[:, 3:].double())[..., None]
    want = torch.einsum("thr,hnr->thn", x, w.double())
    bound = 2.0 ** -8 * want.abs() + 2.0 ** -20 * torch.einsum("thr,hnr->thn", x.abs(), w.double().abs())
    assert ((out.cpu().double() - want).abs() <= bound).all() and torch.isnan(wide[:, H * n:]).all()


@pytest.mark.parametrize("H", [1, 3, 16])
@pytest.mark.parametrize("lengths", [[1, 63, 64, 65], [33, 200, 1, 129], [20], [577, 31]])
def test_latent_attention_of_whole_contexts(H, lengths):
    """Requests that end within a tile, a step of 32 keys or a wavefront's share of them; the tensors around the operands and
    another request's rows are NaN, and reach nothing.  Against float64 on the same numbers: the weights' and the results'
    rounding to bfloat16, 2^-9 each of at most the values' size (4), and as much again for the exponentials and sums."""
    from inferx_amd import ops
    T, dim, rd, vd = sum(lengths) + 70, 128, 64, 128
    scale = (dim + rd) ** -0.5
    q = torch.full((T, H * (dim + rd) + 64), float("nan"), dtype=torch.bfloat16, device=DEV)
    kv = torch.full((T, H * (dim + vd)), float("nan"), dtype=torch.bfloat16, device=DEV)
    rot = torch.full((T, rd), float("nan"), dtype=torch.bfloat16, device=DEV)
    n = sum(lengths)
    q[:n, :H * (dim + rd)] = rnd((n, H * (dim + rd)), 1, 2.0, torch.bfloat16).to(DEV)
    kv[:n] = rnd((n, H * (dim + vd)), 2, 1.0, torch.bfloat16).to(DEV).clamp(-4, 4)
    rot[:n] = rnd((n, rd), 3, 2.0, torch.bfloat16).to(DEV)
    tiles, at = [], 0
    for length in lengths + [70]:
        tiles += [(at + i, min(64, length - i), i) for i in range(0, length, 64)]
        at += length
    out = torch.full((T, H, vd), float("nan"), dtype=torch.bfloat16, device=DEV)
    q3 = q[:, :H * (dim + rd)].unflatten(1, (H, dim + rd))
    ops.latent_whole(q3, kv, rot, torch.tensor(tiles, dtype=torch.int32, device=DEV).t().contiguous(), out, scale)
    at = 0
    for length in lengths:
        r = slice(at, at + length)
        k = torch.cat([kv[r, :H * dim].unflatten(1, (H, dim)), rot[r, None].expand(length, H, rd)], 2).cpu().double()
        v = kv[r, H * dim:].unflatten(1, (H, vd)).cpu().double()
        s = torch.einsum("qhd,khd->hqk", q3[r].cpu().double(), k) * scale
        s = s.masked_fill(torch.ones(length, length, dtype=torch.bool).triu(1), float("-inf"))
        want = torch.einsum("hqk,khd->qhd", s.softmax(2), v)
        err = float((out[r].cpu().double() - want).abs().max())
        assert err <= 4 * 4 * 2.0 ** -9, f"{length}: {err:.2e}"
        at += length
    assert torch.isnan(out[n:]).all()


# the smallest sizes of the kernel's three forms and their largest (128, 320 with a latent of 256, 576), one row of each
# with fewer numbers than the form has room for
@pytest.mark.parametrize("rank,rot", [(16, 16), (96, 0), (112, 16), (128, 32), (144, 48), (256, 64), (272, 16), (512, 0), (512, 64)])
def test_latent_attention_of_prompts_behind_a_launch_that_left_nan(rank, rot):
    """What is behind a row in LDS (here what a launch on a cache of nothing but NaN left there) reaches no result."""
    from inferx_amd import ops
    T, H, page = 75, 6, 16
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    seq, pos, table = i32([0] * T), i32(list(range(T))), i32([[2, 0, 1, 4, 3]])

    def run(rank, rot, seed, fill=None, op=ops.latent_attention_mfma):
        cache = rnd((5, 1, page, rank + rot), seed, 1.0, torch.bfloat16).to(DEV)
        if fill is not None:
            cache.fill_(fill)
        q = rnd((T, H, rank + 64), seed + 1, 2.0, torch.bfloat16).to(DEV)
        out = torch.full((T, H, rank), float("nan"), dtype=torch.bfloat16, device=DEV)
        args = (q[:, :, :rank], q[:, :, rank:rank + rot] if rot else q, cache)
        if op is ops.latent_attention_plain:
            out, args = out.float(), tuple(t.float().contiguous() for t in args)
        op(*args, table, seq, pos, out, rank, rot, (rank + rot) ** -0.5)
        return out.float()

    for _ in range(20):  # (every compute unit's LDS)
        run(512, 64, 5, float("nan"))
    got, want = run(rank, rot, 7), run(rank, rot, 7, op=ops.latent_attention_plain)
    err = float((got - want).abs().max()) / float(want.abs().max())
    assert torch.isfinite(got).all() and err <= 2e-2, f"{err:.2e}"


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("row", [0, 7, 37, 64, 99])
def test_generalized_delta_rule_in_chunks_keeps_what_is_not_finite_to_later_rows(row, bad):
    """A number that is not finite reaches what the recurrence lets it reach and nothing else: a value its column from its row
    on, a reading vector its row, a key, a decay, a removal vector or a direction all columns from its row on.
    Everything else keeps its bits."""
    from inferx_amd import ops
    T, H, D, V = 100, 3, 64, 48  # one chunk and the next one, 36 rows
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    before = rnd((1, H * D * V), 7, 0.3)

    def run(where=None):
        ops_ = [rnd((T, H * D), 1, 0.7, torch.bfloat16), rnd((T, H * D), 2, 0.7, torch.bfloat16), rnd((T, H * V), 3, 1.0, torch.bfloat16),
                torch.exp(-0.6 * torch.sigmoid(rnd((T, H * D), 4))), rnd((T, H * D), 5, D ** -0.5), rnd((T, H * D), 6, D ** -0.5)]
        if where is not None:
            ops_[where][row, (V if where == 2 else D) + 5] = bad  # head 1, number 5
        r, k, v, w, a, b = (t.to(DEV) for t in ops_)
        state, out = before.to(DEV), torch.full((T, H, V), 7.0, device=DEV)
        ops.general_delta_chunks(r, k, v, state, i32([0]), i32([[0, 64], [64, 36]]), i32([[0], [0], [2]]), out, H, D, V, w, a, b)
        return out.cpu(), state.cpu().view(H, V, D)

    want, left = run()
    assert torch.isfinite(want).all() and torch.isfinite(left).all()
    for where in range(6):
        out, state = run(where)
        before_it = torch.ones(T, dtype=torch.bool)
        before_it[row:] = False
        assert torch.equal(out[before_it], want[before_it]), f"operand {where}: an earlier row"
        assert torch.equal(out[:, [0, 2]], want[:, [0, 2]]) and torch.equal(state[[0, 2]], left[[0, 2]]), "another head"
        if where == 2:
            others = torch.arange(V) != 5
            assert torch.equal(out[:, 1, others], want[:, 1, others]) and torch.equal(state[1, others], left[1, others])
            assert not torch.isfinite(out[row:, 1, 5]).any() and not torch.isfinite(state[1, 5, 5]).any()
        elif where == 0:
            later = torch.arange(T) != row
            assert torch.equal(out[later], want[later]) and torch.equal(state, left)
            assert not torch.isfinite(out[row, 1]).any()
        else:
            assert not torch.isfinite(out[row:, 1]).any()


@pytest.mark.parametrize("H,D,V", [(8, 32, 48), (8, 64, 64), (8, 128, 128)])
@pytest.mark.parametrize("decay", [1.0, 0.6065, 0.05, 1e-3])
def test_generalized_delta_rule_in_chunks_is_no_less_exact_than_row_by_row(H, D, V, decay):
    """The distance of the chunked form's results and last states from the float64 recurrence, over sixteen requests, is at
    most that of the form that walks row by row, for decays e^(-decay sigmoid(normal numbers))."""
    from inferx_amd import ops
    lengths = [65 + 13 * s for s in range(16)]
    S, T, starts = len(lengths), sum(lengths), [0]
    for n in lengths:
        starts.append(starts[-1] + n)
    r, k, v = (rnd((T, H * n), s, 0.7, torch.bfloat16).to(DEV) for s, n in ((1, D), (2, D), (3, V)))
    logit = rnd((T, H * D), 4, 2.0)
    w = torch.exp(-decay * torch.sigmoid(logit)).to(DEV)
    u = rnd((T, H, D), 5)
    u = (u / u.norm(dim=2, keepdim=True)).reshape(T, H * D).to(DEV)
    a = (u * torch.sigmoid(rnd((T, H * D), 6)).to(DEV)).contiguous()
    before = rnd((S, H * D * V), 7, 0.3).to(DEV)
    rd, kd, vd, wd, ad, ud = (x.double().view(T, H, -1) for x in (r, k, v, w, a, u))
    M = before.double().view(S, H, V, D).clone()
    want = torch.empty((T, H, V), dtype=torch.float64, device=DEV)
    for t in range(max(lengths)):  # every request's row t
        on = torch.tensor([s for s, n in enumerate(lengths) if t < n], device=DEV)
        at = torch.tensor(starts[:-1], device=DEV)[on] + t
        y = (M[on] * ud[at][:, :, None]).sum(-1)
        now = M[on] * wd[at][:, :, None] - ad[at][:, :, None] * y[..., None] + kd[at][:, :, None] * vd[at][..., None]
        want[at] = (now * rd[at][:, :, None]).sum(-1)
        M[on] = now
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    row0 = [(s, starts[s] + at, min(64, n - at)) for s, n in enumerate(lengths) for at in range(0, n, 64)]
    count = [-(-n // 64) for n in lengths]
    off, slots = [], i32(list(range(S)))
    for chunked in (False, True):
        state, out = before.clone(), torch.empty((T, H, V), device=DEV)
        if chunked:
            ops.general_delta_chunks(r, k, v, state, slots, i32([[x[1] for x in row0], [x[2] for x in row0]]),
                                     i32([list(range(S)), [sum(count[:s]) for s in range(S)], count]), out, H, D, V, w, a, u)
        else:
            rows = ops.StepRows(i32([s for s, n in enumerate(lengths) for _ in range(n)]), i32(starts), slots)
            ops.linear_state(r, k, v, state, rows, out, H, D, V, w_rows=w, a_rows=a, b_rows=u)
        off.append([float((x.double().view(y.shape) - y).norm() / y.norm()) for x, y in ((out, want), (state, M))])
    print(f"decay {decay}, {D} x {V}: rows {off[0][0]:.3e} {off[0][1]:.3e}, chunks {off[1][0]:.3e} {off[1][1]:.3e}")
    assert off[1][0] <= off[0][0] and off[1][1] <= off[0][1], off
