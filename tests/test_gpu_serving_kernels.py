"""The serving kernels at the sizes where their tilings can go wrong, against
the CPU references."""

import math

import pytest
import torch

from agentainer_amd import ops
from agentainer_amd.ops import reference as ref

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _paged(lens, n_kv, D, PS, dtype, width=0, seed=0):
    """Pools holding `lens` random tokens per sequence on shuffled pages.
    Every slot that belongs to no token is NaN: a kernel that multiplies one,
    even by zero, shows it."""
    gen = torch.Generator().manual_seed(seed)
    need = [-(-n // PS) for n in lens]
    perm = torch.randperm(sum(need), generator=gen) + 1
    table = torch.zeros(len(lens), max(width, max(need)), dtype=torch.int32)
    k = torch.full((sum(need) + 1, n_kv, D // 8, PS, 8), math.nan)
    v = torch.full((sum(need) + 1, n_kv, PS, D), math.nan)
    at = 0
    for b, n in enumerate(lens):
        pages = perm[at:at + need[b]]
        at += need[b]
        table[b, :need[b]] = pages.to(torch.int32)
        for i, p in enumerate(pages.tolist()):
            m = min(PS, n - i * PS)
            k[p, :, :, :m] = torch.randn(n_kv, D // 8, m, 8, generator=gen)
            v[p, :, :m] = torch.randn(n_kv, m, D, generator=gen)
    return k.to(dtype), v.to(dtype), table


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n_q,n_kv,PS,specs,width", [
    # (cached, new) per sequence; edges of the 32-row and 64-token tiles
    (32, 8, 16, [(0, 1), (0, 32), (31, 33), (64, 64), (63, 65), (5, 0)], 0),
    (64, 8, 16, [(1, 129), (200, 7)], 0),
    (4, 1, 16, [(0, 63), (17, 95)], 0),       # one kv head
    (12, 1, 32, [(100, 40)], 0),
    (32, 8, 8, [(9, 50), (0, 70)], 0),        # page below a staging group
    (8, 2, 24, [(30, 45)], 0),                # page size no power of two
    # few rows over a long context: the split path, rows whose early and
    # late runs hold no visible key, a run count above the tile count
    (32, 8, 16, [(1200, 45), (0, 19)], 0),
    (16, 4, 16, [(700, 3), (64, 1), (0, 33)], 0),
    (8, 2, 8, [(513, 2)], 200),
])
def test_prefill_attention_edges(dtype, n_q, n_kv, PS, specs, width):
    D = 128
    kc, vc, table = _paged([c + n for c, n in specs], n_kv, D, PS, dtype,
                           width, seed=n_q + PS)
    gen = torch.Generator().manual_seed(3)
    T = sum(n for _c, n in specs)
    # strided rows, as the fused projection hands them over
    q = torch.randn(T, 2 * n_q, D, generator=gen).to(torch.bfloat16)[:, :n_q]
    i32 = dict(dtype=torch.int32)
    lens = torch.tensor([c + n for c, n in specs], **i32)
    starts = torch.tensor([sum(n for _c, n in specs[:i])
                           for i in range(len(specs))], **i32)
    qlens = torch.tensor([n for _c, n in specs], **i32)
    scale = 1.0 / math.sqrt(D)
    out = torch.zeros(T, n_q, D, dtype=torch.bfloat16, device=DEV)
    qd = torch.zeros(T, 2 * n_q, D, dtype=torch.bfloat16, device=DEV)[:, :n_q]
    qd.copy_(q)
    ops.paged_prefill_attention(
        out, qd, kc.to(DEV), vc.to(DEV), table.to(DEV), lens.to(DEV),
        starts.to(DEV), qlens.to(DEV), scale, max_qlen=int(qlens.max()))
    want = torch.zeros(T, n_q, D)
    ref.paged_prefill_attention(want, q.float(), kc.float(), vc.float(),
                                table, lens, starts, qlens, scale)
    # bf16 probabilities and a bf16 result: 2^-9 of the largest value each
    bound = 2.0 ** -8 * float(vc.float().nan_to_num().abs().max())
    assert (out.float().cpu() - want).abs().max().item() <= bound


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n_q,n_kv,PS,lens,width", [
    # edges of the 32-token tiles and of the 128-token runs
    (32, 8, 16, [1, 31, 32, 33, 127, 128, 129, 500], 0),
    (8, 8, 16, [70, 3], 0),                     # one head per kv head
    (16, 8, 16, [255, 257], 0),
    (64, 8, 32, [300, 1], 0),
    (8, 2, 8, [97, 160], 0),                    # page below a load group
    (4, 1, 24, [131, 49], 0),                   # page size no power of two
    (4, 1, 16, [5000], 512),                    # many runs of one sequence
    # more tokens than runs of the shortest length: runs grow
    (1, 1, 16, [8190], 512),
    (8, 8, 16, [600, 9, 1100, 513] * 9, 0),     # 512-token runs
])
def test_decode_attention_edges(dtype, n_q, n_kv, PS, lens, width):
    D, B = 128, len(lens)
    kc, vc, table = _paged(lens, n_kv, D, PS, dtype, width, seed=n_q + PS)
    gen = torch.Generator().manual_seed(4)
    q = torch.randn(B, n_q, D, generator=gen).to(torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32)
    scale = 1.0 / math.sqrt(D)
    qd = torch.zeros(B, n_q + 3, D, dtype=torch.bfloat16, device=DEV)[:, :n_q]
    qd.copy_(q)
    out = torch.zeros(B, n_q, D, dtype=torch.bfloat16, device=DEV)
    ops.paged_decode_attention(out, qd, kc.to(DEV), vc.to(DEV), table.to(DEV),
                               sl.to(DEV), scale)
    want = torch.zeros(B, n_q, D)
    ref.paged_decode_attention(want, q.float(), kc.float(), vc.float(), table,
                               sl, scale)
    # the result's own rounding, and fp32 sums of up to 8190 terms
    err = (out.float().cpu() - want).abs()
    vmax = float(vc.float().nan_to_num().abs().max())
    assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * vmax).all())


@pytest.mark.parametrize("n_q,n_kv", [(8, 8), (32, 8), (64, 8)])
def test_decode_probabilities_keep_32_bits(n_q, n_kv):
    """Two tokens with nearly the same score and opposite values beside one
    without any: the result is the difference of two probabilities near 1/3,
    and shows every bit that one of them lost on its way through the
    product."""
    D, PS, B = 128, 16, 64
    gen = torch.Generator().manual_seed(n_q)
    q = torch.randn(B, n_q, D, generator=gen).to(torch.bfloat16)
    kc = torch.zeros(B, n_kv, D // 8, PS, 8, dtype=torch.bfloat16)
    kc[:, :, :, :2] = (torch.randn(B, n_kv, D // 8, 1, 8, generator=gen)
                       + 2e-3 * torch.randn(B, n_kv, D // 8, 2, 8,
                                            generator=gen))
    vc = torch.zeros(B, n_kv, PS, D, dtype=torch.bfloat16)
    vc[:, :, 0], vc[:, :, 1] = 1.0, -1.0
    table = torch.arange(B, dtype=torch.int32)[:, None]
    sl = torch.full((B,), 3, dtype=torch.int32)
    scale = 0.002
    out = torch.zeros(B, n_q, D, dtype=torch.bfloat16, device=DEV)
    ops.paged_decode_attention(out, q.to(DEV), kc.to(DEV), vc.to(DEV),
                               table.to(DEV), sl.to(DEV), scale)
    keys = kc[:, :, :, :3].double().permute(0, 1, 3, 2, 4).reshape(
        B, n_kv, 3, D).repeat_interleave(n_q // n_kv, dim=1)
    s = (keys @ q.double()[..., None])[..., 0] * scale
    p = torch.softmax(s, -1)
    want = (p[..., 0] - p[..., 1])[..., None]
    assert 1e-5 < want.abs().max() < 1e-3
    # half a bf16 step of the result; two probabilities of 1/3, each off by a
    # few 2^-24 of itself (its exponent, its exponential, the quotient). With
    # 16 bits they are off by 2^-18 of themselves, 1.3e-6 each
    assert bool(((out.double().cpu() - want).abs()
                 <= 2.0 ** -8 * want.abs() + 2.0 ** -22).all())


@pytest.mark.parametrize("n_q,n_kv", [(8, 8), (8, 2), (16, 2)])
def test_decode_infinite_values(n_q, n_kv):
    """An infinite value of a token that is attended to makes the result
    infinite, wherever in a tile, a run or a wave the token is; two of
    opposite signs, or a NaN, make it NaN; the other columns stay."""
    D, PS = 128, 16
    lens = [1, 2, 31, 32, 33, 128, 129, 5000]
    kc, vc, table = _paged(lens, n_kv, D, PS, torch.bfloat16, 512, seed=3)
    inf = math.inf
    for b, n in enumerate(lens):
        for at, col, val in ((n - 1, 3, inf), (0, 70, -inf), (n // 2, 127, inf),
                             (n - 1, 5, math.nan), (n - 1, 6, inf),
                             (0, 6, -inf)):
            vc[table[b, at // PS], :, at % PS, col] = val
    gen = torch.Generator().manual_seed(8)
    q = torch.randn(len(lens), n_q, D, generator=gen).to(torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32)
    out = torch.zeros(len(lens), n_q, D, dtype=torch.bfloat16, device=DEV)
    ops.paged_decode_attention(out, q.to(DEV), kc.to(DEV), vc.to(DEV),
                               table.to(DEV), sl.to(DEV), 0.05)
    want = torch.zeros(len(lens), n_q, D)
    ref.paged_decode_attention(want, q.float(), kc.float(), vc.float(), table,
                               sl, 0.05)
    got = out.float().cpu()
    assert want.isinf().any() and want.isnan().any()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    assert bool(((got - want).abs()[fine]
                 <= 2.0 ** -8 * want.abs()[fine] + 2.0 ** -11).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("width", [0, 512])  # one run, and split runs
def test_prefill_infinite_values(dtype, width):
    """A row's own token, or one that every row sees, with values that are not
    finite. (Rows that a tile masks from such a token get NaN of it.)"""
    n_q, n_kv, D, PS = 8, 2, 128, 16
    specs = [(0, 1), (30, 1), (31, 1), (62, 1), (63, 1), (700, 1), (2, 33)]
    kc, vc, table = _paged([c + n for c, n in specs], n_kv, D, PS,
                           torch.bfloat16, width, seed=4)
    special = math.inf if dtype == torch.bfloat16 else math.nan  # e4m3: no inf
    for b, (c, n) in enumerate(specs):
        for at, col in ((c + n - 1, 3), (0, 127)):
            vc[table[b, at // PS], :, at % PS, col] = special
    kc, vc = kc.to(dtype), vc.to(dtype)
    gen = torch.Generator().manual_seed(9)
    T = sum(n for _c, n in specs)
    q = torch.randn(T, n_q, D, generator=gen).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32)
    lens = torch.tensor([c + n for c, n in specs], **i32)
    starts = torch.tensor([sum(n for _c, n in specs[:i])
                           for i in range(len(specs))], **i32)
    qlens = torch.tensor([n for _c, n in specs], **i32)
    out = torch.zeros(T, n_q, D, dtype=torch.bfloat16, device=DEV)
    ops.paged_prefill_attention(
        out, q.to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), lens.to(DEV),
        starts.to(DEV), qlens.to(DEV), 0.05, max_qlen=int(qlens.max()))
    want = torch.zeros(T, n_q, D)
    ref.paged_prefill_attention(want, q.float(), kc.float(), vc.float(),
                                table, lens, starts, qlens, 0.05)
    last = (starts + qlens - 1).long()
    got, want = out.float().cpu(), want
    assert torch.equal(got[:, :, 127].isfinite(), want[:, :, 127].isfinite())
    got, want = got[last], want[last]
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    bound = 2.0 ** -8 * float(vc.float()[vc.float().isfinite()].abs().max())
    assert (got - want).abs()[fine].max().item() <= bound


def test_rope_append_decode_is_both_steps():
    """Rotation, append and attention in one call against the single ops;
    a padded row (no tokens) is left alone, dirty counters do not matter."""
    n_q, n_kv, D, PS = 32, 8, 128, 16
    lens = [40, 700, 1, 0]
    kc, vc, table = _paged([max(n, 1) for n in lens], n_kv, D, PS,
                           torch.bfloat16, 64, seed=9)
    kc, vc, table = kc.to(DEV), vc.to(DEV), table.to(DEV)
    B = len(lens)
    gen = torch.Generator().manual_seed(5)
    rnd = lambda h: torch.randn(B, h, D, generator=gen).to(  # noqa: E731
        torch.bfloat16).to(DEV)
    q, k, v = rnd(n_q), rnd(n_kv), rnd(n_kv)
    cos_sin = ops.make_cos_sin_table(1024, D, device=DEV)
    pos = torch.tensor([max(n - 1, 0) for n in lens], dtype=torch.int32,
                       device=DEV)
    slots = torch.tensor([int(table[b, (n - 1) // PS]) * PS + (n - 1) % PS
                          if n else -1 for b, n in enumerate(lens)],
                         device=DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    q1, k1, kc1, vc1 = q.clone(), k.clone(), kc.clone(), vc.clone()
    want = torch.full((B, n_q, D), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.rope_append(q1, k1, v, kc1, vc1, cos_sin, pos, slots)
    ops.paged_decode_attention(want, q1, kc1, vc1, table, sl, scale)
    junk = torch.full((4096,), -1, dtype=torch.int32, device=DEV)
    del junk  # what a fresh allocation may hold
    out = torch.full((B, n_q, D), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.rope_append_decode(out, q, k, v, kc, vc, cos_sin, pos, slots, table,
                           sl, scale)
    assert torch.equal(out, want)
    assert torch.equal(q, q1)
    assert torch.equal(kc.view(torch.int16), kc1.view(torch.int16))
    assert torch.equal(vc.view(torch.int16), vc1.view(torch.int16))


def _rel(got, want):
    return ((got.float() - want.float()).norm() / want.float().norm()).item()


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("N,K", [
    (32, 32),          # one k step: most waves have nothing to do
    (96, 160),         # tiles and steps that do not divide
    (4096, 4096), (8192, 1024), (192, 14336),
    (32800, 64),       # the many-tiles path, odd tile count
])
def test_stream_projections(T, N, K):
    """Packed projections against fp32 products of the same bf16 values."""
    gen = torch.Generator(device=DEV).manual_seed(T + N + K)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(  # noqa: E731
        torch.bfloat16)
    x, w = rnd(T, K), rnd(N, K)
    wp = ops.pack_weight(w)
    xp = ops.pack_rows(x)
    want = x.double() @ w.double().t()
    got = ops.stream_linear(xp, T, wp, N, K)
    assert got.shape == (T, N)
    # one bf16 rounding of the result
    assert bool(((got.double() - want).abs()
                 <= 2.0 ** -8 * want.abs() + 1e-4 * K ** 0.5).all())
    parts = ops.stream_parts(xp, T, wp, N, K)
    assert parts.shape[1:] == (T, N)
    assert _rel(parts.sum(0), want) < 1e-5
    if N % 64 == 0:
        act = ops.stream_gate_up(xp, T, wp, N, K)
        g, u = want.chunk(2, dim=1)
        exp = ops.pack_rows((torch.nn.functional.silu(g) * u).to(
            torch.bfloat16))
        sel = _row_slots(T, N // 2)
        assert _rel(act[sel], exp[sel]) < 2.0 ** -8


def _row_slots(T, K):
    """Flat positions of T packed rows of K columns."""
    ms = 1
    while ms * 16 < T:
        ms *= 2
    idx = torch.arange(ms * 16 * K, device=DEV).view(K // 32, ms, 4, 16, 8)
    rows = idx.permute(1, 3, 0, 2, 4).reshape(ms * 16, K)
    return rows[:T].reshape(-1)


@pytest.mark.parametrize("T,H,S", [(1, 512, 0), (5, 4096, 2), (64, 8192, 1),
                                   (33, 4128, 4), (17, 16384, 3),
                                   (65, 512, 8), (128, 4096, 4)])
@pytest.mark.parametrize("packed", [True, False])
def test_add_parts_rmsnorm(T, H, S, packed):
    gen = torch.Generator(device=DEV).manual_seed(T + H)
    res = torch.randn(T, H, generator=gen, device=DEV).to(torch.bfloat16)
    w = torch.randn(H, generator=gen, device=DEV).to(torch.bfloat16)
    parts = (torch.randn(S, T, H, generator=gen, device=DEV) if S else None)
    before = res.clone()
    out = ops.add_parts_rmsnorm(res, parts, w, 1e-5, packed)
    new = before.double() + (parts.double().sum(0) if S else 0)
    # half a bf16 step (7 stored bits: 2^-8 of a value at a power of two),
    # and fp32 sums that may fall across a tie
    assert bool(((res.double() - new).abs()
                 <= 2.0 ** -8 * new.abs() + 1e-5).all())
    ref32 = torch.empty(T, H)
    ref.rmsnorm(ref32, res.float().cpu(), w.float().cpu(), 1e-5)
    rows = out[_row_slots(T, H)].view(T, H) if packed else out
    assert bool(((rows.float().cpu() - ref32).abs()
                 <= 2.0 ** -8 * ref32.abs() + 1e-6).all())


def test_packed_attention_outputs_are_the_rows():
    n_q, n_kv, D, PS = 8, 2, 128, 16
    for T in (3, 17, 40, 70, 128):
        lens = [50 + 7 * i for i in range(T)]
        kc, vc, table = _paged(lens, n_kv, D, PS, torch.bfloat16, seed=T)
        kc, vc, table = kc.to(DEV), vc.to(DEV), table.to(DEV)
        sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
        gen = torch.Generator(device=DEV).manual_seed(T)
        q = torch.randn(T, n_q, D, generator=gen, device=DEV).to(
            torch.bfloat16)
        k = torch.randn(T, n_kv, D, generator=gen, device=DEV).to(
            torch.bfloat16)
        cos_sin = ops.make_cos_sin_table(1024, D, device=DEV)
        pos = sl - 1
        slots = (table.gather(1, (pos // PS).long()[:, None])[:, 0].long()
                 * PS + pos % PS)
        slot = _row_slots(T, n_q * D)
        rows = torch.empty(T, n_q, D, dtype=torch.bfloat16, device=DEV)
        pk = ops.packed_rows(T, n_q * D, DEV)
        args = (k, k, kc, vc, cos_sin, pos, slots, table, sl, 0.1)
        ops.rope_append_decode(rows, q.clone(), *args)
        ops.rope_append_decode(pk, q.clone(), *args, packed=True)
        assert torch.equal(pk[slot], rows.view(-1))
        one = torch.tensor([0], dtype=torch.int32, device=DEV)
        qn = torch.tensor([T], dtype=torch.int32, device=DEV)
        for width in (table.size(1), 128):  # one run, and split runs
            tb = torch.zeros(1, width, dtype=torch.int32, device=DEV)
            tb[0, :table.size(1)] = table[T - 1]
            a2 = (q, kc, vc, tb, sl[T - 1:], one, qn, 0.1)
            ops.paged_prefill_attention(rows, *a2, max_qlen=T)
            pk.zero_()
            ops.paged_prefill_attention(pk, *a2, max_qlen=T, packed=True)
            assert torch.equal(pk[slot], rows.view(-1))


@pytest.mark.parametrize("T,E,top_k,spread", [
    (1, 8, 2, 1.0), (3, 4, 2, 1.0), (16, 8, 2, 1.0), (32, 8, 2, 1.0),
    (64, 8, 2, 1.0), (7, 16, 8, 1.0), (128 // 3, 5, 3, 1.0),
    (64, 8, 2, 0.0),   # every token chooses the same experts: many row groups
    (9, 1, 1, 1.0),
])
def test_stream_experts(T, E, top_k, spread):
    """Routing and both expert projections against the plain computation."""
    H, inter = 256, 512
    gen = torch.Generator(device=DEV).manual_seed(T * E)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(  # noqa: E731
        torch.bfloat16)
    router = rnd(E, H)
    x = rnd(1, H).expand(T, H) * (1 - spread) + rnd(T, H) * max(spread, 1e-3)
    x = x.to(torch.bfloat16).contiguous()
    gus = [rnd(2 * inter, H) * 0.1 for _ in range(E)]
    dns = [rnd(H, inter) * 0.1 for _ in range(E)]
    xp = ops.pack_rows(x)
    choice, weight = ops.route_packed(xp, T, router, top_k)
    logits = x.double() @ router.double().t()
    top, who = torch.softmax(logits, -1).topk(top_k, -1)
    assert torch.equal(choice.long(), who)
    want_w = (top / top.sum(-1, keepdim=True)).float()
    # logits of about 16 summed in fp32
    assert bool(((weight - want_w).abs() <= 1e-4).all())
    gu_w = [ops.pack_weight(w) for w in gus]
    dn_w = [ops.pack_weight(w) for w in dns]
    parts = ops.stream_experts(xp, T, choice, weight, gu_w, dn_w, inter, H)
    assert parts.shape == (top_k, T, H)
    want = torch.zeros(T, H, device=DEV)
    for e in range(E):
        w_e = torch.where(who == e, weight, torch.zeros_like(weight)).sum(-1)
        g, u = (x.float() @ gus[e].float().t()).chunk(2, dim=1)
        act = (torch.nn.functional.silu(g) * u).to(torch.bfloat16)
        y = act.float() @ dns[e].float().t()
        want += w_e[:, None] * y
    # activations may round to the other neighbour (2^-8 of a value)
    assert _rel(parts.sum(0), want) < 2.0 ** -8


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("D,T,pad", [(128, 1, 0), (64, 37, 8), (16, 9, 0),
                                     (128, 5, 3)])
def test_rope_append_pieces(dtype, D, T, pad):
    """16-byte pieces and, where a row stride is no multiple of them (pad 3),
    single values, against the reference; a slot of -1 stores nothing."""
    n_q, n_kv, PS, P = 6, 2, 16, 5
    gen = torch.Generator().manual_seed(D + T)
    width = (n_q + 2 * n_kv) * D + pad
    qkv = torch.randn(T, width, generator=gen).to(torch.bfloat16)
    pos = torch.randint(0, 90, (T,), generator=gen, dtype=torch.int32)
    slots = torch.randperm(P * PS, generator=gen)[:T]
    slots[T // 2] = -1
    cs = ref.make_cos_sin_table(96, D)

    def cut(x):
        q, k, v = x[:, :(n_q + 2 * n_kv) * D].split(
            [n_q * D, n_kv * D, n_kv * D], dim=1)
        return (q.unflatten(1, (n_q, D)), k.unflatten(1, (n_kv, D)),
                v.unflatten(1, (n_kv, D)))

    kc = torch.zeros(P, n_kv, D // 8, PS, 8, device=DEV).to(dtype)
    vc = torch.zeros(P, n_kv, PS, D, device=DEV).to(dtype)
    x = qkv.to(DEV)
    ops.rope_append(*cut(x), kc, vc, cs.to(DEV), pos.to(DEV), slots.to(DEV))
    q, k, v = cut(qkv.clone())
    q, k = q.clone(), k.clone()
    ref.rope_inplace(q, k, cs, pos)
    kr = torch.zeros(P, n_kv, D // 8, PS, 8).to(dtype)
    vr = torch.zeros(P, n_kv, PS, D).to(dtype)
    live = slots >= 0
    ref.kv_append(kr, vr, k[live], v[live], slots[live])
    # one rounding of products summed in fp32 (fp8: of the unrounded key,
    # where the reference rounds to bf16 first)
    step = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -3
    assert bool(((cut(x)[0].float().cpu() - q.float()).abs()
                 <= 2.0 ** -7 * q.float().abs() + 1e-6).all())
    assert bool(((kc.float().cpu() - kr.float()).abs()
                 <= step * kr.float().abs() + 2.0 ** -9).all())
    assert torch.equal(vc.float().cpu(), vr.float())


@pytest.mark.parametrize("T,E,top_k,H", [(65, 8, 2, 512), (1, 1, 1, 8),
                                         (257, 16, 4, 264), (1000, 3, 2, 64)])
def test_expert_rows(T, E, top_k, H):
    """Routing, expert order, gather and weighted return of a prompt's rows."""
    gen = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, H, generator=gen, device=DEV).to(torch.bfloat16)
    router = torch.randn(E, H, generator=gen, device=DEV).to(torch.bfloat16)
    weight, order, place, counts = ops.route_rows(x, router, top_k)
    top, who = torch.softmax(x.double() @ router.double().t(), -1).topk(
        top_k, -1)
    flat = who.reshape(-1)
    want = torch.sort(flat, stable=True).indices
    assert torch.equal(order.long(), want)
    assert torch.equal(place[want].long(), torch.arange(T * top_k,
                                                        device=DEV))
    assert torch.equal(counts.long(), torch.bincount(flat, minlength=E))
    # fp32 sums of logits of about H ** 0.5
    assert bool(((weight - top / top.sum(-1, keepdim=True)).abs()
                 <= 1e-5 * H ** 0.5 + 1e-5).all())
    rows = ops.gather_pairs(x, order, top_k)
    assert torch.equal(rows, x[want // top_k])
    y = torch.randn(T * top_k, H, generator=gen, device=DEV).to(torch.bfloat16)
    back = ops.return_pairs(y, place, weight)
    exp = (weight.double()[:, :, None]
           * y[place.long()].view(T, top_k, H).double()).sum(1)
    assert bool(((back.double() - exp).abs()
                 <= 2.0 ** -8 * exp.abs() + 1e-5).all())


def test_sorted_experts_are_the_gathered_ones():
    from agentainer_amd.models.mixtral import MIXTRAL_CONFIGS, MixtralMoE
    cfg = MIXTRAL_CONFIGS["tiny-mixtral"]
    torch.manual_seed(2)
    with torch.device(DEV), torch.no_grad():
        moe = MixtralMoE(cfg)
        for p in moe.parameters():
            p.normal_(0.0, 0.05)
        h = torch.randn(130, cfg.hidden_size, dtype=torch.bfloat16)
        out = moe(h)
        top, who = torch.softmax(h.double() @ moe.router.double().t(),
                                 -1).topk(cfg.top_k, -1)
        top = (top / top.sum(-1, keepdim=True)).float()
        want = moe._experts_sparse(h, who, top)
    assert _rel(out, want) < 2.0 ** -7  # both round gate, up and result


def test_sorted_experts_in_groups(monkeypatch):
    """Groups of experts: the same bits as all at once, and less memory
    between gate and down."""
    from agentainer_amd.models.mixtral import MIXTRAL_CONFIGS, MixtralMoE
    cfg = MIXTRAL_CONFIGS["tiny-mixtral"]
    torch.manual_seed(4)
    with torch.device(DEV), torch.no_grad():
        moe = MixtralMoE(cfg)
        for p in moe.parameters():
            p.normal_(0.0, 0.05)
        h = torch.randn(5000, cfg.hidden_size, dtype=torch.bfloat16)

        def peak():
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            base = torch.cuda.memory_allocated()
            out = moe(h)
            torch.cuda.synchronize()
            return out, torch.cuda.max_memory_allocated() - base

        moe(h)  # the library's workspaces
        out, used = peak()
        monkeypatch.setattr(MixtralMoE, "SORTED_PAIRS", 1 << 30)
        want, used_at_once = peak()
    assert torch.equal(out, want)
    # 3 * inter columns of bf16 for 10000 pairs against at most 4096 (or one
    # expert's, of four)
    assert used < used_at_once - 3 * cfg.intermediate_size * 2 * 2000


def test_experts_of_a_prompt_under_autograd():
    """With gradients recorded, 65 rows and more take the products that
    autograd accepts, as they did before the rows were sorted."""
    from agentainer_amd.models.mixtral import MIXTRAL_CONFIGS, MixtralMoE
    cfg = MIXTRAL_CONFIGS["tiny-mixtral"]
    torch.manual_seed(3)
    with torch.device(DEV):
        moe = MixtralMoE(cfg)
        with torch.no_grad():
            for p in moe.parameters():
                p.normal_(0.0, 0.05)
        h = torch.randn(70, cfg.hidden_size, dtype=torch.bfloat16)
    out = moe(h)
    assert out.requires_grad
    with torch.no_grad():
        want = moe(h)
    assert not want.requires_grad
    assert _rel(out, want) < 2.0 ** -7  # both round gate, up and result


def test_attention_rows_off_alignment():
    """Query rows and outputs two bytes off a 16-byte boundary, and a row
    stride that is no multiple of one: the same values as aligned ones."""
    n_q, n_kv, D, PS, lens = 8, 2, 128, 16, [40, 75, 9]
    kc, vc, table = _paged(lens, n_kv, D, PS, torch.bfloat16, seed=1)
    kc, vc, table = kc.to(DEV), vc.to(DEV), table.to(DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    B = len(lens)
    gen = torch.Generator(device=DEV).manual_seed(6)
    flat = torch.randn(B * (n_q * D + 3) + 1, generator=gen, device=DEV).to(
        torch.bfloat16)
    q = torch.as_strided(flat, (B, n_q, D), (n_q * D + 3, D, 1), 1)
    buf = torch.zeros(B * n_q * D + 1, dtype=torch.bfloat16, device=DEV)
    out, want = buf[1:].view(B, n_q, D), torch.zeros(B, n_q, D, device=DEV,
                                                     dtype=torch.bfloat16)
    ops.paged_decode_attention(out, q, kc, vc, table, sl, 0.1)
    ops.paged_decode_attention(want, q.contiguous(), kc, vc, table, sl, 0.1)
    assert torch.equal(out, want)
    starts = torch.arange(B, dtype=torch.int32, device=DEV)
    ones = torch.ones(B, dtype=torch.int32, device=DEV)
    args = (kc, vc, table, sl, starts, ones, 0.1)
    out.zero_()
    want.zero_()
    ops.paged_prefill_attention(out, q, *args, max_qlen=1)
    ops.paged_prefill_attention(want, q.contiguous(), *args, max_qlen=1)
    assert torch.equal(out, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n_q,n_kv,PS,lens,width", [
    (32, 8, 16, [1, 63, 64, 65, 511, 512, 513, 900], 0),  # chunks and runs
    (8, 8, 8, [70, 3], 0),
    (16, 8, 24, [255, 2], 64),
    (64, 8, 16, [300, 1], 0),
])
def test_fixed_decode_attention_edges(dtype, n_q, n_kv, PS, lens, width):
    D, B = 128, len(lens)
    kc, vc, table = _paged(lens, n_kv, D, PS, dtype, width, seed=n_q + PS)
    gen = torch.Generator().manual_seed(7)
    q = torch.randn(B, n_q, D, generator=gen).to(torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32)
    scale = 1.0 / math.sqrt(D)
    out = torch.zeros(B + 1, n_q, D, dtype=torch.bfloat16, device=DEV)
    ops.paged_decode_attention_fixed(out[:B], q.to(DEV), kc.to(DEV),
                                     vc.to(DEV), table.to(DEV), sl.to(DEV),
                                     scale)
    qr = q.float()
    if dtype != torch.bfloat16:  # queries in e4m3, one scale per head
        step = qr.abs().amax(-1, keepdim=True).clamp(min=1e-8) / 448.0
        qr = (qr * (1.0 / step)).to(torch.float8_e4m3fn).float() * step
    want = torch.zeros(B, n_q, D)
    ref.paged_decode_attention(want, qr, kc.float(), vc.float(), table, sl,
                               scale)
    # the result's own rounding, and fp32 sums of a few hundred terms
    err = (out[:B].float().cpu() - want).abs()
    vmax = float(vc.float().nan_to_num().abs().max())
    assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * vmax).all())
    assert not out[B].any()


def _decode_state(cfg, lens, kv_dtype, n_layers, seed, PS=16):
    """Caches, metadata and tokens of a decode step over `lens` cached
    tokens."""
    from agentainer_amd.models.llama import AttnMetadata
    caches = []
    for i in range(n_layers):
        kc, vc, table = _paged([n + 1 for n in lens], cfg.n_kv_heads,
                               cfg.head_dim, PS, torch.bfloat16, seed=seed)
        caches.append((kc.nan_to_num().to(kv_dtype).to(DEV),
                       vc.nan_to_num().to(kv_dtype).to(DEV)))
    pos = torch.tensor(lens, dtype=torch.int32)
    slots = torch.stack([table[b, n // PS].long() * PS + n % PS
                         for b, n in enumerate(lens)])
    md = AttnMetadata(page_table=table.to(DEV), seq_lens=(pos + 1).to(DEV),
                      slot_mapping=slots.to(DEV), positions=pos.to(DEV))
    gen = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, cfg.vocab_size, (len(lens),), generator=gen)
    return caches, md, ids.to(DEV)


@pytest.mark.parametrize("name,quant", [
    ("tiny-llama", "fp8"), ("tiny-llama", "mxfp4"),
    ("tiny-mixtral", "fp8"), ("tiny-mixtral", "mxfp4")])
@pytest.mark.parametrize("kv_dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("T", [1, 13, 64])
@torch.no_grad()
def test_quantized_decode_is_row_major(name, quant, kv_dtype, T):
    """A decode step over quantized weights is, bit for bit, the row-major
    chain of the single ops: its codes depend on every order of sums."""
    from agentainer_amd.models.llama import LLAMA_CONFIGS, LlamaForCausalLM
    from agentainer_amd.models.mixtral import (MIXTRAL_CONFIGS,
                                               MixtralForCausalLM)
    moe = name in MIXTRAL_CONFIGS
    cfg = (MIXTRAL_CONFIGS if moe else LLAMA_CONFIGS)[name]
    model = (MixtralForCausalLM if moe else LlamaForCausalLM)(cfg, DEV)
    if moe:
        model.pack_decode_weights(expert_fp8=quant == "fp8",
                                  expert_fp4=quant == "mxfp4")
    else:
        model.pack_decode_weights(dense_quant=quant)
    lens = [3 + 29 * i for i in range(T)]
    caches, md, ids = _decode_state(cfg, lens, kv_dtype, cfg.n_layers, T)
    copies = [(k.clone(), v.clone()) for k, v in caches]
    got = model(ids, md, caches)

    D, nq, nkv, eps = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads, cfg.norm_eps
    x = torch.nn.functional.embedding(ids, model.embed)
    res = None
    for layer, (kc, vc) in zip(model.layers, copies):
        h = torch.empty_like(x)
        if res is None:
            res = x.clone()
            ops.rmsnorm(h, x, layer.input_ln, eps)
        else:
            ops.fused_add_rmsnorm(h, x, res, layer.input_ln, eps)
        at = layer.attn
        qkv = (ops.linear(h, at.qkv_proj, at.qkv_packed) if moe
               else ops.linear_quant(h, at.qkv_q))
        q, k, v = qkv.split([nq * D, nkv * D, nkv * D], dim=1)
        q = q.unflatten(1, (nq, D))
        ops.rope_append(q, k.unflatten(1, (nkv, D)), v.unflatten(1, (nkv, D)),
                        kc, vc, model.cos_sin, md.positions, md.slot_mapping)
        o = torch.empty(T, nq, D, dtype=torch.bfloat16, device=DEV)
        ops.paged_decode_attention_fixed(o, q, kc, vc, md.page_table,
                                         md.seq_lens, at.scale)
        o = o.view(T, nq * D)
        x = (ops.linear(o, at.o_proj, at.o_packed) if moe
             else ops.linear_quant(o, at.o_q))
        h = torch.empty_like(x)
        ops.fused_add_rmsnorm(h, x, res, layer.post_ln, eps)
        if moe:
            x = layer.moe(h)
            continue
        gu = ops.linear_quant(h, layer.mlp.gate_up_q)
        inter = layer.mlp.inter
        act = torch.empty(T, inter, dtype=torch.bfloat16, device=DEV)
        ops.silu_mul(act, gu[:, :inter], gu[:, inter:])
        x = ops.linear_quant(act, layer.mlp.down_q)
    h = torch.empty_like(x)
    ops.fused_add_rmsnorm(h, x, res, model.final_ln, eps)
    want = ops.linear(h, model.lm_head, model.lm_head_packed)
    assert torch.equal(got, want)


def test_attention_outputs_of_other_sizes():
    """An output with more rows than q keeps them; one with fewer than q
    serves sequences that cover no more (prompts only)."""
    n_q, n_kv, D, PS, lens = 8, 2, 128, 16, [40, 75, 9]
    kc, vc, table = _paged(lens, n_kv, D, PS, torch.bfloat16, seed=2)
    kc, vc, table = kc.to(DEV), vc.to(DEV), table.to(DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    B = len(lens)
    gen = torch.Generator(device=DEV).manual_seed(6)
    q = torch.randn(B + 2, n_q, D, generator=gen, device=DEV).to(
        torch.bfloat16)
    new = lambda n: torch.full((n, n_q, D), 7.0, dtype=torch.bfloat16,  # noqa: E731
                               device=DEV)
    want, more = new(B), new(B + 3)
    ops.paged_decode_attention(want, q[:B], kc, vc, table, sl, 0.1)
    ops.paged_decode_attention(more, q[:B], kc, vc, table, sl, 0.1)
    assert torch.equal(more[:B], want) and bool((more[B:] == 7.0).all())
    with pytest.raises(RuntimeError):
        ops.paged_decode_attention(new(B - 1), q[:B], kc, vc, table, sl, 0.1)
    starts = torch.arange(B, dtype=torch.int32, device=DEV)
    ones = torch.ones(B, dtype=torch.int32, device=DEV)
    for tb in (table, torch.nn.functional.pad(table, (0, 64))):  # split runs
        args = (kc, vc, tb, sl, starts, ones, 0.1)
        want, more, fewer = new(B), new(B + 4), new(B)
        ops.paged_prefill_attention(want, q[:B], *args, max_qlen=1)
        ops.paged_prefill_attention(more, q[:B], *args, max_qlen=1)
        ops.paged_prefill_attention(fewer, q, *args, max_qlen=1)
        assert torch.equal(more[:B], want) and bool((more[B:] == 7.0).all())
        assert torch.equal(fewer, want)


@pytest.mark.parametrize("switch", ["SKINNY_DISABLED", "SKINNY_FORCED"])
@torch.no_grad()
def test_projection_switches_reach_the_whole_step(switch, monkeypatch):
    """The switches that choose a projection's kernel choose it for decode
    steps too: none of them streams then."""
    from agentainer_amd.models import llama
    cfg = llama.LLAMA_CONFIGS["tiny-llama"]
    model = llama.LlamaForCausalLM(cfg, DEV)
    model.pack_decode_weights()
    caches, md, ids = _decode_state(cfg, [9, 30, 2], torch.bfloat16,
                                    cfg.n_layers, 1)
    monkeypatch.setattr(ops, switch, True)
    streamed = []
    for name in ("stream_linear", "stream_parts", "stream_gate_up"):
        monkeypatch.setattr(ops, name, lambda *a, n=name, **k:
                            streamed.append(n))
    logits = model(ids, md, caches)
    assert logits.isfinite().all() and not streamed


def test_large_expert_batches_leave_the_graphs_on():
    """A decode batch of a mixture above the captured sizes runs eagerly, by
    itself: smaller ones are still captured, also after it."""
    from agentainer_amd.engine.llm import ModelInstance
    from agentainer_amd.models.mixtral import (MIXTRAL_CONFIGS,
                                               MixtralForCausalLM)
    cfg = MIXTRAL_CONFIGS["tiny-mixtral"]

    def step(graph):
        inst = ModelInstance("tiny-mixtral", cfg, DEV,
                             {"sync_mode": True, "kv_pool_tokens": 4096,
                              "graph_capture": graph},
                             model_cls=MixtralForCausalLM)
        ids = [("a%d" % i, [3 + i, 7, 11 + i]) for i in range(70)]
        inst.forward_step(ids, [[2]] * 70)
        large = inst.forward_step([(s, [5 + i]) for i, (s, _t)
                                   in enumerate(ids)], [[0]] * 70)
        large = large.clone()
        return inst, large, inst.forward_step([(s, [9]) for s, _t in ids[:3]],
                                              [[0]] * 3)

    inst, large, small = step(True)
    assert inst.use_graph
    assert inst._graphs[128]["graph"] is None
    assert inst._graphs[4]["graph"] is not None
    _plain, large0, small0 = step(False)
    assert torch.equal(large, large0) and torch.equal(small, small0)


def _prefill_state(cfg, specs, seed, PS=16):
    """Caches, metadata, tokens and last rows of a prompt step of (cached,
    new) tokens per sequence."""
    from agentainer_amd.models.llama import AttnMetadata
    lens = [c + n for c, n in specs]
    caches = []
    for i in range(cfg.n_layers):
        kc, vc, table = _paged(lens, cfg.n_kv_heads, cfg.head_dim, PS,
                               torch.bfloat16, seed=seed)
        caches.append((kc.nan_to_num().to(DEV), vc.nan_to_num().to(DEV)))
    pos = torch.cat([torch.arange(c, c + n) for c, n in specs])
    seq = torch.repeat_interleave(torch.arange(len(specs)),
                                  torch.tensor([n for _c, n in specs]))
    slots = table[seq, pos // PS].long() * PS + pos % PS
    i32 = dict(dtype=torch.int32, device=DEV)
    starts = [sum(n for _c, n in specs[:i]) for i in range(len(specs))]
    md = AttnMetadata(
        page_table=table.to(DEV), seq_lens=torch.tensor(lens, **i32),
        slot_mapping=slots.to(DEV), positions=pos.to(torch.int32).to(DEV),
        is_prefill=True, query_starts=torch.tensor(starts, **i32),
        query_lens=torch.tensor([n for _c, n in specs], **i32),
        max_qlen=max(n for _c, n in specs))
    gen = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, cfg.vocab_size, (len(pos),), generator=gen)
    last = torch.tensor([s + n - 1 for s, (_c, n) in zip(starts, specs)])
    return caches, md, ids.to(DEV), last.to(DEV)


@pytest.mark.parametrize("family,change", [
    ("llama", {}),
    ("llama", {"qkv_bias": True, "n_heads": 8, "n_kv_heads": 2}),
    ("llama", {"hidden_size": 96, "intermediate_size": 160,
               "vocab_size": 352}),
    # above 64 rows: gate and up by the library, the residual's parts streamed
    ("llama", {"hidden_size": 3072, "intermediate_size": 512}),
    # ... gate and up streamed, and the last projection
    ("llama", {"intermediate_size": 10240, "vocab_size": 20480}),
    # ... and the fused one
    ("llama", {"n_heads": 128, "n_kv_heads": 16, "hidden_size": 3072}),
    ("mixtral", {}),
    # a hidden size of whole fragments, but not of pairs of them
    ("mixtral", {"hidden_size": 96, "intermediate_size": 160}),
])
@pytest.mark.parametrize("T", [1, 17, 64, 65, 128])
@pytest.mark.parametrize("prompt", [False, True])
@torch.no_grad()
def test_streamed_forward_is_the_row_major_one(family, change, T, prompt):
    """The whole step over packed weights and rows against the same model's
    row-major forward."""
    from dataclasses import replace
    from agentainer_amd.models import llama, mixtral
    if family == "llama":
        cfg = replace(llama.LLAMA_CONFIGS["tiny-llama"], **change)
        model = llama.LlamaForCausalLM(cfg, DEV)
    else:
        cfg = replace(mixtral.MIXTRAL_CONFIGS["tiny-mixtral"], **change)
        model = mixtral.MixtralForCausalLM(cfg, DEV)
        # a clear choice of experts: bf16 and fp32 logits choose alike
        for layer in model.layers:
            layer.moe.router.normal_(0.0, 1.0)
    if cfg.qkv_bias:
        for layer in model.layers:
            layer.attn.qkv_bias.normal_(0.0, 0.5)
    model.pack_decode_weights()
    if prompt:
        specs = ([(40, T)] if T < 3 else
                 [(0, T // 3), (33, 1), (16, T - T // 3 - 1)])
        caches, md, ids, last = _prefill_state(cfg, specs, T)
    else:
        caches, md, ids = _decode_state(
            cfg, [5 + 7 * i for i in range(T)], torch.bfloat16, cfg.n_layers,
            T)
        last = None
    copies = [(k.clone(), v.clone()) for k, v in caches]
    streams = llama.can_stream(model, ids)
    assert streams == (T <= 64 or family == "llama" and (
        cfg.hidden_size >= 3072 or cfg.intermediate_size >= 10240))
    got = model(ids, md, caches, last)
    head, model.lm_head_packed = model.lm_head_packed, None
    assert not llama.can_stream(model, ids)
    want = model(ids, md, copies, last)
    assert got.shape == want.shape
    # some 20 bf16 roundings in a row in either, 2^-9 of a value each
    err = (got.float() - want.float()).norm(dim=1) / want.float().norm(dim=1)
    if family == "mixtral":  # a token near a tie may take another expert
        err = err.sort().values[:max(1, T * 9 // 10)]
    assert err.max().item() < 2.0 ** -5
    for (k0, v0), (k1, v1) in zip(caches, copies):
        assert _rel(k0, k1) < 2.0 ** -6 and _rel(v0, v1) < 2.0 ** -6


def _codes(x, kind):
    """What a row-quantized activation holds of bf16 rows x, in 64 bits."""
    top = 448.0 if kind == "fp8" else 6.0
    step = x.float().abs().amax(1, keepdim=True).clamp(min=1e-8) / top
    y = x.float() * (1.0 / step)
    if kind == "fp8":
        q = y.to(torch.float8_e4m3fn).double()
    else:
        grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0],
                            dtype=torch.float64)
        mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0])
        # a magnitude on a midpoint takes the larger code
        q = grid[torch.bucketize(y.abs(), mids, right=True)]
        q = torch.where(y < 0, -q, q)
    return q * step.double()


@pytest.mark.parametrize("kind", ["fp8", "mxfp4"])
@pytest.mark.parametrize("T", [1, 13, 64])
@torch.no_grad()
def test_quantized_experts_against_their_codes(kind, T):
    """A whole mixture layer against 64-bit products of the codes that its
    weights and activations are stored in."""
    from agentainer_amd.models.mixtral import (MIXTRAL_CONFIGS,
                                               MixtralForCausalLM)
    cfg = MIXTRAL_CONFIGS["tiny-mixtral"]
    model = MixtralForCausalLM(cfg, DEV)
    model.pack_decode_weights(expert_fp8=kind == "fp8",
                              expert_fp4=kind == "mxfp4")
    moe = model.layers[1].moe
    gen = torch.Generator().manual_seed(T)
    moe.router.copy_(torch.randn(moe.router.shape, generator=gen))
    h = torch.randn(T, cfg.hidden_size, generator=gen).to(torch.bfloat16)
    got = moe(h.to(DEV)).double().cpu()

    bf = lambda x: x.to(torch.bfloat16).double()  # noqa: E731
    def weight(w):
        N, K = w.shape
        if kind == "mxfp4":
            p, sc = ops.quantize_weight_mxfp4(w)
            return ops.dequantize_mxfp4(p, sc, N, K).double()
        p, sc = ops.quantize_weight_fp8(w)
        q = p.cpu().view(torch.float8_e4m3fn).double().view(
            N // 16, K // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(N, K)
        return q * sc.cpu().double()[:, None]

    # the layer's own bf16 logits: a step of one of them is 0.125
    logits = torch.nn.functional.linear(h.to(DEV), moe.router).double().cpu()
    top, who = torch.softmax(logits, -1).topk(cfg.top_k, -1)
    top = top / top.sum(-1, keepdim=True)
    want = torch.zeros(T, cfg.hidden_size, dtype=torch.float64)
    x = _codes(h, kind)
    for e in range(cfg.n_experts):
        g, u = bf(x @ weight(moe.gate_up[e]).t()).chunk(2, dim=1)
        act = (g / (1.0 + torch.exp(-g)) * u).to(torch.bfloat16)
        y = bf(_codes(act, kind) @ weight(moe.down[e]).t())
        want += torch.where(who == e, top, torch.zeros_like(top)).sum(
            -1, keepdim=True) * y
    # the result's rounding (2^-9), and one activation in some thousands that
    # rounds to the other neighbour and may change its code
    assert ((got - want).norm() / want.norm()).item() < 2.0 ** -7
