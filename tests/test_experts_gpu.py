"""Grouped expert products (``ops.mixers.experts``) against a float64 loop over the experts: both storage types, every
unit, both kernel forms with the edges of their tiles, ragged buckets, identity experts, widths in no whole 16 bytes."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

LIMIT, ALPHA = 1.3, 1.702


def unit64(name, g, u, s):
    if name == "clamped":
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        return g * torch.sigmoid(ALPHA * g) * (u + 1.0)
    if name == "relu2":
        return torch.relu(g) ** 2
    return (F.silu(s * g) if name == "silu" else F.gelu(s * g, approximate="tanh")) * (s * u)


def check(dtype, T, W, F_, E, top, unit, ident=0, skew=False, strided=False):
    from financial_chatbot_llm_amd.ops import mixers as mx
    gen = torch.Generator().manual_seed(T * 131 + W)
    rnd = lambda *s: torch.randn(s, generator=gen)  # noqa: E731
    gated = unit != "relu2"
    first = [[rnd(F_, W) * W ** -0.5 for _ in range(2 if gated else 1)] for _ in range(E)]
    second = [rnd(W, F_) * F_ ** -0.5 for _ in range(E)]
    z = rnd(T, E + ident)
    if skew:                              # most rows want the same few experts
        z[:, :2] += 4.0
    idx = z.topk(top, -1).indices.to(torch.int32)
    scale = torch.rand(T, top, generator=gen) if unit in ("silu", "gelu_tanh") else None
    h = rnd(T, W)
    dev = lambda t: t.to("cuda", dtype)  # noqa: E731
    hd = dev(torch.cat([h, rnd(T, 24)], 1))[:, :W] if strided else dev(h)
    w1 = mx.pack_experts([tuple(dev(m) for m in ms) if gated else dev(ms[0]) for ms in first], dtype)
    w2 = mx.pack_experts([dev(m) for m in second], dtype)
    ys, pos = mx.experts(hd, idx.cuda(), w1, w2, unit, LIMIT, ALPHA, scale.cuda() if scale is not None else None)
    again, pos2 = mx.experts(hd, idx.cuda(), w1, w2, unit, LIMIT, ALPHA, scale.cuda() if scale is not None else None)
    ys, pos = ys.double().cpu(), pos.cpu().long()
    rows = [(t, k) for t in range(T) for k in range(top) if idx[t, k] < E]
    at = torch.tensor([int(pos[t, k]) for t, k in rows], dtype=torch.int64)
    assert len(set(at.tolist())) == len(rows) and (not rows or int(at.max()) == len(rows) - 1)
    assert torch.equal(pos, pos2.cpu().long()) and torch.equal(ys[:len(rows)], again.double().cpu()[:len(rows)])
    h64 = hd.double().cpu()
    q = lambda m: m.to(dtype).double()  # noqa: E731
    want = torch.zeros(len(rows), W, dtype=torch.float64)
    which = torch.tensor([int(idx[t, k]) for t, k in rows])
    for e in set(which.tolist()):
        i = (which == e).nonzero().flatten()
        x = h64[[rows[j][0] for j in i.tolist()]]
        s = torch.tensor([float(scale[rows[j]]) for j in i.tolist()], dtype=torch.float64)[:, None] if scale is not None else 1.0
        g = x @ q(first[e][0]).T
        u = x @ q(first[e][1]).T if gated else None
        want[i] = unit64(unit, g, u, s) @ q(second[e]).T
    if not rows:
        return
    # bf16: the unit's result and the output are rounded once each (2^-9 of a value); f32: sums of W and F terms
    tol = 6e-3 if dtype == torch.bfloat16 else 3e-6
    assert float((ys[at] - want).norm() / want.norm()) < tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,F_,E,top,unit", [
    (1, 256, 128, 4, 2, "clamped"),        # stream form
    (3, 160, 56, 7, 3, "clamped"),         # K and columns in no whole 128 bytes / 16 rows
    (24, 192, 48, 6, 3, "silu"),           # 12 rows on average: the last of bf16's stream form
    (26, 192, 48, 6, 3, "silu"),           # ... and the first of its 64-row tiles
    (50, 192, 48, 6, 3, "relu2"),          # 25: f32's first
    (40, 1056, 544, 32, 4, "clamped"),     # many narrow tiles, the wide stream block
    (64, 1024, 512, 32, 4, "relu2"),
    (140, 160, 72, 5, 2, "relu2"),         # 56: the last of bf16's 64-row tiles
    (143, 160, 72, 5, 2, "gelu_tanh"),     # 57: the first of 128
    (700, 256, 264, 6, 2, "clamped"),      # a column block beyond the last group
    (33, 192, 128, 1, 1, "silu"),          # one expert, three groups of 16 tokens with rows
    (49, 128, 64, 1, 1, "relu2"),          # four, fewer stages of K than the ring holds
    (65, 192, 128, 1, 1, "clamped"),       # one row in the second tile
    (145, 192, 128, 1, 1, "silu"),         # bf16's second tile of 128: an odd number of groups
    (3072, 2048, 64, 1, 1, "clamped"),     # f32's second product in blocks of four row groups ...
    (2900, 2048, 64, 1, 1, "clamped"),     # ... and of eight
    (320, 256, 1024, 8, 2, "silu"),        # f32's first product in blocks of eight
    (515, 192, 128, 2, 2, "silu"),
])
def test_experts_against_float64(dtype, T, W, F_, E, top, unit):
    check(dtype, T, W, F_, E, top, unit)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kw", [dict(ident=3), dict(skew=True), dict(strided=True), dict(ident=60, top=1, T=2)])
def test_experts_identity_skewed_and_strided_rows(dtype, kw):
    a = dict(T=210, W=256, F_=96, E=8, top=4, unit="clamped")
    check(dtype, **{**a, **kw})


@pytest.mark.parametrize("W,F_", [(37, 19), (130, 33)])
def test_experts_widths_in_no_whole_accesses(W, F_):
    for dtype in (torch.bfloat16, torch.float32):
        check(dtype, 21, W, F_, 5, 2, "clamped")
        check(dtype, 600, W, F_, 5, 2, "relu2")


def test_experts_many_experts():
    check(torch.bfloat16, 50, 64, 16, 700, 5, "silu")


@pytest.mark.parametrize("T", [127, 1025, 8200, 16500])
def test_expert_plan_run_lengths(T):
    """The sort's forms by the length of a wave's run (2, 8, 16 and 32 chunks in registers, a loop beyond)."""
    for top in (1, 2):
        check(torch.bfloat16, T, 16, 16, 5, top, "relu2", ident=1)


@pytest.mark.parametrize("E", [8184, 8185, 8192])
def test_most_experts(E):
    """As many as the routing kernels choose from; few pairs, and more than a wave's run of them."""
    check(torch.float32, 40, 8, 8, E, 3, "relu2")
    check(torch.float32, 900, 8, 8, E, 2, "relu2", skew=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,F_,E,top,unit", [
    (100, 512, 1024, 2, 1, "relu2"),       # few experts: tiles of 16 rows far beyond the average from which many take 64
    (130, 2048, 520, 3, 2, "clamped"),
    (700, 512, 1024, 2, 1, "silu"),        # ... and past the line
])
def test_few_experts(dtype, T, W, F_, E, top, unit):
    check(dtype, T, W, F_, E, top, unit)


@pytest.mark.parametrize("T,skew", [(2048, False), (1905, True)])
def test_tiles_of_192(T, skew):
    """Even shares of an expert's rows in one and two tiles of 192, and of thousands of rows beside experts of a few."""
    from financial_chatbot_llm_amd.ops import _native as N
    assert N.load_mixers().mx_experts_tile(T * 4, 32, 0, 64, 32, 64, 16, 1) == 192
    check(torch.bfloat16, T, 1024, 512, 32, 4, "clamped", skew=skew)


def test_tile_rule():
    """Few rows per expert on average keep tiles of 64 whatever the estimate says of even buckets."""
    from financial_chatbot_llm_amd.ops import _native as N
    tile = lambda T, top, E, W, F_: N.load_mixers().mx_experts_tile(T * top, E, 0, F_ // 8, W // 32, W // 16, F_ // 32, 1)     # noqa: E731
    assert [tile(T, 6, 64, 1024, 512) for T in (100, 200, 300, 600, 1000)] == [16, 64, 64, 64, 128]
    assert tile(300, 4, 32, 2048, 1024) == 64 and tile(1100, 4, 32, 2048, 1024) == 128 and tile(5065, 4, 32, 2048, 1024) == 256


@pytest.mark.parametrize("E", [1, 3, 64, 65, 512, 513])
@pytest.mark.parametrize("T", [256, 257, 1023, 1025, 2049, 4097, 8192, 8193])
def test_expert_plan_is_the_stable_sort(E, T):
    """One block (more than 512 experts, or 1024 pairs and fewer) and a block per expert (beyond 32768 pairs in a loop): every pair's place is that of the
    stable sort by expert, identity experts behind; some experts get no pair, one may get nearly all."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    top, W = 4, 8
    g = torch.Generator().manual_seed(T + E)
    for skew in (False, True):
        idx = torch.randint(0, E + 2, (T, top), generator=g)
        if skew:
            idx = torch.where(torch.rand(T, top, generator=g) < 0.9, E // 2, idx)
        w1 = mx.pack_experts([torch.ones(8, W, device="cuda")] * E, torch.float32)
        w2 = mx.pack_experts([torch.ones(W, 8, device="cuda")] * E, torch.float32)
        _, pos = mx.experts(torch.ones(T, W, device="cuda"), idx.int().cuda(), w1, w2, "relu2")
        flat = idx.flatten()
        want = torch.empty(T * top, dtype=torch.int32)
        want[torch.argsort(flat, stable=True)] = torch.arange(T * top, dtype=torch.int32)
        assert torch.equal(pos.cpu().flatten(), torch.where(flat < E, want, 0))


@pytest.mark.parametrize("T,W,F_,E,top,unit,kw", [
    (1700, 2048, 1024, 8, 3, "clamped", {}),             # 637 rows on average: tiles of 256 rows, the last one of half the experts small
    (1600, 2112, 1088, 8, 3, "silu", {"skew": True}),    # an odd number of K tiles; two experts with most of the rows
    (1700, 2048, 1088, 8, 3, "gelu_tanh", {"strided": True, "ident": 1}),      # a column block beyond the last group
    (4000, 768, 1024, 16, 4, "relu2", {"ident": 2}),
    (1700, 2056, 1024, 8, 3, "clamped", {}),             # rows in no whole K tile: 128 tokens
    (300, 256, 136, 64, 6, "silu", {"skew": True}),      # tiles of 64: one and more whole rounds of groups over the XCDs and a rest
    (700, 256, 136, 60, 6, "clamped", {}),
])
def test_experts_of_many_rows(T, W, F_, E, top, unit, kw):
    check(torch.bfloat16, T, W, F_, E, top, unit, **kw)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,E,top,ident,skew", [(1, 64, 1, 0, False), (256, 64, 4, 0, False), (341, 64, 3, 5, True), (342, 64, 3, 0, True), (256, 65, 4, 0, False),
                                                (17, 2, 1, 0, False), (64, 33, 1, 31, True)])
def test_blocks_that_plan_for_themselves(dtype, T, E, top, ident, skew):
    """Around 1024 pairs and 64 experts, beyond which the plan is a launch: buckets of one tile, of several and empty ones, identity entries."""
    check(dtype, T, 256, 64, E, top, "clamped", ident=ident, skew=skew)
    check(dtype, T, 256, 64, E, top, "silu", ident=ident, skew=skew)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_do_not_depend_on_the_step(dtype):
    """A token's expert rows alone and among 64 tokens, both in the stream form: the same bits."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    T, E, W, F_, top = 64, 32, 1024, 512, 4
    g = torch.Generator().manual_seed(2)
    w1 = mx.pack_experts([tuple((torch.randn(F_, W, generator=g) * W ** -0.5).to("cuda", dtype) for _ in range(2)) for _ in range(E)], dtype)
    w2 = mx.pack_experts([(torch.randn(W, F_, generator=g) * F_ ** -0.5).to("cuda", dtype) for _ in range(E)], dtype)
    h, idx = torch.randn(T, W, generator=g).to("cuda", dtype), torch.rand(T, E, generator=g).topk(top, -1).indices.int().cuda()
    ys, pos = mx.experts(h, idx, w1, w2, "clamped", LIMIT, ALPHA)
    for t in (0, 17, 63):
        y1, p1 = mx.experts(h[t:t + 1], idx[t:t + 1].contiguous(), w1, w2, "clamped", LIMIT, ALPHA)
        assert torch.equal(ys[pos[t].long()], y1[p1[0].long()])
