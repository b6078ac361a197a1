"""Windowed and latent attention in the LDS-DMA form: segment lengths, windows and head counts at the edges of its tiles,
with the rows behind each sequence's last token poisoned, against the f32 walk on the CPU."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import mixers as mx

pytestmark = pytest.mark.gpu

# (rows, context) of the segments
SINGLES = [(1, 1), (1, 64), (1, 65), (1, 300)]
RAGGED = [(17, 17), (1, 129), (0, 0), (65, 200), (64, 64)]
LONG = [(150, 700), (40, 64)]


def pages(segs, g):
    need = [(c + 63) // 64 for _, c in segs]
    perm = torch.randperm(sum(need), generator=g).int()
    bt = torch.zeros((len(segs), max(need) + 1), dtype=torch.int32)
    o = 0
    for i, n in enumerate(need):
        bt[i, :n] = perm[o:o + n]
        o += n
    cu = torch.tensor([0] + torch.tensor([n for n, _ in segs]).cumsum(0).tolist(), dtype=torch.int32)
    pos = torch.cat([torch.arange(c - n, c) for n, c in segs]).int()
    return cu, pos, bt, sum(need)


def rows(segs, bt, total, width, dt, g):
    """Cache rows; what lies behind a sequence's last token is NaN, as uninitialised memory may be."""
    cache = torch.full((total, 64, width), float("nan"), dtype=dt)
    for i, (_, c) in enumerate(segs):
        for j in range(c):
            cache[bt[i, j // 64], j % 64] = torch.randn(width, generator=g).to(dt)
    return cache


def check(got, want, dt, weights=0.0):
    # the result's rounding, the rounding of one-term weights, and 32 ulps of the f32 sums (values are within 5)
    e = 2.0 ** -9 if dt == torch.bfloat16 else 2.0 ** -24
    tol = want.abs() * 2 * e + 5 * (weights + 2.0 ** -19)
    bad = (got.float().cpu() - want).abs() > tol
    assert not bad.any() and torch.isfinite(got.float()).all(), (int(bad.sum()), float((got.float().cpu() - want).abs().max()))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("segs", [SINGLES, RAGGED, LONG], ids=["singles", "ragged", "long"])
@pytest.mark.parametrize("heads,opt", [((4, 4), {"window": 1}), ((6, 2), {"window": 63, "keep_first": 5}),
                                       ((70, 1), {"window": 64, "chunked": True, "sink": True}),
                                       ((16, 4), {"window": 1 << 40, "softcap": 7.0, "slopes": True, "gate": "elem"}),
                                       ((8, 1), {"window": 130, "keep_first": 70, "gate": "head", "sink": True})])
def test_window(dt, segs, heads, opt):
    g = torch.Generator().manual_seed(5)
    (H, G), D = heads, 128
    cu, pos, bt, total = pages(segs, g)
    T = int(cu[-1])
    cache = rows(segs, bt, total, G * 2 * D, dt, g)
    q = torch.randn((T, H * D + 8), generator=g).to(dt)
    opt = dict(opt)
    if opt.pop("sink", False):
        opt["sink"] = torch.randn(H, generator=g)
    if opt.pop("slopes", False):
        opt["slopes"] = torch.rand(H, generator=g) * 0.1
    kind = opt.pop("gate", None)
    if kind:
        opt["gate"] = torch.randn((T, H * D if kind == "elem" else H), generator=g).to(dt)
    longest = max(n for n, _ in segs)

    def run(f):
        o = {k: f(v) if torch.is_tensor(v) else v for k, v in opt.items()}
        return mx.window_attend(f(q)[:, :H * D], f(cache), f(cu), f(pos), f(bt), scale=D ** -0.5, max_len=longest, heads=H,
                                kv_heads=G, dim=D, vdim=D, **o)
    check(run(lambda t: t.cuda()), run(lambda t: t.float() if t.is_floating_point() else t), dt)


@pytest.mark.parametrize("segs", [SINGLES, RAGGED, LONG], ids=["singles", "ragged", "long"])
@pytest.mark.parametrize("H,Dr,window,exact", [(1, 32, 1, True), (32, 32, 65, False), (70, 0, 1 << 40, True), (3, 0, 64, False)])
def test_latent(segs, H, Dr, window, exact):
    g = torch.Generator().manual_seed(6)
    dt, R = torch.bfloat16, 256
    cu, pos, bt, total = pages(segs, g)
    T = int(cu[-1])
    cache = rows(segs, bt, total, R + Dr, dt, g)
    ql, qr = (torch.randn((T, H, n), generator=g).to(dt) for n in (R, Dr))
    gate, sink = torch.randn((T, H), generator=g).to(dt), torch.randn(H, generator=g)

    def run(f):
        return mx.latent_attend(f(ql), f(qr), f(cache), f(cu), f(pos), f(bt), window, R ** -0.5, max(n for n, _ in segs),
                                gate=f(gate), sink=f(sink), exact_weights=exact)
    check(run(lambda t: t.cuda()), run(lambda t: t.float() if t.is_floating_point() else t), dt, 0.0 if exact else 2.0 ** -9)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,opt", [((4, 4), {"window": 1 << 40}), ((6, 2), {"window": 40, "keep_first": 3}),
                                       ((16, 4), {"window": 64, "chunked": True, "softcap": 5.0, "slopes": True, "sink": True})])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_window_not_finite(dt, heads, opt, bad):
    """A key or value that is not finite reaches the rows that see its token and no others."""
    g = torch.Generator().manual_seed(9)
    (H, G), D = heads, 128
    segs = [(150, 150), (1, 130), (40, 100)]
    cu, pos, bt, total = pages(segs, g)
    cache = rows(segs, bt, total, G * 2 * D, dt, g)
    q = torch.randn((int(cu[-1]), H * D), generator=g).to(dt)
    opt = dict(opt)
    if opt.pop("sink", False):
        opt["sink"] = torch.randn(H, generator=g)
    if opt.pop("slopes", False):
        opt["slopes"] = torch.rand(H, generator=g) * 0.1

    def run(f, cache):
        o = {k: f(v) if torch.is_tensor(v) else v for k, v in opt.items()}
        return mx.window_attend(f(q), f(cache), f(cu), f(pos), f(bt), scale=D ** -0.5, max_len=150, heads=H, kv_heads=G, dim=D,
                                vdim=D, **o)
    want = run(lambda t: t.float() if t.is_floating_point() else t, cache)
    token = [101, 37, 75]                                             # one of every segment
    sees = torch.zeros(int(cu[-1]), dtype=torch.bool)
    for i, j in enumerate(token):
        for r in range(int(cu[i]), int(cu[i + 1])):
            p = int(pos[r])
            low = p // opt["window"] * opt["window"] if opt.get("chunked") else p - opt["window"] + 1
            sees[r] = j <= p and (j >= low or j < opt.get("keep_first", 0))
        cache[bt[i, j // 64], j % 64, G * D + 5::D] = bad             # a value of every key head
        cache[bt[i, j // 64], j % 64, :G * D:D] = bad if i == 2 else 0.5
    got = run(lambda t: t.cuda(), cache).cpu()
    check(got[~sees], want[~sees], dt)
    assert not torch.isfinite(got[sees].float().view(-1, H, D)[:, :, 5]).any() and 0 < int(sees.sum()) < len(sees)


def test_latent_not_finite():
    g = torch.Generator().manual_seed(10)
    dt, R, Dr, H = torch.bfloat16, 256, 32, 3
    segs = [(100, 130), (1, 70)]
    cu, pos, bt, total = pages(segs, g)
    cache = rows(segs, bt, total, R + Dr, dt, g)
    ql, qr = (torch.randn((101, H, n), generator=g).to(dt) for n in (R, Dr))

    def run(f, cache):
        return mx.latent_attend(f(ql), f(qr), f(cache), f(cu), f(pos), f(bt), 50, R ** -0.5, 100)
    want = run(lambda t: t.float() if t.is_floating_point() else t, cache)
    cache[bt[0, 1], 90 - 64, 7] = float("nan")                        # token 90 of the first segment
    cache[bt[1, 0], 3, 7] = float("inf")                              # left the window long ago
    sees = torch.cat([(pos[:100] >= 90) & (pos[:100] < 140), torch.zeros(1, dtype=torch.bool)])
    got = run(lambda t: t.cuda(), cache).cpu()
    check(got[~sees], want[~sees], dt, 2.0 ** -9)
    assert not torch.isfinite(got[sees].float()).any()


def test_parts_follow_the_walk():
    """Steps of which each split was measured faster: (rows, context) of the segments, 16 heads over 4, window 1 << 30."""
    bf, f32 = torch.bfloat16, torch.float32

    def parts(segs, dt):
        T, S, longest, pages_ = sum(n for n, _ in segs), len(segs), max(n for n, _ in segs), max((c + 63) // 64 for _, c in segs)
        blocks = S * 4 if longest == 1 else (S + T * 4 // 64) * 4
        return mx._key_parts(pages_ * 64, blocks, 1024 if longest == 1 else 512, T * 16, 128, dt)
    for segs in ([(100, 100)] * 8, [(100, 100)], [(512, 512)], [(1000, 1000)], [(40, 40)] * 16, [(1, 100)] * 8):
        assert parts(segs, bf) == 1, segs
    assert parts([(100, 100)] * 8, f32) == parts([(33, 33)], f32) == 1
    assert parts([(300, 900)] + [(1, 700)] * 30, bf) == parts([(1, 100)], f32) == 2
    assert 3 <= parts([(64, 900)], bf) <= 6 and 4 <= parts([(1, 1000)], bf) <= 8 and parts([(64, 900)], f32) >= 6


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("nsplit", [1, 2, 5, 16])
def test_any_number_of_parts(dt, nsplit, monkeypatch):
    """More parts than a row has tiles among them: those are empty."""
    monkeypatch.setattr(mx, "_key_parts", lambda *a: nsplit)
    test_window(dt, LONG, (6, 2), {"window": 63, "keep_first": 5})
    test_window(dt, SINGLES, (8, 1), {"window": 130, "keep_first": 70, "gate": "head", "sink": True})


@pytest.mark.parametrize("nsplit", [63, 64, 65, 128, 150])
def test_more_parts_than_lanes(nsplit, monkeypatch):
    """A merging wave reads the statistics of 64 parts at a time: up to 150 parts, with and without keys of their own, in every group of 64."""
    monkeypatch.setattr(mx, "_key_parts", lambda *a: nsplit)
    segs = [(1, 6000), (2, 70), (1, 4500)]
    test_window(torch.float32, segs, (4, 2), {"window": 1 << 40, "gate": "head", "sink": True})
    test_window(torch.bfloat16, segs, (4, 4), {"window": 5000, "slopes": True, "gate": "elem"})
    test_latent_f32(segs, 8, 32, 1 << 40)


@pytest.mark.parametrize("segs", [SINGLES, RAGGED, LONG], ids=["singles", "ragged", "long"])
@pytest.mark.parametrize("H,Dr,window", [(1, 32, 1), (8, 32, 1024), (70, 0, 1 << 40), (3, 0, 64), (32, 32, 65)])
def test_latent_f32(segs, H, Dr, window):
    g = torch.Generator().manual_seed(16)
    dt, R = torch.float32, 256
    cu, pos, bt, total = pages(segs, g)
    T = int(cu[-1])
    cache = rows(segs, bt, total, R + Dr, dt, g)
    ql, qr = (torch.randn((T, H, n), generator=g).to(dt) for n in (R, Dr))
    gate, sink = torch.randn((T, H), generator=g), torch.randn(H, generator=g)

    def run(f):
        return mx.latent_attend(f(ql), f(qr), f(cache), f(cu), f(pos), f(bt), window, R ** -0.5, max(n for n, _ in segs),
                                gate=f(gate), sink=f(sink) if H > 1 else None)
    check(run(lambda t: t.cuda()), run(lambda t: t), dt)
