"""Projections of up to some two thousand rows in bf16 and 256 in f32 (``ops.gemm.project``) against float64: one launch and slices
of K, all tiles, part-filled ones, edges of the rule, strided rows, and the calls that keep the library's product."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import gemm as G

pytestmark = pytest.mark.gpu


def rows_config(M, N_, K, dtype=torch.bfloat16):
    from financial_chatbot_llm_amd.ops import _native as N
    plan = N.load().penny_linear_rows_plan(M, N_, K, dtype == torch.float32)
    return (plan & 255, plan >> 8 & 255, plan >> 16) if plan else None


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 33, 63, 64, 65, 96, 97, 160, 256, 400, 1000, 1024, 1500, 2048, 2049])
@pytest.mark.parametrize("N_,K", [(512, 64), (528, 128), (2048, 2048), (4096, 2048), (7216, 448), (2064, 3072), (10256, 192),
                                  (10240, 128), (1024, 4096), (1024, 1024), (5168, 1024), (2048, 4160), (500, 128), (512, 96)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_against_float64(dt, M, N_, K):
    g = torch.Generator().manual_seed(M + N_ + K)
    w = (torch.randn((N_, K), generator=g) * K ** -0.5).to(dt).cuda()
    rows = torch.randn((M, K + 24), generator=g).to(dt).cuda()
    e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
    for off in (0, 16, 3):                                   # 3: rows off the kernel's 16 bytes
        x = rows[:, off:off + K]
        y = G.project(x, w)
        want = x.double() @ w.double().t()
        assert y.is_contiguous() and y.shape == (M, N_) and y.dtype == dt
        # one rounding of the result (bf16: to eight significant bits); K f32 products of values of order K^-0.5
        assert ((y.double() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()


def test_every_tile():
    """Each tile and split that the launcher knows, with part-filled tiles on both sides."""
    from financial_chatbot_llm_amd.ops import _native as N
    g = torch.Generator().manual_seed(1)
    w32 = (torch.randn((528, 512), generator=g) * 512 ** -0.5).cuda()
    x32 = torch.randn((150, 512), generator=g).cuda()
    for f32, nf, mt in [(1, nf, mt) for nf, mt in ((2, 2), (2, 4), (4, 2), (2, 6))] + [(0, nf, mt) for nf, mt in ((2, 2), (2, 4), (4, 2), (2, 6), (4, 4), (2, 8), (4, 6), (8, 2), (4, 8), (8, 4), (8, 6), (4, 12), (8, 8))]:
        dt = torch.float32 if f32 else torch.bfloat16
        w, x = w32.to(dt), x32.to(dt)
        want = x.double() @ w.double().t()
        # one rounding of a bf16 result; the f32 sums of 512 products of sums of about 1, each rounded by 2^-24 of the sum so far
        bound = want.abs() * (2.0 ** -22 if f32 else 2.0 ** -8) + 2.0 ** -22 * 512 ** 0.5
        for S in (1, 2, 4, 8) if f32 else (1, 2, 4):
            for paired in (0, 1):
                y = torch.zeros((151, 528), dtype=dt, device="cuda")
                slabs = torch.empty((S, 150, 528), device="cuda") if S > 1 else None
                N.call("penny_linear_rows", N.ptr(x), 512, N.ptr(w), 512, N.ptr(y), 150, 528, N.ptr(slabs), S, nf, mt, f32, paired, N.stream())
                assert ((y[:150].double() - want).abs() <= bound).all(), (f32, nf, mt, S, paired)
                assert (y[150] == 0).all()
    with pytest.raises(RuntimeError):
        N.call("penny_linear_rows", N.ptr(x), 512, N.ptr(w), 512, N.ptr(y), 150, 528, None, 1, 2, 16, 0, 1, N.stream())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [1, 16, 33, 100, 256])
@pytest.mark.parametrize("N_,K", [(520, 64), (536, 512), (3208, 1024), (3112, 1024), (1032, 4096)])
def test_widths_in_eights(dt, M, N_, K):
    """The last sixteen of columns half filled: one launch, slices of K, and the slices left to the reader."""
    g = torch.Generator(device="cuda").manual_seed(M + N_)
    w = (torch.randn((N_, K), generator=g, device="cuda") * K ** -0.5).to(dt)
    x = torch.randn((M, K), generator=g, device="cuda").to(dt)
    want = x.double() @ w.double().t()
    e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
    assert rows_config(M, N_, K, dt) is not None or dt == torch.float32
    y = G.project(x, w)
    assert ((y.double() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()
    p = G.project(x, w, slabs=True)
    assert torch.equal(p.materialize() if isinstance(p, G.Slabs) else p, y)


@pytest.mark.parametrize("f32,nf,mt", [(1, 2, 2), (1, 2, 4), (1, 4, 2), (1, 2, 6), (0, 2, 2), (0, 2, 8), (0, 4, 4), (0, 8, 8), (0, 4, 12)])
def test_widths_in_eights_by_tile(f32, nf, mt):
    """The half-filled last sixteen in the native launch itself, whatever the rule of ``project`` says: tiles that end before, in and behind it, rows in one
    and several chunks, whole K and slices, which are also read as they are left; nothing is written behind the result."""
    from financial_chatbot_llm_amd.ops import _native as N
    g = torch.Generator(device="cuda").manual_seed(nf * 100 + mt)
    dt = torch.float32 if f32 else torch.bfloat16
    for N_, K in ((520, 512), (1032, 1024), (3208, 512)):
        w = (torch.randn((N_, K), generator=g, device="cuda") * K ** -0.5).to(dt)
        for M in (1, 16 * mt, 16 * mt + 1, 3 * 16 * mt - 5):
            x = torch.randn((M, K), generator=g, device="cuda").to(dt)
            want = x.double() @ w.double().t()
            bound = want.abs() * (2.0 ** -22 if f32 else 2.0 ** -8) + 2.0 ** -22 * K ** 0.5        # as in test_every_tile
            for S in (1, 2, 4):
                y = torch.full((M + 1, N_), 7.0, dtype=dt, device="cuda")
                slabs = torch.full((S + 1, M, N_), 7.0, device="cuda") if S > 1 else None
                for out in (y, None) if S > 1 else (y,):
                    N.call("penny_linear_rows", N.ptr(x), K, N.ptr(w), K, N.ptr(out), M, N_, N.ptr(slabs), S, nf, mt, f32, 1, N.stream())
                    if S > 1:
                        assert ((slabs[:S].double().sum(0) - want).abs() <= 2.0 ** -22 * (want.abs() + K ** 0.5)).all(), (N_, M, S)
                        assert (slabs[S] == 7).all()
                assert ((y[:M].double() - want).abs() <= bound).all() and (y[M] == 7).all(), (N_, M, S)


@pytest.mark.parametrize("M,N_,K,here", [(256, 1024, 1024, True), (257, 1024, 1024, True), (384, 1024, 64, True), (338, 520, 32, True), (385, 1024, 64, False),
                                         (338, 6144, 1024, False)])
def test_short_f32_products(M, N_, K, here, monkeypatch):
    """Around the rows up to which short f32 products stay here."""
    from financial_chatbot_llm_amd.ops import _native as N
    calls, call = [], N.call
    monkeypatch.setattr(N, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(M)
    w, x = torch.randn((N_, K), generator=g, device="cuda") * K ** -0.5, torch.randn((M, K), generator=g, device="cuda")
    y = G.project(x, w)
    assert bool(calls) is here
    want = x.double() @ w.double().t()
    assert ((y.double() - want).abs() <= want.abs() * 2.0 ** -20 + 2.0 ** -18 * K ** 0.5).all()


def test_rule():
    assert rows_config(64, 2048, 4096) == (2, 4, 4) and rows_config(64, 4096, 2048) == (2, 2, 1) and rows_config(1, 7216, 2048) == (2, 2, 1)
    assert rows_config(256, 2048, 2048) == (2, 4, 1) and rows_config(512, 1024, 1024) == (2, 4, 1)
    for M, N_, K in ((600, 4096, 2048), (700, 1024, 4096), (300, 12864, 2048), (2049, 512, 64), (1, 500, 128), (1, 504, 128), (1, 512, 96)):
        assert rows_config(M, N_, K) is None


def test_other_calls_keep_the_library():
    w = torch.randn((512, 128), device="cuda")
    x = torch.randn((3, 128), device="cuda")
    assert torch.equal(G.project(x.half(), w.half()), torch.nn.functional.linear(x.half(), w.half()))
    assert rows_config(257, 512, 128, torch.float32) is None
    wb, xb = w.bfloat16(), x.bfloat16()
    assert G.project(xb[None], wb).shape == (1, 3, 512) and G.project(xb[0], wb).shape == (512,)
    assert G.project(xb, wb.clone().requires_grad_()).requires_grad
    with pytest.raises(RuntimeError):
        G.project(xb, w)
    with pytest.raises(RuntimeError):
        G.project(xb[:, :64], wb)


@pytest.mark.parametrize("dt,M,N_,K,eager,graph", [
    (torch.bfloat16, 96, 32000, 1024, True, True), (torch.bfloat16, 128, 12864, 2048, True, False), (torch.bfloat16, 192, 2048, 4096, True, False),
    (torch.bfloat16, 192, 2048, 6144, True, True), (torch.bfloat16, 256, 7232, 2048, True, True), (torch.float32, 32, 3616, 1024, True, True),
    (torch.float32, 48, 3616, 1024, True, False), (torch.float32, 64, 2048, 1024, True, True), (torch.float32, 80, 1024, 1024, True, False),
    (torch.float32, 256, 2048, 32, True, True)])
def test_replayed(dt, M, N_, K, eager, graph, monkeypatch):
    """A step that a graph replays takes only the products that the device runs faster; its warm-up takes the same, other threads do not."""
    import threading
    from financial_chatbot_llm_amd.ops import _native as N
    calls = []
    call = N.call
    monkeypatch.setattr(N, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(M)
    w = (torch.randn((N_, K), generator=g, device="cuda") * K ** -0.5).to(dt)
    x = torch.randn((M, K), generator=g, device="cuda").to(dt)
    native = lambda f: (calls.clear(), f(), bool(calls))[2]                            # noqa: E731
    assert native(lambda: G.project(x, w)) is eager
    with G.replayed():
        assert native(lambda: G.project(x, w)) is graph
        other = []
        t = threading.Thread(target=lambda: other.append(native(lambda: G.project(x, w))))
        t.start()
        t.join()
        assert other == [eager]
        torch.cuda.synchronize()
        cg = torch.cuda.CUDAGraph()
        with torch.cuda.graph(cg):
            y = G.project(x, w)
        assert native(lambda: G.project(x, w)) is graph
    assert native(lambda: G.project(x, w)) is eager
    e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
    for i in range(3):
        x.copy_(torch.randn((M, K), generator=g, device="cuda"))
        cg.replay()
        want = x.double() @ w.double().t()
        assert ((y.double() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()


def test_the_runner_says_so(monkeypatch):
    """The engine's graphs, and the passes that warm them up, are made inside ``replayed``."""
    from financial_chatbot_llm_amd.engine.model_runner import ModelRunner
    seen = []
    monkeypatch.setattr(ModelRunner, "_static_step", lambda self, B, filtered: seen.append((B, filtered, getattr(G._REPLAYED, "on", False))))
    r = ModelRunner.__new__(ModelRunner)
    r._run_static(3)
    r._run_static(4, filtered=True)
    assert seen == [(3, False, True), (4, True, True)] and not getattr(G._REPLAYED, "on", False)


def test_transformed_calls():
    """The head of the layered decoders under vmap, forward mode, a trace and a tensor class; any product under autocast."""
    from types import SimpleNamespace
    from torch.autograd import forward_ad as fw
    from financial_chatbot_llm_amd.models.layered import LayeredDecoder
    g = torch.Generator(device="cuda").manual_seed(3)
    model = SimpleNamespace(head=torch.randn((512, 128), generator=g, device="cuda"))
    logits = lambda h: LayeredDecoder.logits(model, h)                                 # noqa: E731
    h, t = (torch.randn((3, 4, 128), generator=g, device="cuda") for _ in range(2))
    want = torch.nn.functional.linear(h, model.head)
    assert torch.allclose(torch.vmap(logits)(h), want, atol=1e-4)
    with fw.dual_level():
        y, dy = fw.unpack_dual(logits(fw.make_dual(h[0], t[0])))
    assert torch.allclose(y, want[0], atol=1e-4) and torch.allclose(dy, t[0] @ model.head.t(), atol=1e-4)
    y, dy = torch.func.jvp(logits, (h[0],), (t[0],))
    assert torch.allclose(dy, t[0] @ model.head.t(), atol=1e-4)
    traced = torch.jit.trace(logits, h[0], check_trace=False)
    assert torch.allclose(traced(h[1]), want[1], atol=1e-4)
    assert isinstance(logits(torch.nn.Parameter(h[0], requires_grad=False)), torch.Tensor) and logits(h[0]).dtype == torch.float32
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert logits(h[0]).dtype == torch.bfloat16


RING = [(64, 64, 4), (64, 128, 4), (128, 64, 2), (128, 96, 2), (128, 128, 2), (128, 160, 2), (128, 192, 2), (128, 256, 2), (256, 128, 1), (256, 160, 1)]


@pytest.mark.parametrize("tile", range(1, 11))
def test_ring_tiles(tile):
    """Each tile with less than one of it, whole ones and part-filled ones on both sides; K of one step, fewer than the ring's stages and more; strided
    rows; nothing written behind the result."""
    from financial_chatbot_llm_amd.ops import _native as N
    tn, tm, kg = RING[tile - 1]
    g = torch.Generator().manual_seed(tile)
    for M, N_ in ((1, 8), (tm, tn), (tm + 1, tn + 8), (9 * tm - 15, 2 * tn - 24), (3 * tm + 16, 5 * tn + 64)):
        for K in sorted({32 * max(kg, 2), 64 * max(kg, 2), 384, 1152}):
            x = torch.randn((M, K + 8), generator=g).bfloat16().cuda()[:, :K]
            w = (torch.randn((N_, K), generator=g) * K ** -0.5).bfloat16().cuda()
            y = torch.full((M + 1, N_), 7.0, dtype=torch.bfloat16, device="cuda")
            N.call("penny_linear_ring", N.ptr(x), K + 8, N.ptr(w), K, N.ptr(y), N_, None, 0, M, N_, tile, N.stream())
            want = x.double() @ w.double().t()
            # one rounding to eight significant bits; f32 sums of K products of values of order K^-0.5, as above
            assert ((y[:M].double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -18 * K ** 0.5).all(), (M, N_, K)
            assert (y[M] == 7).all()
            r = torch.randn((M, N_ + 16), generator=g).bfloat16().cuda()[:, :N_]
            want = (y[:M].float() + r.float()).bfloat16()           # added to the rounded product, in place
            N.call("penny_linear_ring", N.ptr(x), K + 8, N.ptr(w), K, N.ptr(r), N_ + 16, N.ptr(r), N_ + 16, M, N_, tile, N.stream())
            assert torch.equal(r, want)
    for bad in ((K + 4, 64, K), (K + 8, 60, K), (K + 8, 64, K - 32), (64, 64, K)):
        with pytest.raises(RuntimeError):
            N.call("penny_linear_ring", N.ptr(x), bad[0], N.ptr(w), bad[2], N.ptr(y), N_, None, 0, 1, bad[1], tile, N.stream())


def test_ring_rule():
    """One round of blocks, and the shortest: the streaming tiles and the library keep the rest."""
    from financial_chatbot_llm_amd.ops import _native as N
    plan = N.load().penny_linear_ring_plan
    assert plan(1188, 2048, 2048) == 4 and plan(400, 7216, 2048) == 5 and plan(300, 12288, 2048) > 0 and plan(2600, 2048, 2048) == 7
    assert plan(256, 2048, 2048) == plan(3073, 1024, 1024) == plan(1000, 12288, 2048) == plan(400, 2044, 2048) == plan(400, 2048, 2080) == 0
    assert plan(300, 512, 1024) == 0                                    # shorter on the streaming tiles
    for M in range(257, 3100, 61):
        for N_ in (512, 1000, 2048, 3208, 7216, 8192, 12864):
            for K in (64, 192, 1024, 6144):
                t = plan(M, N_, K)
                assert t == 0 or (-(-M // RING[t - 1][1]) * -(-N_ // RING[t - 1][0]) <= 256 and K % (32 * RING[t - 1][2]) == 0)


def test_ring_leaves_even_widths_in_large_tiles_to_the_library():
    from financial_chatbot_llm_amd.ops import _native as N
    ring, plan = N.load().penny_linear_ring_plan, N.load().penny_project_ring_plan
    assert plan(1600, 4096, 2048) == plan(2557, 4096, 2048) == plan(1300, 5120, 2048) == plan(2600, 2560, 1024) == 0
    assert ring(1600, 4096, 2048) == 8 and ring(2557, 4096, 2048) == 10 and ring(2600, 2560, 1024) == 9      # sums in place stay there
    assert plan(1600, 5168, 2048) == 10 and plan(2123, 2048, 64) == 9 and plan(1300, 4096, 2048) == 7
    for M in range(257, 3100, 61):
        for N_, K in ((512, 1024), (3592, 1024), (2048, 6144), (4096, 512)):
            assert plan(M, N_, K) == ring(M, N_, K) or (N_ % 256 == 0 and K >= 1024 and ring(M, N_, K) >= 8)


@pytest.mark.parametrize("M,N_,K", [(257, 3208, 1024), (400, 7216, 2048), (1188, 2048, 6144), (3072, 1024, 1024)])
def test_ring_projections(M, N_, K, monkeypatch):
    """Through ``project``, not-a-numbers and infinities where they belong; rows off the alignment and replays keep their paths."""
    from financial_chatbot_llm_amd.ops import _native as N
    calls = []
    call = N.call
    monkeypatch.setattr(N, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(M)
    w = (torch.randn((N_, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    rows = torch.randn((M, K + 8), generator=g, device="cuda").bfloat16()
    for off in (0, 8, 4):
        x = rows[:, off:off + K]
        x[5, 7], x[M - 1, K - 1] = float("nan"), float("inf")
        calls.clear()
        y, want = G.project(x, w), x.double() @ w.double().t()
        assert calls == (["penny_linear_ring"] if off % 8 == 0 else [])
        assert y[5].isnan().all() and torch.allclose(y[M - 1].double(), want[M - 1], equal_nan=True)
        y[5] = y[M - 1] = want[5] = want[M - 1] = 0
        assert ((y.double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -18 * K ** 0.5).all()
    with G.replayed():
        calls.clear()
        G.project(rows[:, :K], w)
        assert "penny_linear_ring" not in calls


@pytest.mark.parametrize("tile", range(1, 11))
def test_ring_slabs(tile):
    from financial_chatbot_llm_amd.ops import _native as N
    tn, tm, kg = RING[tile - 1]
    g = torch.Generator().manual_seed(tile)
    step = 64 if kg == 1 else 32 * kg
    for M, N_, S, n in ((1, 8, 1, 1), (tm + 5, tn + 40, 2, 1), (2 * tm + 16, 3 * tn - 8, 3, 7), (tm, tn, 4, 5)):
        K = S * n * step + (64 - S * n * step % 64) % 64
        K = K if K % (S * step) == 0 else S * n * step * 2
        x = torch.randn((M, K + 8), generator=g).bfloat16().cuda()[:, :K]
        w = (torch.randn((N_, K), generator=g) * K ** -0.5).bfloat16().cuda()
        P = G.ring_slabs(x, w, S, tile)
        want = torch.stack([a.double() @ b.double().t() for a, b in zip(x.chunk(S, 1), w.chunk(S, 1))])
        assert ((P.double() - want).abs() <= 2.0 ** -18 * K ** 0.5 * K ** -0.5 * K ** 0.5).all(), (M, N_, S, K)


@pytest.mark.parametrize("tile", range(3, 11))
@pytest.mark.parametrize("Hq,Hkv,qs", [(2, 1, 1.0), (5, 1, 0.13)])
def test_qkv_ring(tile, Hq, Hkv, qs):
    """Rotated queries and the paged caches of every tile that holds a head, against the torch path: part-filled tiles, a last half tile
    of heads, tokens without a slot."""
    from financial_chatbot_llm_amd.ops import _native as N
    tn, tm, kg = RING[tile - 1]
    g = torch.Generator().manual_seed(tile)
    K, N_ = 384, (Hq + 2 * Hkv) * 128
    for M in (1, tm, 2 * tm + 17):
        x, w = torch.randn((M, K + 8), generator=g).bfloat16(), (torch.randn((N_, K), generator=g) * K ** -0.5).bfloat16()
        f = torch.rand((300, 64), generator=g) * 6.28
        cs, pos, nb = torch.cat([f.cos(), f.sin()], 1), torch.randint(0, 300, (M,), generator=g).int(), M // 64 + 2
        slots = torch.randperm(nb * 64, generator=g)[:M].int()
        slots[M // 2] = -1
        kc, vc = (torch.zeros((nb, Hkv, 64 * 128), dtype=torch.bfloat16) for _ in range(2))
        dk, dv = kc.cuda(), vc.cuda()
        dx, dw, dc, dp, ds = x.cuda()[:, :K], w.cuda(), cs.cuda(), pos.cuda(), slots.cuda()
        q = torch.zeros((M + 1, Hq, 128), dtype=torch.bfloat16, device="cuda")
        N.call("penny_qkv_ring", N.ptr(dx), K + 8, N.ptr(dw), K, M, N.ptr(dp), N.ptr(dc), N.ptr(ds), N.ptr(q), N.ptr(dk), N.ptr(dv), Hq, Hkv,
               qs, tile, N.stream())
        want = G.prefill_qkv_rope(x[:, :K], w, pos, cs, slots, kc, vc, Hq, Hkv, qs)
        # a sum next to the middle of two bf16 values may be rounded either way: their spacing is up to 2^-7 of them.  That of each of
        # the pair that turns, and of the result
        turn = torch.cat([want.float()[..., :64], want.float()[..., 64:]], -1).view(M, Hq, 2, 64).norm(dim=2).repeat(1, 1, 2)
        assert ((q[:M].cpu().float() - want.float()).abs() <= 2.0 ** -7 * (1.5 * turn + want.float().abs()) + 1e-5).all()
        assert (q[M] == 0).all()
        assert ((dv.cpu().float() - vc.float()).abs() <= 2.0 ** -7 * vc.float().abs() + 1e-5).all()
        assert (dk.cpu().float() - kc.float()).norm() <= 2.0 ** -8 * kc.float().norm() and ((dk.cpu() == 0) == (kc == 0)).float().mean() > 0.999


def test_qkv_and_slabs_take_the_ring(monkeypatch):
    from financial_chatbot_llm_amd.ops import _native as N
    calls = []
    call = N.call
    monkeypatch.setattr(N, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(5)
    x, w = torch.randn((300, 14336), generator=g, device="cuda").bfloat16(), torch.randn((4096, 14336), generator=g, device="cuda").bfloat16()
    r = torch.randn((300, 4096), generator=g, device="cuda").bfloat16()
    P = G.linear(x, w, slabs=True, fuse_residual=r)
    assert calls == ["penny_ring_slabs"] and isinstance(P, G.Slabs) and P.P.shape == (4, 300, 4096)
    want = x.double() @ w.double().t()
    assert ((P.P.double().sum(0) - want).norm() / want.norm()) < 5e-6              # f32 sums of 14336 products
    calls.clear()
    x, r = (torch.randn((1300, n), generator=g, device="cuda").bfloat16() for n in (14336, 4096))
    before = r.clone()
    y = G.linear(x[:, :4096], w[:, :4096].contiguous(), slabs=True, fuse_residual=r)
    assert calls == ["penny_linear_ring"] and isinstance(y, G.ResidualSum) and y.t is r
    want = x[:, :4096].double() @ w[:, :4096].double().t()
    assert ((r.double() - before.double() - want).abs() <= 2.0 ** -7 * (want.abs() + before.double().abs()) + 1e-3).all()
    monkeypatch.setenv("PENNY_PREFILL_GEMM", "force")
    calls.clear()
    G.linear(x[:, :4096], w[:, :4096].contiguous(), slabs=True, fuse_residual=r)
    assert calls == ["penny_gemm_prefill"]


@pytest.mark.parametrize("M,ring", [(2049, True), (2560, True), (2561, False)])
def test_long_sums_take_the_ring_where_whole_tiles_leave_cus_idle(M, ring, monkeypatch):
    """4096 x 14336 with the residual sum: 129 - 160 tiles of 256 x 256 run on the ring instead, and the two agree."""
    from financial_chatbot_llm_amd.ops import _native as N
    calls = []
    call = N.call
    monkeypatch.setattr(N, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w, r = ((torch.randn(s, generator=g, device="cuda") * f).bfloat16() for s, f in (((M, 14336), 1.0), ((4096, 14336), 0.01), ((M, 4096), 1.0)))
    before = r.clone()
    G.linear(x, w, slabs=True, fuse_residual=r)
    assert calls == ["penny_linear_ring" if ring else "penny_gemm_prefill"]
    want = x.float() @ w.float().t()
    # the product and the sum are rounded to bf16 one after the other, half a step of at most 2^-7 each
    assert ((r.float() - before.float() - want).abs() <= 2.0 ** -7 * (want.abs() + before.float().abs()) + 1e-3).all()


@pytest.mark.parametrize("stride", [0, 8])
def test_rows_that_overlap_are_read_as_before(stride):
    """Rows of a stride below their length, of which prefill products take any multiple of eight: QKV, slabs and the sum in place."""
    M, K, N_ = 300, 4096, 4096
    g = torch.Generator(device="cuda").manual_seed(stride)
    x = torch.randn(M * 8 + K, generator=g, device="cuda").bfloat16().as_strided((M, K), (stride, 1))
    w = (torch.randn((N_, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    want = x.double() @ w.double().t()
    y = G.linear(x, w, slabs=True)
    y = y.P.double().sum(0) if isinstance(y, G.Slabs) else y.double()
    assert ((y - want).norm() / want.norm()) < 2.0 ** -8
    r = torch.randn((M, N_), generator=g, device="cuda").bfloat16()
    before = r.double()
    s = G.linear(x, w, fuse_residual=r)
    s = s.t.double() if isinstance(s, G.ResidualSum) else s.double() + before
    assert ((s - before - want).abs() <= 2.0 ** -7 * (want.abs() + before.abs()) + 1e-3).all()
    qkv = (torch.randn((6144, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    cos_sin = torch.cat([torch.ones(1, 64), torch.zeros(1, 64)], 1).cuda()
    none = torch.full((M,), -1, dtype=torch.int32, device="cuda")
    caches = [torch.zeros(1, 8, 64 * 128, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    q = G.prefill_qkv_rope(x, qkv, torch.zeros_like(none), cos_sin, none, *caches, 32, 8)
    want = x.double() @ qkv[:4096].double().t()
    assert ((q.view(M, 4096).double() - want).norm() / want.norm()) < 2.0 ** -7
