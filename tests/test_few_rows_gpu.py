"""Projections of one to four rows with their norm, SiLU or residual add (``ops.gemm.few_rows``) against float64 of the same
roundings, at both LDS sizes and part-filled threads, and the decoder's step of few rows against the general one."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import gemm as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("form,N_,K,norm", [("slab", 48, 512, True), ("slab", 96, 4096, True), ("slab", 32, 1536, True), ("add", 16, 512, False),
                                            ("add", 80, 4096, False), ("add", 48, 14336, False), ("silu", 32, 512, True),
                                            ("silu", 96, 2560, True), ("silu", 64, 4096, True)])
def test_against_float64(M, form, N_, K, norm):
    gen = torch.Generator().manual_seed(M + N_ + K)
    rnd = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16).cuda()          # noqa: E731
    x, w, res = rnd(M, K + 8)[:, :K], rnd(N_, K) * K ** -0.5, rnd(M, N_)
    nw = 1 + 0.1 * rnd(K) if norm else None
    h = x.double()
    if norm:
        h = (x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5)).bfloat16()
        h = (h.float() * nw.float()).bfloat16().double()
    want = h @ w.double().t()
    # a half unit of a norm that falls the other way moves a value of h by 2^-8 of it: a sum of K of them, few of which do
    tol = 2.0 ** -18 * K ** 0.5 + (2.0 ** -8 * 4 * K ** -0.5 * h.abs().max() if norm else 0.0)
    ulp = lambda t: t.abs() * 2.0 ** -8                                                # noqa: E731
    before = res.clone()
    y = G.few_rows(x, G.tile_weight(w), form, nw, 1e-5, residual=res)
    if form == "slab":
        assert y.P.shape == (1, M, N_) and ((y.P[0].double() - want).abs() <= tol + want.abs() * 2.0 ** -20).all()
    elif form == "add":
        assert y is res and ((y.double() - (before.double() + want)).abs() <= tol + ulp(want) + ulp(before.double() + want)).all()
    else:
        gate, up = (want.view(M, -1, 2, 16)[:, :, i].reshape(M, -1) for i in (0, 1))
        ref = gate * torch.sigmoid(gate) * up
        # gate, up, their unit and the product are each rounded once; the unit's slope is 1.1 at most
        bound = ulp(ref) * 2 + (ulp(gate) + tol) * 1.1 * up.abs() + (ulp(up) + tol) * gate.abs() + tol
        assert y.shape == (M, N_ // 2) and ((y.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("M,Hq,Hkv,K", [(1, 32, 8, 4096), (2, 3, 1, 512), (3, 8, 2, 1024), (4, 4, 4, 4096)])
def test_qkv_rope(M, Hq, Hkv, K):
    """The rotating, cache-writing form against the two launches that it stands for: a skipped slot, both ends of a page."""
    from financial_chatbot_llm_amd import ops
    gen = torch.Generator().manual_seed(M + K)
    x, w = (torch.randn(s, generator=gen).to(torch.bfloat16).cuda() for s in ((M, K), ((Hq + 2 * Hkv) * 128, K)))
    wt, nw, cs = G.tile_weight(w * K ** -0.5), torch.ones(K, device="cuda").bfloat16(), torch.randn((300, 128), generator=gen).cuda()
    pos = torch.tensor([0, 299, 64, 17][:M], dtype=torch.int32, device="cuda")
    slots = torch.tensor([64, 191, -1, 0][:M], dtype=torch.int32, device="cuda")
    caches = [torch.full((3, Hkv, 64 * 128), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(4)]
    q = G.few_qkv_rope(x, wt, nw, 1e-5, pos, cs, slots, caches[0], caches[1], Hq, Hkv)
    want = ops.rope_kv_write(G.few_rows(x, wt, "slab", nw, 1e-5), pos, cs, slots, caches[2], caches[3], Hq, Hkv, 128)
    for a, b in ((q, want), (caches[0], caches[2]), (caches[1], caches[3])):
        # the f32 sums of K differ in their order: another rounding to eight bits before the rotation and after it, of values up to the largest
        assert a.shape == b.shape and (a.float() - b.float()).abs().max() <= 4 * 2.0 ** -8 * b.float().abs().max()
        assert ((a == 7.0) == (b == 7.0)).float().mean() > 0.999            # the same places are written


def test_refused():
    x, wt = torch.zeros((2, 4096), device="cuda", dtype=torch.bfloat16), G.tile_weight(torch.zeros((64, 4096), device="cuda", dtype=torch.bfloat16))
    assert G.few_ok(4, wt, True) and not G.few_ok(5, wt, True) and not G.few_ok(1, None, False)
    assert not G.few_ok(1, torch.empty((4, 256, 64, 8), device="cuda", dtype=torch.bfloat16), True)       # a norm over 8192 columns
    with pytest.raises(RuntimeError):
        G.few_rows(torch.zeros((5, 4096), device="cuda", dtype=torch.bfloat16), wt, "slab", norm=x[0])
    with pytest.raises(RuntimeError):
        G.few_rows(x, wt, "slab")
    with pytest.raises(RuntimeError):
        G.few_rows(x, wt, "add", norm=x[0], residual=torch.zeros((2, 64), device="cuda", dtype=torch.bfloat16))


@pytest.mark.parametrize("T", [1, 3, 4])
def test_decoder_step(T, monkeypatch):
    """The same step through :meth:`forward_few` and through the general layers, from the same cache."""
    from financial_chatbot_llm_amd.models.common import AttentionMetadata, KVCache
    from financial_chatbot_llm_amd.models.configs import ModelConfig
    from financial_chatbot_llm_amd.models.llama import LlamaModel
    from financial_chatbot_llm_amd.ops.attention import DecodeWorkspace
    cfg = ModelConfig(name="few", arch="llama", vocab_size=512, hidden_size=1024, intermediate_size=2048, num_layers=2, num_heads=8,
                      num_kv_heads=2, head_dim=128, max_position=512)
    model = LlamaModel(cfg, device="cuda").init_random(3)
    assert not model.takes_few(T)                            # no streamed copies of these sizes
    model.wt = {n: G.tile_weight(w) for n, w in model.w.items() if n.endswith((".qkv", ".o", ".down", ".gate_up"))}
    assert model.takes_few(T) and not model.takes_few(5)
    pos = torch.full((T,), 70, dtype=torch.int32, device="cuda")
    ids = torch.arange(T, dtype=torch.int32, device="cuda") * 7
    bt = torch.arange(2 * T, dtype=torch.int32, device="cuda").view(T, 2)
    outs = []
    for few in (True, False):
        kv = KVCache(cfg.num_layers, 2 * T, 2, 128, device="cuda")
        for i in range(cfg.num_layers):
            for c in (kv.k(i), kv.v(i)):
                c.copy_(torch.randn(c.shape, generator=torch.Generator().manual_seed(i)).to(c.dtype))
        meta = AttentionMetadata(num_prefill_tokens=0, num_decode=T, slots=(bt[:, 1].long() * 64 + 6).to(torch.int32),
                                 ctx_lens_d=pos + 1, block_tables_d=bt, decode_ws=DecodeWorkspace.create(T, 8, 128, 512, "cuda"))
        monkeypatch.setattr(LlamaModel, "takes_few", lambda self, t, few=few: few)
        outs.append((model.forward(ids, pos, meta, kv).float(), kv.k(1).float(), kv.v(1).float()))
    for a, b in zip(*outs):
        # both round the same values to eight bits in a different order of f32 sums: at most a unit per layer of the largest
        assert (a - b).abs().max() <= 4 * 2.0 ** -8 * b.abs().max()


# The most rows of x that a block holds (7168 chunks of 16 bytes), and one step of K beyond
@pytest.mark.parametrize("M,K", [(1, 57344), (2, 28672), (3, 18944), (4, 14336)])
def test_widest_rows(M, K):
    gen = torch.Generator().manual_seed(K)
    rnd = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16).cuda()          # noqa: E731
    x, w = rnd(M, K + 512), rnd(32, K + 512) * K ** -0.5
    res = torch.zeros((M, 32), dtype=torch.bfloat16, device="cuda")
    wide = G.tile_weight(w)
    assert not G.few_ok(M, wide, False)
    with pytest.raises(RuntimeError):
        G.few_rows(x, wide, "add", residual=res)
    x, w = x[:, :K], w[:, :K].contiguous()
    wt = G.tile_weight(w)
    assert G.few_ok(M, wt, False)
    y, want = G.few_rows(x, wt, "add", residual=res), x.double() @ w.double().t()
    assert ((y.double() - want).abs() <= 2.0 ** -18 * K ** 0.5 + want.abs() * 2.0 ** -8).all()


def test_operands():
    """Rows and a norm off 16 bytes give the same as aligned ones; what does not fit the weight is refused before any launch."""
    gen = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16).cuda()          # noqa: E731
    K, Hq, Hkv = 512, 2, 1
    wt, x, nw, res = G.tile_weight(rnd(512, K)), rnd(3, K + 9), rnd(K + 3), rnd(3, 512)
    for xo in (x[:, 3:K + 3], x[:, 8:K + 8], rnd(K, 3).t()):
        assert torch.equal(G.few_rows(xo, wt, "slab", nw[3:]).P, G.few_rows(xo.contiguous().clone(), wt, "slab", nw[3:].clone()).P)
    xo, nw = x[:, :K].contiguous(), nw[:K].contiguous()
    for bad in (lambda: G.few_rows(x[:, :K - 32], wt, "slab", nw), lambda: G.few_rows(rnd(3, 2 * K), wt, "add", residual=res),
                lambda: G.few_rows(xo.float(), wt, "slab", nw), lambda: G.few_rows(xo, wt.float(), "slab", nw),
                lambda: G.few_rows(xo, wt, "silu", nw.float()), lambda: G.few_rows(xo, wt, "silu", nw[:-8]),
                lambda: G.few_rows(xo, wt, "add"), lambda: G.few_rows(xo, wt, "add", residual=res.float()),
                lambda: G.few_rows(xo, wt, "add", residual=res[:2]), lambda: G.few_rows(xo, wt, "add", residual=rnd(512, 3).t())):
        with pytest.raises(ValueError):
            bad()
    with pytest.raises(RuntimeError):                        # added in place: it cannot be cloned
        G.few_rows(xo, wt, "add", residual=rnd(3 * 516 + 1)[1:].view(3, 516)[:, :512])
    pos, cs, cache = torch.zeros(3, dtype=torch.int32, device="cuda"), torch.zeros((4, 128), device="cuda"), rnd(1, 1, 64 * 128)
    good = dict(x=xo, wt=wt, norm=nw, eps=1e-5, positions=pos, cos_sin=cs, slots=pos, k_cache=cache, v_cache=cache.clone(), Hq=Hq, Hkv=Hkv)
    assert G.few_qkv_rope(**good).shape == (3, Hq, 128)
    for k, v in dict(x=rnd(3, K - 32), norm=nw.float(), positions=pos.long(), slots=pos[:2], cos_sin=cs.half(), k_cache=cache.float(), Hq=3).items():
        with pytest.raises(ValueError):
            G.few_qkv_rope(**dict(good, **{k: v}))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("prompts,rows", [([(70, 3)], []), ([(0, 4)], []), ([(64, 1)], []), ([(127, 2)], [40]), ([(0, 1), (62, 2)], [130]), ([], [5, 64, 191])])
def test_decoder_step_of_prompts(D, prompts, rows, monkeypatch):
    """Heads that take the slab form and its rotation pass, and short prompts -- whole ones, tails behind a cached prefix and over a page's
    end -- alone and beside decoding rows, through :meth:`forward_few` and through the general layers."""
    from financial_chatbot_llm_amd.models.common import AttentionMetadata, KVCache
    from financial_chatbot_llm_amd.models.configs import ModelConfig
    from financial_chatbot_llm_amd.models.llama import LlamaModel
    from financial_chatbot_llm_amd.ops.attention import DecodeWorkspace
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")                  # noqa: E731
    cfg = ModelConfig(name="few", arch="llama", vocab_size=512, hidden_size=1024, intermediate_size=2048, num_layers=2, num_heads=1024 // D,
                      num_kv_heads=256 // D, head_dim=D, max_position=512)
    model = LlamaModel(cfg, device="cuda").init_random(4)
    model.wt = {n: G.tile_weight(w) for n, w in model.w.items() if n.endswith((".qkv", ".o", ".down", ".gate_up"))}
    segs = prompts + [(c, 1) for c in rows]
    T, tp, n = sum(k for _, k in segs), sum(k for _, k in prompts), len(prompts)
    assert model.takes_few(T)
    pos = [a + j for a, k in segs for j in range(k)]
    bt = torch.arange(4 * len(segs), dtype=torch.int32, device="cuda").view(len(segs), 4)
    slots = i32([(4 * i + (a + j) // 64) * 64 + (a + j) % 64 for i, (a, k) in enumerate(segs) for j in range(k)])
    meta = AttentionMetadata(slots=slots, num_prefill_tokens=tp, num_decode=len(rows), decode_ws=DecodeWorkspace.create(4, model.hq, D, 512, "cuda"))
    if prompts:
        meta.cu_q, meta.ctx_lens_p = i32([sum(k for _, k in prompts[:i]) for i in range(n + 1)]), i32([a + k for a, k in prompts])
        meta.block_tables_p, meta.max_q_len = bt[:n].contiguous(), max(k for _, k in prompts)
    if rows:
        meta.ctx_lens_d, meta.block_tables_d = i32([c + 1 for c in rows]), bt[n:].contiguous()
    outs = []
    for few in (True, False):
        kv = KVCache(cfg.num_layers, 4 * len(segs), model.hkv, D, device="cuda")
        for i in range(cfg.num_layers):
            for c in (kv.k(i), kv.v(i)):
                c.copy_(torch.randn(c.shape, generator=torch.Generator().manual_seed(i)).to(c.dtype))
        monkeypatch.setattr(LlamaModel, "takes_few", lambda self, t, few=few: few)
        outs.append((model.forward(i32(range(3, 3 + T)), i32(pos), meta, kv).float(), kv.k(0).float(), kv.k(1).float(), kv.v(1).float()))
    for a, b in zip(*outs):
        # both round the same values to eight bits in a different order of f32 sums: at most a unit per layer of the largest
        assert (a - b).abs().max() <= 4 * 2.0 ** -8 * b.abs().max()
