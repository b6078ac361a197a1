"""Encoder projections on the LDS ring's tiles (``penny_bias_rows_plan``): every tile it chooses, part-filled ones, strided rows, the
edges of the rule, and the native walk of longer batches against the calls that it stands for."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("M", [33, 64, 65, 97, 192, 193, 257, 385, 500, 769, 1024, 1025, 1365, 1500, 2048])
@pytest.mark.parametrize("N,K", [(2304, 768), (768, 768), (768, 3072), (3072, 768), (1152, 384), (4096, 1024), (1040, 64), (48, 192)])
def test_against_float64(M, N, K, gelu):
    from financial_chatbot_llm_amd.ops import _native as nat, gemm
    assert (nat.load().penny_bias_rows_plan(M, N, K) > 0) <= (M <= 2048 if N % 256 == 0 else M <= 1024)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g, device="cuda").to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    got = gemm.linear_bias(x, w, b, gelu).double()
    want = x.double() @ w.double().T + b.double()
    e = want.abs() * 2.0 ** -8 + 2.0 ** -18 * K ** 0.5                  # one rounding to eight bits; K f32 products
    if gelu:
        want = F.gelu(want)
        e = 1.13 * e + want.abs() * 2.0 ** -8 + 2.0 ** -18              # through a slope of 1.13 at most, and rounded again
    assert ((got - want).abs() <= e).all()


def test_every_tile():
    from financial_chatbot_llm_amd.ops import _native as nat
    seen = {nat.load().penny_bias_rows_plan(M, N, 768) for M in range(33, 2049, 5) for N in (256, 512, 768, 1024, 1536, 2304, 3072, 4096, 8192)}
    assert {t & 255 | (t >> 8) << 8 for t in seen if t} <= {nf | mt << 8 for nf, mt in (
        (2, 2), (2, 4), (4, 2), (2, 6), (4, 4), (2, 8), (4, 6), (8, 2), (4, 8), (8, 4), (8, 6), (4, 12), (8, 8))}
    g = torch.Generator(device="cuda").manual_seed(2)
    for t in sorted(seen - {0}):                             # each tile by a shape that it is chosen for
        M, N = next((M, N) for M in range(33, 2049, 5) for N in (256, 512, 768, 1024, 1536, 2304, 3072, 4096, 8192)
                    if nat.load().penny_bias_rows_plan(M, N, 768) == t)
        x = torch.randn(M, 768, generator=g, device="cuda").to(torch.bfloat16)
        w = (torch.randn(N, 768, generator=g, device="cuda") * 768 ** -0.5).to(torch.bfloat16)
        b, y = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16), torch.zeros(M + 1, N, dtype=torch.bfloat16, device="cuda")
        nat.call("penny_gemm_bias_small", nat.ptr(x), 768, nat.ptr(w), 768, nat.ptr(y), N, nat.ptr(b), M, N, 0, nat.stream())
        want = x.double() @ w.double().T + b.double()
        assert ((y[:M].double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -18 * 768 ** 0.5).all() and (y[M] == 0).all(), (t & 255, t >> 8)


@pytest.mark.parametrize("lens", [[64] * 3, [40, 9] * 8, [500, 268, 3], [64] * 20, [64] * 20 + [1]])
def test_walk_of_longer_batches(lens, monkeypatch):
    """Up to 1280 tokens (one round of blocks for the widest projection) in one native call, bit by bit the per-layer calls."""
    from financial_chatbot_llm_amd.models import bert
    from financial_chatbot_llm_amd.models.configs import get_model_config
    g = torch.Generator().manual_seed(sum(lens))
    cfg = get_model_config("bge-base-en")
    m = bert.BertEncoder.build(cfg, device="cuda", seed=3)
    ids = [torch.randint(0, cfg.vocab_size, (n,), generator=g).tolist() for n in lens]
    calls = []
    walk = m._small_batch
    monkeypatch.setattr(m, "_small_batch", lambda *a: calls.append(walk(*a)) or calls[-1])
    x, _ = m.forward(ids)
    assert calls == [sum(lens) <= 1280]
    monkeypatch.setattr(m, "_small_batch", lambda *a: False)
    y, _ = m.forward(ids)
    assert torch.equal(x, y)


def test_rule():
    """Slices of K and the ring only where they are the faster way."""
    from financial_chatbot_llm_amd.ops import _native as nat
    lib = nat.load()
    assert [lib.penny_encoder_slices(*a) for a in ((7, 1024, 1024), (18, 1024, 1024), (150, 1024, 1024), (16, 512, 2048), (17, 512, 3008),
                                                   (16, 768, 3072), (192, 768, 3072), (193, 768, 3072), (18, 1024, 4096), (18, 256, 3136))] == \
        [1, 1, 1, 1, 1, 4, 4, 1, 4, 1]
    assert [lib.penny_bias_rows_plan(*a) > 0 for a in ((32, 1024, 1024), (33, 1024, 1024), (190, 1024, 1024), (1024, 2048, 8192), (1025, 2048, 8192),
                                                       (2048, 1024, 4096), (33, 1152, 384), (33, 1152, 1088))] == \
        [False, True, True, True, False, True, True, False]


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("N,K", [(2304, 768), (768, 768), (3072, 768), (768, 3072), (1024, 4096), (1024, 1024), (1152, 384), (512, 2048), (256, 3136), (512, 3072), (2048, 4096), (1280, 1536),
                                 (48, 192), (1040, 64), (1040, 1600), (256, 96)])
def test_rows_do_not_depend_on_their_batch(N, K, gelu):
    """A row's values bit by bit the same by blocks of few rows, in slices and on the ring's tiles; the last two: sizes that neither takes."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x = torch.randn(1024, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    ref = gemm.linear_bias(x[:16], w, b, gelu)
    for M in (17, 33, 40, 64, 65, 100, 130, 192, 193, 300, 512, 768) + ((1000, 1024) if N % 256 == 0 or K <= 1024 else ()):
        if gemm.small_bias_wins(M, N, K) or gemm.N.load().penny_bias_rows_plan(M, N, K):
            assert torch.equal(gemm.linear_bias(x[:M], w, b, gelu)[:16], ref), M


def test_embeddings_do_not_depend_on_their_batch():
    """A text embedded alone and beside any others, up to the number of tokens that one native call takes."""
    from financial_chatbot_llm_amd.models import bert
    from financial_chatbot_llm_amd.models.configs import get_model_config
    g = torch.Generator().manual_seed(1)
    cfg = get_model_config("bge-base-en")
    m = bert.BertEncoder.build(cfg, device="cuda", seed=3)
    text = lambda n: torch.randint(5, cfg.vocab_size, (n,), generator=g).tolist()      # noqa: E731
    q = text(14)
    ref = m.encode([q])
    for others in (1, 2, 3, 5, 8, 12, 20, 40, 60, 80):
        assert torch.equal(m.encode([q] + [text(6 + i % 14) for i in range(others)])[0], ref[0]), others


@pytest.mark.parametrize("M,N,K", [(7, 1024, 1024), (18, 1024, 1024), (33, 1024, 1024), (190, 1024, 1024), (16, 512, 2048), (17, 512, 2048), (40, 1152, 384)])
def test_at_the_rule(M, N, K):
    test_against_float64(M, N, K, False)
