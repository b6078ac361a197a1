"""The encoder's own kernels against plain float32: attention over packed rows (tile edges, one-token texts, both head
sizes, rows wider than q | k | v) and the biased projections of small batches (edges of the token and row tiles)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H", [(64, 12), (64, 3), (128, 2)])
@pytest.mark.parametrize("lens", [[1], [18], [64, 63, 65, 1, 16], [130, 7, 200], [300]])
@pytest.mark.parametrize("pad", [0, 8])
def test_encoder_attention(D, H, lens, pad):
    from financial_chatbot_llm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(D + sum(lens))
    T = sum(lens)
    x = torch.randn(T, 3 * H * D + pad, generator=g, device="cuda").to(torch.bfloat16)
    qkv = x[:, :3 * H * D]
    cu = torch.tensor([0] + lens).cumsum(0).to("cuda", torch.int32)
    scale = 1.7 * D ** -0.5
    if pad:                          # the op's row stride comes from the tensor, the head size from its width
        assert qkv.stride(0) == 3 * H * D + pad
    got = ops.encoder_attention(qkv, cu, max(lens), H, scale).float()
    a = 0
    for n in lens:
        q, k, v = qkv[a:a + n].float().reshape(n, 3, H, D).permute(1, 2, 0, 3).contiguous()
        p = torch.softmax(torch.matmul(q, k.transpose(1, 2).contiguous()) * scale, -1)
        want = torch.matmul(p, v).permute(1, 0, 2).reshape(n, H * D)
        # weights and output are rounded to bf16 once each
        assert float((got[a:a + n] - want).norm() / want.norm()) < 6e-3
        assert float((got[a:a + n] - want).abs().max()) < 0.03 * float(want.abs().max())
        a += n


def test_encoder_attention_takes_bf16_rows(monkeypatch):
    from financial_chatbot_llm_amd import ops
    from financial_chatbot_llm_amd.ops import _native
    g = torch.Generator(device="cuda").manual_seed(3)
    lens, H, D = [5, 70, 0, 1], 2, 64
    qkv = torch.randn(sum(lens), 3 * H * D, generator=g, device="cuda").to(torch.bfloat16)
    cu = torch.tensor([0] + lens).cumsum(0).cuda()                            # 64-bit bounds
    for x in (qkv.float(), qkv.half(), qkv.t().contiguous().t(), qkv[:, :-1]):
        with pytest.raises(ValueError):
            ops.encoder_attention(x, cu, 70, H, 0.125)
    got = ops.encoder_attention(qkv, cu, 70, H, 0.125)
    monkeypatch.setattr(_native, "_FORCE_TORCH_OPS", True)                     # plain torch on the same device
    for x in (qkv, torch.cat([qkv, qkv], 1)[:, :3 * H * D]):
        want = ops.encoder_attention(x, cu, 70, H, 0.125)
        assert want.device == qkv.device and float((got.float() - want.float()).norm() / want.float().norm()) < 8e-3


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 128, 129, 768])
@pytest.mark.parametrize("N,K", [(768, 768), (48, 96), (3072, 768), (768, 3072), (16, 32)])
@pytest.mark.parametrize("gelu", [False, True])
def test_small_batch_projection(M, N, K, gelu):
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g, device="cuda").to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    b = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    assert gemm.small_bias_ok(x, w) and M <= gemm.BGE_SMALL_MAX_M
    got = gemm.linear_bias(x, w, b, gelu).float()
    want = x.float() @ w.float().T + b.float()
    if gelu:
        want = F.gelu(want)
    # f32 sums; the result (with gelu also its argument) is rounded to bf16 once
    assert float((got - want).norm() / want.norm()) < 4e-3


def test_projections_the_small_kernel_does_not_take():
    """What the library product takes is answered by it, what it refuses is refused."""
    from financial_chatbot_llm_amd.ops import gemm
    g = torch.Generator(device="cuda").manual_seed(5)
    M, N, K = 9, 48, 96
    flat = torch.randn(N * K + M * K + N + 8, generator=g, device="cuda").to(torch.bfloat16)
    x, w, b = flat[:M * K].view(M, K), flat[M * K:M * K + N * K].view(N, K), flat[-N - 8:-8]
    off = flat[1:1 + N * K].view(N, K)                                        # two bytes off the kernel's 16
    for args in ((x, w, None), (x, off, b), (x, w, flat[3:3 + N]), (x, w, flat[:2 * N:2]), (flat[1:1 + M * K].view(M, K), w, b)):
        want = args[0].float() @ args[1].float().T + (args[2].float() if args[2] is not None else 0.0)
        assert float((gemm.linear_bias(*args).float() - want).norm() / want.norm()) < 4e-3      # one rounding to bf16
    for args in ((x, w, b.float()), (x[:, :64], w, b), (x, w, b[:16]), (x, w.float(), b)):
        with pytest.raises(RuntimeError):
            gemm.linear_bias(*args)


def test_a_layer_weight_off_the_alignment():
    from financial_chatbot_llm_amd.models.bert import BertEncoder
    from financial_chatbot_llm_amd.models.configs import get_model_config
    m = BertEncoder.build(get_model_config("bert-tiny"), "cuda")
    want = m.encode([[5, 6, 7]])
    for name in ("layers.0.o_b", "layers.1.ln1_g"):                          # slices of a flat buffer
        t = m.w[name]
        m.w[name] = torch.cat([t.new_zeros(4), t])[4:]
    assert torch.allclose(m.encode([[5, 6, 7]]), want, atol=2e-2)            # other kernels, bf16 activations


def test_gelu_over_all_bf16():
    from financial_chatbot_llm_amd import ops
    bits = torch.arange(1 << 16, dtype=torch.int32)
    x = torch.cat([bits[:0x7f81], bits[0x8000:0xff80]]).to(torch.int16).view(torch.bfloat16)   # finite values and +inf
    x = torch.cat([x, x.new_zeros(-x.numel() % 8)])
    got = ops.gelu_(x.cuda().clone().view(1, -1)).cpu().view(-1).double()
    z = x.double()
    want = 0.5 * z * torch.special.erfc(-z * 0.5 ** 0.5)
    want[torch.isneginf(want) | torch.isnan(want)] = 0.0
    fin = torch.isfinite(z)
    assert torch.isposinf(got[~fin]).all()
    # one rounding to bf16 (8 significant bits: half a unit in the last place is at most 2^-8; below 2^-126 to zero), and
    # 3e-7 of x for x > 0, 1e-4 of the result in the negative tail
    tol = want.abs() * (2.0 ** -8 + 1e-4) + 3e-7 * z.clamp(min=0) * (z.abs() < 10) + 2.0 ** -126
    assert ((got - want).abs() <= tol)[fin].all(), float(((got - want).abs() / tol)[fin].max())


@pytest.mark.parametrize("lens", [[1], [18], [5, 1, 40, 64, 65], [16] * 48, [500, 268], [500, 269]])
def test_small_batches_in_one_call(lens, monkeypatch):
    """The native walk over the layers against the per-layer calls it stands for, bit by bit; 769 tokens take the latter."""
    from financial_chatbot_llm_amd.models import bert
    from financial_chatbot_llm_amd.models.configs import get_model_config
    g = torch.Generator().manual_seed(sum(lens))
    cfg = get_model_config("bge-base-en")
    m = bert.BertEncoder.build(cfg, device="cuda", seed=3)
    ids = [torch.randint(0, cfg.vocab_size, (n,), generator=g).tolist() for n in lens]
    x, cu = m.forward(ids)
    e = m.encode(ids)
    monkeypatch.setattr(m, "_small_batch", lambda *a: False)
    y, _ = m.forward(ids)
    assert cu == [0] + torch.tensor(lens).cumsum(0).tolist() and torch.equal(x, y)
    want = F.normalize(y[torch.tensor(cu[:-1], device="cuda")].float(), dim=-1)
    assert e.shape == want.shape and float((e - want).abs().max()) < 1e-6      # f32 sums of 768 squares in another order


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257])
@pytest.mark.parametrize("N,K", [(256, 1024), (512, 2080), (768, 3072), (1024, 4096), (768, 1536), (1024, 96)])
def test_sliced_projection(M, N, K):
    """A long K over few columns goes by slices where those fill the chip; the norm behind it adds them up to the same values."""
    from financial_chatbot_llm_amd.ops import _native as nat, gemm
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    x, w, b = r(M, K + 8)[:, :K], r(N, K) * K ** -0.5, r(N)
    S = nat.load().penny_encoder_slices(M, N, K)
    assert 1 <= S <= max(1, K // 512) and nat.load().penny_encoder_slices(18, 768, 3072) == 4
    got = gemm.linear_bias(x, w, b).float()
    want = x.double() @ w.double().T + b.double()
    assert float((got - want).norm() / want.norm()) < 4e-3                        # one rounding to bf16


def test_encoder_embed_edges():
    """Fused embedding rows against the separate ops: last and out-of-table ids, every supported width."""
    from financial_chatbot_llm_amd import ops
    from financial_chatbot_llm_amd.ops import _native as N
    for H in (256, 512, 768, 1024):
        g = torch.Generator().manual_seed(H)
        r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()  # noqa: E731
        word, position, kind, w, b = r(50, H), r(9, H), r(2, H), r(H), r(H)
        ids = torch.tensor([0, 49, 50, 7, 3], dtype=torch.int32, device="cuda")
        pos = torch.tensor([0, 8, 1, 9, 4], dtype=torch.int32, device="cuda")
        y = torch.empty(5, H, dtype=torch.bfloat16, device="cuda")
        N.call("penny_encoder_embed", N.ptr(ids), N.ptr(pos), N.ptr(word), 50, N.ptr(position), 9, N.ptr(kind), N.ptr(w),
               N.ptr(b), N.ptr(y), 5, H, 1e-12, N.stream())
        ep = (ops.embedding(pos, position).float() + kind[0].float()).to(torch.bfloat16)
        want = ops.layer_norm(ops.embedding(ids, word), w, b, 1e-12, residual=ep)
        assert float((y.float() - want.float()).abs().max()) <= 2.0 ** -6      # a rounding to bf16 below 4


def test_ids_that_travel_with_the_launch(monkeypatch):
    """Small batches whose ids are the launch's own arguments against ids copied to the device, bit by bit: the largest that fits and the
    first that does not (960 ints of ids, positions and bounds), ids outside the table, positions beyond theirs, calls in a row."""
    from financial_chatbot_llm_amd.models import bert
    from financial_chatbot_llm_amd.models.configs import ModelConfig
    cfg = ModelConfig("bert-r", "bert", 300, 256, 2, 4, 4, 64, 512, max_position=160, norm_eps=1e-12, type_vocab_size=2)
    m = bert.BertEncoder.build(cfg, device="cuda", seed=3)
    batches = [[[(5 * i + j) % 300 for j in range(n)] for i, n in enumerate(lens)]
               for lens in ([1], [4], [5, 1, 18], [479], [480], [3] * 137, [3] * 138, [2, 0, 3])]
    batches += [[[-1, 299, 300, 2]], [[2 ** 31 - 1, 0, 1]]]
    got = [m.encode(b) for b in batches for _ in range(2)]
    with pytest.raises(OverflowError):
        m.encode([[2 ** 31]])
    monkeypatch.setattr(bert, "EMBED_ARGS", 0)
    want = [m.encode(b) for b in batches for _ in range(2)]
    assert all(torch.equal(a.nan_to_num(), b.nan_to_num()) for a, b in zip(got, want))


def test_projection_form_follows_its_shape():
    """Shapes of which each form was measured faster."""
    from financial_chatbot_llm_amd.ops.gemm import small_bias_wins as small
    assert all(small(*s) for s in ((768, 2304, 768), (768, 768, 3072), (400, 1152, 384), (18, 384, 1536), (64, 8192, 2048), (511, 4096, 1024)))
    assert not any(small(*s) for s in ((769, 768, 768), (512, 1152, 384), (64, 384, 1536), (128, 8192, 2048), (768, 4096, 1024)))


def test_activations_of_tile_products_over_all_bf16():
    """The tile kernel's tables of GELU and SiLU give what the row kernels work out, bit for bit, for every bf16 value."""
    from financial_chatbot_llm_amd import ops
    from financial_chatbot_llm_amd.ops import gemm
    K, M = 128, 257
    values = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    # GELU: products of zero, every value as a bias
    x, w = torch.zeros(M, K, dtype=torch.bfloat16, device="cuda"), torch.zeros(1 << 16, K, dtype=torch.bfloat16, device="cuda")
    got = gemm.prefill_gemm(x, w, "bias_gelu", bias=values)
    want = ops.gelu_(values.clone().view(1, -1)).view(-1)
    bits = lambda t: torch.nan_to_num(t, 7.0, 8.0, 9.0).view(torch.int16)  # noqa: E731  (and the sign of zeros)
    assert torch.equal(bits(got), bits(want).expand(M, -1))
    # SiLU: row m's entries 1 .. 127 of X reach a gate each through unit rows of W, entry 0 is the factor 1.5 of every `up`
    fin = values[torch.isfinite(values)]
    fin = torch.cat([fin, fin.new_zeros(-fin.numel() % (K - 1))]).view(-1, K - 1)
    x = torch.cat([fin.new_full((fin.shape[0], 1), 1.5), fin], 1).contiguous()
    eye = torch.eye(K, dtype=torch.bfloat16, device="cuda")
    up = torch.zeros_like(eye)
    up[:, 0] = 1.0
    got = gemm.prefill_gemm(x, gemm.interleave16(eye, up).contiguous(), "silu")
    want = ops.silu_mul(torch.cat([x + 0.0, x[:, :1].expand(-1, K)], 1).contiguous())          # a sum is no -0
    assert torch.equal(bits(got), bits(want))
    # gates beyond what f32 holds
    x[:, 1::2], x[:, 2::2] = 3e38, -3e38
    got = gemm.prefill_gemm(x, gemm.interleave16(2 * eye, up).contiguous(), "silu")
    want = ops.silu_mul(torch.cat([2 * x, x[:, :1].expand(-1, K)], 1).contiguous())
    assert torch.isinf(want[:, 1]).all() and torch.isnan(want[:, 2]).all() and torch.equal(bits(got), bits(want))


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("N,K,over", [(2304, 768, 7), (2304, 768, 600), (768, 768, 250), (3072, 768, 1), (512, 1024, 300)])
def test_rows_behind_the_last_full_round(N, K, over, gelu):
    """The rows that a last, nearly empty round of tiles would take go to smaller tiles: the same bits as in whole tiles."""
    from financial_chatbot_llm_amd.ops import _native, gemm
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nt = N // 256
    M = (cus // nt if cus // nt else 1) * (1 if cus % nt == 0 else 2) * 256 + over     # row tiles of one or two full rounds, and a few rows
    peeled = _native.load().penny_bias_peeled_rows
    assert peeled(M, N, K, cus, gelu) == over and peeled(M, N, K, 0, gelu) == 0          # the two sides below are two paths
    assert peeled(M - over, N, K, cus, gelu) == 0 and peeled(M, N, K + 1024, cus, gelu) == 0
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = (torch.randn(s, generator=g, device="cuda").to(torch.bfloat16) for s in ((M, K), (N, K)))
    b = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    y, want = torch.empty((M, N), dtype=torch.bfloat16, device="cuda"), gemm.prefill_gemm(x, w, "bias_gelu" if gelu else "bias", bias=b)
    _native.call("penny_gemm_prefill", _native.ptr(x), K, _native.ptr(w), K, _native.ptr(y), N, _native.ptr(b), 0, M, N, 1, 6 if gelu else 5,
                 None, 0, None, 0, 0, _native.stream())                                # no count of CUs: whole tiles only
    assert torch.equal(want, y)
