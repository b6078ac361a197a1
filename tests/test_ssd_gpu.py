"""The chunked state-space scan against a float64 recurrence and beside the token-by-token kernel: chunk edges, fresh and
continued segments, padding rows, mixed lengths, slow and very fast decays."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def recurrence(u, dtr, bias, A_log, D, S, H, P, N, G):
    y = torch.zeros(u.shape[0], H, P, dtype=torch.float64)
    x, B, C = u[:, :H * P].view(-1, H, P), u[:, H * P:H * P + G * N].view(-1, G, N), u[:, H * P + G * N:].view(-1, G, N)
    B, C = (t.repeat_interleave(H // G, 1) for t in (B, C))
    dt = F.softplus(dtr + bias)
    keep = torch.exp(-torch.exp(A_log) * dt)
    for t in range(u.shape[0]):
        S = keep[t, :, None, None] * S + (dt[t, :, None] * x[t])[:, :, None] * B[t][:, None]
        y[t] = (S * C[t][:, None]).sum(-1) + D[:, None] * x[t]
    return y.reshape(-1, H * P), S


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,P,N,G,decay", [(2, 64, 128, 2, 1.0), (4, 16, 64, 1, 8.0), (2, 48, 256, 2, 0.1), (4, 32, 128, 2, 60.0)])
@pytest.mark.parametrize("lens", [[64], [32, 1, 31, 63, 65], [200, 5, 129], [1, 128]])
def test_chunked_scan(dtype, H, P, N, G, decay, lens):
    from financial_chatbot_llm_amd.ops import mixers as mx
    g = torch.Generator().manual_seed(sum(lens) + N)
    rnd = lambda *s: torch.randn(s, generator=g)  # noqa: E731
    T, S = sum(lens) + 1, len(lens) + 1           # one padding row at the end
    cu = torch.tensor([0] + lens + [1]).cumsum(0)
    slot = torch.tensor([S + 2 - i for i in range(len(lens))] + [-1])
    starts = [0 if i % 2 == 0 else 70 for i in range(len(lens))] + [0]
    pos = torch.cat([torch.arange(a, a + n) for a, n in zip(starts, lens + [1])])
    u, dtr = rnd(T, H * P + 2 * G * N), (rnd(T, H) * 0.5).to(dtype)
    bias, A_log, D = rnd(H) * 0.5 - 2.0, torch.log(decay * (0.5 + torch.rand(H, generator=g))), rnd(H)
    state = rnd(S + 3, H, P, N)
    dev = lambda t: t.cuda() if t.is_floating_point() else t.to("cuda", torch.int32)  # noqa: E731
    got = {}
    for name, most in (("chunks", max(lens)), ("tokens", 1)):
        st = state.cuda()
        y = mx.ssm_scan(u.cuda(), dtr.cuda(), dev(bias), dev(A_log), dev(D), st, dev(cu), dev(slot), dev(pos), H, P, N, G, most)
        got[name] = (y.double().cpu(), st.double().cpu())
    off = {"chunks": 0.0, "tokens": 0.0}
    for i, n in enumerate(lens):
        a = int(cu[i])
        s0 = torch.zeros(H, P, N, dtype=torch.float64) if starts[i] == 0 else state[slot[i]].double()
        y, s1 = recurrence(u[a:a + n].double(), dtr[a:a + n].double(), bias.double(), A_log.double(), D.double(), s0, H, P, N, G)
        for name, (gy, gs) in got.items():
            off[name] = max(off[name], float((gy[a:a + n] - y).norm() / y.norm()), float((gs[slot[i]] - s1).norm() / s1.norm()))
    used = set(slot[:-1].tolist())
    for _, gs in got.values():                    # no other slot is touched
        for k in range(S + 3):
            assert k in used or torch.equal(gs[k], state[k].double())
    # f32 sums of up to N + 64 products and one exponential per pair of tokens
    assert off["chunks"] < 2e-6 and off["chunks"] < 2.0 * off["tokens"] + 3e-7, off


def test_not_finite():
    """An infinite input reaches no earlier token and no other channel."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    H, P, N, G, T = 2, 32, 64, 1, 150
    g = torch.Generator().manual_seed(1)
    u, dtr = torch.randn(T, H * P + 2 * G * N, generator=g), torch.randn(T, H, generator=g)
    bias, A_log, D = torch.zeros(H), torch.zeros(H), torch.ones(H)
    cu, slot, pos = torch.tensor([0, T]), torch.tensor([0]), torch.arange(T)
    dev = lambda t: t.cuda() if t.is_floating_point() else t.to("cuda", torch.int32)  # noqa: E731
    out = []
    for bad in (None, 85):
        v, st = u.clone(), torch.zeros(1, H, P, N).cuda()
        if bad is not None:
            v[bad, 5] = float("inf")
        y = mx.ssm_scan(*(dev(t) for t in (v, dtr, bias, A_log, D)), st, dev(cu), dev(slot), dev(pos), H, P, N, G, T)
        out.append((y.cpu(), st.cpu()))
    (y, st), (z, sz) = out
    assert torch.equal(y[:85], z[:85]) and not torch.isfinite(z[85:, 5]).any() and not torch.isfinite(sz[0, 0, 5]).any()
    y[:, 5], z[:, 5], st[0, 0, 5], sz[0, 0, 5] = 0, 0, 0, 0
    assert torch.equal(y, z) and torch.equal(st, sz)


@pytest.mark.parametrize("n", [0, 1, 20, 31, 40])
@pytest.mark.parametrize("most", [[], [40]])
def test_one_segment_in_a_longer_buffer(n, most):
    """The rows behind the last segment belong to nobody: ``max_len`` left out, or given as the buffer's rows, is a bound."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    H, P, N, G, T = 2, 16, 64, 1, 40
    g = torch.Generator().manual_seed(n)
    args = [torch.randn(T, H * P + 2 * G * N, generator=g), torch.randn(T, H, generator=g), torch.randn(H, generator=g) - 2.0,
            torch.zeros(H), torch.ones(H)]
    state = torch.randn(3, H, P, N, generator=g)
    meta = [torch.tensor([0, n]), torch.tensor([2]), torch.arange(T) + 9]
    dev = lambda t: t.cuda() if t.is_floating_point() else t.to("cuda", torch.int32)  # noqa: E731
    got_state, want_state = state.cuda(), state.clone()
    got = mx.ssm_scan(*map(dev, args), got_state, *map(dev, meta), H, P, N, G, *most)
    want = mx.ssm_scan(*args, want_state, *meta, H, P, N, G)
    # f32 sums of up to N + 40 products on both sides
    assert torch.allclose(got[:n].cpu(), want[:n], rtol=1e-5, atol=1e-4) and torch.allclose(got_state.cpu(), want_state, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("lens", [[1] * 40 + [96] + [1] * 30 + [33, 31, 300], [32] * 9 + [31, 2, 640], [5, 0, 70, 1, 0, 64, 65] * 4])
def test_short_segments_beside_long_ones(lens):
    """The chunks' scratch is numbered past the short segments, which have none."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    H, P, N, G = 4, 16, 64, 2
    g = torch.Generator().manual_seed(len(lens))
    T, S = sum(lens), len(lens)
    assert mx._ssm_in_chunks(T, S, max(lens), H * P * N)
    args = [torch.randn(T, H * P + 2 * G * N, generator=g), torch.randn(T, H, generator=g), torch.randn(H, generator=g) - 2.0,
            torch.zeros(H), torch.ones(H)]
    state = torch.randn(S, H, P, N, generator=g)
    meta = [torch.tensor([0] + lens).cumsum(0), torch.randperm(S, generator=g),
            torch.cat([torch.arange(n) + (i % 3) for i, n in enumerate(lens)])]
    dev = lambda t: t.cuda() if t.is_floating_point() else t.to("cuda", torch.int32)  # noqa: E731
    got_state, want_state = state.cuda(), state.clone()
    got = mx.ssm_scan(*map(dev, args), got_state, *map(dev, meta), H, P, N, G, max(lens))
    want = mx.ssm_scan(*args, want_state, *meta, H, P, N, G)
    # f32 sums of up to N + 64 products on both sides
    assert torch.allclose(got.cpu(), want, rtol=2e-5, atol=2e-4) and torch.allclose(got_state.cpu(), want_state, rtol=2e-5, atol=2e-4)


def test_form_follows_the_step():
    """Steps of which each form was measured faster (64 heads of 64 x 128, then 32)."""
    from financial_chatbot_llm_amd.ops.mixers import _ssm_in_chunks as chunks
    for H, tokens, chunked in ((64, [[31] * 16, [32], [48], [40] * 2, [32] * 8, [64] + [1] * 8, [192] + [1] * 64, [48] * 4 + [1] * 64],
                                [[64], [64] * 2, [40] * 4, [96] + [1] * 8, [256] + [1] * 64, [32] * 16, [2048] * 2]),
                               (32, [[32] * 8, [40] * 4, [64] + [1] * 8, [128] + [1] * 64, [96] * 4 + [1] * 64],
                                [[40] * 8, [128] * 4 + [1] * 64, [96] + [1] * 8])):
        for lens in tokens + chunked:
            assert chunks(sum(lens), len(lens), max(lens), H * 64 * 128) == (lens in chunked), (H, lens)
