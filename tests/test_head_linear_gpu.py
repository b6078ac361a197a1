"""A matrix per head on strided rows of heads (``ops.mixers.HeadLinear``) against float64: both kernel forms, edges of the token
tiles, odd numbers of column groups, views off the kernel's 16 bytes, and the sizes that keep the batched product."""
import pytest
import torch

from financial_chatbot_llm_amd.ops import mixers as mx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 2, 15, 17, 64, 512, 513, 1000])
@pytest.mark.parametrize("H,N,K", [(16, 256, 96), (3, 96, 256), (1, 16, 32), (2, 48, 64), (5, 40, 24), (2, 512, 160)])
def test_against_float64(dt, T, H, N, K):
    g = torch.Generator().manual_seed(T + N)
    w = (torch.randn((H, N, K), generator=g) * K ** -0.5).to(dt).cuda()
    q = torch.randn((T, H * (K + 32) + 8), generator=g).to(dt).cuda()
    f = mx.HeadLinear(w)
    assert f.native == (N % 16 == 0 and K % 32 == 0)
    for off in (0, 8, 3):                                    # 3: rows off the kernel's 16 bytes
        x = q[:, off:off + H * (K + 32)].unflatten(1, (H, K + 32))[:, :, :K]
        y = f(x)
        want = torch.einsum("thk,hnk->thn", x.double().cpu(), w.double().cpu())
        assert y.is_contiguous() and y.shape == (T, H, N)
        # one rounding of the result to eight significant bits (half a unit: 2^-8 of it at most); sums of K f32 products
        e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
        assert ((y.double().cpu() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()


def test_weights_off_16_bytes():
    """A part of a flat buffer of weights, as a loader may hand it over."""
    w, x = torch.randn(3 * 32 * 64 + 3, device="cuda")[3:].view(3, 32, 64), torch.randn((5, 3, 64), device="cuda")
    assert ((mx.HeadLinear(w)(x).double() - (x.double()[:, :, None] * w.double()).sum(-1)).abs() <= 2.0 ** -18 * 64).all()


@pytest.mark.parametrize("dt,T,H,N,K,native", [
    (torch.bfloat16, 8192, 32, 128, 256, True), (torch.bfloat16, 8193, 32, 128, 256, False), (torch.float32, 1024, 32, 128, 256, True),
    (torch.float32, 1025, 32, 128, 256, False), (torch.float32, 1025, 32, 256, 128, True), (torch.bfloat16, 3, 2, 512, 96, False),
    (torch.bfloat16, 3, 2, 256, 128, True), (torch.bfloat16, 3, 2, 256, 160, False)])
def test_rule(dt, T, H, N, K, native, monkeypatch):
    """Large matrices, and a long K beside many rows, keep the batched product."""
    from financial_chatbot_llm_amd.ops import _native as nat
    calls = []
    mcall = nat.mcall
    monkeypatch.setattr(nat, "mcall", lambda name, *a: (calls.append(name), mcall(name, *a))[1])
    g = torch.Generator(device="cuda").manual_seed(T)
    w = torch.randn((H, N, K), generator=g, device="cuda").mul_(K ** -0.5).to(dt)
    x = torch.randn((T, H, K), generator=g, device="cuda").to(dt)
    y = mx.HeadLinear(w)(x)
    assert calls == (["mx_head_linear"] if native else [])
    want = (x[:50].double()[:, :, None] * w.double()).sum(-1)
    e = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -20
    assert ((y[:50].double() - want).abs() <= want.abs() * e + 2.0 ** -18 * K ** 0.5).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,N_,K", [(16, 96, 224), (40, 16, 32), (9, 48, 480), (17, 240, 64)])
def test_many_tokens_through_lds(dtype, H, N_, K):
    """Beyond 8192 rows of heads the tokens go through LDS: the sums of few tokens, bit for bit, at the edges of its tiles."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    g = torch.Generator().manual_seed(H + K)
    lin = mx.HeadLinear((torch.randn((H, N_, K), generator=g) * K ** -0.5).to(dtype).cuda())
    few = 8192 // H
    for T in (few + 1, (few // 64 + 1) * 64, (few // 64 + 1) * 64 + 1):
        x = torch.randn((T, H, K + 32), generator=g).to(dtype).cuda()[:, :, 16:K + 16]
        assert torch.equal(lin(x), torch.cat([lin(x[:few]), lin(x[few:])]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nq,nk,nv", [(8, 16, 8), (2048, 512, 512), (2056, 264, 2080), (4096, 8, 16), (8192, 1024, 1024), (8200, 40, 48)])
def test_query_and_key_norm_by_sixteen_bytes(dtype, nq, nk, nv):
    """Rows by 16 bytes and by single entries (columns that start between two of them) against 64 bits."""
    from financial_chatbot_llm_amd.ops import mixers as mx
    g = torch.Generator().manual_seed(nq)
    T, rows = 7, [3, -1, 0, 8, 5, 1, 2]
    qw, kw = torch.rand(nq, generator=g) + 0.5, torch.rand(nk, generator=g) + 0.5
    for off in (0, 8, 1):
        buf = torch.randn((T, nq + nk + nv + 24), generator=g).to(dtype)
        q, k, v = buf[:, off:off + nq], buf[:, off + nq:off + nq + nk], buf[:, off + nq + nk:off + nq + nk + nv]
        for norm in (True, False):
            cache = torch.full((9, nk + nv), 7.0, dtype=dtype, device="cuda")
            d = buf.cuda()
            got = mx.qk_norm_write(d[:, off:off + nq], d[:, off + nq:off + nq + nk], d[:, off + nq + nk:off + nq + nk + nv],
                                   qw.cuda() if norm else None, kw.cuda() if norm else None, 1e-5, torch.tensor(rows, dtype=torch.int32, device="cuda"), cache)
            rms = lambda x, w: x.double() / (x.double().pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * w.double() if norm else x.double()  # noqa: E731
            # one rounding to the type, f32 sums before it
            tol = 2.0 ** -8 if dtype == torch.bfloat16 else 2e-6
            for a, b in ((got, rms(q, qw)), (torch.stack([cache[r] for r in rows if r >= 0]),
                                            torch.cat([rms(k, kw), v.double()], 1)[[i for i, r in enumerate(rows) if r >= 0]])):
                assert ((a.double().cpu() - b).abs() <= tol * b.abs() + 1e-6).all()
            assert (cache[[r for r in range(9) if r not in rows]] == 7.0).all()
